"""Emulator cases (TEST INFRASTRUCTURE ONLY) for the FP64 Riccati factorisation by launch
path, factors, reciprocal diagonals and their flags (sv: ux and pi too) against the oracle:
  direct  no plan: stages of at most 32 rows (one wave each), and a batch of up to one
          instance per CU (four waves each);
  plan    the class launches, one, two and four waves per instance (a knob of a class
          that the hint admits sends the batch there);
  beyond  instances larger than the hint, on both paths: factorised all the same;
  knobs   which launches a knob changes: of the FP64 sweep those of batches whose hint
          admits its class, none of the FP32 sweep (of the mixed-precision solve);
  join    an event record or wait that fails: the call reports it, and every helper stream
          that waits on the caller's is waited for by it.
Usage: python case_ric_paths.py <trf | sv> <direct | plan | beyond | knobs | join> <ps>"""
import ctypes
import sys

import numpy as np

from case_ric import HINT, split
from emu_harness import Block, bfa, compare, emu_lib, oracle
from blasfeo_amd.riccati import RiccatiBatch, RiccatiSv, HostRiccati, HostRiccatiSv

SMALL = ([1, 3, 8, 11, 17, 24, 15, 29, 16], [0, 2, 3, 4, 9, 6, 1, 2, 15])
MIXED = ([1, 3, 8, 17, 30, 40, 64, 64, 50, 12], [0, 2, 5, 16, 1, 33, 20, 63, 9, 4])


def check(entry, ps, nxs, nus, hint, knob):
    sv = entry == "sv"
    rb = RiccatiBatch(nxs, nus, N=3, ps=ps, aug=sv)
    inp = rb.fill_inputs(np.random.default_rng(40 + ps))
    in_blocks, fix_in = split(rb.inp, inp, ("mem", "pA", "dA"))
    out_blocks, fix_out = split(rb.out, rb.out.host_buffer(), ("mem", "pA", "dA"))
    babt, rsq, L, work, nx, nu = rb.tables(0, 0)
    fix_in(babt), fix_in(rsq), fix_out(L), fix_out(work)
    tbl = {}
    for k, v in (("babt", babt), ("rsq", rsq), ("L", L), ("work", work), ("nx", nx), ("nu", nu)):
        tbl[k] = Block(v.nbytes)
        tbl[k].write(v)
    if sv:
        rs = RiccatiSv(rb).rs
        vtab = rs.table(0)
        vblocks = []
        for r in vtab:
            b = Block(int(r["memsize"]))
            b.write(np.zeros(int(r["memsize"]), np.uint8))
            r["mem"] = r["pa"] = b.addr
            vblocks.append(b)
        tbl["v"] = Block(vtab.nbytes)
        tbl["v"].write(vtab)
        a = RiccatiSv(rb).args(*(tbl[k].addr for k in ("v", "babt", "rsq", "L", "work", "nx", "nu")))
        host = HostRiccatiSv(rb, inp)
        oracle.lib().or_dric_sv_batch(ps, rb.batch, host.argv.ctypes.data)
        hout, hL = host.fac.outbuf, host.fac.t[2]
    else:
        a = rb.args(*(tbl[k].addr for k in ("babt", "rsq", "L", "work", "nx", "nu")))
        host = HostRiccati(rb, inp)
        oracle.lib().or_dric_trf_batch(ps, rb.batch, host.argv.ctypes.data)
        hout, hL = host.outbuf, host.t[2]
    ablk = Block(a.nbytes)
    ablk.write(a)
    E = emu_lib("emu_lapack")
    E.blasfeo_amd_tune_set(b"ric_per_cu", 0, knob)
    print("emu d_back_ric_%s ps=%d batch=%d hint=%r knob=%d" % (entry, ps, rb.batch, hint, knob), flush=True)
    rc = getattr(E, "blasfeo_amd_d_back_ric_%s_batched" % entry)(ps, rb.batch, ctypes.c_void_p(ablk.addr),
                                                                 ctypes.byref(HINT(*hint)), None)
    E.blasfeo_amd_tune_set(b"ric_per_cu", 0, 0)
    assert rc == 0, E.emu_last_error()
    Lout = tbl["L"].read(bfa.DMAT)
    for i in range(rb.batch):
        for k in range(rb.N + 1):
            j = rb.i_L[i][k]
            m, n, pm, cn = rb.out.geom(j)
            got = out_blocks[j].read(np.float64)
            want = np.frombuffer(hout[rb.out.offsets[j]: rb.out.offsets[j] + out_blocks[j].nbytes], np.float64)
            what = "%s instance %d stage %d (%dx%d)" % (entry, i, k, m, n)
            compare(np.tril(bfa.pm_unpack(got[: pm * cn], ps, cn, m, n)).ravel(),
                    np.tril(bfa.pm_unpack(want[: pm * cn], ps, cn, m, n)).ravel(), 1e-11, "factor " + what)
            ud = int(Lout[i * (rb.N + 1) + k]["use_dA"])
            assert ud == int(hL[i * (rb.N + 1) + k]["use_dA"]), ("use_dA", what, ud)
            if ud:
                compare(got[pm * cn: pm * cn + n], want[pm * cn: pm * cn + n], 1e-11, "dA " + what)
        for kind, ks in (("ux", range(rb.N + 1)), ("pi", range(rb.N))) if sv else ():
            for k in ks:
                j = rs.index(i, kind, k)
                compare(vblocks[j].read(np.float64, int(rs.sizes[j])), rs.vec(host.vbuf, i, kind, k), 1e-11,
                        "%s[%d] instance %d" % (kind, k, i))


def knobs(entry, ps):
    E = emu_lib("emu_lapack")

    def launches(f, knob, cls, value):
        E.blasfeo_amd_tune_set(knob, cls, value)
        n = E.emu_launches(0), E.emu_launches(1)
        f()
        E.blasfeo_amd_tune_set(knob, cls, 0)
        return E.emu_launches(0) - n[0], E.emu_launches(1) - n[1]

    small = lambda: check(entry, ps, *SMALL, (31, 29, 0), 0)  # noqa: E731
    plain = launches(small, b"ric_per_cu", 1, 0)
    assert plain[0] <= 2, plain   # the sweep, and sv's forward substitution
    for cls in range(2, 8):
        assert launches(small, b"ric_per_cu", cls, 1) == plain, cls
        assert launches(small, b"ric_threads", cls, 256) == plain, cls
    assert launches(small, b"ric_per_cu", 1, 1)[0] > 2
    if entry == "trf":
        import case_ric
        case_ric.NXS, case_ric.NUS = SMALL   # classes 0 and 1 of the FP64 sweep
        mixed = lambda: case_ric.run_mixed(ps)  # noqa: E731
        assert launches(mixed, b"ric_threads", 4, 128) == launches(mixed, b"ric_threads", 4, 0)


def join(entry, ps):
    E = emu_lib("emu_lapack")
    E.emu_fail_stream(0)
    check(entry, ps, [5], [2], (7, 5, 0), 2)
    helpers = E.emu_waits(1)
    assert helpers == E.emu_waits(0) > 0
    # the fork's record, its waits, then a record and a wait for each helper's join
    for n in range(1, 1 + 1 + 3 * helpers):
        E.emu_fail_stream(n)
        try:
            check(entry, ps, [5], [2], (7, 5, 0), 2)
            failed = False
        except AssertionError as e:
            failed = b"helper streams" in e.args[0]
        assert failed, n
        broken = n > 1 + helpers   # a helper whose own join failed cannot be waited for
        assert E.emu_waits(0) == E.emu_waits(1) - broken, (n, E.emu_waits(0), E.emu_waits(1))
    E.emu_fail_stream(0)


def run(entry, path, ps):
    top = 127 if entry == "sv" else 128
    if path == "knobs":
        knobs(entry, ps)
    elif path == "join":
        join(entry, ps)
    elif path == "direct":
        check(entry, ps, *SMALL, (31, 29, 0), 0)
        check(entry, ps, *MIXED, (127, 64, 0), 0)
    elif path == "plan":
        check(entry, ps, *SMALL, (31, 29, 0), 2)
        check(entry, ps, *MIXED, (top, 64, 0), 2)
    else:
        # one-wave and four-wave direct launches, then the plan with the same bounds;
        # nx = 70 is within the rows of the second bound (trf only)
        wide = ([70, 8], [20, 3]) if entry == "trf" else ([8], [3])
        for knob in (0, 2):
            check(entry, ps, *MIXED, (14, 8, 0), knob)
            check(entry, ps, MIXED[0] + wide[0], MIXED[1] + wide[1], (100, 64, 0), knob)
    print("ok", flush=True)


if __name__ == "__main__":
    run(sys.argv[1], sys.argv[2], int(sys.argv[3]))
