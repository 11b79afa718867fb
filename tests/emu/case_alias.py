"""Emulator case (TEST INFRASTRUCTURE ONLY): getrf in place through two descriptors of
one buffer, the second with its base a panel and two columns further on and its
offsets as much smaller.  Pivots exactly, factors at the reference's rule.
Usage: python case_alias.py <getrf_rp | getrf_np> <ps>"""
import ctypes
import sys

import numpy as np

from emu_harness import Block, Mat, compare, emu_lib, oracle, records, bfa


def run(op, ps):
    E = emu_lib("emu_lapack")
    rng = np.random.default_rng(ps)
    for m, n in ((40, 40), (40, 70), (130, 90), (200, 200)):
        A = rng.uniform(-1, 1, (m, n)) + (m * np.eye(m, n) if op == "getrf_np" else 0)
        S = np.zeros((ps + 1 + m, 3 + n))
        S[ps + 1:, 3:] = A
        C, ref = Mat(ps, *S.shape), Mat(ps, *S.shape)
        C.fill(S)
        ref.fill(S)
        D = Mat(ps, 1 + m, 1 + n)
        d = C.desc.read(bfa.DMAT)
        d["pA"] += 8 * (ps * C.cn + 2 * ps)
        d["dA"] = D.buf.addr + 8 * D.pm * D.cn
        D.desc.write(d)
        piv = [Block(4 * min(m, n)) for _ in range(2)]
        print("emu %s in place, ps=%d %d x %d" % (op, ps, m, n), flush=True)
        blk = records(bfa.DFACT_ARG, [dict(m=m, n=n, ci=ps + 1, cj=3, di=1, dj=1, sC=C, sD=D, ipiv=piv[0].addr)])
        rc = getattr(E, "blasfeo_amd_d%s_batched" % op)(ps, 1, ctypes.c_void_p(blk.addr), ctypes.byref(bfa.HINT(m, n, 0)), None)
        assert rc == 0, E.emu_last_error()
        a = [ps, m, n, ref.desc.addr, ps + 1, 3, ref.desc.addr, ps + 1, 3]
        oracle.fn("d", op)(*(a + [piv[1].addr] if op == "getrf_rp" else a))
        if op == "getrf_rp":
            np.testing.assert_array_equal(piv[0].read(np.int32), piv[1].read(np.int32))
        k = C.pm * C.cn
        compare(C.content()[:k], ref.content()[:k], 1e-11, "%s ps=%d %d x %d" % (op, ps, m, n))
    print("ok", flush=True)


if __name__ == "__main__":
    run(sys.argv[1], int(sys.argv[2]))
