"""Emulator cases (TEST INFRASTRUCTURE ONLY) for the LU factorisations on the record
sets of tests/lu_cases.py, checked against the oracle: pivots exactly, factors at
the reference's rule, NaN and Inf included.
The instances of more than half the bound (all of them for 64).
Usage: python case_lu.py <getrf_rp | getrf_np> <ps> <bound of the rows>"""
import ctypes
import sys

import numpy as np

from emu_harness import Block, records, emu_lib, to_mats, bfa, oracle
import lu_cases


def run(op, ps, bound):
    E = emu_lib("emu_lapack")
    re, ro = to_mats(ps, [c for c in lu_cases.lu(ps, 60 + ps, op == "getrf_rp") if bound // 2 * (bound > 64) < c[1]["m"] <= bound])
    piv = [[Block(4 * min(r["m"], r["n"])) for r in s] for s in (re, ro)]
    for s, p in zip((re, ro), piv):
        for r, b in zip(s, p):
            b.write(np.full(b.nbytes // 4, -7, np.int32))
            r["ipiv"] = b.addr
    blk = records(bfa.DFACT_ARG, re)
    print("emu %s ps=%d batch=%d" % (op, ps, len(re)), flush=True)
    rc = getattr(E, "blasfeo_amd_d%s_batched" % op)(ps, len(re), ctypes.c_void_p(blk.addr),
                                                    ctypes.byref(bfa.HINT(bound, 300, 0)), None)
    assert rc == 0, E.emu_last_error()
    f = oracle.fn("d", op)
    for r in ro:
        a = [ps, r["m"], r["n"], r["sC"].desc.addr, r["ci"], r["cj"], r["sD"].desc.addr, r["di"], r["dj"]]
        f(*(a + [r["ipiv"]] if op == "getrf_rp" else a))
    for i, (x, y) in enumerate(zip(re, ro)):
        what = "%s ps=%d instance %d (%d x %d)" % (op, ps, i, x["m"], x["n"])
        np.testing.assert_array_equal(piv[0][i].read(np.int32), piv[1][i].read(np.int32), err_msg=what)
        g, w = x["sD"].content(), y["sD"].content()
        with np.errstate(invalid="ignore"):
            same = (g == w) | (np.isnan(g) & np.isnan(w)) | (np.abs(g - w) <= 1e-11 * (np.abs(g) + np.abs(w)) + 1e-11)
        assert same.all(), "%s: %d differ, first %s emu=%r ref=%r" % (what, int((~same).sum()), np.argwhere(~same)[:1].tolist(), g[~same][:1], w[~same][:1])
        assert x["sD"].use_dA() == y["sD"].use_dA(), what
    print("ok", flush=True)


if __name__ == "__main__":
    run(sys.argv[1], int(sys.argv[2]), int(sys.argv[3]))
