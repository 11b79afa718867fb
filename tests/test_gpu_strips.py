"""GPU parity of the kernels that keep 16-row strips in registers, at the edges of
their strips, blocks and launches, against the CPU oracle: potrf_l(_mn) with one
and with several waves per instance, syrk_dpotrf_ln, trsm_rltn; and of the gemm
family's tiles."""
import numpy as np
import pytest

import blasfeo_amd as bfa
import oracle
from blasfeo_amd import autotune
from helpers import Batch, run_both, compare_buffers
import chol_cases
import gemm_cases
import trsm_cases

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 79, 80, 81, 95, 96, 97, 111, 112, 113, 127, 128]
LARGE = [129, 144, 145, 176, 177, 208, 240, 241, 255, 256]


def _panel_sizes(prec):
    return [4, 8] if prec == "d" else [4, 8, 16]


@pytest.mark.parametrize("bound", [32, 64, 128, 256])
@pytest.mark.parametrize("bw", [1, 2])
@pytest.mark.parametrize("prec,ps", [(p, q) for p in "ds" for q in _panel_sizes(p)])
def test_potrf(gpu, prec, ps, bw, bound):
    sizes = [n for n in EDGES + LARGE if n <= bound]
    b = Batch(prec, ps, seed=3)
    recs = chol_cases.to_batch(b, chol_cases.potrf(ps, "potrf_l", sizes, 40 + ps, inplace_at=len(sizes) - 1))
    f = oracle.fn(prec, "potrf_l")
    autotune.set_knob("potrf_bw", 0, bw)
    try:
        g, gd, rr, rd = run_both(b, b.host(), bfa.DFACT_ARG, recs, prec + "potrf_l",
                                 lambda h, r: f(ps, r["m"], h.desc_addr(r["sC"]), r["ci"], r["cj"], h.desc_addr(r["sD"]), r["di"], r["dj"]),
                                 (bound, bound, 0))
    finally:
        autotune.set_knob("potrf_bw", 0, 0)
    compare_buffers(b, g, rr, "potrf_l", tol=1e-11 if prec == "d" else 2e-3)
    assert (gd["use_dA"] == rd["use_dA"]).all()


@pytest.mark.parametrize("bw", [1, 2])
@pytest.mark.parametrize("ps", [4, 8])
def test_potrf_mn(gpu, ps, bw):
    """trapezoids: rows below the factored block in its last strip and in later ones"""
    b = Batch("d", ps, seed=4)
    recs = chol_cases.to_batch(b, chol_cases.potrf(ps, "potrf_l_mn", [n for n in EDGES if n <= 108], 60 + ps))
    f = oracle.fn("d", "potrf_l_mn")
    autotune.set_knob("potrf_bw", 0, bw)
    try:
        g, gd, rr, rd = run_both(b, b.host(), bfa.DFACT_ARG, recs, "dpotrf_l_mn",
                                 lambda h, r: f(ps, r["m"], r["n"], h.desc_addr(r["sC"]), r["ci"], r["cj"], h.desc_addr(r["sD"]), r["di"], r["dj"]),
                                 (128, 128, 0))
    finally:
        autotune.set_knob("potrf_bw", 0, 0)
    compare_buffers(b, g, rr, "potrf_l_mn")
    assert (gd["use_dA"] == rd["use_dA"]).all()


@pytest.mark.parametrize("bound", [32, 64, 128])
@pytest.mark.parametrize("ps", [4, 8])
def test_syrk_potrf(gpu, ps, bound):
    """k around the 16-column chunks, B = A and B a matrix of its own, m > n"""
    rng = np.random.default_rng(80 + ps)
    b = Batch("d", ps, seed=5)
    recs = []
    for i, m in enumerate([n for n in EDGES if n <= bound]):
        n = m if i % 3 else max(1, m - i)
        k = [0, 1, 3, 4, 15, 16, 17, 32, 33, 70][i % 10]
        ai, bi, ci, di = (int(x) for x in rng.integers(0, 2 * ps, 4)) if i % 2 else (0, 0, 0, 0)
        A = rng.standard_normal((ai + m, k + 2))
        mats = {"sA": (ai + m, k + 2, A)}
        if i % 4 == 2:   # B: A's rows scaled, at another offset
            Bm = np.zeros((bi + m, k + 1))
            Bm[bi:, 1:] = 0.5 * A[ai:, 2:]
            mats["sB"], rb = (bi + m, k + 1, Bm), dict(bi=bi, bj=1)
        else:
            mats["sB"], rb = "=sA", dict(bi=ai, bj=2)
        mats["sC"] = (ci + m, n, np.vstack([np.zeros((ci, n)), m * np.eye(m)[:, :n] + 0.01 * rng.standard_normal((m, n))]))
        mats["sD"] = (di + m, n, -1.0)
        recs.append((mats, dict(m=m, n=n, k=k, ai=ai, aj=2, ci=ci, cj=0, di=di, dj=0, **rb)))
    recs = chol_cases.to_batch(b, recs)
    f = oracle.fn("d", "syrk_potrf_ln_mn")

    def ocall(h, r):
        f(ps, r["m"], r["n"], r["k"], h.desc_addr(r["sA"]), r["ai"], r["aj"], h.desc_addr(r["sB"]), r["bi"], r["bj"],
          h.desc_addr(r["sC"]), r["ci"], r["cj"], h.desc_addr(r["sD"]), r["di"], r["dj"])

    g, gd, rr, rd = run_both(b, b.host(), bfa.DSYRK_DPOTRF_ARG, recs, "dsyrk_dpotrf_ln", ocall, (bound, bound, 70))
    compare_buffers(b, g, rr, "syrk_dpotrf_ln")
    assert (gd["use_dA"] == rd["use_dA"]).all()


@pytest.mark.parametrize("finite", [True, False])
@pytest.mark.parametrize("prec,ps", [(p, q) for p in "ds" for q in _panel_sizes(p)])
def test_trsm_rltn(gpu, prec, ps, finite):
    b = Batch(prec, ps, seed=6)
    recs = chol_cases.to_batch(b, trsm_cases.rltn(ps, 100 + ps, finite))
    f = oracle.fn(prec, "trsm_rltn")

    def ocall(h, r):
        f(ps, r["m"], r["n"], r["alpha"], h.desc_addr(r["sA"]), r["ai"], r["aj"], h.desc_addr(r["sB"]), r["bi"], r["bj"],
          h.desc_addr(r["sD"]), r["di"], r["dj"])

    with np.errstate(invalid="ignore"):
        g, gd, rr, rd = run_both(b, b.host(), bfa.DTRSM_ARG if prec == "d" else bfa.STRSM_ARG, recs, prec + "trsm_rltn", ocall, (130, 256, 0))
        if finite:
            compare_buffers(b, g, rr, "trsm_rltn")
        else:
            for i in range(len(b.layout)):
                x, y = b.layout.view(g, i), b.layout.view(rr, i)
                tol = 1e-11 if prec == "d" else 9e-4
                same = (x == y) | (np.isnan(x) & np.isnan(y)) | (np.abs(x - y) <= tol * (np.abs(x) + np.abs(y)) + tol)
                assert same.all(), "matrix %d: %d differ" % (i, int((~same).sum()))
    assert (gd["use_dA"] == rd["use_dA"]).all()


@pytest.mark.parametrize("tile", [1, 2])
@pytest.mark.parametrize("op", ["gemm_nt", "gemm_nn", "syrk_ln", "syrk_ln_mn"])
@pytest.mark.parametrize("prec,ps", [(p, q) for p in "ds" for q in _panel_sizes(p)])
def test_gemm_pieces(gpu, prec, ps, op, tile):
    """rows on piece boundaries; four times over: a batch above the one that is spread over the XCDs"""
    if prec == "s" and op == "syrk_ln_mn":
        pytest.skip("no FP32 syrk_ln_mn entry")
    f = oracle.fn(prec, op)

    def ocall(h, r):
        mn = (r["m"],) if op == "syrk_ln" else (r["m"], r["n"])
        f(ps, *mn, r["k"], r["alpha"], h.desc_addr(r["sA"]), r["ai"], r["aj"], h.desc_addr(r["sB"]), r["bi"], r["bj"],
          r["beta"], h.desc_addr(r["sC"]), r["ci"], r["cj"], h.desc_addr(r["sD"]), r["di"], r["dj"])

    autotune.set_knob("gemm_wave", 0, tile)
    try:
        for times in (1, 4):
            b = Batch(prec, ps, seed=7)
            recs = chol_cases.to_batch(b, gemm_cases.pieces(ps, op, 120 + ps) * times)
            g, gd, rr, rd = run_both(b, b.host(), bfa.DGEMM_ARG if prec == "d" else bfa.SGEMM_ARG, recs, prec + op, ocall, (130, 130, 33))
            compare_buffers(b, g, rr, "%s%s ps=%d" % (prec, op, ps))
            assert (gd["use_dA"] == rd["use_dA"]).all()
    finally:
        autotune.set_knob("gemm_wave", 0, 0)
