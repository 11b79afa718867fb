"""GPU parity of the LU of instances of up to 256 rows (one, two and four waves per
instance by the bound) against the CPU oracle, on the records of tests/lu_cases.py."""
import numpy as np
import pytest

import blasfeo_amd as bfa
import oracle
from helpers import Batch, run_both
import chol_cases
import lu_cases
from test_gpu_lapack import _check_fp32_getrf, _run_getrf

pytestmark = pytest.mark.gpu


def _records(b, op, bound, ps, sizes_only=False):
    cases = [c for c in lu_cases.lu(ps, 200 + ps, op == "getrf_rp") if c[1]["m"] <= bound]
    if sizes_only:
        cases = cases[:sum(m <= bound for m, _ in lu_cases.SIZES)]
    recs = chol_cases.to_batch(b, cases)
    b.host_buf = b.host()
    return recs


def _same(b, recs, g, rr):
    for r in recs:
        x, y = b.layout.view(g, r["sD"]), b.layout.view(rr, r["sD"])
        with np.errstate(invalid="ignore"):
            same = (x == y) | (np.isnan(x) & np.isnan(y)) | (np.abs(x - y) <= 1e-11 * (np.abs(x) + np.abs(y)) + 1e-11)
        assert same.all(), "%d x %d: %d differ" % (r["m"], r["n"], int((~same).sum()))


@pytest.mark.parametrize("bound", [64, 128, 256])
@pytest.mark.parametrize("ps", [4, 8])
def test_getrf_rp(gpu, ps, bound):
    b = Batch("d", ps, seed=8)
    recs = _records(b, "getrf_rp", bound, ps)
    with np.errstate(invalid="ignore"):
        g, gd, rr, rd, gp, hp = _run_getrf(b, "d", recs, (bound, 300, 0))
    np.testing.assert_array_equal(gp, hp)
    _same(b, recs, g, rr)
    assert (gd["use_dA"] == rd["use_dA"]).all()


@pytest.mark.parametrize("bound", [64, 128, 256])
@pytest.mark.parametrize("ps", [4, 8, 16])
def test_sgetrf_rp(gpu, ps, bound):
    b = Batch("s", ps, seed=8)
    recs = _records(b, "getrf_rp", bound, ps, sizes_only=True)
    g, gd, rr, rd, gp, hp = _run_getrf(b, "s", recs, (bound, 300, 0))
    _check_fp32_getrf(b, recs, g, rr, gp, hp, 2e-3)
    assert (gd["use_dA"] == rd["use_dA"]).all()


@pytest.mark.parametrize("bound", [64, 128, 256])
@pytest.mark.parametrize("ps", [4, 8])
def test_getrf_np(gpu, ps, bound):
    b = Batch("d", ps, seed=8)
    recs = _records(b, "getrf_np", bound, ps)
    f = oracle.fn("d", "getrf_np")
    g, gd, rr, rd = run_both(b, b.host_buf, bfa.DFACT_ARG, recs, "dgetrf_np",
                             lambda h, r: f(ps, r["m"], r["n"], h.desc_addr(r["sC"]), r["ci"], r["cj"], h.desc_addr(r["sD"]), r["di"], r["dj"]),
                             (bound, 300, 0))
    _same(b, recs, g, rr)
    assert (gd["use_dA"] == rd["use_dA"]).all()
