"""trsm_rltn of batches that take several launches (more than 2^31 threads)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code", ["d", "s"])
def test_large_batch_large_bound(gpu, code):
    """140000 solves of 2 x 2 with a bound of 4096 rows: every one of them is made,
    against the solution of the shared factor."""
    import torch
    import blasfeo_amd as bfa
    batch, ps, n = 140000, 4, 2
    f = np.float64 if code == "d" else np.float32
    tdt = torch.float64 if code == "d" else torch.float32
    dm, dt = (bfa.DMAT, bfa.DTRSM_ARG) if code == "d" else (bfa.SMAT, bfa.STRSM_ARG)
    size = bfa.memsize(f, ps, n, n) // np.dtype(f).itemsize
    dev = "cuda:0"
    mem = torch.zeros((batch + 1) * size, dtype=tdt, device=dev)
    v = mem.view(batch + 1, size)
    L = np.array([[2.0, 0.0], [0.5, 4.0]])
    B = torch.arange(batch * n, dtype=tdt, device=dev).view(batch, n) % 97
    for j in range(n):
        v[1:, j * ps] = B[:, j]   # row 0 of each B
        for i in range(n):
            v[0, j * ps + i] = float(L[i, j])
    d = np.zeros(batch + 1, dm)
    isz = np.dtype(f).itemsize
    d["mem"] = d["pA"] = np.uint64(mem.data_ptr()) + np.arange(batch + 1, dtype=np.uint64) * np.uint64(size * isz)
    d["dA"] = d["pA"] + np.uint64(ps * 4 * isz)
    d["m"], d["n"], d["pm"], d["cn"] = n, n, ps, 4
    desc = torch.from_numpy(d.view(np.uint8).copy()).to(dev)
    r = np.zeros(batch, dt)
    at = np.uint64(desc.data_ptr()) + np.arange(1, batch + 1, dtype=np.uint64) * np.uint64(dm.itemsize)
    r["m"], r["n"], r["alpha"], r["sA"], r["sB"], r["sD"] = 1, n, 1.0, desc.data_ptr(), at, at
    recs = torch.from_numpy(r.view(np.uint8).copy()).to(dev)
    bfa.call(code + "trsm_rltn", ps, batch, recs.data_ptr(), (4096, 256, 0), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    x = torch.stack([v[1:, 0], v[1:, ps]], 1).double().cpu().numpy()
    want = np.linalg.solve(L, B.double().cpu().numpy().T).T
    np.testing.assert_allclose(x, want, rtol=1e-11 if code == "d" else 1e-5, atol=1e-11 if code == "d" else 1e-5)
