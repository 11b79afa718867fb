"""Matrices of more than 4 GiB on the GPU: tests/wide_cases.py, by numpy."""
import numpy as np
import pytest

import wide_cases as w

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("geom", ["stride", "deep"])
@pytest.mark.parametrize("ps", [4, 8])
def test_more_than_4_gib(gpu, ps, geom):
    import torch
    import blasfeo_amd as bfa
    from blasfeo_amd import autotune
    rows, cn, _ = w.GEOM[geom]
    big = torch.zeros(rows * cn, dtype=torch.float64, device="cuda:0")

    def put(i, v):
        big[torch.from_numpy(i).to(big.device)] = torch.from_numpy(np.ascontiguousarray(v)).to(big.device)

    def upload(a):
        t = torch.from_numpy(a.view(np.uint8).copy()).to(big.device)
        return t.data_ptr(), t

    def lib(entry, batch, args, hint):
        print("gpu wide %s %s ps=%d" % (geom, entry, ps), flush=True)
        bfa.call(entry, ps, batch, args, hint, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()

    for op in w.OPS:
        if op == "ric_trf" and geom == "deep":
            continue   # its matrices have no row offset
        store = w.Store(ps, geom, big.data_ptr(), put, lambda i: big[torch.from_numpy(i).to(big.device)].cpu().numpy())
        for k, v in w.knobs(op).items():
            autotune.set_knob(k, 0, v)
        try:
            w.run(op, ps, geom, store, upload, lib)
        finally:
            for k in w.knobs(op):
                autotune.set_knob(k, 0, 0)
