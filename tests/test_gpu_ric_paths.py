"""GPU parity of the FP64 Riccati factorisation by launch path, against the CPU oracle:
the direct launches (stages of at most 32 rows: one wave per instance; a batch of at
most one instance per CU: four waves), the planned class launches, instances larger
than the hint on both, and the planned path captured and replayed."""
import ctypes

import numpy as np
import pytest

import blasfeo_amd as bfa
import oracle
from blasfeo_amd import autotune
from blasfeo_amd.riccati import RiccatiBatch, DeviceRiccati, HostRiccati, DeviceRiccatiSv, HostRiccatiSv
from helpers import assert_close

pytestmark = pytest.mark.gpu


def _check(entry, rb, inp, what):
    import torch
    sv = entry == "sv"
    dev = (DeviceRiccatiSv if sv else DeviceRiccati)(rb, inp)
    print("riccati %s %s ps=%d batch=%d" % (entry, what, rb.ps, rb.batch), flush=True)
    dev.run()
    torch.cuda.synchronize()
    host = (HostRiccatiSv if sv else HostRiccati)(rb, inp)
    getattr(oracle.lib(), "or_dric_%s_batch" % entry)(rb.ps, rb.batch, host.argv.ctypes.data)
    fd, fh = (dev.fac, host.fac) if sv else (dev, host)
    g, gL, hL = fd.outbuf.cpu().numpy(), fd.t_dev[2].cpu().numpy().view(bfa.DMAT), fh.t[2]
    for i in range(rb.batch):
        for k in range(rb.N + 1):
            j, r = rb.i_L[i][k], i * (rb.N + 1) + k
            w = "%s instance %d stage %d" % (what, i, k)
            assert_close(np.tril(rb.out.get(g, j)), np.tril(rb.out.get(fh.outbuf, j)), 1e-11, w)
            assert gL[r]["use_dA"] == hL[r]["use_dA"], w
            if gL[r]["use_dA"]:
                assert_close(rb.out.dview(g, j), rb.out.dview(fh.outbuf, j), 1e-11, w + " dA")
        if sv:
            rs, v = host.sv.rs, dev.vectors()
            for kind, ks in (("ux", range(rb.N + 1)), ("pi", range(rb.N))):
                for k in ks:
                    assert_close(rs.vec(v, i, kind, k), rs.vec(host.vbuf, i, kind, k), 1e-11, "%s %s[%d]" % (what, kind, k))


@pytest.mark.parametrize("path", ["direct", "plan"])
@pytest.mark.parametrize("sizes", ["small", "mixed", "beyond one wave", "beyond four waves"])
@pytest.mark.parametrize("ps", [4, 8])
@pytest.mark.parametrize("entry", ["trf", "sv"])
def test_paths(gpu, entry, ps, sizes, path):
    rng = np.random.default_rng(670 + ps)
    if sizes == "small":
        nxs, nus = list(rng.integers(1, 27, 20)) + [29, 16], list(rng.integers(0, 5, 20)) + [2, 15]
    else:
        nxs, nus = list(rng.integers(1, 65, 20)) + [64, 64], list(rng.integers(0, 20, 20)) + [63, 20]
    rb = RiccatiBatch(nxs, nus, N=3, ps=ps, aug=entry == "sv")
    inp = rb.fill_inputs(rng)
    if sizes == "beyond one wave":
        rb.max_nk, rb.max_nx = 14, 8
    elif sizes == "beyond four waves":
        rb.max_nk, rb.max_nx = 60, 20
    try:
        # a knob of a class that the hint admits sends the batch to the plan
        autotune.set_knob("ric_per_cu", 0, 2 if path == "plan" else 0)
        _check(entry, rb, inp, "%s %s" % (path, sizes))
    finally:
        autotune.reset()


def _planned(rng, extra, N, hi=65):
    """A batch that no direct launch serves: more instances than CUs, more than 32 rows."""
    import torch
    n = torch.cuda.get_device_properties(0).multi_processor_count + extra
    return RiccatiBatch([40] + list(rng.integers(1, hi, n - 1)), [9] + list(rng.integers(1, 17, n - 1)), N=N, ps=4)


def test_planned_graph_replay(gpu):
    """Zero-fill, plan and class launches with their helper streams in a graph: three
    replays, eager work and synchronisation between them, each the eager result."""
    import torch
    rng = np.random.default_rng(671)
    rb = _planned(rng, 40, 3)
    dev = DeviceRiccati(rb, rb.fill_inputs(rng))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        dev.run(s.cuda_stream)
    torch.cuda.synchronize()
    ref = dev.outbuf.clone()
    g = dev.capture(s)
    for rep in range(3):
        dev.outbuf.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            g.replay()
        torch.cuda.synchronize()
        assert torch.equal(dev.outbuf, ref), "replay %d" % rep


def test_planned_graph_replay_after_growth(gpu):
    """The graph of a planned batch after a larger planned batch has replaced the
    stream's plan workspace: the block that the graph holds stays allocated."""
    import torch
    rng = np.random.default_rng(672)
    rb = _planned(rng, 8, 2)
    dev = DeviceRiccati(rb, rb.fill_inputs(rng))
    big = _planned(rng, 40000, 1, 9)
    dbig = DeviceRiccati(big, big.fill_inputs(rng))
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        dev.run(s.cuda_stream)
    torch.cuda.synchronize()
    ref = dev.outbuf.clone()
    g = dev.capture(s)
    with torch.cuda.stream(s):
        dbig.run(s.cuda_stream)
    torch.cuda.synchronize()
    for rep in range(2):
        dev.outbuf.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(s):
            g.replay()
        torch.cuda.synchronize()
        assert torch.equal(dev.outbuf, ref), "replay %d" % rep


def test_planned_noalloc_twice(gpu):
    """The allocation-free entry, planned both times: the second call, smaller and
    shorter, finds the first one's counts, heads and lists in the fixed scratch."""
    import torch
    rng = np.random.default_rng(673)
    for extra, N, hi in ((80, 4, 65), (8, 2, 40)):
        rb = _planned(rng, extra, N, hi)
        inp = rb.fill_inputs(rng)
        ref, dev = DeviceRiccati(rb, inp), DeviceRiccati(rb, inp)
        ref.run()
        h = bfa.HINT(rb.max_nk, rb.max_nx, 0)
        rc = bfa.lib().blasfeo_amd_d_back_ric_trf_batched_noalloc(4, rb.batch, ctypes.c_void_p(dev.args.data_ptr()), ctypes.byref(h), None)
        bfa.check(rc, "d_back_ric_trf_batched_noalloc")
        torch.cuda.synchronize()
        assert torch.equal(dev.outbuf, ref.outbuf)
