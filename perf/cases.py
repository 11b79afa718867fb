"""Performance cases of the batched BLASFEO hot path.

Each case is one call sequence that a program makes on device-resident
batches through ``blasfeo_amd.call``: the argument records, descriptors and
buffers are laid out once (``prepare``) and the calls are then made on them
again and again (``run``), as an optimiser does from one iteration to the next.

The sizes of a ragged batch come from the case itself, the values in the
matrices from the seed.
"""
import math

import numpy as np
import torch

import blasfeo_amd as bfa

DEV = "cuda"
CHUNK = 1 << 25  # padded elements worked on at a time where inputs or references are formed


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # One controller's control step, the problem of the reference's Riccati
        # example (N = 10, nx = 8, nu = 3): factorise and solve a single
        # system, so launches and the latency of the stage chain are all there is.
        dict(name="ric_one", op="ric_solve", batch=1, N=10, nx_lo=8, nx_hi=8, nu_lo=3, nu_hi=3, ps=4),
        # The batched Riccati factorisation of the benchmark: uneven systems, 20 stages.
        dict(name="ric_trf", op="ric_trf", batch=8192, N=20, nx_lo=8, nx_hi=64, nu_lo=2, nu_hi=16, ps=4),
        # Factorise and solve in one recursion (an interior-point step over many
        # scenarios of a medium-sized system), ps = 8 layout.
        dict(name="ric_sv", op="ric_sv", batch=2048, N=15, nx_lo=6, nx_hi=40, nu_lo=1, nu_hi=10, ps=8),
        # Many small Cholesky factorisations of one size (the benchmark's 4096 x 32 x 32).
        dict(name="potrf_32", op="potrf", batch=4096, lo=32, hi=32, ps=4, dtype="d"),
        # Condensed Hessians: rank-k update and Cholesky in one call, uneven sizes.
        dict(name="syrk_potrf", op="syrk_potrf", batch=32768, lo=8, hi=128, ps=4),
        # Many small uneven products and rank-k updates (the benchmark's U{4..128}).
        dict(name="gemm_syrk", op="gemm_syrk", batch=32768, lo=4, hi=128, ps=4, dtype="d"),
        # Products of larger uneven matrices in the ps = 8 layout.
        dict(name="gemm_nn_large", op="gemm_nn", batch=1024, lo=64, hi=512, ps=8, dtype="d"),
        # The single-precision product and rank-k update (FP32 twins).
        dict(name="sgemm_ssyrk", op="gemm_syrk", batch=8192, lo=16, hi=256, ps=8, dtype="s"),
        # SPD systems: Cholesky, then both triangular solves with 4 right-hand
        # sides (the benchmark's FP64 SPD solve, 2048 x 256 x 256).
        dict(name="spd_solve", op="spd_solve", batch=2048, lo=256, hi=256, nrhs=4, ps=4),
        # Rows below a factored block: right-side triangular solves, uneven sizes.
        dict(name="trsm_rltn", op="trsm", batch=8192, lo=16, hi=256, ps=4, dtype="d"),
        # General systems: pivoted LU, then row swaps and both triangular solves.
        dict(name="lu_solve", op="lu_solve", batch=8192, lo=16, hi=256, nrhs=4, ps=4),
        # Column-major data in and out of the panel-major layout on the device.
        dict(name="pack_unpack", op="pack", batch=8192, lo=16, hi=256, tran=False, ps=4),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _range(rng, lo, hi):
    """A size range inside lo..hi: ragged more often than uniform."""
    a, b = sorted((rng.randint(lo, hi), rng.randint(lo, hi)))
    return (b, b) if rng.random() < 0.3 else (a, b)


def draw(rng):
    """One more case of the ranges above, its batch cut so that it costs no
    more than the largest listed case where its sizes are near their upper end."""
    op = rng.choice(("ric_solve", "ric_trf", "ric_sv", "potrf", "syrk_potrf", "gemm_syrk", "gemm_nn",
                     "gemm_syrk_s", "spd_solve", "trsm", "lu_solve", "pack"))
    ps = rng.choice((4, 4, 8))
    batch = lambda lo, hi, per, most: max(1, min(_log(rng, lo, hi), int(most / per)))  # noqa: E731
    if op in ("ric_solve", "ric_trf", "ric_sv"):
        if op == "ric_solve":  # control of small systems, from one to many of them
            nx, nu, N, b = _range(rng, 4, 24), _range(rng, 1, 6), rng.randint(5, 30), _log(rng, 1, 2048)
        else:
            nx, nu, N = _range(rng, 8, 64), _range(rng, 2, 16), rng.randint(5, 20)
            b = batch(256, 8192, N * nx[1] ** 2, 2e8)
        return dict(op=op, batch=b, N=N, nx_lo=nx[0], nx_hi=nx[1], nu_lo=nu[0], nu_hi=nu[1], ps=ps)
    if op == "potrf":
        lo, hi = _range(rng, 8, 128)
        return dict(op=op, batch=_log(rng, 256, 16384), lo=lo, hi=hi, ps=ps, dtype=rng.choice("dds"))
    if op == "syrk_potrf":
        lo, hi = _range(rng, 8, 128)
        return dict(op=op, batch=batch(1024, 32768, hi ** 2, 2.3e8), lo=lo, hi=hi, ps=ps)
    if op == "gemm_syrk":
        lo, hi = _range(rng, 4, 128)
        return dict(op=op, batch=batch(1024, 32768, hi ** 3, 4e10), lo=lo, hi=hi, ps=ps, dtype="d")
    if op == "gemm_nn":
        lo, hi = _range(rng, 64, 512)
        return dict(op=op, batch=batch(64, 1024, hi ** 3, 8e10), lo=lo, hi=hi, ps=ps, dtype=rng.choice("dds"))
    if op == "gemm_syrk_s":
        lo, hi = _range(rng, 16, 256)
        return dict(op="gemm_syrk", batch=batch(512, 8192, hi ** 3, 5e10), lo=lo, hi=hi, ps=rng.choice((4, 8, 8)), dtype="s")
    if op == "spd_solve":
        lo, hi = _range(rng, 96, 256)
        return dict(op=op, batch=_log(rng, 128, 2048), lo=lo, hi=hi, nrhs=rng.randint(1, 8), ps=ps)
    if op == "trsm":
        lo, hi = _range(rng, 16, 256)
        return dict(op=op, batch=batch(512, 8192, hi ** 2, 1.8e8), lo=lo, hi=hi, ps=ps, dtype=rng.choice("dds"))
    if op == "lu_solve":
        lo, hi = _range(rng, 16, 256)
        return dict(op=op, batch=batch(512, 8192, hi ** 2, 1.8e8), lo=lo, hi=hi, nrhs=rng.randint(1, 6), ps=ps)
    lo, hi = _range(rng, 16, 256)
    return dict(op="pack", batch=_log(rng, 512, 8192), lo=lo, hi=hi, tran=rng.random() < 0.4, ps=ps)


# ---------------------------------------------------------------------------
# batches of panel-major matrices in GPU memory
# ---------------------------------------------------------------------------
def _dt(code):
    return (np.float64, torch.float64) if code == "d" else (np.float32, torch.float32)


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a).view(np.uint8).reshape(-1).copy()).to(DEV)


class Mats:
    """Matrices of the given sizes in one zeroed GPU buffer, with their descriptors."""

    def __init__(self, code, ps, ms, ns):
        self.np_dt, self.dt = _dt(code)
        self.ps, self.ms, self.ns = ps, np.asarray(ms, np.int64), np.asarray(ns, np.int64)
        item = np.dtype(self.np_dt).itemsize
        _, _, total = bfa.bulk_layout(self.np_dt, ps, self.ms, self.ns, 0)
        self.buf = torch.zeros(total // item, dtype=self.dt, device=DEV)
        self.desc, offs, _ = bfa.bulk_layout(self.np_dt, ps, self.ms, self.ns, self.buf.data_ptr())
        self.cn = self.desc["cn"].astype(np.int64)
        self.off = offs // item
        self.doff = (self.desc["dA"].astype(np.int64) - self.buf.data_ptr()) // item
        self.dev = _dev(self.desc)

    def use_dA(self, values):
        self.desc["use_dA"] = values
        self.dev.copy_(_dev(self.desc))

    def addr(self):
        return np.uint64(self.dev.data_ptr()) + np.arange(len(self.ms), dtype=np.uint64) * np.uint64(bfa.DMAT.itemsize)

    def _index(self, sel, M, N):
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a[sel])).to(DEV)[:, None, None]  # noqa: E731
        i = torch.arange(M, device=DEV)[None, :, None]
        j = torch.arange(N, device=DEV)[None, None, :]
        ok = (i < t(self.ms)) & (j < t(self.ns))
        at = t(self.off) + (i - i % self.ps) * t(self.cn) + j * self.ps + i % self.ps
        return at, ok

    def put(self, sel, dense, lower=False):
        """dense[b, :, :] into the matrices sel (the part that fits each)."""
        at, ok = self._index(sel, dense.shape[1], dense.shape[2])
        if lower:
            ok = ok & torch.ones(dense.shape[1:], dtype=torch.bool, device=DEV).tril()[None]
        self.buf[at[ok]] = dense[ok].to(self.dt)

    def get(self, sel, M, N):
        """The matrices sel as float64, zero outside each one's size."""
        at, ok = self._index(sel, M, N)
        return torch.where(ok, self.buf[torch.where(ok, at, torch.zeros_like(at))].double(), 0.0)

    def put_diag(self, sel, diag, sizes):
        """diag[b, :sizes] into the reciprocal-diagonal blocks."""
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)[:, None]  # noqa: E731
        j = torch.arange(diag.shape[1], device=DEV)[None, :]
        ok = (j < t(sizes)).expand(diag.shape)
        self.buf[(t(self.doff[sel]) + j)[ok]] = diag[ok].to(self.dt)


def _chunks(count, per):
    step = max(1, CHUNK // max(1, per))
    return [np.arange(a, min(count, a + step)) for a in range(0, count, step)]


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape, dtype=torch.float64):
    return torch.randn(*shape, generator=g, device=DEV, dtype=dtype)


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64) * 2 - 1


def _sizes(case, what, lo="lo", hi="hi"):
    key = [case["batch"], case[lo], case[hi], what, case["ps"], sum(map(ord, case["op"]))]
    return np.random.default_rng(key).integers(case[lo], case[hi] + 1, size=case["batch"])


def _records(dtype, batch, **fields):
    a = np.zeros(batch, dtype=dtype)
    for k, v in fields.items():
        a[k] = v
    return _dev(a)


def _pad_eye(sizes, n):
    """1 on the diagonal beyond each size, so that a padded factorisation leaves the padding alone."""
    d = torch.arange(n, device=DEV)[None, :] >= torch.from_numpy(np.asarray(sizes)).to(DEV)[:, None]
    return torch.diag_embed(d.double())


def _spd(g, sizes, n):
    """B B^T + size I, B ~ U[-1, 1], each in the leading block of an n x n matrix (zero outside)."""
    B = _uniform(g, len(sizes), n, n)
    s = torch.from_numpy(np.asarray(sizes)).to(DEV)
    B = B * (torch.arange(n, device=DEV)[None, None, :] < s[:, None, None])
    A = torch.matmul(B, B.transpose(1, 2).contiguous())
    return A + torch.diag_embed(s.double()[:, None].expand(-1, n))


# ---------------------------------------------------------------------------
# products
# ---------------------------------------------------------------------------
def _gemm_prepare(c, seed):
    g, code, ps, n = _gen(seed), c["dtype"], c["ps"], c["batch"]
    m, nn, k = (_sizes(c, w) for w in (1, 2, 3))
    rec = bfa.DGEMM_ARG if code == "d" else bfa.SGEMM_ARG
    s = dict(case=c)
    if c["op"] == "gemm_nn":
        A, B = Mats(code, ps, m, k), Mats(code, ps, k, nn)
    else:
        A, B = Mats(code, ps, m, k), Mats(code, ps, nn, k)
    C, D = Mats(code, ps, m, nn), Mats(code, ps, m, nn)
    mats = [A, B, C]
    s["args"] = _records(rec, n, m=m, n=nn, k=k, alpha=1, beta=1, sA=A.addr(), sB=B.addr(), sC=C.addr(), sD=D.addr())
    s["hint"] = (int(m.max()), int(nn.max()), int(k.max()))
    s["D"] = D
    if c["op"] == "gemm_syrk":
        m2, k2 = _sizes(c, 4), _sizes(c, 5)
        A2, C2, D2 = Mats(code, ps, m2, k2), Mats(code, ps, m2, m2), Mats(code, ps, m2, m2)
        s["args2"] = _records(rec, n, m=m2, n=m2, k=k2, alpha=1, beta=1, sA=A2.addr(), sB=A2.addr(), sC=C2.addr(), sD=D2.addr())
        s["hint2"] = (int(m2.max()), int(m2.max()), int(k2.max()))
        s["D2"] = D2
        mats += [A2, C2]
    for M in mats:
        M.buf.normal_(generator=g)
    s["mats"] = mats
    return s


def _gemm_run(s):
    c = s["case"]
    p, ps, n, st = c["dtype"], c["ps"], c["batch"], _stream()
    if c["op"] == "gemm_nn":
        bfa.call(p + "gemm_nn", ps, n, s["args"].data_ptr(), s["hint"], st)
        return s["D"].buf
    bfa.call(p + "gemm_nt", ps, n, s["args"].data_ptr(), s["hint"], st)
    bfa.call(p + "syrk_ln", ps, n, s["args2"].data_ptr(), s["hint2"], st)
    return s["D"].buf, s["D2"].buf


def _gemm_exact(c, seed):
    s = _gemm_prepare(c, seed)
    h, dbl = c["hi"], dict(c, dtype="d")
    outs = []

    def layout(D):
        return Mats("d", c["ps"], D.ms, D.ns) if c["dtype"] == "d" else _F64As(c["ps"], D.ms, D.ns)

    A, B, C = s["mats"][:3]
    R = layout(s["D"])
    for sel in _chunks(dbl["batch"], 4 * h * h):
        b = B.get(sel, h, h)
        if c["op"] != "gemm_nn":
            b = b.transpose(1, 2).contiguous()
        R.put(sel, C.get(sel, h, h) + torch.matmul(A.get(sel, h, h), b))
    outs.append(R.buf)
    if c["op"] == "gemm_syrk":
        A2, C2 = s["mats"][3:]
        R = layout(s["D2"])
        for sel in _chunks(dbl["batch"], 4 * h * h):
            a = A2.get(sel, h, h)
            R.put(sel, C2.get(sel, h, h) + torch.matmul(a, a.transpose(1, 2).contiguous()), lower=True)
        outs.append(R.buf)
    return outs[0] if c["op"] == "gemm_nn" else tuple(outs)


class _F64As(Mats):
    """Float64 values at the places that a float batch has them."""

    def __init__(self, ps, ms, ns):
        super().__init__("s", ps, ms, ns)
        self.dt = torch.float64
        self.buf = self.buf.double()


def _layout_like(code, ps, ms, ns):
    return Mats("d", ps, ms, ns) if code == "d" else _F64As(ps, ms, ns)


def _gemm_work(c):
    m, n, k = (_sizes(c, w).astype(float) for w in (1, 2, 3))
    b, f = (m * k + n * k + 2 * m * n).sum(), (2 * m * n * k).sum()
    if c["op"] == "gemm_syrk":
        m, k = _sizes(c, 4).astype(float), _sizes(c, 5).astype(float)
        b, f = b + (m * k + m * (m + 1)).sum(), f + (m * (m + 1) * k).sum()
    return {"bytes": b * (8 if c["dtype"] == "d" else 4), "flops": f}


# ---------------------------------------------------------------------------
# Cholesky, rank-k update with Cholesky, SPD solve
# ---------------------------------------------------------------------------
def _potrf_prepare(c, seed):
    g, ps, n = _gen(seed), c["ps"], c["batch"]
    code = c.get("dtype", "d")
    m = _sizes(c, 1)
    C, D = Mats(code, ps, m, m), Mats(code, ps, m, m)
    for sel in _chunks(n, 3 * c["hi"] ** 2):
        C.put(sel, _spd(g, m[sel], c["hi"]))
    s = dict(case=c, m=m, C=C, D=D)
    h = int(m.max())
    s["hint"] = (h, h, 0)
    if c["op"] == "syrk_potrf":
        k = _sizes(c, 2)
        A = Mats("d", ps, m, k)
        A.buf.normal_(generator=g)
        s["A"], s["k"] = A, k
        s["args"] = _records(bfa.DSYRK_DPOTRF_ARG, n, m=m, n=m, k=k, sA=A.addr(), sB=A.addr(), sC=C.addr(), sD=D.addr())
        s["hint"] = (h, h, int(k.max()))
    else:
        s["args"] = _records(bfa.DFACT_ARG, n, m=m, n=m, sC=C.addr(), sD=D.addr())
    if c["op"] == "spd_solve":
        r = c["nrhs"]
        B, X = Mats("d", ps, m, np.full(n, r)), Mats("d", ps, m, np.full(n, r))
        B.buf.normal_(generator=g)
        s["B"], s["X"] = B, X
        s["args1"] = _records(bfa.DTRSM_ARG, n, m=m, n=r, alpha=1, sA=D.addr(), sB=B.addr(), sD=X.addr())
        s["args2"] = _records(bfa.DTRSM_ARG, n, m=m, n=r, alpha=1, sA=D.addr(), sB=X.addr(), sD=X.addr())
        s["hint2"] = (h, r, 0)
    return s


def _potrf_run(s):
    c = s["case"]
    ps, n, st = c["ps"], c["batch"], _stream()
    if c["op"] == "syrk_potrf":
        bfa.call("dsyrk_dpotrf_ln", ps, n, s["args"].data_ptr(), s["hint"], st)
        return s["D"].buf
    bfa.call(c.get("dtype", "d") + "potrf_l", ps, n, s["args"].data_ptr(), s["hint"], st)
    if c["op"] == "potrf":
        return s["D"].buf
    bfa.call("dtrsm_llnn", ps, n, s["args1"].data_ptr(), s["hint2"], st)
    bfa.call("dtrsm_lltn", ps, n, s["args2"].data_ptr(), s["hint2"], st)
    return s["D"].buf, s["X"].buf


def _potrf_exact(c, seed):
    s = _potrf_prepare(c, seed)
    code, h, m = c.get("dtype", "d"), c["hi"], s["m"]
    R = _layout_like(code, c["ps"], m, m)
    X = Mats("d", c["ps"], m, np.full(c["batch"], c["nrhs"])) if c["op"] == "spd_solve" else None
    for sel in _chunks(c["batch"], 4 * h * h):
        M = s["C"].get(sel, h, h)
        if c["op"] == "syrk_potrf":
            a = s["A"].get(sel, h, h)
            M = M + torch.matmul(a, a.transpose(1, 2).contiguous())
        M = M.tril() + M.tril(-1).transpose(1, 2) + _pad_eye(m[sel], h)
        L = torch.linalg.cholesky(M)
        R.put(sel, L, lower=True)
        R.put_diag(sel, 1.0 / torch.diagonal(L, dim1=1, dim2=2), m[sel])
        if X is not None:
            X.put(sel, torch.cholesky_solve(s["B"].get(sel, h, c["nrhs"]), L))
    return R.buf if X is None else (R.buf, X.buf)


def _potrf_work(c):
    m = _sizes(c, 1).astype(float)
    b, f = (m * (m + 1) + m).sum(), (m ** 3 / 3).sum()
    if c["op"] == "syrk_potrf":
        k = _sizes(c, 2).astype(float)
        b, f = b + (m * k).sum(), f + (m * (m + 1) * k).sum()
    if c["op"] == "spd_solve":
        b, f = b + (2 * m * c["nrhs"]).sum(), f + (2 * m * m * c["nrhs"]).sum()
    return {"bytes": b * (8 if c.get("dtype", "d") == "d" else 4), "flops": f}


# ---------------------------------------------------------------------------
# triangular solve from the right
# ---------------------------------------------------------------------------
def _trsm_prepare(c, seed):
    g, code, ps, n = _gen(seed), c["dtype"], c["ps"], c["batch"]
    m, nn = _sizes(c, 1), _sizes(c, 2)
    A, B, D = Mats(code, ps, nn, nn), Mats(code, ps, m, nn), Mats(code, ps, m, nn)
    B.buf.normal_(generator=g)
    # a factor with its reciprocal diagonal, as a Cholesky leaves it
    h = c["hi"]
    for sel in _chunks(n, 3 * h * h):
        sz = torch.from_numpy(nn[sel]).to(DEV).double()[:, None, None]
        L = _randn(g, len(sel), h, h).tril(-1) * (0.5 / sz.sqrt())
        d = 1.0 + torch.rand(len(sel), h, generator=g, device=DEV, dtype=torch.float64)
        A.put(sel, L + torch.diag_embed(d), lower=True)
        A.put_diag(sel, 1.0 / d.to(A.dt).double(), nn[sel])
    A.use_dA(nn)
    rec = bfa.DTRSM_ARG if code == "d" else bfa.STRSM_ARG
    args = _records(rec, n, m=m, n=nn, alpha=1, sA=A.addr(), sB=B.addr(), sD=D.addr())
    return dict(case=c, m=m, n=nn, A=A, B=B, D=D, args=args, hint=(int(m.max()), int(nn.max()), 0))


def _trsm_run(s):
    c = s["case"]
    bfa.call(c["dtype"] + "trsm_rltn", c["ps"], c["batch"], s["args"].data_ptr(), s["hint"], _stream())
    return s["D"].buf


def _trsm_exact(c, seed):
    s = _trsm_prepare(c, seed)
    h = c["hi"]
    R = _layout_like(c["dtype"], c["ps"], s["m"], s["n"])
    for sel in _chunks(c["batch"], 4 * h * h):
        L = s["A"].get(sel, h, h) + _pad_eye(s["n"][sel], h)
        Xt = torch.linalg.solve_triangular(L, s["B"].get(sel, h, h).transpose(1, 2).contiguous(), upper=False)
        R.put(sel, Xt.transpose(1, 2).contiguous())
    return R.buf


def _trsm_work(c):
    m, n = _sizes(c, 1).astype(float), _sizes(c, 2).astype(float)
    return {"bytes": (n * (n + 1) / 2 + 2 * m * n).sum() * (8 if c["dtype"] == "d" else 4), "flops": (m * n * n).sum()}


# ---------------------------------------------------------------------------
# LU solve
# ---------------------------------------------------------------------------
def _lu_prepare(c, seed):
    g, ps, n, r = _gen(seed), c["ps"], c["batch"], c["nrhs"]
    m = _sizes(c, 1)
    C, D = Mats("d", ps, m, m), Mats("d", ps, m, m)
    B, X = Mats("d", ps, m, np.full(n, r)), Mats("d", ps, m, np.full(n, r))
    h = c["hi"]
    # A ~ U[-1, 1] with one larger entry (0.7 sqrt(n)) in each row and column,
    # at random places, so that the pivots are all over the rows and no system
    # is near singular; right-hand sides whose solutions are of order one
    for sel in _chunks(n, 3 * h * h):
        sz = torch.from_numpy(m[sel]).to(DEV)
        A = _uniform(g, len(sel), h, h) + torch.diag_embed((0.7 * sz.double().sqrt())[:, None].expand(-1, h))
        key = torch.rand(len(sel), h, generator=g, device=DEV, dtype=torch.float64)
        row = torch.arange(h, device=DEV)[None, :]
        order = torch.argsort(torch.where(row < sz[:, None], key, 2.0 + row.double()), dim=1)
        C.put(sel, _rows(A, order))
        A = C.get(sel, h, h)
        B.put(sel, torch.matmul(A, _randn(g, len(sel), h, r)))
    first = np.concatenate([[0], np.cumsum(m)[:-1]])
    ipiv = torch.zeros(int(m.sum()), dtype=torch.int32, device=DEV)
    s = dict(case=c, m=m, C=C, D=D, B=B, X=X, ipiv=ipiv)
    pv = np.uint64(ipiv.data_ptr()) + first.astype(np.uint64) * np.uint64(4)
    s["args"] = _records(bfa.DFACT_ARG, n, m=m, n=m, sC=C.addr(), sD=D.addr(), ipiv=pv)
    s["args1"] = _records(bfa.DROWPE_ARG, n, kmax=m, ipiv=pv, sA=X.addr())
    s["args2"] = _records(bfa.DTRSM_ARG, n, m=m, n=r, alpha=1, sA=D.addr(), sB=X.addr(), sD=X.addr())
    s["hint"], s["hint2"] = (int(m.max()), int(m.max()), 0), (int(m.max()), r, 0)
    return s


def _lu_run(s):
    c = s["case"]
    ps, n, st = c["ps"], c["batch"], _stream()
    bfa.call("dgetrf_rp", ps, n, s["args"].data_ptr(), s["hint"], st)
    s["X"].buf.copy_(s["B"].buf)
    bfa.call("drowpe", ps, n, s["args1"].data_ptr(), s["hint2"], st)
    bfa.call("dtrsm_llnu", ps, n, s["args2"].data_ptr(), s["hint2"], st)
    bfa.call("dtrsm_lunn", ps, n, s["args2"].data_ptr(), s["hint2"], st)
    return s["D"].buf, s["ipiv"], s["X"].buf


def _lu_exact(c, seed):
    s = _lu_prepare(c, seed)
    m, r = s["m"], c["nrhs"]
    R, X = Mats("d", c["ps"], m, m), Mats("d", c["ps"], m, np.full(c["batch"], r))
    order = np.argsort(m, kind="stable")  # by size, so that little is padding; LAPACK on the host
    for part in np.array_split(order, max(1, min(64, len(order) // 32))):
        h = int(m[part].max())
        LU, piv = torch.linalg.lu_factor((s["C"].get(part, h, h) + _pad_eye(m[part], h)).cpu())
        sol = torch.linalg.lu_solve(LU, piv, s["B"].get(part, h, r).cpu())
        LU = LU.to(DEV)
        R.put(part, LU)
        R.put_diag(part, 1.0 / torch.diagonal(LU, dim1=1, dim2=2), m[part])
        X.put(part, sol.to(DEV))
    return R.buf, None, X.buf


def _lu_work(c):
    m, r = _sizes(c, 1).astype(float), c["nrhs"]
    return {"bytes": (8 * (2 * m * m + m + 2 * m * r) + 4 * m).sum(), "flops": (2 * m ** 3 / 3 + 2 * m * m * r).sum()}


# ---------------------------------------------------------------------------
# column-major <-> panel-major
# ---------------------------------------------------------------------------
def _pack_prepare(c, seed):
    g, ps, n = _gen(seed), c["ps"], c["batch"]
    m, nn = _sizes(c, 1), _sizes(c, 2)
    P = Mats("d", ps, nn, m) if c["tran"] else Mats("d", ps, m, nn)
    pm, pn = (nn, m) if c["tran"] else (m, nn)
    first = np.concatenate([[0], np.cumsum(m * nn)[:-1]])
    A = _randn(g, int((m * nn).sum()))
    out = torch.zeros_like(A)
    a = lambda t: np.uint64(t.data_ptr()) + first.astype(np.uint64) * np.uint64(8)  # noqa: E731
    return dict(case=c, m=m, n=nn, pm=pm, pn=pn, first=first, A=A, out=out, P=P, hint=(int(pm.max()), int(pn.max()), 0),
                args=_records(bfa.DPACK_ARG, n, m=m, n=nn, lda=m, A=a(A), sA=P.addr()),
                args2=_records(bfa.DPACK_ARG, n, m=pm, n=pn, lda=pm, A=a(out), sA=P.addr()))


def _pack_run(s):
    c = s["case"]
    bfa.call("dpack_tran" if c["tran"] else "dpack", c["ps"], c["batch"], s["args"].data_ptr(), s["hint"], _stream())
    bfa.call("dunpack", c["ps"], c["batch"], s["args2"].data_ptr(), s["hint"], _stream())
    return s["P"].buf, s["out"]


def _pack_exact(c, seed):
    s = _pack_prepare(c, seed)
    h, R, out = c["hi"], s["P"], torch.zeros_like(s["A"])
    for sel in _chunks(c["batch"], 4 * h * h):
        t = lambda a: torch.from_numpy(a[sel]).to(DEV)[:, None, None]  # noqa: E731
        i, j = torch.arange(h, device=DEV)[None, :, None], torch.arange(h, device=DEV)[None, None, :]
        ok = (i < t(s["m"])) & (j < t(s["n"]))
        at = t(s["first"]) + i + j * t(s["m"])
        dense = torch.where(ok, s["A"][torch.where(ok, at, torch.zeros_like(at))], 0.0)
        if c["tran"]:
            dense = dense.transpose(1, 2).contiguous()
        R.put(sel, dense)
        ok = (i < t(s["pm"])) & (j < t(s["pn"]))
        out[(t(s["first"]) + i + j * t(s["pm"]))[ok]] = dense[ok]
    return R.buf, out


def _pack_work(c):
    m, n = _sizes(c, 1).astype(float), _sizes(c, 2).astype(float)
    return {"bytes": 32 * (m * n).sum(), "flops": 0}


# ---------------------------------------------------------------------------
# Riccati recursion
# ---------------------------------------------------------------------------
class Vecs:
    """Vectors of the given sizes in one zeroed GPU buffer, with their descriptors."""

    def __init__(self, ps, sizes):
        self.sizes = np.asarray(sizes, np.int64)
        pm = -(-self.sizes // ps) * ps
        mem = -(-(pm * 8) // 64) * 64
        offs = np.concatenate([[0], np.cumsum(mem)[:-1]])
        self.off = offs // 8
        self.buf = torch.zeros(int(mem.sum()) // 8, dtype=torch.float64, device=DEV)
        d = np.zeros(len(self.sizes), dtype=bfa.DVEC)
        d["mem"] = d["pa"] = np.uint64(self.buf.data_ptr()) + offs.astype(np.uint64)
        d["m"], d["pm"], d["memsize"] = self.sizes, pm, mem
        self.dev = _dev(d)

    def addr(self, per):
        """Address of the descriptor array of each instance (`per` vectors each)."""
        count = len(self.sizes) // per
        return np.uint64(self.dev.data_ptr()) + np.arange(count, dtype=np.uint64) * np.uint64(per * bfa.DVEC.itemsize)

    def put(self, sel, dense):
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a[sel])).to(DEV)[:, None]  # noqa: E731
        j = torch.arange(dense.shape[1], device=DEV)[None, :]
        ok = j < t(self.sizes)
        self.buf[(t(self.off) + j)[ok]] = dense[ok]


def _ric_dense(c, g, nx, nu, NX, NU, aug):
    """Inputs of some instances with inputs padded to NU and states to NX:
    A = I + N(0,1)/10 (scaled so that larger systems do not grow faster than
    ones of 8 states), B ~ N(0,1), Q = R = I, and with aug b, r, q ~ N(0,1)."""
    k = len(nx)
    tx = torch.from_numpy(np.asarray(nx)).to(DEV)[:, None]
    tu = torch.from_numpy(np.asarray(nu)).to(DEV)[:, None]
    okx = torch.arange(NX, device=DEV)[None, :] < tx
    oku = torch.arange(NU, device=DEV)[None, :] < tu
    scale = 0.1 * (8.0 / torch.clamp(tx, min=8).double()).sqrt()[:, :, None]
    A = torch.eye(NX, device=DEV, dtype=torch.float64) + scale * _randn(g, k, NX, NX)
    A = A * okx[:, :, None] * okx[:, None, :]
    B = _randn(g, k, NX, NU) * okx[:, :, None] * oku[:, None, :]
    C = torch.cat([B, A], 2).transpose(1, 2).contiguous()  # [B^T; A^T]
    vec = lambda ok: _randn(g, *ok.shape) * ok  # noqa: E731
    extra = (vec(okx), vec(torch.cat([oku, okx], 1)), vec(okx)) if aug else None
    return C, extra


def _compact(nx, nu, NX, NU, n):
    """Where entry i of an instance's [u; x] is in the padded [u; x]."""
    t = lambda a: torch.from_numpy(np.asarray(a)).to(DEV)[:, None]  # noqa: E731
    i = torch.arange(n, device=DEV)[None, :]
    return torch.where(i < t(nu), i, torch.clamp(i - t(nu) + NU, max=NU + NX - 1))


def _rows(M, at):
    return torch.gather(M, 1, at[:, :, None].expand(-1, -1, M.shape[2]))


def _cols(M, at):
    return torch.gather(M, 2, at[:, None, :].expand(-1, M.shape[1], -1))


def _ric_sizes(c):
    return _sizes(c, 1, "nx_lo", "nx_hi"), _sizes(c, 2, "nu_lo", "nu_hi")


def _ric_prepare(c, seed, keep=None):
    g, ps, n, N = _gen(seed), c["ps"], c["batch"], c["N"]
    nx, nu = _ric_sizes(c)
    nk = nx + nu
    aug = 1 if c["op"] == "ric_sv" else 0
    NX, NU = c["nx_hi"], c["nu_hi"]
    C, R, Q = Mats("d", ps, nk + aug, nx), Mats("d", ps, nk + aug, nk), Mats("d", ps, nx + aug, nx)
    stage = lambda a, last: np.concatenate([np.repeat(a[:, None], N, 1), last[:, None]], 1).reshape(-1)  # noqa: E731
    L = Mats("d", ps, stage(nk + aug, nx + aug), stage(nk, nx))
    work = Mats("d", ps, nk + aug, nx)
    solve = c["op"] == "ric_solve"
    vecs = {}
    if solve or aug:
        kinds = (("b", nx, None), ("rq", nk, nx), ("Pb", nx, None)) if solve else ()
        for kind, size, last in kinds + (("ux", nk, nx), ("pi", nx, None), ("work", nx[:, None], None)):
            if kind == "work":
                vecs[kind] = Vecs(ps, nx)
            else:
                vecs[kind] = Vecs(ps, np.repeat(size, N) if last is None else stage(size, last))
    chunks = _chunks(n, 8 * (NX + NU) ** 2)
    for sel in chunks:
        Cd, extra = _ric_dense(c, g, nx[sel], nu[sel], NX, NU, aug)
        at = _compact(nx[sel], nu[sel], NX, NU, NX + NU)
        e = torch.eye(NX + NU, device=DEV, dtype=torch.float64).expand(len(sel), -1, -1)
        Cc, Rc, Qc = _rows(Cd, at), e, e[:, :NX, :NX]
        if keep is not None:
            keep.append((sel, Cd, extra))
        if aug:
            place = lambda M, sizes, row: torch.cat([M, torch.zeros_like(M[:, :1])], 1).scatter(  # noqa: E731
                1, torch.from_numpy(sizes).to(DEV)[:, None, None].expand(-1, 1, M.shape[2]), row[:, None, :])
            b, rq, q = extra
            # rows beyond a size hold nothing: put() takes size + 1 rows
            mask = lambda M, sizes: M * (torch.arange(M.shape[1], device=DEV)[None, :, None] < torch.from_numpy(sizes).to(DEV)[:, None, None])  # noqa: E731
            Cc = place(mask(Cc, nk[sel]), nk[sel], b)
            Rc = place(mask(Rc, nk[sel]), nk[sel], torch.gather(rq, 1, at))
            Qc = place(mask(Qc, nx[sel]), nx[sel], q)
        C.put(sel, Cc)
        R.put(sel, Rc)
        Q.put(sel, Qc)
    if solve:
        # dense vectors in the batch's own order, one stage after the other
        for kind in ("b", "rq"):
            v = vecs[kind]
            for sel in _chunks(len(v.sizes), NX + NU):
                v.put(sel, _randn(g, len(sel), NX + NU))
    rep = lambda M, count: np.repeat(M.desc, count)  # noqa: E731
    rsq = np.concatenate([rep(R, N).reshape(n, N), Q.desc[:, None]], 1).reshape(-1)
    t = [_dev(rep(C, N)), _dev(rsq), L.dev, work.dev, _dev(np.repeat(nx, N + 1).astype(np.int32)),
         _dev(stage(nu, np.zeros_like(nu)).astype(np.int32))]
    idx = np.arange(n, dtype=np.uint64)
    at = lambda x, size: np.uint64(x.data_ptr()) + idx * np.uint64(size)  # noqa: E731
    f = dict(N=N, nx=at(t[4], 4 * (N + 1)), nu=at(t[5], 4 * (N + 1)), BAbt=at(t[0], bfa.DMAT.itemsize * N),
             L=at(t[2], bfa.DMAT.itemsize * (N + 1)))
    rsq_at = at(t[1], bfa.DMAT.itemsize * (N + 1))
    s = dict(case=c, tabs=t, mats=(C, R, Q, work), L=L, vecs=vecs, nx=nx, nu=nu,
             hint=(int(nk.max()), int(nx.max()), 0))
    if aug:
        s["args"] = _records(bfa.RICCATI_SV_ARG, n, RSQrq=rsq_at, work_mat=at(t[3], bfa.DMAT.itemsize),
                             work_vec=vecs["work"].addr(1), ux=vecs["ux"].addr(N + 1), pi=vecs["pi"].addr(N), **f)
    else:
        s["args"] = _records(bfa.RICCATI_ARG, n, RSQrq=rsq_at, work=at(t[3], bfa.DMAT.itemsize), **f)
    if solve:
        per = dict(b=N, rq=N + 1, Pb=N, ux=N + 1, pi=N, work=1)
        s["args2"] = _records(bfa.RICCATI_TRS_ARG, n, **f, **{k: vecs[k].addr(per[k]) for k in per})
    return s


def _ric_run(s):
    c = s["case"]
    ps, n, st = c["ps"], c["batch"], _stream()
    if c["op"] == "ric_sv":
        bfa.call("d_back_ric_sv", ps, n, s["args"].data_ptr(), s["hint"], st)
        return s["L"].buf, s["vecs"]["ux"].buf, s["vecs"]["pi"].buf
    bfa.call("d_back_ric_trf", ps, n, s["args"].data_ptr(), s["hint"], st)
    if c["op"] == "ric_trf":
        return s["L"].buf
    bfa.call("d_back_ric_trs", ps, n, s["args2"].data_ptr(), s["hint"], st)
    return s["L"].buf, s["vecs"]["Pb"].buf, s["vecs"]["ux"].buf, s["vecs"]["pi"].buf


def _ric_exact(c, seed):
    keep = []
    s = _ric_prepare(c, seed, keep)
    N, n, NX, NU, ps = c["N"], c["batch"], c["nx_hi"], c["nu_hi"], c["ps"]
    nx, nu = s["nx"], s["nu"]
    nk = nx + nu
    aug = c["op"] == "ric_sv"
    solve = c["op"] == "ric_solve"
    R = Mats("d", ps, s["L"].ms, s["L"].ns)
    out = {k: Vecs(ps, s["vecs"][k].sizes) for k in ("Pb", "ux", "pi") if k in s["vecs"]}
    mv = lambda M, v: torch.matmul(M, v[:, :, None])[:, :, 0]  # noqa: E731
    T = lambda M: M.transpose(1, 2).contiguous()  # noqa: E731
    tri = lambda M, v, up=False: torch.linalg.solve_triangular(M, v[:, :, None], upper=up)[:, :, 0]  # noqa: E731
    for sel, C, extra in keep:
        k = len(sel)
        at = _compact(nx[sel], nu[sel], NX, NU, NX + NU)

        def emit(stage, Lk, row, last=False):
            where = sel * (N + 1) + stage
            size = nx[sel] if last else nk[sel]
            D = Lk if last else _cols(_rows(Lk, at), at)
            diag = torch.diagonal(D, dim1=1, dim2=2)
            D = D * (torch.arange(D.shape[2], device=DEV)[None, None, :] < torch.from_numpy(size).to(DEV)[:, None, None])
            D = D.tril()
            if row is not None:
                r = row if last else torch.gather(row, 1, at)
                D = torch.cat([D, torch.zeros_like(D[:, :1])], 1).scatter(
                    1, torch.from_numpy(size).to(DEV)[:, None, None].expand(-1, 1, D.shape[2]), r[:, None, :])
            R.put(where, D)
            R.put_diag(where, 1.0 / diag, size)

        def vector(v, kind, stage, per, only=None):
            where = sel * per + stage
            size, st = s["vecs"][kind].sizes[where], s["vecs"][kind]
            j = torch.arange(int(size.max()), device=DEV)[None, :]
            o = torch.from_numpy(np.ascontiguousarray(st.off[where])).to(DEV)[:, None]
            ok = j < torch.from_numpy(size).to(DEV)[:, None]
            d = torch.where(ok, st.buf[torch.where(ok, o + j, torch.zeros_like(j))], 0.0)
            return d

        def padded(v, is_x):
            """A vector in an instance's own order, at its padded place."""
            size = nx[sel] if is_x else nk[sel]
            ok = torch.arange(v.shape[1], device=DEV)[None, :] < torch.from_numpy(size).to(DEV)[:, None]
            if is_x:
                w = torch.zeros(k, NX, device=DEV, dtype=torch.float64)
                w[:, :v.shape[1]] = v * ok
                return w
            w = torch.zeros(k, NU + NX, device=DEV, dtype=torch.float64)
            return w.scatter_add(1, at[:, :v.shape[1]], v * ok)

        Lxx = torch.eye(NX, device=DEV, dtype=torch.float64).expand(k, -1, -1).contiguous()
        p = rowx = None
        if aug:
            b_all, rq_all, q = extra
            p, rowx = q, q  # P_N = I
        if solve:
            p = padded(vector(None, "rq", N, N + 1), True)
        emit(N, Lxx, rowx, True)
        Ls, vs, Ps, ps_ = [None] * N, [None] * N, [None] * (N + 1), [None] * (N + 1)
        Ps[N], ps_[N] = Lxx, p
        for st in range(N - 1, -1, -1):
            W = torch.matmul(C, Lxx)
            M = torch.eye(NU + NX, device=DEV, dtype=torch.float64) + torch.matmul(W, T(W))
            Lk = torch.linalg.cholesky(M)
            row = None
            if aug or solve:
                if aug:
                    b, rq = b_all, rq_all
                else:
                    b = padded(vector(None, "b", st, N), True)
                    rq = padded(vector(None, "rq", st, N + 1), False)
                Pb = mv(Lxx, mv(T(Lxx), b))
                if solve:
                    out["Pb"].put(sel * N + st, Pb)
                v = rq + mv(C, Pb + p)
                row = tri(Lk, v)
                Ls[st], vs[st] = Lk, row
                p = mv(Lk[:, NU:, NU:], row[:, NU:])
            emit(st, Lk, row if aug else None)
            Lxx = Lk[:, NU:, NU:].contiguous()
            Ps[st], ps_[st] = Lxx, p
        if aug or solve:
            z = -tri(T(Ls[0]), vs[0], True)
            for st in range(N):
                if st > 0:
                    Lk = Ls[st]
                    u = -tri(T(Lk[:, :NU, :NU]), vs[st][:, :NU] + mv(T(Lk[:, NU:, :NU]), x), True)  # noqa: F821
                    z = torch.cat([u, x], 1)  # noqa: F821
                out["ux"].put(sel * (N + 1) + st, torch.gather(z, 1, at))
                b = b_all if aug else padded(vector(None, "b", st, N), True)
                x = mv(T(C), z) + b
                Pk = Ps[st + 1]
                out["pi"].put(sel * N + st, ps_[st + 1] + mv(Pk, mv(T(Pk), x)))
            out["ux"].put(sel * (N + 1) + N, x)
    if aug:
        return R.buf, out["ux"].buf, out["pi"].buf
    return (R.buf, out["Pb"].buf, out["ux"].buf, out["pi"].buf) if solve else R.buf


def _ric_work(c):
    nx, nu = (v.astype(float) for v in _ric_sizes(c))
    nk, N = nx + nu, c["N"]
    tri = lambda v: v * (v + 1) / 2  # noqa: E731
    b = 8 * (nk * nx + tri(nk) + tri(nx) + N * (tri(nk) + nk) + tri(nx) + nx).sum()
    f = N * (nk * nx * nx + nk * nk * nx + nk ** 3 / 3).sum() + (nx ** 3 / 3).sum()
    if c["op"] != "ric_trf":
        b += 8 * (N * (nk + nx)).sum()
        f += N * (4 * nx * nx + 4 * nk * nx + 2 * nk * nk).sum()
    if c["op"] == "ric_solve":
        b += 8 * (N * (nk + 2 * nx)).sum()
    return {"bytes": float(b), "flops": float(f)}


# ---------------------------------------------------------------------------
_OPS = {
    "ric_solve": (_ric_prepare, _ric_run, _ric_exact, _ric_work),
    "ric_trf": (_ric_prepare, _ric_run, _ric_exact, _ric_work),
    "ric_sv": (_ric_prepare, _ric_run, _ric_exact, _ric_work),
    "potrf": (_potrf_prepare, _potrf_run, _potrf_exact, _potrf_work),
    "syrk_potrf": (_potrf_prepare, _potrf_run, _potrf_exact, _potrf_work),
    "spd_solve": (_potrf_prepare, _potrf_run, _potrf_exact, _potrf_work),
    "gemm_syrk": (_gemm_prepare, _gemm_run, _gemm_exact, _gemm_work),
    "gemm_nn": (_gemm_prepare, _gemm_run, _gemm_exact, _gemm_work),
    "trsm": (_trsm_prepare, _trsm_run, _trsm_exact, _trsm_work),
    "lu_solve": (_lu_prepare, _lu_run, _lu_exact, _lu_work),
    "pack": (_pack_prepare, _pack_run, _pack_exact, _pack_work),
}


def _stream():
    return torch.cuda.current_stream().cuda_stream


def prepare(case, seed):
    return _OPS[case["op"]][0](case, seed)


def run(state):
    return _OPS[state["case"]["op"]][1](state)


def exact(case, seed):
    return _OPS[case["op"]][2](case, seed)


def work(case):
    w = _OPS[case["op"]][3](case)
    return {"bytes": float(w["bytes"]), "flops": float(w["flops"])}
