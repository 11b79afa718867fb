"""Blocks of matrices of more than 4 GiB, shared by the GPU test and the CPU kernel
emulator: 70 x 70 blocks whose byte offsets pass 2^32 within the block ("stride", a
panel stride of 10 million columns) or before it ("deep", below row 400 of a matrix of
1.5 million columns).  All matrices share one buffer, each with columns and a descriptor
of its own; the results are compared with numpy."""
import ctypes

import numpy as np

import blasfeo_amd as bfa

GEOM = {"stride": (80, 10_000_000, 3), "deep": (488, 1_500_000, 403)}   # rows, panel stride, first row of a block
N = 70
SLOT = 96          # columns of a matrix
OPS = ["gemm_nt", "gemm_nn", "syrk_ln", "trsm_rltn", "trsm_llnn", "trsm_lltn", "trsm_llnu", "trsm_lunn", "potrf_l",
       "potrf_l one wave", "syrk_dpotrf_ln", "getrf_rp", "getrf_np", "ric_trf"]


class Store:
    """The shared buffer: element (i, j) of matrix s, through put and get of flat indices."""

    def __init__(self, ps, geom, base, put, get):
        self.ps, self.base, self.put, self.get = ps, base, put, get
        self.rows, self.cn, self.r0 = GEOM[geom]
        self.used = 0

    def at(self, s, i, j):
        i, j = np.broadcast_arrays(np.asarray(i, np.int64)[:, None], np.asarray(j, np.int64)[None, :] + s)
        return (i // self.ps * self.cn + j) * self.ps + i % self.ps

    def new(self, A, ri, cj):
        # the last columns of the stride, counted down
        self.used += SLOT
        s = self.cn - self.used
        m, n = A.shape
        self.put(self.at(s, ri + np.arange(m), cj + np.arange(n)).ravel(), A.ravel())
        return dict(slot=s, ri=ri, cj=cj, shape=A.shape)

    def read(self, M):
        m, n = M["shape"]
        return self.get(self.at(M["slot"], M["ri"] + np.arange(m), M["cj"] + np.arange(n)).ravel()).reshape(m, n)

    def desc(self, mats, diag):
        """Descriptors of mats; diag: address of 128 doubles for each."""
        d = np.zeros(len(mats), bfa.DMAT)
        for i, M in enumerate(mats):
            d[i]["mem"] = d[i]["pA"] = self.base + 8 * self.ps * M["slot"]
            d[i]["dA"] = diag + 1024 * i
            d[i]["m"], d[i]["n"] = self.rows, SLOT
            d[i]["pm"], d[i]["cn"] = self.rows, self.cn
        return d


def spd(rng, n):
    B = rng.uniform(-1, 1, (n, n))
    return B @ B.T + n * np.eye(n)


def lu(A, pivot):
    A, p = A.copy(), []
    for j in range(len(A)):
        k = j + int(np.argmax(np.abs(A[j:, j]))) if pivot else j
        p.append(k)
        A[[j, k]] = A[[k, j]]
        A[j + 1:, j] /= A[j, j]
        A[j + 1:, j + 1:] -= np.outer(A[j + 1:, j], A[j, j + 1:])
    return A, p


def run(op, ps, geom, store, upload, lib):
    """One call of op on the store; upload(array) -> (address, handle), lib(entry, batch, records'
    address, hint) runs it."""
    rng = np.random.default_rng(17)
    r0 = store.r0
    keep, mats = [], []

    def up(a):
        addr, h = upload(np.ascontiguousarray(a))
        keep.append((addr, h))
        return addr

    def new(A, ri=None, cj=2):
        M = store.new(A, r0 if ri is None else ri, cj)
        mats.append(M)
        return M

    def call(entry, dtype, rec, hint):
        desc = up(store.desc(mats, up(np.zeros(128 * len(mats)))))
        r = np.zeros(1, dtype)
        for k, v in rec.items():
            r[0][k] = desc + mats.index(v) * bfa.DMAT.itemsize if isinstance(v, dict) else v
        lib(entry, 1, up(r), hint)

    def close(M, want, mask=None):
        got = store.read(M)
        if mask is not None:
            got, want = got * mask, want * mask
        np.testing.assert_allclose(got, want, rtol=1e-11, atol=1e-11, err_msg="%s %s ps=%d" % (op, geom, ps))

    A, B, C = (rng.uniform(-1, 1, (N, N)) for _ in range(3))
    low = np.tril(np.ones((N, N)))
    at = lambda f, M: {f + "i": M["ri"], f + "j": M["cj"]}  # noqa: E731
    if op in ("gemm_nt", "gemm_nn", "syrk_ln"):
        a, b, c, d = new(A), new(B), new(C, r0 + 1), new(np.zeros((N, N)))
        call("d" + op, bfa.DGEMM_ARG, dict(m=N, n=N, k=N, alpha=1.5, beta=-0.5, sA=a, sB=b, sC=c, sD=d,
                                           **at("a", a), **at("b", b), **at("c", c), **at("d", d)), (N, N, N))
        close(d, 1.5 * A @ (B if op == "gemm_nn" else B.T) - 0.5 * C, low if op == "syrk_ln" else None)
    elif op.startswith("trsm"):
        T = np.tril(A) / N + 2 * np.eye(N)
        T = {"trsm_llnu": np.tril(T, -1) + np.eye(N), "trsm_lunn": T.T}.get(op, T)
        n = N if op == "trsm_rltn" else 3
        R = B[:, :n]
        a, b, d = new(T), new(R), new(np.zeros((N, n)))
        call("d" + op, bfa.DTRSM_ARG, dict(m=N, n=n, alpha=1.0, sA=a, sB=b, sD=d, **at("a", a), **at("b", b), **at("d", d)),
             (N, n, 0))
        close(d, np.linalg.solve(T, R.T).T if op == "trsm_rltn" else np.linalg.solve(T.T if op == "trsm_lltn" else T, R))
    elif op.startswith("potrf"):
        S = spd(rng, N)
        c, d = new(S), new(np.zeros((N, N)))
        call("dpotrf_l", bfa.DFACT_ARG, dict(m=N, n=N, sC=c, sD=d, **at("c", c), **at("d", d)), (N, N, 0))
        close(d, np.linalg.cholesky(S), low)
    elif op == "syrk_dpotrf_ln":
        S = spd(rng, N)
        a, c, d = new(A), new(S), new(np.zeros((N, N)))
        call("dsyrk_dpotrf_ln", bfa.DSYRK_DPOTRF_ARG, dict(m=N, n=N, k=N, sA=a, sB=a, sC=c, sD=d, **at("a", a), **at("b", a),
                                                           **at("c", c), **at("d", d)), (N, N, N))
        close(d, np.linalg.cholesky(S + A @ A.T), low)
    elif op.startswith("getrf"):
        S = A if op == "getrf_rp" else A + N * np.eye(N)
        c, d = new(S), new(np.zeros((N, N)))
        piv = up(np.zeros(N, np.int32))
        call("d" + op, bfa.DFACT_ARG, dict(m=N, n=N, sC=c, sD=d, ipiv=piv, **at("c", c), **at("d", d)), (N, N, 0))
        close(d, lu(S, op == "getrf_rp")[0])
    else:
        # one stage of 60 states and 10 inputs, its matrices from row 0 on
        nx, nu = 60, 10
        BA = rng.uniform(-1, 1, (N, nx)) / 8
        R, Q = spd(rng, N), spd(rng, nx)
        b, r, q, l0, l1, w = (new(M, 0, 0) for M in (BA, R, Q, np.zeros((N, N)), np.zeros((nx, nx)), np.zeros((N, nx))))
        desc = up(store.desc(mats, up(np.zeros(128 * len(mats)))))
        row = lambda M: desc + mats.index(M) * bfa.DMAT.itemsize  # noqa: E731
        rec = np.zeros(1, bfa.RICCATI_ARG)
        rec[0]["N"], rec[0]["BAbt"], rec[0]["RSQrq"], rec[0]["L"], rec[0]["work"] = 1, row(b), row(r), row(l0), row(w)
        rec[0]["nx"], rec[0]["nu"] = up(np.array([nx, nx], np.int32)), up(np.array([nu, 0], np.int32))
        lib("d_back_ric_trf", 1, up(rec), (N, nx, 0))
        L1 = np.linalg.cholesky(Q)
        W = BA @ L1
        close(l1, L1, low[:nx, :nx])
        close(l0, np.linalg.cholesky(R + W @ W.T), low)


def knobs(op):
    if op == "potrf_l one wave":
        return {"potrf_bw": 1}
    return {"trsm_thin": 1} if op.startswith("trsm_l") else {}


def hint(h):
    return ctypes.byref(bfa.HINT(*h))
