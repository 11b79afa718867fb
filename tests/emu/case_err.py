"""Emulator cases (TEST INFRASTRUCTURE ONLY): rounding errors of factorisations against
extended precision, beside those of the same factorisation in numpy's float64 with the
finished blocks' products summed from zero and the matrix element joined last.  A sum begun at the
element is rounded at the element's size in every step, and on these inputs the errors
are then more than twice as large; 1.25 leaves room for the order of the sums.
Usage: python case_err.py <getrf | syrk_dpotrf | riccati>"""
import ctypes
import sys

import numpy as np

from emu_harness import Block, Mat, emu_lib, records, bfa

PS = 4


def mat(A):
    M = Mat(PS, *A.shape)
    M.fill(A)
    return M


def get(M, m, n):
    return bfa.pm_unpack(M.content()[: M.pm * M.cn], PS, M.cn, m, n)


def call(E, entry, dtype, recs, hint):
    blk = records(dtype, recs)
    rc = getattr(E, "blasfeo_amd_%s_batched" % entry)(PS, len(recs), ctypes.c_void_p(blk.addr), ctypes.byref(bfa.HINT(*hint)), None)
    assert rc == 0, E.emu_last_error()


def rms(x, ref):
    d = (x - ref).astype(float)
    return np.sqrt((d * d).mean() / (ref.astype(float) ** 2).mean())


def products(L, U):
    s = np.zeros((L.shape[0], U.shape[1]), L.dtype)
    for k in range(L.shape[1]):
        s = s + np.outer(L[:, k], U[k])
    return s


def lu(A, nb=16):
    """L and U of A without pivoting in A's type, by rows and columns of nb, as the kernel
    takes them: the finished columns' products summed from zero, then a panel and a
    block row column by column."""
    A, n = A.copy(), len(A)
    for c in range(0, n, nb):
        e = min(c + nb, n)
        A[c:, c:e] -= products(A[c:, :c], A[:c, c:e])
        A[c:e, e:] -= products(A[c:e, :c], A[:c, e:])
        for j in range(c, e):
            A[j + 1:, j] *= A.dtype.type(1) / A[j, j]
            A[j + 1:, j + 1:e] -= np.outer(A[j + 1:, j], A[j, j + 1:e])
            A[j + 1:e, e:] -= np.outer(A[j + 1:e, j], A[j, e:])
    return A


def run_getrf(E):
    rng = np.random.default_rng(5)
    kernel, plain = [], []
    for n in (96, 130, 200, 256):
        # row by row the largest entry in another place: the pivots' order is known
        A = rng.uniform(-1, 1, (n, n)) + 0.7 * np.sqrt(n) * np.eye(n)
        p = rng.permutation(n)
        D, piv = mat(np.zeros((n, n))), Block(4 * n)
        print("emu error of dgetrf_rp n=%d" % n, flush=True)
        call(E, "dgetrf_rp", bfa.DFACT_ARG, [dict(m=n, n=n, sC=mat(A[p]), sD=D, ipiv=piv.addr)], (n, n, 0))
        B = A[p]
        for i, j in enumerate(piv.read(np.int32)):
            B[[i, j]] = B[[j, i]]
        exact = lu(B.astype(np.longdouble))
        kernel.append(rms(get(D, n, n), exact))
        plain.append(rms(lu(B), exact))
    return kernel, plain


def chol(A):
    A, n = A.copy(), len(A)
    for j in range(n):
        A[j:, j] *= A.dtype.type(1) / np.sqrt(A[j, j])
        A[j + 1:, j + 1:] -= np.outer(A[j + 1:, j], A[j + 1:, j])
    return np.tril(A)


def spd(rng, n):
    B = rng.standard_normal((n, n))
    return B @ B.T / n + np.eye(n)


def run_syrk_dpotrf(E):
    rng = np.random.default_rng(6)
    kernel, plain = [], []
    for n in (32, 64, 90, 128):
        C, A = 10 * spd(rng, n), 0.1 * rng.standard_normal((n, n))
        a, D = mat(A), mat(np.zeros((n, n)))
        print("emu error of dsyrk_dpotrf_ln n=%d" % n, flush=True)
        call(E, "dsyrk_dpotrf_ln", bfa.DSYRK_DPOTRF_ARG, [dict(m=n, n=n, k=n, sA=a, sB=a, sC=mat(C), sD=D)], (n, n, n))
        X = A.astype(np.longdouble)
        exact = chol(C.astype(np.longdouble) + products(X, X.T))
        kernel.append(rms(np.tril(get(D, n, n)), exact))
        plain.append(rms(chol(C + products(A, A.T)), exact))
    return kernel, plain


class Table:
    """An array in its own block, as a field of a record."""

    def __init__(self, a):
        self.desc = Block(a.nbytes)
        self.desc.write(a)


def run_riccati(E):
    """One stage, RSQ large beside W W^T: the factor of stage 0."""
    rng = np.random.default_rng(7)
    kernel, plain = [], []
    for nx, nu in ((20, 6), (40, 12), (64, 20), (64, 60)):
        n = nx + nu
        BA, R, Q = 0.1 * rng.standard_normal((n, nx)), 10 * spd(rng, n), spd(rng, nx)
        b, r, q, l0, l1, w = (mat(M) for M in (BA, R, Q, np.zeros((n, n)), np.zeros((nx, nx)), np.zeros((n, nx))))
        desc = lambda *ms: Table(np.concatenate([m.desc.read(bfa.DMAT) for m in ms]))  # noqa: E731
        print("emu error of d_back_ric_trf nx=%d nu=%d" % (nx, nu), flush=True)
        call(E, "d_back_ric_trf", bfa.RICCATI_ARG,
             [dict(N=1, nx=Table(np.array([nx, nx], np.int32)).desc.addr, nu=Table(np.array([nu, 0], np.int32)).desc.addr,
                   BAbt=desc(b).desc.addr, RSQrq=desc(r, q).desc.addr, L=desc(l0, l1).desc.addr, work=w)], (n, nx, 0))
        for f, out in ((np.longdouble, None), (np.float64, plain)):
            W = products(BA.astype(f), chol(Q.astype(f)))
            L = chol(R.astype(f) + products(W, W.T))
            if out is None:
                exact = L
            else:
                out.append(rms(L, exact))
        kernel.append(rms(np.tril(get(l0, n, n)), exact))
    return kernel, plain


if __name__ == "__main__":
    kernel, plain = globals()["run_" + sys.argv[1]](emu_lib("emu_lapack"))
    print("kernel", kernel, "plain", plain)
    assert np.mean(kernel) <= 1.25 * np.mean(plain), (kernel, plain)
    print("ok", flush=True)
