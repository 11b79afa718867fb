"""Record sets of the LU tests shared by the GPU tests and the CPU kernel emulator
(tests/emu/); same case format as tests/chol_cases.py."""
import numpy as np

# at the edges of 16-row and 16-column blocks, of the 64 rows a lane slot holds and
# of the 256 rows a workgroup takes; tall and wide
SIZES = [(1, 1), (5, 5), (15, 16), (16, 15), (17, 17), (16, 40), (40, 16), (33, 64), (64, 33), (65, 65), (100, 7), (7, 100),
         (63, 80), (128, 129), (150, 70), (70, 150), (193, 192), (192, 193), (256, 256), (256, 20), (20, 256), (65, 300), (255, 272)]


def lu(ps, seed, pivot=True):
    """getrf of SIZES, offsets on every second one, in place on every third (the
    two combined now and then), then ties in every column, a permutation, a
    zero column, a NaN and an Inf (with pivoting only)."""
    rng = np.random.default_rng(seed)
    out = []

    def add(A, r):
        m, n = A.shape
        ci, di = ((int(rng.integers(0, 2 * ps)), int(rng.integers(0, 2 * ps))) if r % 2 else (0, 0))
        cj, dj = ((int(rng.integers(0, 3)), int(rng.integers(0, 3))) if r % 2 else (0, 0))
        S = np.zeros((ci + m, cj + n))
        S[ci:, cj:] = A
        mats = {"sC": (ci + m, cj + n, S)}
        if r % 3 == 2:
            mats["sD"] = "=sC"
            di, dj = ci, cj
        else:
            mats["sD"] = (di + m, dj + n, -1.0)
        out.append((mats, dict(m=m, n=n, ci=ci, cj=cj, di=di, dj=dj)))

    for r, (m, n) in enumerate(SIZES):
        A = rng.uniform(-1, 1, (m, n))
        if not pivot:
            A[np.arange(min(m, n)), np.arange(min(m, n))] += m
        add(A, r)
    if pivot:
        for r in range(6):   # in both forms
            add(np.ones((70, 70)) + np.eye(70), r)
        for r in range(3):
            add(np.eye(137)[rng.permutation(137)], r)
            Z = rng.integers(-2, 3, (40, 44)).astype(float)
            Z[:, 4] = 0.0
            add(Z, r)
            N = rng.uniform(-1, 1, (90, 90))
            N[70, 0] = np.nan
            add(N, r)
            N = rng.uniform(-1, 1, (90, 70))
            N[80, 3] = np.inf
            add(N, r)
    return out
