"""The drop-in LU interface at the edges of its sweeps' columns (8x8 points),
chunks (8 steps) and rounds (32 steps): random couplings, different in the two
directions, with and without the phi wrap, against the ILU(0) solve of the same
FP32 matrix in float64.

Tolerance: the matrix is diagonally dominant (the couplings of a row add up to
at most 6/8 of its diagonal), so a sweep damps what each point adds, a handful
of FP32 roundings (6e-8) of values no larger than the largest: 1e-5 of it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

OFFS = ((0, 0, -1), (0, -1, 0), (-1, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1))  # (i, j, k)


def _matrix(dims, wrap, seed):
    """1-based CSR in the driver's order of columns, and per row and offset
    the neighbour (-1: none) and coupling."""
    a, b, c = dims
    n = a * b * c
    rng = np.random.default_rng(seed)
    p = np.arange(n)
    i, j, k = p % a, (p // a) % b, p // (a * b)
    nb = np.full((6, n), -1, dtype=np.int64)
    for q, (di, dj, dk) in enumerate(OFFS):
        kk = k + dk
        ok = (0 <= i + di) & (i + di < a) & (0 <= j + dj) & (j + dj < b)
        ok &= np.full(n, True) if wrap else (0 <= kk) & (kk < c)
        nb[q] = np.where(ok, (i + di) + a * ((j + dj) + b * (kk % c)), -1)
    v = (-rng.uniform(0.2, 1.0, (6, n))).astype(np.float32)
    dg = rng.uniform(8.0, 9.0, n).astype(np.float32)
    ia, ja, av = [1], [], []
    for r in range(n):
        # the wrap to the last plane (row of plane 0) comes last, the one to
        # plane 0 (row of the last plane) first: by the column it would have
        at = []
        for q, (di, dj, dk) in enumerate(OFFS):
            if nb[q, r] >= 0:
                at.append((r + di + a * (dj + b * dk), int(nb[q, r]), float(v[q, r])))
        at.append((r, r, float(dg[r])))
        at.sort()
        for part in ([e for e in at if e[0] >= n], [e for e in at if 0 <= e[0] < n],
                     [e for e in at if e[0] < 0]):
            for _, col, val in part:
                ja.append(col + 1)
                av.append(val)
        ia.append(len(ja) + 1)
    return (np.array(ia, np.int32), np.array(ja, np.int32), np.array(av, np.float32),
            nb, v.astype(np.float64), dg.astype(np.float64))


def _ilu_solve(dims, nb, v, dg, x):
    """The D-ILU solve (equal to ILU(0) on this pattern) in float64."""
    a, b, c = dims
    n = a * b * c
    p = np.arange(n)
    lev = p % a + (p // a) % b + p // (a * b)
    levels = [np.flatnonzero(lev == s) for s in range(int(lev.max()) + 1)]
    lower = [(nb[q] >= 0) & (nb[q] < p) for q in range(6)]
    upper = [(nb[q] >= 0) & (nb[q] > p) for q in range(6)]
    back = [5, 4, 3, 2, 1, 0]  # the neighbour's offset back to the row
    d, t, z = np.zeros(n + 1), np.zeros(n + 1), np.zeros(n + 1)
    y = np.zeros(n)
    for s in levels:
        d[s], y[s] = dg[s], x[s]
        for q in range(6):
            m = np.where(lower[q][s], nb[q][s], n)
            d[s] -= np.where(m < n, v[q][s] * v[back[q]][np.minimum(m, n - 1)], 0.0) / np.where(
                m < n, d[m], 1.0)
            y[s] -= np.where(m < n, v[q][s] * t[m], 0.0)
        t[s] = y[s] / d[s]
    for s in reversed(levels):
        z[s] = y[s]
        for q in range(6):
            m = np.where(upper[q][s], nb[q][s], n)
            z[s] -= np.where(m < n, v[q][s] * z[m], 0.0)
        z[s] /= d[s]
    return z[:n]


@pytest.mark.parametrize("wrap", [True, False])
@pytest.mark.parametrize("dims", [(2, 2, 8), (8, 8, 9), (9, 17, 11), (3, 5, 40), (17, 8, 33),
                                  (24, 17, 36), (12, 30, 64)])
def test_legacy_lu_columns(dims, wrap):
    from pot3d_amd import _lib
    L = _lib.load()
    ia, ja, av, nb, v, dg = _matrix(dims, wrap, 7)
    n = len(ia) - 1
    x = np.random.default_rng(8).standard_normal(n)
    ref = _ilu_solve(dims, nb, v, dg, x)
    L.load_external_lu_solver(av.ctypes.data, ia.ctypes.data, ja.ctypes.data, n, len(av))
    first = None
    for _ in range(3):
        y = x.copy()
        L.external_lu_solver(y.ctypes.data)
        assert np.max(np.abs(y - ref)) <= 1e-5 * np.max(np.abs(ref)), (dims, wrap)
        first = y if first is None else first
        assert np.array_equal(y, first)
    L.unload_external_lu_solver()
