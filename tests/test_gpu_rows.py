"""Power step of levels without long rows (csrc/mi_rows.hip: 64 rows per
slice, 4 entries per group, sorted windows of 2048 rows) at the sizes where
it can go wrong: the edges of a slice and of a window, rows of no entries, of
whole and ragged groups, of 128 entries (the longest taken) and 129 (which the
streaming step takes), unit weights, weights at the edge of 16 bits and past
it, and a loop that ends after its first iteration.  With normLap the same
levels take the streaming step.

Reference: numpy FP64 of the same formulas (eigensolve_kokkos.h:102-206).  A
product with a row of k entries differs by at most (k + 3) eps times the sum
of the absolute terms; for the loop's vectors see test_gpu_small.py (1e-11).  With
normLap the runs' vectors differ by e = |u - u_host|, the constant's part too,
and two dot products of unit vectors by at most 2 e on either side (the step's
norm is at least 1/2): 8 e are allowed on their change, which must stay far
below tol."""
import numpy as np
import pytest
import scipy.sparse as sp

from ipdps_2021_graph_coarsening_amd import graphs

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _ring(n, degrees, longest, wmax, rng):
    """Symmetric: vertex v joined to v +- 1 .. d(v) / 2 as far as both ends
    want it, d those of blocks of 50 vertices in turn; vertex n / 3 joined to
    more, so that its row has `longest` entries."""
    d = np.array(degrees)[(np.arange(n) // 50) % len(degrees)]
    us, vs = [], []
    for k in range(1, max(degrees) // 2 + 1):
        u = np.arange(n - k)
        keep = (d[u] >= 2 * k) & (d[u + k] >= 2 * k)
        us.append(u[keep])
        vs.append(u[keep] + k)
    h, reach = n // 3, max(degrees) // 2 + 1
    far = np.flatnonzero(np.abs(np.arange(n) - h) > reach)
    has = sum(int(((u == h) | (v == h)).sum()) for u, v in zip(us, vs))
    if longest:
        to = rng.choice(far, longest - has, replace=False)
        us.append(np.minimum(to, h))
        vs.append(np.maximum(to, h))
    u, v = np.concatenate(us), np.concatenate(vs)
    w = None if wmax is None else rng.integers(1, wmax + 1, len(u)).astype(np.uint32)
    if w is not None and len(w):
        w[len(w) // 2] = wmax
    rows, cols = np.concatenate([u, v]), np.concatenate([v, u])
    order = np.lexsort((cols, rows))
    rp = np.zeros(n + 1, np.uint32)
    np.cumsum(np.bincount(rows, minlength=n), out=rp[1:])
    assert not longest or np.diff(rp).max() == longest
    return rp, cols[order].astype(np.uint32), None if w is None else np.concatenate([w, w])[order]


def _matrix(rp, col, w):
    n = len(rp) - 1
    return sp.csr_matrix((np.ones(len(col)) if w is None else w.astype(np.float64), col, rp), shape=(n, n))


@pytest.mark.parametrize("wmax", [None, 1, 65535, 65536])
@pytest.mark.parametrize("n,degrees,longest", [
    (2, [2], 0), (63, [2, 6], 0), (64, [8], 31), (65, [8, 10], 0), (300, [4, 2], 128), (300, [4, 2], 129),
    (1000, [32], 0), (2047, [2, 0, 14], 127), (2048, [6], 128), (2049, [0, 4, 18], 128), (9000, [26, 30, 0], 129),
    (20001, [12, 8], 128)])
def test_product(ctx, n, degrees, longest, wmax):
    rng = np.random.default_rng(n)
    rp, col, w = _ring(n, degrees, longest, wmax, rng)
    x = rng.uniform(-1, 1, n)
    g = ctx.graph(rp, col, w)
    y = g.spmv_shift(x)
    assert np.array_equal(y, g.spmv_shift(x))
    g.close()
    A = _matrix(rp, col, w)
    deg = np.asarray(A.sum(axis=1)).ravel()
    gb = max(2 * deg.max(), 2)
    ref = (gb - deg) * x + A @ x
    bound = (np.diff(rp) + 3) * EPS * ((gb - deg) * np.abs(x) + A @ np.abs(x))
    assert np.all(np.abs(y - ref) <= bound)


@pytest.mark.parametrize("normLap", [0, 1])
@pytest.mark.parametrize("n,degrees,longest,wmax,tol", [
    (7169, [4, 10], 128, 9, 1e-7), (8192, [6], 0, None, 1e-7), (8193, [20, 12], 127, 70000, 1e-7),
    (20001, [26, 8], 129, 3, 1e-6), (40000, [4, 6], 0, None, 1e-6), (9000, [8], 0, 5, 2.0)])
def test_loop(ctx, n, degrees, longest, wmax, tol, normLap):
    rng = np.random.default_rng(n)
    rp, col, w = _ring(n, degrees, longest, wmax, rng)
    u0 = rng.uniform(-1, 1, n)
    g = ctx.graph(rp, col, w)
    if tol > 1 and not normLap:  # dot products below gb, the first of them compared with 0
        tol = 1e9
    u, it, most = g.power_iter(u0, normLap=normLap, tol=tol)
    u2, it2, _ = g.power_iter(u0, normLap=normLap, tol=tol)
    g.close()
    assert it2 == it and np.array_equal(u, u2) and not most
    if tol > 1:
        assert it == 1
    A = _matrix(rp, col, w)
    deg = np.asarray(A.sum(axis=1)).ravel()
    c = 1 / np.sqrt(n)
    v = u0 - (u0.sum() * c) * c if not normLap else u0 - (u0 * deg).sum() * c / (c * c * deg.sum()) * c
    v = v / np.linalg.norm(v)
    gb = max(2 * deg.max(), 2)
    dots = [1e300, 0.0]
    for _ in range(it):
        h = v
        v = 0.5 * h + 0.5 * (A @ h) / deg if normLap else (gb - deg) * h + A @ h
        if not normLap:
            v = v - (v.sum() * c) * c
        v = v / np.linalg.norm(v)
        dots.append(h @ v)
    d = u - h
    slack = 8 * np.linalg.norm(d) if normLap else 1e-6 * tol
    assert slack <= 0.1 * tol
    if normLap:  # (the constant vector: see test_gpu_small.py)
        span = np.stack([np.ones(n), h], axis=1)
        d = d - span @ np.linalg.lstsq(span, d, rcond=None)[0]
    assert np.linalg.norm(d) <= 1e-11
    assert abs(dots[-1] - dots[-2]) <= tol + slack
    assert abs(dots[-2] - dots[-3]) > tol - slack
