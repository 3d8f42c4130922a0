"""Small levels' power iteration (one workgroup: csrc/mi_small.hip, under the
normalised Laplacian k_power_small_lds in csrc/mi_eigen.hip) at the
sizes where the former's layout changes: one wavefront (<= 64 rows), 4 / 8 / 16
wavefronts, the largest level and the one after it, rows of very different
lengths (a hub makes a wavefront's stream too long for registers, then for
LDS), rows without entries, and weights past the packed entry's 19 bits.

Reference: numpy FP64, the reference's formulas (eigensolve_kokkos.h:102-206)
run for the number of iterations the device reports.  Both start from the
same vector and each step is a contraction up to rounding, so the vectors
differ by at most a few eps per iteration: 300 iterations of 1e-15 stay below
1e-12; 1e-11 is allowed.  With normLap the loop takes the constant vector out
only once, before the first iteration, and its component, of rounding size in
both runs, then grows towards the others (its eigenvalue is the largest) and
rescales the normalised vector: the constant and the vector itself are
projected out of the difference there.  The iteration count itself is checked by
the change of u . v at the device's last and last but one iteration against
tol.  With normLap the device's constant component is read off its vector and
followed back (an iteration divides it by the norm before normalising), and
the dot products are those of the host's vectors with it.  What is left of the
difference, at most 1e-11, moves a dot product of unit vectors by at most
twice that on either side (the step's norm is at least 1/2): 1e-10 is allowed
on the change of two, a thousandth of tol."""
import numpy as np
import pytest
import scipy.sparse as sp

import ipdps_2021_graph_coarsening_amd as mi
from ipdps_2021_graph_coarsening_amd import graphs

pytestmark = pytest.mark.gpu

TOL = 1e-7


def _host(rp, col, w, u, normLap, iters, device=None):
    n = len(rp) - 1
    A = sp.csr_matrix((np.ones(len(col)) if w is None else w.astype(np.float64), col, rp), shape=(n, n))
    deg = np.asarray(A.sum(axis=1)).ravel()
    c = 1 / np.sqrt(n)
    u = u - (u @ np.full(n, c)) * c if not normLap else u - (u * deg).sum() * c / (c * c * deg.sum()) * c
    v = u / np.linalg.norm(u)
    gb = max(2 * deg.max(), 2)
    dots, inputs, norms = [1.0, 0.0], [], []
    step = lambda u: 0.5 * u + 0.5 * (A @ u) / deg if normLap else (gb - deg) * u + A @ u
    for _ in range(iters):
        u = v
        v = step(u)
        if not normLap:
            v = v - (v.sum() * c) * c
        inputs.append(u)
        norms.append(np.linalg.norm(v))
        v = v / norms[-1]
        dots.append(u @ v)
    if normLap and device is not None:
        # device = p u + q 1 + rest: the constant per unit of the host's vector
        p, q = np.linalg.lstsq(np.stack([u, np.ones(n)], axis=1), device, rcond=None)[0]
        const = q / p
        for k in range(iters - 1, max(iters - 4, -1), -1):
            x = inputs[k] + const
            x = x / np.linalg.norm(x)
            y = step(x)
            dots[k + 2] = x @ y / np.linalg.norm(y)
            const *= norms[k - 1]
    return u, dots


def _star(n, extra, rng):
    """A hub joined to every vertex, plus random edges."""
    i = np.arange(1, n)
    u = np.concatenate([np.zeros(n - 1, np.int64), rng.integers(0, n, extra)])
    v = np.concatenate([i, rng.integers(0, n, extra)])
    return graphs.from_edges(n, u, v, None, lcc=False)


def _sparse(n, m, rng, wmax):
    u, v = rng.integers(0, n, m), rng.integers(0, n, m)
    k = np.arange(n - 1)
    return graphs.from_edges(n, np.concatenate([u, k]), np.concatenate([v, k + 1]),
                             rng.integers(1, wmax + 1, m + n - 1), lcc=False)


def _case(name):
    rng = np.random.default_rng(7)
    kind, n = name.rsplit("-", 1)
    n = int(n)
    if kind == "path":
        return graphs.path(n)
    if kind == "star":
        return _star(n, 3 * n, rng)
    if kind == "dense":
        return _sparse(n, 20 * n, rng, 9)
    if kind == "wide":
        return _sparse(n, 3 * n, rng, 1 << 24)
    if kind == "w17":
        return _sparse(n, 3 * n, rng, 1 << 17)
    return _sparse(n, 2 * n, rng, 16)


@pytest.mark.parametrize("name", [
    "path-2", "path-3", "mesh-17", "star-40", "mesh-63", "mesh-64", "mesh-65", "star-64", "wide-50", "wide-300",
    "mesh-128", "mesh-129", "mesh-1023", "mesh-1024", "mesh-1025", "star-1000", "star-3000", "dense-900",
    "dense-2100", "w17-700", "w17-1500", "wide-1500", "wide-6000", "mesh-4096", "mesh-6500", "mesh-7168", "mesh-7169",
    "star-7168", "dense-4000"])
@pytest.mark.parametrize("normLap", [0, 1])
def test_small_level_against_numpy(ctx, name, normLap):
    rp, col, w = _case(name)
    n = len(rp) - 1
    u0 = np.random.default_rng(n).uniform(-1, 1, n)
    g = ctx.graph(rp, col, w)
    u, it, mr = g.power_iter(u0, normLap=normLap, tol=TOL)
    try:
        ctx.set_small_levels(1 << 17, 3)  # three iterations per launch
        u3, it3, _ = g.power_iter(u0, normLap=normLap, tol=TOL)
    finally:
        ctx.set_small_levels()
    g.close()
    assert it3 == it and np.array_equal(u3, u)
    assert not mr
    if n == 2:  # (the only vector besides the constant maps to 0)
        return
    hu, dots = _host(rp, col, w, u0, normLap, it, u)
    d = u - hu
    slack = 1e-10 if normLap else 1e-6 * TOL
    if normLap:
        span = np.stack([np.ones(n), hu], axis=1)
        d = d - span @ np.linalg.lstsq(span, d, rcond=None)[0]
    assert np.linalg.norm(d) <= 1e-11 * np.linalg.norm(hu)
    assert abs(dots[-1] - dots[-2]) <= TOL + slack
    assert it == 1 or abs(dots[-2] - dots[-3]) > TOL - slack


def _blocks(sizes, rng, wmax):
    """Complete graphs joined in a path by one edge each: dense, and slow to
    converge."""
    us, vs, at = [], [], 0
    for k in sizes:
        i, j = np.triu_indices(k, 1)
        us += [i + at, [at]]
        vs += [j + at, [at + k]]
        at += k
    u, v = np.concatenate(us[:-1]), np.concatenate(vs[:-1])
    w = rng.integers(1, 9, len(u))
    w[::97] = wmax
    return graphs.from_edges(at, u, v, w, lcc=False)


@pytest.mark.parametrize("sizes,wmax", [
    ([102] * 5, 9),           # 128 steps per wavefront: eight hold the level in registers
    ([104] * 5, 9),           # 144: sixteen
    ([90, 80, 70], 65535),    # the largest weight of the register form
    ([90, 80, 70], 65536)])   # ... past it
def test_level_passed_on_to_sixteen_wavefronts(ctx, sizes, wmax):
    """Levels whose rows or weights the registers of eight wavefronts do not
    hold go on in sixteen, alone and as the last of a chain: against numpy, and
    launches of one, three and 8192 iterations give the same bits."""
    rng = np.random.default_rng(11)
    rp, col, w = _blocks(sizes, rng, wmax)
    n = len(rp) - 1
    u0 = rng.uniform(-1, 1, n)
    g = ctx.graph(rp, col, w)
    runs, sols = [], []
    try:
        for chunk in (0, 3, 1):
            ctx.set_small_levels(1 << 17, chunk)
            u, it, most = g.power_iter(u0, tol=TOL)
            assert not most
            runs.append((u, it))
            H = g.hierarchy(5)
            ev, st, _ = H.fiedler(9, tol=TOL)
            sols.append((ev, st["level_iters"]))
            H.close()
    finally:
        ctx.set_small_levels()
        g.close()
    for u, it in runs[1:]:
        assert it == runs[0][1] and np.array_equal(u, runs[0][0])
    for ev, iters in sols[1:]:
        assert iters == sols[0][1] and np.array_equal(ev, sols[0][0])
    hu, dots = _host(rp, col, w, u0, 0, runs[0][1])
    assert np.linalg.norm(runs[0][0] - hu) <= 1e-11
    assert abs(dots[-1] - dots[-2]) <= TOL * (1 + 1e-6)


def test_level_passed_on_inside_a_chain(ctx):
    """A finest level whose weights fit 16 bits, coarser ones whose sums do not:
    eight wavefronts leave those to sixteen and take the finest again.  Whole
    chains in launches of 1, 50 and 8192 iterations, alone and in a batch with
    a chain that needs no sixteen, give the same bits; against the launches
    per iteration the vectors agree to 1e-6 (the same stop, other sums)."""
    rp, col, _ = graphs.grid2d(75)
    rng = np.random.default_rng(4)
    r = np.repeat(np.arange(len(rp) - 1), np.diff(rp))
    w = rng.integers(20000, 60001, len(col)).astype(np.uint32)
    key = np.minimum(r, col).astype(np.int64) * len(rp) + np.maximum(r, col)
    w = w[np.unique(key, return_index=True)[1]][np.searchsorted(np.unique(key), key)]  # symmetric
    g, plain = ctx.graph(rp, col, w), ctx.graph(*graphs.grid2d(60))
    H = g.hierarchy(5)
    a = [H.level(l) for l in range(H.nlevels)]
    eight = [l for l in range(H.nlevels)
             if (a[l]["rowptr"][-1] > 5120 or len(a[l]["rowptr"]) > 1025)]
    assert len(eight) >= 2 and a[0]["w"].max() <= 65535 and all(a[l]["w"].max() > 65535 for l in eight[1:])
    cfg = mi.Config(4, 0, 0, 1, 1e-10, 2)
    sols, parts = [], []
    try:
        for chunk in (0, 50, 1):
            ctx.set_small_levels(1 << 17, chunk)
            ev, st, _ = H.fiedler(9)
            sols.append((ev, st["level_iters"]))
            res, _ = mi.bisect_batch(ctx, [plain, g, plain], cfg, hec_seeds=[5] * 3, pcg_states=[9] * 3)
            parts.append([x.part for x in res])
        one = mi.partition_graph(ctx, g, cfg, hec_seed=5, pcg_state=9).part
        ctx.set_small_levels(0)
        ev, _, _ = H.fiedler(9)
    finally:
        ctx.set_small_levels()
        H.close()
        g.close()
        plain.close()
    for k in (1, 2):
        assert sols[k][1] == sols[0][1] and np.array_equal(sols[k][0], sols[0][0])
        assert all(np.array_equal(x, y) for x, y in zip(parts[k], parts[0]))
    assert np.array_equal(parts[0][1], one) and np.array_equal(parts[0][0], parts[0][2])
    assert abs(ev @ sols[0][0]) >= (1 - 1e-6) * np.linalg.norm(ev) * np.linalg.norm(sols[0][0])


def test_rows_without_entries(ctx):
    """Isolated vertices (their rows come last in the layout, in slices of no
    steps): y = (gb - 0) x there."""
    rng = np.random.default_rng(3)
    for n, k in ((60, 20), (700, 300), (5000, 4000)):
        rp, col, w = _sparse(k, 3 * k, rng, 5)
        rp = np.concatenate([rp, np.full(n - k, rp[-1], np.uint32)])
        u0 = rng.uniform(-1, 1, n)
        g = ctx.graph(rp, col, w)
        u, it, _ = g.power_iter(u0, tol=TOL)
        g.close()
        hu, dots = _host(rp, col, w, u0, 0, it)
        assert np.linalg.norm(u - hu) <= 1e-11 * np.linalg.norm(hu)
        assert abs(dots[-1] - dots[-2]) <= TOL * (1 + 1e-6)
