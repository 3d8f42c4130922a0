"""The maps of a hierarchy against the same levels coarsened one by one: a
hierarchy draws the random stream once and filters each level's permutation
out of the finer level's (csrc/mi_hec.hip, 2048 entries per workgroup), a
single level draws and sorts its own.  Integers, compared exactly; each
hierarchy's own levels against the oracle: test_gpu_parity.py."""
import itertools

import numpy as np
import pytest

import oracle
from ipdps_2021_graph_coarsening_amd import graphs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,variant", [
    *itertools.product([51, 255, 2047, 2048, 2049, 4097, 70001], [0, 1, 3, 4]),
    (2048 * 1024, 0), (2048 * 1024 + 1, 0)])  # 1024 workgroups, and one more (their counts are scanned)
def test_levels_one_by_one(ctx, n, variant):
    rng = np.random.default_rng(n)
    k = np.arange(n - 1)
    extra = n if n < 1 << 20 else n // 50
    u, v = np.concatenate([k, rng.integers(0, n, extra)]), np.concatenate([k + 1, rng.integers(0, n, extra)])
    rp, col, w = graphs.from_edges(n, u, v, rng.integers(1, 9, len(u)), lcc=False)
    ctx.set_coarsening(variant)
    try:
        g = ctx.graph(rp, col, w)
        H = g.hierarchy(5)
        assert H.nlevels > 1
        for l in range(H.nlevels - 1):
            a = H.level(l)
            one = ctx.graph(a["rowptr"], a["col"], a["w"])
            vcmap = one.hec_level(l + 1, 5)[0]
            one.close()
            assert np.array_equal(vcmap, a["vcmap"])
        H.close()
        g.close()
    finally:
        ctx.set_coarsening(0)


@pytest.mark.parametrize("n", [1, 2, 65, 1023, 1024, 1025, 4095, 4096, 4097])
def test_map_in_one_workgroup(ctx, n):
    """Maps of at most 4096 vertices are made in one workgroup's LDS: against
    the oracle, with isolated vertices too (prefilled maps: test_gpu_gosh2.py)."""
    rng = np.random.default_rng(n)
    k = np.arange(n - 1)
    for chain in (True, False):
        u, v = rng.integers(0, n, n), rng.integers(0, n, n)
        if chain:
            u, v = np.concatenate([k, u]), np.concatenate([k + 1, v])
        rp, col, w = graphs.from_edges(n, u, v, rng.integers(1, 4, len(u)), lcc=False)
        for level in (1, 2):
            g = ctx.graph(rp, col, w)
            vc, nc, vperm, hn = g.hec_level(level, 11)
            ovc, onc, ovperm, ohn = oracle.coarsen_hec(level, rp, col, w, 11)
            assert np.array_equal(vperm, ovperm) and np.array_equal(hn, ohn)
            assert nc == onc and np.array_equal(vc, ovc)
            g.close()
