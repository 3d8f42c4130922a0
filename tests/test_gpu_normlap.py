"""Bisections under the normalised Laplacian against recorded ones.

The power iteration of that path takes the constant vector out once, before
the first iteration (eigensolve_kokkos.h:118-150); what rounding leaves of it
grows against the rest, so the iteration at which a level stops, and with it
the partition, depends on the order of every sum.  That order is therefore
part of the results: the same levels, iteration counts, partitions and cuts
as tests/golden/normlap_bisections.json, whatever form a level runs in."""
import hashlib
import json
import os

import numpy as np
import pytest

import ipdps_2021_graph_coarsening_amd as mi
from ipdps_2021_graph_coarsening_amd import graphs

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "normlap_bisections.json")

# name: (graph, mixed precision from this many entries on, hec_seed)
CASES = {
    "grid2d-45": (lambda: graphs.grid2d(45), None, 3),
    "grid2d-64": (lambda: graphs.grid2d(64), None, 1),
    "grid2d-100": (lambda: graphs.grid2d(100), None, 2),  # 10,000 vertices: vectors not all in LDS
    "grid2d-231w": (lambda: graphs.grid2d(231, "uniform16", 5), None, 3),
    "grid3d-13": (lambda: graphs.grid3d(13, None), None, 4),
    "grid3d-26w": (lambda: graphs.grid3d(26), None, 5),
    "grid3d-35w-mixed": (lambda: graphs.grid3d(35), 1 << 14, 6),
    "rgg-7428": (lambda: graphs.rgg(7428, seed=2), None, 7),
    "rgg-34337-mixed": (lambda: graphs.rgg(34337, seed=2), 1 << 14, 8),
    "rmat-12": (lambda: graphs.rmat(12, 16, seed=1), None, 9),
    "rmat-14-mixed": (lambda: graphs.rmat(14, 8, seed=1), 1 << 14, 10),
    "rmat-16": (lambda: graphs.rmat(16, 12, seed=1), None, 11),
}


def _digest(part):
    return hashlib.sha256(np.ascontiguousarray(part, dtype=np.int32).tobytes()).hexdigest()


def _outcome(r):
    return dict(levels=[int(x) for x in r.stats["level_n"]], iters=[int(x) for x in r.stats["level_iters"]],
                cut=int(r.edge_cut), part=_digest(r.part))


def bisect(ctx, name, batch=False):
    make, mixed, seed = CASES[name]
    g = ctx.graph(*make())
    cfg = mi.Config(4, 1, 0, 1, 1e-10, 2)
    try:
        ctx.set_precision(mixed is not None, mixed or 0)
        if batch:
            res, _ = mi.bisect_batch(ctx, [g, g], cfg, hec_seeds=[seed, seed], pcg_states=[seed, seed])
            assert _outcome(res[0]) == _outcome(res[1])
            return _outcome(res[0])
        return _outcome(mi.partition_graph(ctx, g, cfg, hec_seed=seed, pcg_state=seed))
    finally:
        ctx.set_precision(False)
        g.close()


def fourway(ctx):
    g = ctx.graph(*graphs.grid3d(20))
    r = mi.partition_4way(ctx, g, mi.Config(4, 1, 0, 1, 1e-10, 4), hec_seed=12, pcg_state=12)
    g.close()
    return dict(cuts=[int(x) for x in r.extra["cuts"]], part=_digest(r.part))


def recorded(ctx):
    """What the file holds (written once, by the streaming step and the
    one-workgroup loops that add in its order)."""
    out = {name: bisect(ctx, name) for name in CASES}
    for limit in (0, 1 << 20):  # one workgroup for no level, and for larger ones
        ctx.set_small_levels(limit)
        out["rmat-14 small levels %d" % limit] = bisect(ctx, "rmat-14-mixed")
        out["grid2d-100 small levels %d" % limit] = bisect(ctx, "grid2d-100")
    ctx.set_small_levels()
    out["4way"] = fourway(ctx)
    return out


@pytest.fixture(scope="module")
def golden():
    with open(GOLDEN) as f:
        return json.load(f)


@pytest.mark.parametrize("name", list(CASES))
def test_bisection(ctx, golden, name):
    assert bisect(ctx, name) == golden[name]


@pytest.mark.parametrize("name", ["grid2d-45", "grid2d-231w", "rmat-12", "rgg-34337-mixed"])
def test_batch(ctx, golden, name):
    assert bisect(ctx, name, batch=True) == golden[name]


@pytest.mark.parametrize("chunk", [1, 7])
def test_resumed_launches(ctx, golden, chunk):
    try:
        ctx.set_small_levels(1 << 17, chunk)
        for name in ("grid2d-45", "grid2d-100", "rmat-12"):
            assert bisect(ctx, name) == golden[name]
    finally:
        ctx.set_small_levels()


@pytest.mark.parametrize("limit", [0, 1 << 20])
def test_small_level_limit(ctx, golden, limit):
    try:
        ctx.set_small_levels(limit)
        assert bisect(ctx, "rmat-14-mixed") == golden["rmat-14 small levels %d" % limit]
        assert bisect(ctx, "grid2d-100") == golden["grid2d-100 small levels %d" % limit]
    finally:
        ctx.set_small_levels()


def test_fourway(ctx, golden):
    assert fourway(ctx) == golden["4way"]
