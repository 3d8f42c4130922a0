"""The calls that the speed of this framework is measured on.

A case is one call (or the two calls that belong together) of a program that
partitions graphs: the graph's edges are in hand, drawn on the GPU from the
seed and brought to the host as a file reader would leave them; the context
is kept from call to call; partitions come back as host arrays.

Keys of a case:
- ``call``: "bisect" (partition_graph of a resident graph), "batch"
  (bisect_batch of resident graphs), "fourway" (partition_4way of a resident
  graph), "convert" (graph_from_edges of a host edge list, then
  partition_graph), "power" (power_iter: one level's power iteration);
- ``graph`` and ``size``: "grid2d" size x size, "grid3d" size^3, "rmat"
  2^size vertices with ``edge_factor`` edges each, "rgg" random geometric
  graph of size vertices with mean degree 10 ("batch": ``count`` graphs,
  their sizes spread over [1000, size] evenly in the logarithm);
- ``weights``: edge weights uniform in 1..16 on meshes, summed duplicates on
  R-MAT; without it every edge weighs 1;
- ``mode``: "fp64" (plain), "mixed" (FP32 vectors above the finest level),
  "fm" (FM refinement instead of the eigensolve);
- ``norm_lap``: 1 for the normalised Laplacian (the config's refine_alg);
- ``variant``: the coarsening map (0 HEC, 1 matching, 2 mt-metis, 3 HEC v3,
  5 MIS-2, 6 GOSH).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import ipdps_2021_graph_coarsening_amd as mi

_contexts: dict = {}


def _case(call, graph, size, mode="fp64", weights=False, edge_factor=16, norm_lap=0, variant=0, count=1):
    return dict(call=call, graph=graph, size=size, mode=mode, weights=weights, edge_factor=edge_factor,
                norm_lap=norm_lap, variant=variant, count=count)


def listed():
    return [
        # a small mesh, the size of a block in a larger ordering or of a test: latency only
        dict(name="grid2d64-bisect", **_case("bisect", "grid2d", 64)),
        # the plain bisection of a 256 x 256 five-point grid, a usual first example
        dict(name="grid2d256-bisect", **_case("bisect", "grid2d", 256)),
        # an unstructured mesh of an odd size under the normalised Laplacian
        dict(name="rgg100003-normlap", **_case("bisect", "rgg", 100003, norm_lap=1)),
        # the same kind of graph through another coarsening, as in comparisons of coarsenings
        dict(name="rgg150001-match", **_case("bisect", "rgg", 150001, weights=True, variant=1)),
        # a power-law graph that fits the caches, plain double precision
        dict(name="rmat20-bisect", **_case("bisect", "rmat", 20, weights=True)),
        # a weighted three-dimensional mesh in mixed precision
        dict(name="grid3d128-mixed", **_case("bisect", "grid3d", 128, mode="mixed", weights=True)),
        # many small unequal graphs at once (subdomains, collections of meshes)
        dict(name="rgg-batch192", **_case("batch", "rgg", 200000, mode="mixed", count=192)),
        # four parts by recursive bisection of a large power-law graph
        dict(name="rmat21-4way-mixed", **_case("fourway", "rmat", 21, mode="mixed", weights=True)),
        # the largest: a power-law graph of half a billion stored entries
        dict(name="rmat24-bisect", **_case("bisect", "rmat", 24, weights=True)),
        # the FM flow on a mesh, the other refinement a user picks
        dict(name="grid2d400-fm", **_case("bisect", "grid2d", 400, mode="fm")),
        # from an edge list on the host to a partition on the host
        dict(name="rmat18-convert", **_case("convert", "rmat", 18)),
        # one level's power iteration with the vector in hand
        dict(name="rmat17-power", **_case("power", "rmat", 17, weights=True)),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _mesh(rng, lo, hi):
    """A mesh of about lo to hi vertices: (graph, size)."""
    n = _log(rng, lo, hi)
    graph = rng.choice(("grid2d", "grid3d", "rgg"))
    return graph, max(4, {"grid2d": round(n ** 0.5), "grid3d": round(n ** (1 / 3)), "rgg": n}[graph])


def draw(rng):
    call = rng.choice(("mesh", "mesh", "rmat", "rmat", "variant", "batch", "fourway", "fm", "convert", "power"))
    if call == "mesh":
        graph, size = _mesh(rng, 2000, 2_000_000)
        return _case("bisect", graph, size, mode=rng.choice(("fp64", "mixed")), weights=rng.random() < 0.5,
                     norm_lap=int(rng.random() < 0.25))
    if call == "rmat":
        return _case("bisect", "rmat", rng.randint(12, 23), mode=rng.choice(("fp64", "mixed")),
                     weights=rng.random() < 0.7, edge_factor=rng.randint(6, 24))
    if call == "variant":
        graph, size = _mesh(rng, 5000, 300_000)
        return _case("bisect", graph, size, weights=rng.random() < 0.5, variant=rng.choice((1, 2, 3, 5, 6)))
    if call == "batch":
        return _case("batch", "rgg", _log(rng, 5000, 150_000), mode=rng.choice(("fp64", "mixed")),
                     count=_log(rng, 8, 160))
    if call == "fourway":
        if rng.random() < 0.5:
            return _case("fourway", "rmat", rng.randint(14, 21), mode="fp64", weights=True,
                         edge_factor=rng.randint(6, 24))
        graph, size = _mesh(rng, 5000, 1_000_000)
        return _case("fourway", graph, size, mode="fp64", weights=rng.random() < 0.5)
    if call == "fm":
        graph, size = _mesh(rng, 3000, 200_000)
        return _case("bisect", graph, size, mode="fm", weights=rng.random() < 0.3)
    if call == "convert":
        if rng.random() < 0.5:
            return _case("convert", "rmat", rng.randint(12, 20), edge_factor=rng.randint(6, 24))
        graph, size = _mesh(rng, 2000, 500_000)
        return _case("convert", graph, size)
    if rng.random() < 0.5:
        return _case("power", "rmat", rng.randint(11, 18), weights=True, edge_factor=rng.randint(6, 24))
    graph, size = _mesh(rng, 2000, 200_000)
    return _case("power", graph, size, weights=True)


# ---------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _vertices(case):
    size = case["size"]
    return {"rmat": 1 << size, "rgg": size, "grid2d": size ** 2, "grid3d": size ** 3}[case["graph"]]


def _grid_edges(shape):
    idx = torch.arange(math.prod(shape), dtype=torch.int32, device="cuda").reshape(shape)
    us, vs = [], []
    for d in range(len(shape)):
        us.append(idx.narrow(d, 0, shape[d] - 1).reshape(-1))
        vs.append(idx.narrow(d, 1, shape[d] - 1).reshape(-1))
    return torch.cat(us), torch.cat(vs)


def _rmat_edges(scale, edge_factor, gen):
    """Chakrabarti et al. with (a, b, c, d) = (0.57, 0.19, 0.19, 0.05)."""
    m = edge_factor << scale
    u = torch.zeros(m, dtype=torch.int32, device="cuda")
    v = torch.zeros(m, dtype=torch.int32, device="cuda")
    for bit in range(scale):
        r = torch.rand(m, generator=gen, device="cuda")
        u |= (r >= 0.76).int() << bit
        v |= (((r >= 0.57) & (r < 0.76)) | (r >= 0.95)).int() << bit
    return u, v


def _rgg_edges(n, gen):
    """Points in the unit square, joined below the distance that gives a mean
    degree of 10: neighbours are sought in the 3 x 3 cells around a point."""
    r = math.sqrt(10.0 / (math.pi * n))
    k = max(1, int(1.0 / r))
    p = torch.rand(n, 2, generator=gen, device="cuda", dtype=torch.float64)
    cell = (p * k).long().clamp_(max=k - 1)
    order = torch.argsort(cell[:, 0] * k + cell[:, 1], stable=True)
    p, cell = p[order], cell[order]
    count = torch.bincount(cell[:, 0] * k + cell[:, 1], minlength=k * k)
    start = torch.cumsum(count, 0) - count
    us, vs = [], []
    for dx, dy in ((0, 0), (0, 1), (1, -1), (1, 0), (1, 1)):
        x, y = cell[:, 0] + dx, cell[:, 1] + dy
        inside = (x < k) & (y >= 0) & (y < k)
        c = torch.where(inside, x * k + y, 0)
        cnt = torch.where(inside, count[c], 0)
        i = torch.repeat_interleave(torch.arange(n, device="cuda"), cnt)
        j = start[c][i] + torch.arange(len(i), device="cuda") - (torch.cumsum(cnt, 0) - cnt)[i]
        keep = ((p[i] - p[j]) ** 2).sum(1) < r * r
        if dx == 0 and dy == 0:
            keep &= i < j
        us.append(order[i[keep]])
        vs.append(order[j[keep]])
    return torch.cat(us).int(), torch.cat(vs).int()


def _edges(case, seed):
    """(n, u, v, w or None) on the GPU."""
    gen = _generator(seed)
    graph, size, n = case["graph"], case["size"], _vertices(case)
    if graph == "rmat":
        u, v = _rmat_edges(size, case["edge_factor"], gen)
        return n, u, v, torch.ones_like(u) if case["weights"] else None
    if graph == "rgg":
        u, v = _rgg_edges(n, gen)
    else:
        shape = (size,) * (2 if graph == "grid2d" else 3)
        u, v = _grid_edges(shape)
    w = torch.randint(1, 17, u.shape, generator=gen, device="cuda", dtype=torch.int32) if case["weights"] else None
    return n, u, v, w


def _host(t):
    return None if t is None else t.cpu().numpy().view(np.uint32)


def _context(case):
    """The context that a program with these settings keeps."""
    key = (case["mode"], case["variant"])
    if key not in _contexts:
        c = mi.Context(0)
        c.set_precision(case["mode"] == "mixed")
        c.set_refinement(case["mode"] == "fm")
        c.set_coarsening(case["variant"])
        _contexts[key] = c
    return _contexts[key]


def _batch_sizes(case):
    k = case["count"]
    return [int(round(1000 * (case["size"] / 1000) ** ((i + 0.5) / k))) for i in range(k)]


def _resident(ctx, case, seed):
    """A resident graph: duplicates merged, largest connected component.  An
    R-MAT graph with summed weights, a mesh as it is."""
    n, u, v, w = _edges(case, seed)
    u, v, w = _host(u), _host(v), _host(w)
    torch.cuda.empty_cache()
    return ctx.graph_from_edges(n, u, v, w, lcc=True)


def prepare(case, seed):
    ctx = _context(case)
    parts = 4 if case["call"] == "fourway" else 2
    s = dict(case=case, ctx=ctx, seed=seed % (1 << 31) + 1, config=mi.Config(4, case["norm_lap"], 0, 1, 1e-10, parts))
    sizes = _batch_sizes(case) if case["call"] == "batch" else [_vertices(case)]
    s["part"] = np.full(sum(sizes), -1, dtype=np.int32)
    s["level_n"] = np.zeros((len(sizes), mi.MAX_LEVELS), dtype=np.int64)
    if case["call"] == "batch":
        s["graphs"] = [_resident(ctx, dict(case, size=n), seed * 1009 + i) for i, n in enumerate(sizes)]
        s["seeds"] = [s["seed"] + i for i in range(case["count"])]
        s["at"] = np.concatenate([[0], np.cumsum(sizes)[:-1]])
    elif case["call"] == "convert":
        n, u, v, w = _edges(case, seed)
        s.update(n=n, u=_host(u), v=_host(v), w=_host(w))
    else:
        s["graph"] = _resident(ctx, case, seed)
        if case["call"] == "power":
            s["u"] = _start_vector(s["graph"].n, seed)
            s["vector"] = np.zeros(sizes[0])
    torch.cuda.empty_cache()
    return s


def _start_vector(n, seed):
    return np.random.default_rng(seed).uniform(-1.0, 1.0, n)


# ---------------------------------------------------------------- the calls
# The largest component's size depends on the seed: results go to the front
# of the program's own arrays, which hold the graph before that reduction.
def _answer(s, results, at=(0,)):
    """Partitions, cuts (figures of merit of the partitions) and level sizes."""
    for r, a, levels in zip(results, at, s["level_n"]):
        s["part"][a:a + len(r.part)] = r.part
        levels[:] = 0
        levels[:len(r.stats["level_n"])] = r.stats["level_n"]
    return dict(part=s["part"], cut=np.array([r.edge_cut for r in results], dtype=np.float64), level_n=s["level_n"])


def run(s):
    ctx, cfg, seed, call = s["ctx"], s["config"], s["seed"], s["case"]["call"]
    if call == "bisect":
        return _answer(s, [mi.partition_graph(ctx, s["graph"], cfg, hec_seed=seed, pcg_state=seed)])
    if call == "batch":
        res, _ = mi.bisect_batch(ctx, s["graphs"], cfg, hec_seeds=s["seeds"], pcg_states=s["seeds"])
        return _answer(s, res, s["at"])
    if call == "fourway":
        r = mi.partition_4way(ctx, s["graph"], cfg, hec_seed=seed, pcg_state=seed)
        s["part"][:len(r.part)] = r.part
        return dict(part=s["part"], cuts=np.array(r.extra["cuts"], dtype=np.float64))
    if call == "convert":
        g = ctx.graph_from_edges(s["n"], s["u"], s["v"], s["w"], lcc=True)
        r = _answer(s, [mi.partition_graph(ctx, g, cfg, hec_seed=seed, pcg_state=seed)])
        g.close()
        return r
    u, iters, _ = s["graph"].power_iter(s["u"], 0, 1e-10)
    s["vector"][:len(u)] = u
    return dict(u=s["vector"], iters=iters)


# ---------------------------------------------------------------- what they cost and give
def _sizes(case):
    """About (vertices, stored entries) of a case's graph."""
    if case["graph"] == "rmat":
        return 0.6 * 2 ** case["size"], 0.93 * 2 * case["edge_factor"] * 2 ** case["size"]
    if case["graph"] == "rgg":
        return case["size"], 10.0 * case["size"]
    d = 2 if case["graph"] == "grid2d" else 3
    return case["size"] ** d, 2 * d * (case["size"] - 1) * case["size"] ** (d - 1)


def work(case):
    """The CSR graph (or edge list) read once and the result written once; one
    product of its matrix with a vector."""
    if case["call"] == "batch":
        each = [work(dict(case, call="bisect", size=n)) for n in _batch_sizes(case)]
        return {k: sum(w[k] for w in each) for k in ("bytes", "flops")}
    n, m = _sizes(case)
    per_entry = 8 if case["weights"] else 4
    if case["call"] == "convert":
        return {"bytes": per_entry * m + 4 * n, "flops": 2 * m}
    return {"bytes": 4 * (n + 1) + per_entry * m + (16 if case["call"] == "power" else 4) * n, "flops": 2 * m}


def tolerance(case):
    """Measured with the sums in other orders (other loop and vertex orders of
    the levels): vectors of one power iteration agreed to 2e-15; of 50
    partitions one changed, by two vertices that tie, which is 1e-3 of the
    smallest graphs.  Mixed precision was 2e-4 of the vertices from double
    precision at most."""
    if case["mode"] == "fm":
        return "exact"  # integers throughout
    if case["call"] == "power":
        return {"rel": 1e-12}
    return {"rel": 1e-3, "differ": 1e-3}


def _largest_component(n, u, v):
    """Which vertices belong to the largest component (of equals, the one
    with the smallest vertex)."""
    lab = torch.arange(n, device="cuda")
    while True:
        new = lab.scatter_reduce(0, u, lab[v], reduce="amin").scatter_reduce(0, v, lab[u], reduce="amin")
        new = new[new]
        if torch.equal(new, lab):
            break
        lab = new
    size = torch.bincount(lab, minlength=n)
    return lab == int(torch.nonzero(size == size.max())[0])


def exact(case, seed):
    """A partition has no 64-bit value of its own; one power iteration has:
    u <- (gb - D + A) u with gb = max(2 max(D), 2), the constant vector taken
    out and the norm put to 1, until the dot product of the vectors before and
    after a step changes by at most 1e-10."""
    if case["call"] != "power":
        return None
    n, a, b, w = _edges(case, seed)
    a, b = a.long(), b.long()
    w = torch.ones_like(a) if w is None else w.long()
    keep = a != b
    a, b, w = a[keep], b[keep], w[keep]
    inside = _largest_component(n, a, b)
    new = torch.cumsum(inside.long(), 0) - 1
    e = inside[a]
    a, b, w, n = new[a[e]], new[b[e]], w[e], int(inside.sum())
    key, at = torch.unique(torch.cat([a * n + b, b * n + a]), return_inverse=True)
    w = torch.zeros(len(key), dtype=torch.float64, device="cuda").index_add_(0, at, torch.cat([w, w]).double())
    row, col = key // n, key % n
    ptr = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    ptr[1:] = torch.cumsum(torch.bincount(row, minlength=n), 0)
    A = torch.sparse_csr_tensor(ptr, col, w, size=(n, n))
    deg = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, row, w)
    shift = torch.clamp(2 * deg.max(), min=2.0) - deg
    v = torch.from_numpy(_start_vector(n, seed)).cuda()
    v = v - v.sum() / n
    v = v / v.norm()
    before, dot = 1.0, 0.0
    while abs(dot - before) > 1e-10:
        u, before = v, dot
        v = A @ u + shift * u
        v = v - v.sum() / n
        v = v / v.norm()
        dot = float(u @ v)
    full = np.zeros(_vertices(case))
    full[:n] = u.cpu().numpy()
    return dict(u=full, iters=None)  # the vector that entered the last product
