"""The workloads whose speed this framework is judged by.

Every case is one call (or one call per pass) of the package's public entry
points on data that is resident in HBM, as the drivers, the benchmark and the
tests make them: a breadth-first search, a batch of searches on one graph,
searches on several graphs at once, a maximal independent set, a spanning
forest.  Graph families and sizes are those of the benchmark configurations:
RMAT, the random-local graph and the 3D torus, from a few thousand vertices
(launch latency counts) to 2^24 (memory traffic counts), in uint32 and int64
offsets, with the deterministic and the any-parent rule.
"""
import math

import numpy as np
import torch

import pbbsbench_amd as pb

# RMAT quadrant probabilities (a, b, c): the Graph500 mix of the large search
# workloads, the rMatGraph mix of the set and forest inputs, and the flatter
# mix of the small search workload.
SKEW = {"g500": (0.57, 0.19, 0.19), "pbbs": (0.55, 0.125, 0.125), "flat": (0.5, 0.1, 0.1)}

_context = None


def context():
    """The process's one context on GPU 0, as a program that works on several
    graphs keeps it."""
    global _context
    if _context is None:
        _context = pb.Context(0)
    return _context


def listed():
    return [
        # BFS(start, G) as the drop-in user calls it, parents in host memory,
        # on the smallest graph in earnest use: latency only.
        dict(name="bfs_call_rmat12", kind="bfs", graph="rmat", scale=12, draws=8 << 12,
             skew="g500", wide=False, any_parent=False, host=True),
        # The small search workload: 2^16 vertices, outputs stay in HBM.
        dict(name="bfs_rmat16", kind="bfs", graph="rmat", scale=16, draws=1 << 19,
             skew="flat", wide=False, any_parent=False, host=False),
        # An ordinary skewed graph under the any-parent rule (backForwardBFS).
        dict(name="bfs_any_rmat22", kind="bfs", graph="rmat", scale=22, draws=1 << 26,
             skew="g500", wide=False, any_parent=True, host=False),
        # The headline search: 2^24 vertices, 2^28 draws, int64 offsets.
        dict(name="bfs_rmat24_i64", kind="bfs", graph="rmat", scale=24, draws=1 << 28,
             skew="g500", wide=True, any_parent=False, host=False),
        # Random-local graph, no hubs: 10M vertices, 10 draws each.
        dict(name="bfs_randlocal10m_i64", kind="bfs", graph="randlocal", n=10_000_000, k=10,
             wide=True, any_parent=False, host=False),
        # Deep graph: 216^3 torus, hundreds of levels of small frontiers.
        dict(name="bfs_torus216", kind="bfs", graph="torus", side=216,
             wide=False, any_parent=False, host=False),
        # A full batch of 64 sources in one traversal.
        dict(name="batch64_rmat22", kind="batch", graph="rmat", scale=22, draws=1 << 26,
             skew="g500", wide=False, sources=64),
        # A ragged batch on a smaller graph, as a serving loop merges them.
        dict(name="batch12_rmat18", kind="batch", graph="rmat", scale=18, draws=16 << 18,
             skew="g500", wide=False, sources=12),
        # One query on each of 16 small graphs of uneven size, one call.
        dict(name="multi16_rmat10_17", kind="multi", lo=10, hi=17, jobs=16),
        # rMatGraph_JR: the independent-set input, relabelled at random.
        dict(name="mis_rmat24_jr", kind="mis", graph="rmat", scale=24, draws=12 * 16_000_000,
             skew="pbbs", wide=False),
        # 3Dgrid_JR: the sparse independent-set input (degree 6), relabelled.
        dict(name="mis_torus256_jr", kind="mis", graph="torus", side=256, wide=False),
        # rMatGraph_E: the spanning-forest input, edges in random order.
        dict(name="st_rmat24_e", kind="st", scale=24, draws=12 * 16_000_000, skew="pbbs"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_rmat(rng, lo, hi, skew):
    scale = rng.randint(lo, hi)
    # average draws per vertex 4..16, odd totals among them
    return dict(graph="rmat", scale=scale, draws=int((1 << scale) * rng.uniform(4, 16)),
                skew=skew)


def draw(rng):
    kind = rng.choice(["bfs", "bfs", "bfs", "bfs", "batch", "batch", "multi", "mis", "mis", "st"])
    wide = rng.random() < 0.5
    if kind == "bfs":
        graph = rng.choice(["rmat", "rmat", "randlocal", "torus"])
        if graph == "rmat":
            c = _draw_rmat(rng, 10, 24, rng.choice(["g500", "flat"]))
            n = 1 << c["scale"]
        elif graph == "randlocal":
            n = _log_int(rng, 1_000, 10_000_000)
            c = dict(graph="randlocal", n=n, k=rng.randint(4, 10))
        else:
            side = _log_int(rng, 8, 216)
            n = side ** 3
            c = dict(graph="torus", side=side)
        return dict(kind="bfs", wide=wide, any_parent=rng.random() < 0.3,
                    host=n <= 1 << 20 and rng.random() < 0.5, **c)
    if kind == "batch":
        return dict(kind="batch", wide=wide, sources=rng.randint(2, 64),
                    **_draw_rmat(rng, 10, 22, "g500"))
    if kind == "multi":
        lo = rng.randint(8, 12)
        return dict(kind="multi", lo=lo, hi=rng.randint(lo, 17), jobs=rng.randint(2, 16))
    if kind == "mis":
        if rng.random() < 0.6:
            return dict(kind="mis", wide=wide, **_draw_rmat(rng, 10, 23, "pbbs"))
        return dict(kind="mis", wide=wide, graph="torus", side=_log_int(rng, 12, 256))
    c = _draw_rmat(rng, 12, 23, "pbbs")
    return dict(kind="st", scale=c["scale"], draws=c["draws"], skew="pbbs")


# ------------------------------------------------------------------- inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _upload(off, adj, wide):
    g = pb.HostGraph(off.cpu().numpy(), adj.cpu().numpy())
    return context().upload(g, wide_offsets=wide)


def _randlocal(n, k, seed, wide):
    """Vertex i draws k neighbours i +- floor(n^u) mod n; symmetrised, loops
    and duplicates dropped, rows ascending."""
    gen = _generator(seed)
    i = torch.arange(n, device="cuda").repeat_interleave(k)
    step = (float(n) ** torch.rand(n * k, device="cuda", dtype=torch.float64, generator=gen)).long()
    sign = torch.randint(0, 2, (n * k,), device="cuda", generator=gen) * 2 - 1
    j = (i + sign * step) % n
    keep = i != j
    i, j = i[keep], j[keep]
    keys = torch.unique(torch.cat([i * n + j, j * n + i]))
    rows = keys // n
    off = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    off[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    return _upload(off, (keys - rows * n).int(), wide)


def _torus_relabelled(side, seed, wide):
    """side^3 torus with its vertices relabelled by a random permutation, rows
    ascending."""
    n = side ** 3
    label = torch.randperm(n, device="cuda", generator=_generator(seed))
    grid = label.view(side, side, side)
    nbrs = [grid.roll(s, d).reshape(-1) for d in range(3) for s in (1, -1)]
    rows = torch.empty(n, 6, dtype=torch.int32, device="cuda")
    rows[label] = torch.stack(nbrs, 1).int().sort(1).values
    off = torch.arange(n + 1, device="cuda") * 6
    return _upload(off, rows.reshape(-1), wide)


def _rmat_edges(scale, draws, skew, seed):
    """Distinct undirected RMAT edges without loops, vertices relabelled at
    random and edges in random order (an unordered edge-array file's shape)."""
    gen = _generator(seed)
    a, b, c = SKEW[skew]
    u = torch.zeros(draws, dtype=torch.int64, device="cuda")
    v = torch.zeros_like(u)
    for _ in range(scale):
        r = torch.rand(draws, device="cuda", generator=gen)
        u.mul_(2).add_(r >= a + b)
        v.mul_(2).add_(((r >= a) & (r < a + b)) | (r >= a + b + c))
    label = torch.randperm(1 << scale, device="cuda", generator=gen)
    u, v = label[u], label[v]
    keys = torch.unique((torch.minimum(u, v) << scale) + torch.maximum(u, v))
    keys = keys[torch.randperm(keys.numel(), device="cuda", generator=gen)]
    u, v = (keys >> scale).int(), (keys & ((1 << scale) - 1)).int()
    keep = u != v
    return u[keep], v[keep]


def _graph(case, seed, relabel=0):
    wide = case.get("wide", False)
    if case["graph"] == "rmat":
        a, b, c = SKEW[case["skew"]]
        return context().gen_rmat(case["scale"], case["draws"], a, b, c, seed=seed + 1,
                                  permute_seed=relabel, wide_offsets=wide)
    if case["graph"] == "randlocal":
        return _randlocal(case["n"], case["k"], seed, wide)
    if relabel:
        return _torus_relabelled(case["side"], seed, wide)
    return context().gen_grid3d(case["side"], wide_offsets=wide)


def _sources(dg, count, seed):
    """Random vertices of vertex 0's component (an RMAT graph's largest)."""
    parent = torch.empty(dg.n, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    dg.bfs_device(0, parent_ptr=parent.data_ptr())
    reached = torch.nonzero(parent >= 0).view(-1).cpu().numpy()
    return np.random.default_rng(seed).choice(reached, count, replace=len(reached) < count)


def prepare(case, seed):
    kind = case["kind"]
    s = dict(kind=kind)
    if kind == "st":
        u, v = _rmat_edges(case["scale"], case["draws"], case["skew"], seed)
        s.update(n=1 << case["scale"], u=u, v=v)
        s["forest"] = torch.full((s["n"] - 1,), -1, dtype=torch.int32, device="cuda")
    elif kind == "multi":
        rng = np.random.default_rng(seed)
        a, b, c = SKEW["g500"]
        span = case["hi"] - case["lo"] + 1
        graphs = []
        for j in range(case["jobs"]):
            scale = case["lo"] + j * span // case["jobs"]
            graphs.append(context().gen_rmat(scale, 16 << scale, a, b, c,
                                             seed=int(rng.integers(1, 1 << 30))))
        for dg in graphs:
            dg.prepare(single=True, batch=False)
        s.update(graphs=graphs, sources=[int(_sources(dg, 1, seed)[0]) for dg in graphs])
    else:
        dg = _graph(case, seed, relabel=seed + 2 if kind == "mis" else 0)
        s["graph"] = dg
        if kind == "mis":
            s["flags"] = torch.empty(dg.n, dtype=torch.int32, device="cuda")
        elif kind == "batch":
            dg.prepare(single=False, batch=True)
            s["sources"] = _sources(dg, case["sources"], seed)
            s["parent"] = torch.empty(case["sources"], dg.n, dtype=torch.int32, device="cuda")
            s["depth"] = torch.empty_like(s["parent"])
        else:
            dg.prepare(single=True, batch=False)
            s.update(any_parent=case["any_parent"], host=case["host"],
                     source=int(_sources(dg, 1, seed)[0]))
            if not case["host"]:
                s["parent"] = torch.empty(dg.n, dtype=torch.int32, device="cuda")
                s["depth"] = torch.empty_like(s["parent"])
    # the outputs are written on the context's own stream
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- a pass
def run(s):
    kind = s["kind"]
    if kind == "bfs":
        if s["host"]:
            if s["any_parent"]:
                parent, depth, _ = s["graph"].bfs(s["source"], any_parent=True)
                return parent, depth
            return pb.BFS(s["source"], s["graph"])
        s["graph"].bfs_device(s["source"], s["parent"].data_ptr(), s["depth"].data_ptr(),
                              any_parent=s["any_parent"])
        return s["parent"], s["depth"]
    if kind == "batch":
        s["graph"].bfs_batch_device(s["sources"], s["parent"].data_ptr(), s["depth"].data_ptr())
        return s["parent"], s["depth"]
    if kind == "multi":
        return [(p, d) for p, d, _ in context().bfs_multi(s["graphs"], s["sources"])]
    if kind == "mis":
        s["graph"].mis_device(s["flags"].data_ptr())
        return s["flags"]
    count, _ = context().spanning_forest_device(s["n"], s["u"].numel(), s["u"].data_ptr(),
                                                s["v"].data_ptr(), s["forest"].data_ptr())
    return s["forest"], count


# ------------------------------------------------------- what a pass must move
def _size(case):
    """(vertices, directed CSR entries).  An RMAT draw leaves about 1.9 entries
    once loops and duplicates are gone, a random-local one about 1.9."""
    if case.get("graph") == "torus":
        return case["side"] ** 3, 6 * case["side"] ** 3
    if case.get("graph") == "randlocal":
        return case["n"], int(1.9 * case["n"] * case["k"])
    return 1 << case["scale"], int(1.9 * case["draws"])


def work(case):
    """Each offset and adjacency entry read once, each output written once;
    integer work, so no floating-point operations."""
    kind = case["kind"]
    if kind == "multi":
        span = case["hi"] - case["lo"] + 1
        sizes = [1 << (case["lo"] + j * span // case["jobs"]) for j in range(case["jobs"])]
        return dict(bytes=sum(4 * n + 4 * 2 * 16 * 0.8 * n + 8 * n for n in sizes), flops=0)
    n, m = _size(case)
    if kind == "st":   # every edge's two ends, the forest's ids
        return dict(bytes=4 * m + 4 * n, flops=0)
    graph = (8 if case["wide"] else 4) * (n + 1) + 4 * m
    out = {"bfs": 8 * n, "mis": 4 * n, "batch": 8 * n * case.get("sources", 0)}[kind]
    if kind == "bfs" and case["host"] and not case["any_parent"]:
        out = 4 * n
    return dict(bytes=graph + out, flops=0)


def exact(case, seed):
    """Every output is a whole number (vertex and edge ids, depths, flags)."""
    return None
