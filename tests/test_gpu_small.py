"""Small graphs by one workgroup at their edges: the largest vertex count and
edge count that take it and the next, rows longer and shorter than a step's
edges, frontiers past the workgroup's size, isolated sources, directed and
unsorted rows.  Parents and depths equal the oracle's exactly, alone and among
several graphs, with host and device outputs."""
import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu


def random_graph(n, m, seed, directed=False):
    rng = np.random.default_rng(seed)
    return pb.from_edges(n, rng.integers(0, n, m), rng.integers(0, n, m),
                         symmetrise=not directed)


def exact(n, m):
    """n vertices, exactly m directed edges: consecutive neighbours, rows unsorted."""
    deg = np.full(n, m // n)
    deg[:m % n] += 1
    src = np.repeat(np.arange(n), deg)
    k = np.arange(m) - np.repeat(np.cumsum(deg) - deg, deg)
    return pb.HostGraph(np.r_[0, np.cumsum(deg)], ((src * 7 + k + 1) % n).astype(np.int32))


def star(n):
    return pb.from_edges(n, np.zeros(n - 1, np.int64), np.arange(1, n))


CASES = {
    "n1": lambda: pb.HostGraph(np.array([0, 0]), np.zeros(0, np.int32)),
    "isolated source": lambda: pb.from_edges(9, [1, 2], [2, 3]),
    "one edge": lambda: pb.from_edges(2, [0], [1]),
    "path": lambda: pb.from_edges(3000, np.arange(2999), np.arange(1, 3000)),
    "star": lambda: star(16384),
    "star past it": lambda: star(16385),
    "frontier of a chunk": lambda: star(1025),
    "frontier past a chunk": lambda: star(1026),
    "a step's edges": lambda: star(4097),
    "a step's edges and one": lambda: star(4098),
    "two hubs": lambda: pb.from_edges(
        16384, np.r_[np.zeros(9000, np.int64), np.full(9000, 16383)],
        np.r_[np.arange(1, 9001), np.arange(7000, 16000)]),
    "most edges": lambda: exact(5000, 80000),
    "past most edges": lambda: exact(5000, 80001),
    "directed": lambda: random_graph(16384, 60000, 1, directed=True),
    "sparse": lambda: random_graph(16384, 20000, 2),
    "torus": lambda: pb.grid3d(16),
}


@pytest.mark.parametrize("wide", [False, True])
def test_small_graphs(ctx, wide):
    jobs = []
    for name, make in CASES.items():
        g = make()
        dg = ctx.upload(g, wide_offsets=wide)
        for s in {0, g.n // 2, g.n - 1}:
            print("[case]", name, "source", s, flush=True)
            wp, wd = oracle.serial_bfs(g.offsets, g.adj, s)
            p, d, st = dg.bfs(s)
            assert np.array_equal(p, wp) and np.array_equal(d, wd), (name, s)
            assert st["reached"] == (wd < g.n).sum() and st["levels"] == wd[wd < g.n].max() + 1
            assert st["edges_reached"] == g.degrees()[wd < g.n].sum()
            st = dg.bfs_device(s)
            assert st["reached"] == (wd < g.n).sum()
            if dg.info["symmetric"]:   # the checker's rules read rows as in-neighbours
                r = dg.check_device(s, *ctx.outputs())
                assert r["valid"] == 1 and r["max_rule_bad"] == 0 and r["depth_bad"] == 0, (name, r)
            if s == g.n - 1:
                jobs.append((name, dg, s, wp, wd))
    # several graphs: with the two past the limits, and without
    for some in (jobs, [j for j in jobs if j[0] not in ("star past it", "past most edges")]):
        res = ctx.bfs_multi([j[1] for j in some], [j[2] for j in some])
        for (name, _, s, wp, wd), (p, d, st) in zip(some, res):
            assert np.array_equal(p, wp) and np.array_equal(d, wd), (name, s)
            assert st["reached"] == (wd < len(wd)).sum()
