"""Deep graphs of short rows (persistent launches that meet every few levels):
parents and depths equal the oracle's exactly, on frontiers that stay with one
workgroup, spread over all of them, outgrow their lists (the run then takes
the other path, now and later), on rows at the longest length taken and one
past it, unsorted rows, and launches that give up waiting."""
import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu


def strip(w, l):
    i = np.arange(w * l)
    x, y = i % w, i // w
    return pb.from_edges(w * l, np.r_[i[x < w - 1], i[y < l - 1]],
                         np.r_[i[x < w - 1] + 1, i[y < l - 1] + w])


def tree(levels, fan=2):
    n = (fan ** levels - 1) // (fan - 1)
    v = np.arange(1, n)
    return pb.from_edges(n, (v - 1) // fan, v)


def beads(length, fan):
    """Hubs in a line, each with `fan` leaves: hub rows of fan + 2 entries."""
    n = length * (fan + 1)
    hub = np.arange(length) * (fan + 1)
    leaf = np.setdiff1d(np.arange(n), hub)
    return pb.from_edges(n, np.r_[hub[:-1], np.repeat(hub, fan)], np.r_[hub[1:], leaf])


def two_parts():
    g = strip(3, 200)
    u = np.repeat(np.arange(g.n), g.degrees())
    return pb.from_edges(2 * g.n + 5, np.r_[u, u + g.n + 5], np.r_[g.adj, g.adj + g.n + 5])


def reverse_rows(g):
    src = np.repeat(np.arange(g.n), g.degrees())
    return pb.HostGraph(g.offsets, g.adj[np.lexsort((-g.adj.astype(np.int64), src))])


GRAPHS = {
    "torus7": (lambda: pb.grid3d(7), [0, 171]),
    "torus40": (lambda: pb.grid3d(40), [0, 31999]),
    "torus40 relabelled": (lambda: pb.permute(pb.grid3d(40), 5), [3, 777]),
    "path": (lambda: strip(1, 3000), [0, 1500]),
    "strip": (lambda: strip(30, 500), [0, 7]),
    "square": (lambda: strip(300, 300), [0, 45150]),
    "tree": (lambda: tree(15), [0, 20000]),
    "rows of 64": (lambda: beads(100, 62), [0, 3150]),
    "rows of 65": (lambda: beads(100, 63), [0, 3150]),
    "two parts": (two_parts, [0, 602, 1204]),
}


@pytest.mark.parametrize("tune", [dict(persist=1), dict(persist=1, grid_blocks=3),
                                  dict(persist=1, td_to_bu_div=0), dict()])
@pytest.mark.parametrize("name", GRAPHS)
def test_deep_shapes(name, tune):
    build, sources = GRAPHS[name]
    g = build()
    with pb.Context(0) as c:
        c.set_tuning(**tune)
        for wide in (False, True):
            dg = c.upload(g, wide_offsets=wide)
            for s in sources:
                print("[case] deep", name, tune, wide, s, flush=True)
                want = oracle.serial_bfs(g.offsets, g.adj, s)
                for _ in range(2):   # by itself the second run on a graph is the deep one
                    p, d, st = dg.bfs(s)
                    assert np.array_equal(p, want[0]) and np.array_equal(d, want[1])
                    reached = want[0] >= 0
                    assert st["reached"] == reached.sum()
                    assert st["edges_reached"] == g.degrees()[reached].sum()
                    assert st["levels"] == want[1][reached].max() + 1
            dg.free()


@pytest.mark.parametrize("tune,graph", [
    (dict(persist=1, grid_blocks=1), "torus40"),                       # lists overflow
    (dict(persist=1, grid_blocks=1, td_to_bu_div=0), "tree"),          # claims overflow
    (dict(persist=1, persist_wait_us=0), "square"),                    # the first wait gives up
])
def test_deep_falls_back(tune, graph):
    build, sources = GRAPHS[graph]
    g = build()
    with pb.Context(0) as c:
        c.set_tuning(**tune)
        dg = c.upload(g)
        for s in sources + sources:
            print("[case] deep falls back", graph, tune, s, flush=True)
            want = oracle.serial_bfs(g.offsets, g.adj, s)
            p, d, _ = dg.bfs(s)
            assert np.array_equal(p, want[0]) and np.array_equal(d, want[1])
        dg.free()


def test_deep_unsorted_rows():
    g = reverse_rows(strip(20, 400))
    with pb.Context(0) as c:
        c.set_tuning(persist=1)
        dg = c.upload(g, assume_symmetric=True)
        assert not dg.info["sorted"]
        print("[case] deep, unsorted rows", flush=True)
        p, d, _ = dg.bfs(11)
        want = oracle.serial_bfs(g.offsets, g.adj, 11)
        assert np.array_equal(p, want[0]) and np.array_equal(d, want[1])
        dg.free()
