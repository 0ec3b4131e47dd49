"""Searches that meet at the barrier of a few workgroups, at the rule's edges:
the most vertices and the next, the fewest above the one-workgroup graphs, wide,
directed and unsorted forms, isolated sources, and two contexts at once (one
holds the device's persistent launch, the other runs its levels).  Parents and
depths equal the oracle's; any-parent outputs equal those of a launch a level."""
import threading

import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu


def random_graph(n, m, seed, directed=False):
    rng = np.random.default_rng(seed)
    return pb.from_edges(n, rng.integers(0, n, m), rng.integers(0, n, m) ** 2 // n,
                         symmetrise=not directed)


def reversed_rows(g):
    at = np.arange(g.m) - np.repeat(g.offsets[:-1], g.degrees())
    return pb.HostGraph(g.offsets, g.adj[np.repeat(g.offsets[1:] - 1, g.degrees()) - at])


CASES = {
    "fewest": lambda: random_graph(16385, 9_000, 1),
    "one workgroup's edges and more": lambda: random_graph(3_000, 90_000, 2),
    "half of the most vertices": lambda: random_graph(1 << 17, 700_000, 3),
    "past half of the most vertices": lambda: random_graph((1 << 17) + 1, 700_000, 4),
    "most vertices": lambda: random_graph(1 << 18, 600_000, 9),
    "past most vertices": lambda: random_graph((1 << 18) + 1, 600_000, 10),
    "dense": lambda: random_graph(20_000, 2_000_000, 5),
    "directed": lambda: random_graph(60_001, 400_000, 6, directed=True),
    "reversed rows": lambda: reversed_rows(random_graph(60_001, 400_000, 7)),
    "rmat": lambda: pb.rmat(16, 16 << 16, 0.57, 0.19, 0.19, seed=8),
    "path": lambda: pb.from_edges(20_000, np.arange(19_999), np.arange(1, 20_000)),
}


@pytest.mark.parametrize("name", CASES)
def test_few_groups(ctx, name):
    g = CASES[name]()
    t = ctx.tuning
    for wide in (False, True):
        dg = ctx.upload(g, wide_offsets=wide)
        for s in (0, g.n // 2, g.n - 1):
            print("[case]", name, "wide" if wide else "", "source", s, flush=True)
            wp, wd = oracle.serial_bfs(g.offsets, g.adj, s)
            p, d, st = dg.bfs(s)
            assert np.array_equal(p, wp) and np.array_equal(d, wd)
            assert st["reached"] == (wd < g.n).sum()
            ap, ad, _ = dg.bfs(s, any_parent=True)
            ctx.set_tuning(persist=0)
            lp, ld, _ = dg.bfs(s, any_parent=True)
            ctx.set_tuning(persist=t.persist)
            assert np.array_equal(ad, wd) and np.array_equal(ap, lp) and np.array_equal(ad, ld)
        dg.free()


def test_two_contexts_at_once():
    g = CASES["rmat"]()
    sources = [int(s) for s in np.flatnonzero(g.degrees() > 0)[::4000][:8]]
    want = [oracle.serial_bfs(g.offsets, g.adj, s) for s in sources]
    bad = []

    def run():
        c = pb.Context(0)
        dg = c.upload(g)
        for _ in range(10):
            for s, (wp, wd) in zip(sources, want):
                p, d, _ = dg.bfs(s)
                if not (np.array_equal(p, wp) and np.array_equal(d, wd)):
                    bad.append(s)
        dg.free()
        c.close()

    threads = [threading.Thread(target=run) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
