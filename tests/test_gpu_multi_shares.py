"""Several graphs of short rows in one call: outputs equal the oracle's, with shares
of the workgroups set by vertices, by edges and by the device, and the call takes
no longer than the searches one after another."""
import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu


def directed(n, per, seed):
    r = np.random.default_rng(seed)
    return pb.from_edges(n, r.integers(0, n, n * per), r.integers(0, n, n * per), symmetrise=False)


LISTS = {
    "tori": lambda: [pb.grid3d(k) for k in (13, 24, 32, 40)],
    "directed": lambda: [directed(30_000, 5, 1), directed(60_000, 5, 2), directed(100_000, 10, 3)],
    "sparse and skewed": lambda: [pb.from_edges(300_000, np.arange(60), np.arange(1, 61)),
                                  pb.rmat(15, 16 << 15, 0.57, 0.19, 0.19, seed=3)],
    "whole device": lambda: [directed(600_000, 2, s) for s in range(8)],
}


@pytest.mark.parametrize("name", LISTS)
def test_outputs(ctx, name):
    graphs = LISTS[name]()
    dgs = [ctx.upload(g) for g in graphs]
    src = [7 + 5 * i for i in range(len(graphs))]
    print("[case]", name, [(g.n, g.m) for g in graphs], flush=True)
    for g, s, (p, d, st) in zip(graphs, src, ctx.bfs_multi(dgs, src)):
        wp, wd = oracle.serial_bfs(g.offsets, g.adj, s)
        assert np.array_equal(p, wp) and np.array_equal(d, wd)
        assert st["reached"] == (wd < g.n).sum()
    for dg in dgs:
        dg.free()


def test_no_slower_than_one_by_one(ctx):
    dgs = [ctx.upload(g) for g in LISTS["directed"]()]
    t = ctx.tuning
    shared = min(ctx.bfs_multi(dgs, [1] * 3)[0][2]["device_ms"] for _ in range(30))
    try:
        ctx.set_tuning(persist=0)
        alone = sum(min(dg.bfs_device(1)["device_ms"] for _ in range(30)) for dg in dgs)
    finally:
        ctx.set_tuning(persist=t.persist)
    print("[case] shared", shared, "alone", alone, flush=True)
    assert shared < 1.1 * alone
    for dg in dgs:
        dg.free()
