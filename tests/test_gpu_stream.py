"""Levels that stream the adjacency (small frontiers of hubs on graphs of 2^26
entries or more): whole and cut groups of rows, a last word and group that are
not full, few and many workgroups, frontiers from one vertex up.
The GPU checker's BFS, max-parent and depth rules hold at every vertex."""
import numpy as np
import pytest

import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu

M = 2 ** 26


def ragged(g, rows):
    """g without its last vertices: n is no multiple of 64."""
    n = g.n - rows
    src = np.repeat(np.arange(g.n, dtype=np.int32), g.degrees())
    keep = (src < n) & (g.adj < n)
    off = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(src[keep], minlength=n), out=off[1:])
    return pb.HostGraph(off, g.adj[keep])


@pytest.fixture(scope="module")
def host(ctx):
    dg = ctx.gen_rmat(21, 2 ** 26, 0.57, 0.19, 0.19, seed=3)
    g = dg.download()
    dg.free()
    assert g.m >= M
    return g


@pytest.mark.parametrize("form", ["as generated", "ragged", "wide"])
def test_stream_levels(ctx, host, form):
    g = ragged(host, 37) if form == "ragged" else host
    assert g.m >= M
    dg = ctx.upload(g, wide_offsets=form == "wide")
    deg = g.degrees()
    rng = np.random.default_rng(5)
    low = np.flatnonzero((deg > 0) & (deg < 4))
    sources = [int(np.argmax(deg)), *(int(s) for s in rng.choice(low, 3, replace=False))]
    t = ctx.tuning
    usual = {"td_to_bu_div": t.td_to_bu_div, "grid_blocks": t.grid_blocks}
    try:
        # the second switches at a 200th of the usual degree sums
        for tune in ({}, {"td_to_bu_div": 4000}, {"td_to_bu_div": 4000, "grid_blocks": 3}):
            ctx.set_tuning(**tune)
            for s in sources:
                print("[case]", form, tune, "source", s, "degree", deg[s], flush=True)
                st = dg.bfs_device(s)
                r = dg.check_device(s, *ctx.outputs())
                assert r["valid"] == 1 and r["cycle"] == 0, r
                assert r["max_rule_bad"] == 0 and r["depth_bad"] == 0, r
                assert r["reached"] == st["reached"] and r["max_level"] + 1 == st["levels"]
            ctx.set_tuning(**usual)
    finally:
        ctx.set_tuning(**usual)
        dg.free()
