"""Which levels stream the adjacency: of a small frontier, those whose edges are
between m / (2 td_to_bu_div) and m / 10 (there a bottom-up level below m /
td_to_bu_div edges is a streamed one), not those with more, where the general
bottom-up level ends sooner, and none from the fourth level on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SMALL = 8192


@pytest.fixture(scope="module")
def graph(ctx):
    dg = ctx.gen_rmat(21, 2 ** 26, 0.57, 0.19, 0.19, seed=3)
    assert dg.m >= 2 ** 26
    yield dg
    dg.free()


def levels(ctx, dg, s, div):
    usual = ctx.tuning.td_to_bu_div
    ctx.set_tuning(td_to_bu_div=div)
    try:
        return dg.profile(s)[1]
    finally:
        ctx.set_tuning(td_to_bu_div=usual)


def small_frontiers(ctx, dg):
    """{source: (level, its edges)} where a small frontier first has many edges."""
    deg = np.diff(dg.download().offsets)
    found = {}
    for s in np.random.default_rng(7).choice(np.flatnonzero((deg > 0) & (deg < 30)), 60, False):
        for l in levels(ctx, dg, int(s), 20):
            if l["frontier"] > SMALL:
                break
            if l["frontier_edges"] * 35 > dg.m:
                found[int(s)] = (l["level"], l["frontier_edges"])
                break
    return found


def test_range(ctx, graph):
    found = small_frontiers(ctx, graph)
    streamed = general = 0
    for s, (k, e) in found.items():
        div = (graph.m - SMALL * 20) // e    # |F| + edges stay within m / div: not bottom-up by itself
        if div < 1 or 2 * div * e <= graph.m:
            continue
        print("[case] source", s, "level", k, "edges", e, "of", graph.m, "div", div, flush=True)
        mode = levels(ctx, graph, s, div)[k]["mode"]
        if e * 10 <= graph.m:
            assert mode == "BU"
            streamed += 1
        else:
            assert mode == "TD"
            general += 1
    assert streamed and general, found


@pytest.mark.parametrize("graphs", [0, 1])
@pytest.mark.parametrize("chunk", [1, 2, 3, 4, 5])
def test_chunks(ctx, graph, chunk, graphs):
    t = ctx.tuning
    usual = {k: getattr(t, k) for k in ("chunk_levels", "use_graphs")}
    dg = ctx.gen_rmat(21, 2 ** 26, 0.57, 0.19, 0.19, seed=3)   # no run yet: chunks from the first
    try:
        ctx.set_tuning(chunk_levels=chunk, use_graphs=graphs)
        for s in list(small_frontiers(ctx, graph))[:2] + [0]:
            print("[case] chunk", chunk, "graphs", graphs, "source", s, flush=True)
            for _ in range(2):
                st = dg.bfs_device(s)
                r = dg.check_device(s, *ctx.outputs())
                assert r["valid"] == 1 and r["max_rule_bad"] == 0 and r["depth_bad"] == 0, r
                assert r["reached"] == st["reached"] and r["max_level"] + 1 == st["levels"]
    finally:
        ctx.set_tuning(**usual)
        dg.free()
