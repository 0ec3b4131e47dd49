"""Which searches meet at the barrier of a few workgroups (one launch) and which
take a launch a level: by the entries a vertex has where every level is top-down,
and by the levels of the last search on the smallest graphs.  Outputs equal the
oracle's either way."""
import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu


def directed(n, m):
    """Exactly m entries, m / n a row."""
    deg = np.full(n, m // n)
    deg[:m % n] += 1
    src = np.repeat(np.arange(n), deg)
    k = np.arange(m) - np.repeat(np.cumsum(deg) - deg, deg)
    return pb.HostGraph(np.r_[0, np.cumsum(deg)], ((src * 31 + k * 977 + 1) % n).astype(np.int32))


def uniform(n, m):
    r = np.random.default_rng(3)
    return pb.from_edges(n, r.integers(0, n, m), r.integers(0, n, m))


def tail(fan, length=30):
    """A path of `length` vertices to one with a row of `fan` entries; 5 starts it."""
    ids = np.r_[5, np.arange(6, 6 + length - 1)]
    hub = ids[-1]
    leaves = hub + 1 + np.arange(fan - 1)
    return pb.from_edges(int(leaves[-1]) + 1, np.r_[ids[:-1], np.full(fan - 1, hub)],
                         np.r_[ids[1:], leaves])


# graph, any-parent, tuning, one launch on the first search and on the next
CASES = {
    "directed, 6 entries a row": (lambda: directed(60_000, 360_000), False, {}, 1, 1),
    "directed, one entry more": (lambda: directed(60_000, 360_001), False, {}, 0, 0),
    "directed, 20 entries a row": (lambda: directed(30_000, 600_000), True, {}, 0, 0),
    "directed, most vertices": (lambda: directed(1 << 17, 5 << 17), False, {}, 1, 1),
    "directed, one more": (lambda: directed((1 << 17) + 1, 5 << 17), False, {}, 0, 0),
    "no bottom-up levels": (lambda: uniform(30_000, 300_000), False, {"td_to_bu_div": 0}, 0, 0),
    "bottom-up levels": (lambda: uniform(30_000, 300_000), False, {}, 1, 1),
    "few levels": (lambda: uniform(12_000, 150_000), True, {}, 1, 1),
    "many levels, small": (lambda: pb.grid3d(24), True, {}, 0, 0),
    "13 levels, small": (lambda: pb.grid3d(8), True, {}, 0, 0),
    "many levels, a long row": (lambda: tail(16), True, {}, 0, 0),
    "many levels, a longer row": (lambda: tail(17), True, {}, 1, 0),
    "few levels, short rows": (lambda: tail(3, 4), True, {}, 0, 1),
    "many levels": (lambda: pb.grid3d(27), True, {}, 1, 1),
    "set grid": (lambda: uniform(30_000, 300_000), False, {"grid_blocks": 64}, 0, 0),
}


@pytest.mark.parametrize("name", CASES)
def test_rule(ctx, name):
    make, any_parent, tune, first, later = CASES[name]
    g = make()
    t = ctx.tuning
    usual = {k: getattr(t, k) for k in ("td_to_bu_div", "grid_blocks")}
    dg = ctx.upload(g)
    wp, wd = oracle.serial_bfs(g.offsets, g.adj, 5)
    try:
        ctx.set_tuning(**tune)
        for one in (first, later, later):
            print("[case]", name, g.n, g.m, flush=True)
            p, d, st = dg.bfs(5, any_parent=any_parent)
            assert np.array_equal(d, wd) and (any_parent or np.array_equal(p, wp))
            assert (st["launches"] == 1) == bool(one), st
    finally:
        ctx.set_tuning(**usual)
        dg.free()
