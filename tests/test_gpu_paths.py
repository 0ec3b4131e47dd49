"""Which path a search takes, as its stats show it.  A launch a level: several
launches.  One launch: a deep graph's and a small graph's search have no bottom-up
levels, whatever the switch to them; the persistent launch of level kernels has."""
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


def beads(length, fan):
    """Hubs in a line, each with `fan` leaves: hub rows of fan + 2 entries."""
    n = length * (fan + 1)
    hub = np.arange(length) * (fan + 1)
    leaf = np.setdiff1d(np.arange(n), hub)
    return pb.from_edges(n, np.r_[hub[:-1], np.repeat(hub, fan)], np.r_[hub[1:], leaf])


def path_of(st):
    if st["launches"] > 1:
        return "levels"
    return "persistent" if st["bu_levels"] else "deep or small"


# graph, td_to_bu_div under which level kernels go bottom-up, other tuning, paths of
# the first search and the later ones.  The graphs of the deep path are past the
# one-workgroup limits.
CASES = {
    "torus": (lambda: pb.grid3d(40), 40, {}, "persistent", "deep or small"),
    "torus, at once": (lambda: pb.grid3d(40), 40, {"persist": 1}, "deep or small", "deep or small"),
    "torus, unsorted": (lambda: reverse_rows(pb.grid3d(40)), 40, {"persist": 1}, "deep or small",
                        "deep or small"),
    "strip": (lambda: strip(20, 1000), 900, {}, "persistent", "deep or small"),
    "rows of 64": (lambda: beads(300, 62), 300, {}, "persistent", "deep or small"),
    "rows of 65": (lambda: beads(300, 63), 300, {}, "persistent", "persistent"),
    "a launch a level": (lambda: pb.grid3d(40), 40, {"persist": 0}, "levels", "levels"),
    "small": (lambda: pb.grid3d(16), 1000, {}, "deep or small", "deep or small"),
    "small, too many edges": (lambda: pb.rmat(13, 16 << 13, 0.57, 0.19, 0.19, seed=2), 20, {},
                              "persistent", "persistent"),
    "small, a set grid": (lambda: pb.grid3d(10), 1000, {"grid_blocks": 8}, "levels", "levels"),
    "few workgroups": (lambda: pb.rmat(16, 8 << 16, 0.57, 0.19, 0.19, seed=2), 20, {}, "persistent",
                       "persistent"),
    "past few workgroups": (lambda: pb.rmat(19, 4 << 19, 0.57, 0.19, 0.19, seed=2), 20, {}, "levels",
                            "levels"),
}


def reverse_rows(g):
    src = np.repeat(np.arange(g.n), g.degrees())
    return pb.HostGraph(g.offsets, g.adj[np.lexsort((-g.adj.astype(np.int64), src))])


def search(dg, g, s, want):
    p, d, st = dg.bfs(s)
    assert np.array_equal(p, want[0]) and np.array_equal(d, want[1])
    return path_of(st)


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("name", CASES)
def test_path(name, wide):
    make, div, tune, first, later = CASES[name]
    g = make()
    s = int(np.flatnonzero(g.degrees())[0])
    want = oracle.serial_bfs(g.offsets, g.adj, s)
    with pb.Context(0) as c:
        c.set_tuning(td_to_bu_div=div, **tune)
        dg = c.upload(g, wide_offsets=wide, assume_symmetric=True)
        for path in (first, later, later):
            print("[case]", name, g.n, g.m, flush=True)
            assert search(dg, g, s, want) == path
        dg.free()


def test_deep_launch_that_gives_up_runs_by_levels():
    g = pb.grid3d(40)
    want = oracle.serial_bfs(g.offsets, g.adj, 0)
    with pb.Context(0) as c:
        c.set_tuning(persist=1, persist_wait_us=0)
        dg = c.upload(g)
        print("[case] gives up", flush=True)
        for _ in range(2):
            assert search(dg, g, 0, want) == "levels"
        c.set_tuning(persist_wait_us=200_000, td_to_bu_div=40)
        assert search(dg, g, 0, want) == "deep or small"
        dg.free()


def test_refusal_belongs_to_its_tuning():
    """One workgroup's lists overflow on the torus.  The same graph is searched the
    deep way with the usual ones."""
    g = pb.grid3d(40)
    want = oracle.serial_bfs(g.offsets, g.adj, 0)
    with pb.Context(0) as c:
        c.set_tuning(persist=1, td_to_bu_div=40, grid_blocks=1)
        dg = c.upload(g)
        print("[case] refused", flush=True)
        assert search(dg, g, 0, want) == "levels"          # overflowed, ran again
        assert search(dg, g, 0, want) == "persistent"      # not tried again
        c.set_tuning(grid_blocks=0)
        assert search(dg, g, 0, want) == "deep or small"
        c.set_tuning(grid_blocks=1)
        assert search(dg, g, 0, want) == "persistent"      # still known
        dg.free()
