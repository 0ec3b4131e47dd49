"""Which independent sets run in one workgroup: sets equal the oracle's on graphs
at and past every line of the rule (vertices, entries with the vertices, entries
of graphs with short rows, the longest of those rows), and a dense graph takes no
longer for being small enough by its vertices alone."""
import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu


def exact(n, m):
    """n vertices, m directed entries in rows of equal length (to one).  Not
    symmetric, rows unsorted: the rule reads rows."""
    deg = np.full(n, m // n, np.int64)
    deg[n - m % n:] += 1
    src = np.repeat(np.arange(n), deg)
    k = np.arange(m) - np.repeat(np.cumsum(deg) - deg, deg)
    return pb.HostGraph(np.r_[0, np.cumsum(deg)], ((src * 7 + k * 5 + 3) % n).astype(np.int32))


def rows_of(longest, n=9000, m=599_000):
    """Short rows but one, of `longest` entries."""
    deg = np.full(n, (m - longest) // (n - 1), np.int64)
    deg[:m - longest - deg[0] * (n - 1)] += 1
    deg[-1] = longest
    src = np.repeat(np.arange(n), deg)
    k = np.arange(m) - np.repeat(np.cumsum(deg) - deg, deg)
    return pb.HostGraph(np.r_[0, np.cumsum(deg)], ((src * 3 + k + 1) % n).astype(np.int32))


CASES = {
    "cost at the line": lambda: exact(1000, 770_000 - 30 * 1000),
    "cost past it": lambda: exact(1000, 770_001 - 30 * 1000),
    "short rows, most entries": lambda: exact(16384, 600_000),
    "short rows, one entry more": lambda: exact(16384, 600_001),
    "most vertices and one": lambda: exact(16385, 100_000),
    "longest short row": lambda: rows_of(128),
    "a longer row": lambda: rows_of(129),
    "few vertices, dense": lambda: exact(520, 900_000 // 520 * 520),
}


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("name", CASES)
def test_lines(ctx, name, wide):
    g = CASES[name]()
    dg = ctx.upload(g, wide_offsets=wide)
    print("[case]", name, g.n, g.m, dg.info["max_degree"], flush=True)
    flags, st = dg.mis()
    want = oracle.mis(g.offsets, g.adj)
    assert np.array_equal(flags, want) and st["members"] == (want == 1).sum()
    dg.free()


def test_dense_graph_is_not_kept_to_one_workgroup(ctx):
    """2^14 vertices and 1.08M entries, and the same with an isolated vertex more."""
    dg = ctx.gen_rmat(14, 40 << 14, 0.55, 0.125, 0.125, seed=5, permute_seed=7)
    g = dg.download()
    more = ctx.upload(pb.HostGraph(np.r_[g.offsets, g.offsets[-1]], g.adj))
    print("[case] dense", g.n, g.m, flush=True)
    best = [min(d.mis_device()["device_ms"] for _ in range(30)) for d in (dg, more)]
    assert best[0] < 1.3 * best[1], best
    dg.free()
    more.free()
