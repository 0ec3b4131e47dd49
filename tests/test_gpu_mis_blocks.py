"""The independent set's blocks at their edges: one workgroup's limit, block
and 64-vertex boundaries, rows of every length around a look's 2 or 4 entries,
rows ending at the adjacency's last entry, directed and unsorted rows, long
chains across blocks.  Flags equal the oracle's exactly."""
import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu


def random_graph(n, degree, seed, directed=False):
    rng = np.random.default_rng(seed)
    m = int(n * degree)
    return pb.from_edges(n, rng.integers(0, n, m), rng.integers(0, n, m),
                         symmetrise=not directed)


def unsorted(g, seed):
    src = np.repeat(np.arange(g.n), g.degrees())
    return pb.HostGraph(g.offsets, g.adj[np.lexsort((np.random.default_rng(seed).random(g.m), src))])


def stepped(n):
    """Vertex v joined to v - 1 .. v - (v % 11): rows of 0 to 20 entries."""
    v = np.repeat(np.arange(n), np.arange(n) % 11)
    k = np.concatenate([np.arange(1, d + 1) for d in np.arange(n) % 11]) if n > 1 else v
    keep = v - k >= 0
    return pb.from_edges(n, v[keep], (v - k)[keep])


CASES = {
    "n1": lambda: pb.HostGraph(np.array([0, 0]), np.zeros(0, np.int32)),
    "one edge": lambda: pb.from_edges(2, [0], [1]),
    "block less one": lambda: random_graph(1023, 3, 1),
    "block and one": lambda: random_graph(1025, 12, 2),
    "one workgroup": lambda: random_graph(16384, 6, 3),
    "past one workgroup": lambda: random_graph(16385, 6, 4),
    "wide rows past it": lambda: random_graph(16449, 30, 5),
    "blocks of 512": lambda: random_graph(4 * 8192 - 1, 9, 6),
    "many blocks": lambda: random_graph(3_000_001, 2, 7),
    "many blocks, wide rows": lambda: random_graph(700_003, 20, 8),
    "stepped": lambda: stepped(20_000),
    "stepped small": lambda: stepped(777),
    "directed": lambda: random_graph(40_000, 8, 9, directed=True),
    "directed small": lambda: random_graph(5_000, 8, 10, directed=True),
    "unsorted": lambda: unsorted(random_graph(40_000, 12, 11), 1),
    "unsorted small": lambda: unsorted(random_graph(9_000, 12, 12), 2),
    "clique, then its tail": lambda: pb.from_edges(
        20_000, *np.r_[np.stack(np.triu_indices(300, 1), 1),
                       np.stack([np.arange(299, 19_999), np.arange(300, 20_000)], 1)].T),
}


@pytest.mark.parametrize("name", CASES)
def test_mis_blocks(ctx, name):
    g = CASES[name]()
    want = oracle.mis(g.offsets, g.adj)
    for wide in (False, True):
        print("[case] mis blocks", name, g.n, g.m, wide, flush=True)
        dg = ctx.upload(g, wide_offsets=wide)
        f, st = dg.mis()
        assert np.array_equal(f, want)
        assert st["members"] == (want == 1).sum()
        dg.free()
