"""The forest's round tiles and the large tree's bitmap at their edges: tile
counts and iterates per thread at the sizes where they change, vertex counts
on either side of the bitmap's threshold and off a whole word, trees that
never grow large, and a bad edge met while the bitmap filters.  Ids and round
counts equal the oracle's exactly."""
import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb

pytestmark = pytest.mark.gpu

N = 2 ** 20   # the bitmap is kept above this many vertices


def edges(n, m, seed, span=None):
    """Random ends, with self-loops and repeats; span: ends at most this far apart."""
    rng = np.random.default_rng(seed)
    u = rng.integers(0, n, m).astype(np.int32)
    if span is None:
        return u, rng.integers(0, n, m).astype(np.int32)
    return u, ((u + rng.integers(0, span, m)) % n).astype(np.int32)


@pytest.mark.parametrize("n,m,span", [
    (N, 6 * N, None),             # no bitmap
    (N + 1, 6 * N, None),         # bitmap, one vertex in its last word
    (N + 65, 25500, None),        # one round is one tile less an edge: no large tree
    (N + 65, 25600, None),        # two tiles
    (3 * N + 7, 9 * N, 3),        # long thin components
    (2 * N, 1024 * 256 * 100 - 1, None),   # 1024 tiles of one iterate a thread
    (2 * N, 1024 * 256 * 100, None),       # four a thread
])
def test_st_tiles(ctx, n, m, span):
    print("[case] forest tiles", n, m, span, flush=True)
    u, v = edges(n, m, seed=n % 1000 + m % 1000, span=span)
    got, st = ctx.spanning_forest(n, u, v)
    want, rounds = oracle.st(n, u, v)
    assert np.array_equal(got, want) and st["rounds"] == rounds


def test_st_bad_edge_under_the_bitmap(ctx):
    n, m = N + 65, 8 * N
    u, v = edges(n, m, seed=3)
    v[m - 5] = n
    with pytest.raises(pb.PbbsError, match="outside"):
        ctx.spanning_forest(n, u, v)
    u, v = edges(n, m, seed=4)   # and the context still works
    got, _ = ctx.spanning_forest(n, u, v)
    assert np.array_equal(got, oracle.st(n, u, v)[0])
