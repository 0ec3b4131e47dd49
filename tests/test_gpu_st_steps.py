"""Forests whose rounds are so large that a workgroup takes its tile in more than one
step: the edges where the second step begins, without and with the large tree's
bitmap.  Ids and round counts equal the oracle's exactly."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

ONE_STEP = 1024 * 8 * 256 * 100   # edges from which 1024 tiles of 2048 iterates do not hold a round


@pytest.mark.parametrize("n,m", [(1 << 16, ONE_STEP - 1), (1 << 16, ONE_STEP),
                                 ((1 << 21) + 1, ONE_STEP + 12345)])
def test_st_steps(ctx, n, m):
    print("[case] forest steps", n, m, flush=True)
    rng = np.random.default_rng(n + m)
    u = rng.integers(0, n, m, dtype=np.int32)
    v = rng.integers(0, n, m, dtype=np.int32)
    got, st = ctx.spanning_forest(n, u, v)
    want, rounds = oracle.st(n, u, v)
    assert np.array_equal(got, want) and st["rounds"] == rounds
