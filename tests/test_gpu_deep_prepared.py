"""A prepared deep graph: after the first search no search allocates device memory,
the first on the deep path included."""
import ctypes

import numpy as np
import pytest

import oracle
import pbbsbench_amd as pb
from pbbsbench_amd.core import hip_runtime

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip_runtime().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("order", ["small first", "large first"])
def test_no_allocation_after_the_first_search(order):
    sides = (28, 40) if order == "small first" else (40, 28)
    with pb.Context(0) as c:
        for side in sides:
            g = pb.grid3d(side)
            dg = c.upload(g)
            dg.prepare(single=True, batch=False)
            want = oracle.serial_bfs(g.offsets, g.adj, 9)
            assert c.set_tuning(td_to_bu_div=40) is None
            print("[case] prepared torus", side, flush=True)
            st = dg.bfs_device(9)
            before = free_bytes()
            for _ in range(3):
                st = dg.bfs_device(9)
            assert free_bytes() >= before
            assert st["launches"] == 1 and st["bu_levels"] == 0   # the deep path
            p, d, _ = dg.bfs(9)
            assert np.array_equal(p, want[0]) and np.array_equal(d, want[1])
            dg.free()
