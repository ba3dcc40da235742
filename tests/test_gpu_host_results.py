"""Single-source results for host memory at the edge of the size that goes through the
query's pinned memory (1 MB), natural and permuted, against the oracle; an unaligned
destination, and a word after it that must stay."""
import ctypes as C

import numpy as np
import pytest
from conftest import progress

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 262143, 262144, 262145])
@pytest.mark.parametrize("permuted", [False, True])
def test_host_result_sizes(blest, oracle, n, permuted):
    progress(f"case host result {n} permuted={permuted}")
    lib = blest._lib.load()
    v = np.arange(1, n)
    g = blest.CSC.from_edges(n, (v - 1) // 3, v)
    cp, rows = g.arrays()
    inv = None
    if permuted:
        inv = np.random.default_rng(2).permutation(n).astype(np.uint32)
        g.apply_permutation(inv)
    k = blest.BVSSBFSKernel(blest.DeviceGraph(blest.BVSS().construct_from_csc(g), g, inv))
    out = np.empty(n + 2, np.int32)
    for r in (0, n - 1):
        out[:] = -7
        blest.check(lib.blest_bfs(k.q._h, r, out[1:].ctypes.data_as(blest._lib.I32P),
                                  C.byref(blest._lib.BfsStats())))
        np.testing.assert_array_equal(out[1 : n + 1], oracle.bfs(n, cp, rows, r))
        assert out[0] == out[n + 1] == -7
