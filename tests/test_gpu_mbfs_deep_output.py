"""Multi-source levels past the kept history (16), merged with the kept ones by the closing kernel
512 vertices and four at a time: vertex counts around its tiles, root counts around its words,
vertices that no root reaches, results in device and host memory."""
import ctypes as C

import numpy as np
import pytest
from conftest import progress
from test_gpu_result_ranges import DeviceBuffer

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [511, 512, 513, 514, 1024, 1539])
@pytest.mark.parametrize("permuted", [False, True])
def test_deep_rows(blest, oracle, n, permuted):
    progress(f"case multi-source deep rows n={n} permuted={permuted}")
    # a path through the even vertices, a star among the odd ones from 101 on, the odd ones before alone
    even, odd = np.arange(0, n, 2), np.arange(101, n, 2)
    g = blest.CSC.from_edges(n, np.concatenate([even[:-1], np.full(len(odd) - 1, 101)]),
                             np.concatenate([even[1:], odd[1:]]))
    cp, rows = g.arrays()
    inv = None
    if permuted:
        inv = np.random.default_rng(4).permutation(n).astype(np.uint32)
        g.apply_permutation(inv)
    dg = blest.DeviceGraph(blest.BVSS().construct_from_csc(g), g, inv)
    q = blest._Query(dg, 128)
    lib, st = blest._lib.load(), blest._lib.BfsStats()
    for k in (1, 31, 33, 64, 65, 128):
        srcs = (np.arange(k) * 7 % n).astype(np.uint32)
        want = np.stack([oracle.bfs(n, cp, rows, int(r)) for r in srcs])
        o = blest._lib.MbfsOpts(0, 128 if k > 64 else 64)
        buf, host = DeviceBuffer(4 * n * k), np.empty((k, n), dtype=np.int32)
        for out in (buf.i32(), host.ctypes.data_as(blest._lib.I32P)):
            blest.check(lib.blest_mbfs(q._h, srcs.ctypes.data_as(blest._lib.U32P), k, out, C.byref(o), C.byref(st)))
        np.testing.assert_array_equal(buf.numpy(np.int32, n * k).reshape(k, n), want, err_msg=f"device k={k}")
        np.testing.assert_array_equal(host, want, err_msg=f"host k={k}")
