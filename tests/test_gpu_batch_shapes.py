"""GPU parity of the graph batch against the oracle where its workgroup's steps can go wrong:
hub lists around the lane's own share and a wave, deep graphs (bottom-up never taken), one
vertex, words and waves partly filled, the largest size, host and device results."""
import ctypes as C

import numpy as np
import pytest
from conftest import progress
from test_gpu_result_ranges import DeviceBuffer

pytestmark = pytest.mark.gpu


def star(B, leaves, n=None):
    return B.CSC.from_edges(n or leaves + 1, np.zeros(leaves, dtype=np.int64), np.arange(1, leaves + 1))


def path(B, n):
    return B.CSC.from_edges(n, np.arange(n - 1), np.arange(1, n))


def double_star(B, leaves):
    """Two hubs joined through one leaf: the far hub is found from a full list of unreached leaves."""
    a = np.arange(2, 2 + leaves)
    return B.CSC.from_edges(2 + 2 * leaves, np.concatenate([np.zeros(leaves, dtype=np.int64), np.ones(leaves, dtype=np.int64), [1]]),
                            np.concatenate([a, a + leaves, [2]]))


def graphs(B):
    out = [path(B, 1 + k) for k in (0, 1, 63, 64, 300)]
    out += [star(B, k) for k in (7, 31, 32, 33, 95, 96, 97, 289, 5000)]
    out += [double_star(B, k) for k in (40, 3000)]
    out += [B.CSC.rmat(11, 16, seed=4), B.CSC.rmat(15, 8, seed=5), B.CSC.grid(90, 0.9, 0.0, 6),
            B.CSC.erdos_renyi(131072, 6.0, seed=7), B.CSC.erdos_renyi(131071, 1.5, seed=8),
            B.CSC.erdos_renyi(4097, 20.0, seed=9)]
    return out


def test_batch_shapes(blest, oracle):
    progress("case batch shapes")
    gs = graphs(blest)
    patterns = [g.arrays() for g in gs]
    batch = blest.GraphBatch(gs)
    total = sum(g.n for g in gs)
    buf = DeviceBuffer(4 * total)
    for pick in ("first", "last", "middle"):
        roots = np.array([{"first": 0, "last": g.n - 1, "middle": g.n // 2}[pick] for g in gs], dtype=np.uint32)
        want = [oracle.bfs(g.n, cp, rows, int(r)) for g, (cp, rows), r in zip(gs, patterns, roots)]
        got, _ = batch.bfs(roots)
        for i, (w, lv) in enumerate(zip(want, got)):
            np.testing.assert_array_equal(lv, w, err_msg=f"graph {i} root {pick}")
        blest.check(blest._lib.load().blest_graph_batch_bfs(batch._h, roots.ctypes.data_as(blest._lib.U32P),
                                                            buf.i32(), None))
        np.testing.assert_array_equal(buf.numpy(np.int32, total), np.concatenate(want))
