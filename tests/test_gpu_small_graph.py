"""The one-workgroup BFS of small graphs against the oracle and against the level kernels
(fuse_quads < 0) on the same graphs: sizes around words, the bounds of the path, hub lists,
deep graphs, permutations; results on the host, in a device array and in the query's own."""
import ctypes as C

import numpy as np
import pytest
from conftest import progress
from test_gpu_batch_shapes import double_star, path, star
from test_gpu_result_ranges import DeviceBuffer

pytestmark = pytest.mark.gpu

GRAPHS = {
    "one": lambda B: path(B, 1),
    "path65": lambda B: path(B, 65),
    "star33": lambda B: star(B, 33),
    "star5000": lambda B: star(B, 5000, n=5100),
    "double_star": lambda B: double_star(B, 3000),
    "rmat13": lambda B: B.CSC.rmat(13, 8, seed=3),
    "grid200": lambda B: B.CSC.grid(200, 0.9, 0.01, 5),
    "vertices_at_bound": lambda B: B.CSC.erdos_renyi(16384, 9.0, seed=4),
    "vertices_over": lambda B: B.CSC.erdos_renyi(16385, 9.0, seed=4),
    "edges_over": lambda B: B.CSC.erdos_renyi(20000, 14.0, seed=2),
}


@pytest.mark.parametrize("name", GRAPHS)
@pytest.mark.parametrize("permuted", [False, True])
def test_small_graph_parity(blest, oracle, name, permuted):
    progress(f"case small graph {name} permuted={permuted}")
    lib = blest._lib.load()
    g = GRAPHS[name](blest)
    cp, rows = g.arrays()
    n = g.n
    inv = None
    if permuted:
        inv = np.random.default_rng(1).permutation(n).astype(np.uint32)
        g.apply_permutation(inv)
    dg = blest.DeviceGraph(blest.BVSS().construct_from_csc(g), g, inv, use_graphs=2)
    k = blest.BVSSBFSKernel(dg)
    buf = DeviceBuffer(4 * n)
    st = blest._lib.BfsStats()
    roots = [0, n // 2, n - 1]
    for r in roots:
        want = oracle.bfs(n, cp, rows, r)
        for fuse in (0, -1):
            dg.set_fuse(fuse)
            res = k.run(r)
            np.testing.assert_array_equal(res.levels, want, err_msg=f"root {r} fuse {fuse}")
            assert res.total_levels == want.max() + 1 and res.no_visited == (want >= 0).sum()
            assert res.edges_in_component == np.diff(cp.astype(np.int64))[want >= 0].sum() // 2
            assert res.td_levels + res.bu_levels == res.total_levels
            blest.check(lib.blest_bfs(k.q._h, r, buf.i32(), C.byref(st)))
            np.testing.assert_array_equal(buf.numpy(np.int32, n), want)
            # into the query's own level array
            own = C.cast(C.c_void_p(lib.blest_query_levels_device(k.q._h)), blest._lib.I32P)
            blest.check(lib.blest_bfs(k.q._h, r, own, C.byref(st)))
            back = np.empty(n, dtype=np.int32)
            assert buf.hip.hipMemcpy(back.ctypes.data_as(C.c_void_p), C.cast(own, C.c_void_p), 4 * n, 2) == 0
            np.testing.assert_array_equal(back, want)


@pytest.mark.parametrize("permuted", [False, True])
def test_multi_source_into_device_rows(blest, oracle, permuted):
    """Rows written by the closing kernel, levels past the kept history among them."""
    progress(f"case multi-source device rows permuted={permuted}")
    g = path(blest, 500)
    cp, rows = g.arrays()
    inv = None
    if permuted:
        inv = np.random.default_rng(2).permutation(g.n).astype(np.uint32)
        g.apply_permutation(inv)
    dg = blest.DeviceGraph(blest.BVSS().construct_from_csc(g), g, inv)
    q = blest._Query(dg, 128)
    for k in (3, 70):
        srcs = np.arange(k, dtype=np.uint32) * 7
        buf = DeviceBuffer(4 * g.n * k)
        o, st = blest._lib.MbfsOpts(0, 128 if k > 64 else 64), blest._lib.BfsStats()
        blest.check(blest._lib.load().blest_mbfs(q._h, srcs.ctypes.data_as(blest._lib.U32P), k, buf.i32(), C.byref(o),
                                                 C.byref(st)))
        got = buf.numpy(np.int32, g.n * k).reshape(k, g.n)
        for j, r in enumerate(srcs):
            np.testing.assert_array_equal(got[j], oracle.bfs(g.n, cp, rows, int(r)), err_msg=f"k={k} root {r}")
