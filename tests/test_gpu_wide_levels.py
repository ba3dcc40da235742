"""Short-list graphs with few, wide levels, which belong on the bit-matrix levels: told by their
bottom-up levels, which vertex queues do not have."""
import ctypes as C

import numpy as np
import pytest
from conftest import progress
from test_gpu_result_ranges import DeviceBuffer

pytestmark = pytest.mark.gpu


def tree(B, n, arity):
    """Complete arity-ary tree, and its vertices' depths."""
    v = np.arange(1, n)
    depth, first, width = np.empty(n, dtype=np.int32), 0, 1
    for d in range(64):
        depth[first:first + width] = d
        first, width = first + width, width * arity
        if first >= n:
            break
    return B.CSC.from_edges(n, (v - 1) // arity, v), depth


def noalloc(blest, dg, root, n):
    buf, st = DeviceBuffer(4 * n), blest._lib.BfsStats()
    blest.check(blest._lib.load().blest_bfs_noalloc(dg._h, root, buf.i32(), C.byref(st), None))
    return buf.numpy(np.int32, n), st


def test_verdict_is_the_graphs(blest):
    """One traversal tells; queries made after it and the allocation-free call know."""
    progress("case wide levels verdict")
    g, depth = tree(blest, 300000, 7)  # 8 levels of 37,500 vertices on average: past 32,768
    bv = blest.BVSS().construct_from_csc(g)
    dg = blest.DeviceGraph(bv, g, None)
    first = blest.BVSSBFSKernel(dg).run(0)
    np.testing.assert_array_equal(first.levels, depth)
    for rep in range(2):
        res = blest.BVSSBFSKernel(dg).run(0)
        np.testing.assert_array_equal(res.levels, depth)
        assert res.bu_levels > 0
        levels, st = noalloc(blest, dg, 0, g.n)
        np.testing.assert_array_equal(levels, depth)
        assert st.bu_levels > 0 and st.total_levels == depth.max() + 1
    # told by the allocation-free call itself
    dg = blest.DeviceGraph(bv, g, None)
    for rep in range(3):
        levels, st = noalloc(blest, dg, 0, g.n)
        np.testing.assert_array_equal(levels, depth)
        assert rep == 0 or st.bu_levels > 0


@pytest.mark.parametrize("n, arity", [(1_000_000, 7), (600_000, 5), (500_000, 31)])
def test_more_discoveries_than_are_held(blest, n, arity):
    """Queue levels (the first traversal of a graph) whose workgroups write out more than once; with
    31 children each, 512 entries alone discover more than fits."""
    progress(f"case wide levels n={n} arity={arity}")
    g, depth = tree(blest, n, arity)
    perm = np.random.default_rng(6).permutation(n).astype(np.uint32)
    mixed, _ = tree(blest, n, arity)
    mixed.apply_permutation(perm)
    for graph, inv in ((g, None), (mixed, perm)):
        dg = blest.DeviceGraph(blest.BVSS().construct_from_csc(graph), graph, inv)
        res = blest.BVSSBFSKernel(dg).run(0)
        np.testing.assert_array_equal(res.levels, depth)
        assert res.bu_levels == 0 and res.no_visited == n and res.edges_in_component == n - 1


def test_first_wide_traversal(blest):
    """It may not cost several of those that follow on the bit matrix (it was seven times theirs)."""
    progress("case wide levels first traversal time")
    g, depth = tree(blest, 4_000_000, 7)
    bv = blest.BVSS().construct_from_csc(g)
    st, first, later = blest._lib.BfsStats(), [], []
    for rep in range(4):
        k = blest.BVSSBFSKernel(blest.DeviceGraph(bv, g, None))
        for out in (first, later, later):
            blest.check(blest._lib.load().blest_bfs(k.q._h, 0, None, C.byref(st)))
            assert st.total_levels == depth.max() + 1
            out.append(st.kernel_ms)
    assert np.median(first) <= 3 * np.median(later), (first, later)
