"""GPU parity of the connected components against the oracle where the seeded forest can go
wrong: equal-sized large components, hub lists around one and several waves, vertices whose
list is shorter than the sampled part, counts around whole waves, and no CSR at all."""
import ctypes as C

import numpy as np
import pytest
from conftest import progress
from test_gpu_result_ranges import DeviceBuffer

pytestmark = pytest.mark.gpu
HIP_H2D = 1


def star_pair(n, hub):
    """Two stars of `hub` leaves, interleaved over the IDs, and isolated vertices after them."""
    leaves = np.arange(2, 2 + 2 * hub)
    return n, leaves % 2, leaves


def paths(n, length):
    """Paths of `length` vertices: every tree small, no giant."""
    v = np.arange(n - 1)
    v = v[(v + 1) % length != 0]
    return n, v, v + 1


def two_blocks(n, degree, seed):
    """Two random graphs of the same size on the even and the odd vertices."""
    rng = np.random.default_rng(seed)
    e = rng.integers(0, n // 2, size=(2, n * degree // 2)) * 2
    odd = rng.integers(0, 2, size=e.shape[1])
    return n, e[0] + odd, e[1] + odd


CASES = {
    "star_pair_66": lambda: star_pair(200, 66),            # one entry more than the sampled part + a lane's list
    "star_pair_67": lambda: star_pair(201, 68),
    "star_pair_5000": lambda: star_pair(10240, 5000),
    "pairs": lambda: paths(4097, 2),
    "paths_7": lambda: paths(65535, 7),
    "path": lambda: paths(3000, 3000),
    "two_blocks": lambda: two_blocks(60000, 3, 1),
    "two_blocks_sparse": lambda: two_blocks(300002, 1, 2),
    "wave": lambda: paths(64, 64),
    "wave_less": lambda: paths(63, 5),
}


@pytest.mark.parametrize("name", CASES)
def test_cc_forest_parity(blest, oracle, name):
    progress(f"case cc forest {name}")
    n, src, dst = CASES[name]()
    g = blest.CSC.from_edges(n, src, dst)
    cp, rows = g.arrays()
    want, comps = oracle.cc(n, cp, rows)
    perm = np.random.default_rng(7).permutation(n).astype(np.uint32)
    shuffled = blest.CSC.from_arrays(n, cp, rows)
    shuffled.apply_permutation(perm)
    for label, graph, inv, opts in (("csr", g, None, {}), ("csr_unsorted", g, None, {"bu_probe": -1}),
                                    ("permuted", shuffled, perm, {}),
                                    ("slices", g, None, {"keep_csr": 0, "direction": 1}),
                                    ("slices_permuted", shuffled, perm, {"keep_csr": 0, "direction": 1})):
        kernel = blest.BVSSCCKernel(blest.BVSS().construct_from_csc(graph), graph, inv, **opts)
        for rep in range(2):
            res = kernel.run()
            np.testing.assert_array_equal(res.components, want, err_msg=f"{label} rep={rep}")
            assert res.no_components == comps, label


def test_cc_into_device_labels(blest, oracle):
    """Labels written straight into the caller's device array, and only into it."""
    progress("case cc device labels")
    g = blest.CSC.rmat(13, 4, seed=3)
    cp, rows = g.arrays()
    want, comps = oracle.cc(g.n, cp, rows)
    inv = g.reorder(blest.Reorder.RCM)
    kernel = blest.BVSSCCKernel(blest.BVSS().construct_from_csc(g), g, inv)
    buf = DeviceBuffer(4 * (g.n + 16))
    mark = np.full(g.n + 16, 0xDEADBEEF, dtype=np.uint32)
    assert buf.hip.hipMemcpy(buf.ptr, mark.ctypes.data_as(C.c_void_p), mark.nbytes, HIP_H2D) == 0
    st = blest._lib.CcStats()
    out = C.cast(C.c_void_p(buf.ptr.value + 32), blest._lib.U32P)
    blest.check(blest._lib.load().blest_cc(kernel.q._h, 0, out, C.byref(st)))
    got = buf.numpy(np.uint32, g.n + 16)
    np.testing.assert_array_equal(got[8:8 + g.n], want)
    assert (got[:8] == mark[0]).all() and (got[8 + g.n:] == mark[0]).all()
    assert st.no_components == comps
    blest.check(blest._lib.load().blest_cc(kernel.q._h, 0, None, C.byref(st)))
    assert st.no_components == comps
