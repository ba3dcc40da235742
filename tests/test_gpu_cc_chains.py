"""Connected components of graphs whose seed forest is made of long chains: vertices numbered
along their paths, with ends around the tiles that the seed kernel shortens chains in."""
import ctypes as C

import numpy as np
import pytest
from conftest import progress

pytestmark = pytest.mark.gpu


def strided(n, step):
    """`step` interleaved paths: each vertex is joined to the one `step` before it."""
    v = np.arange(n - step)
    return n, v, v + step


def comb(n, leg):
    """A spine with paths of `leg` vertices hung from it."""
    spine = np.arange(n // leg - 1) * leg
    v = np.arange(n)
    v = v[v % leg != leg - 1]
    return n, np.concatenate([spine, v]), np.concatenate([spine + leg, v + 1])


def ring(n):
    v = np.arange(n)
    return n, v, (v + 1) % n


CASES = {
    "path_1023": lambda: strided(1023, 1),
    "path_1024": lambda: strided(1024, 1),
    "path_1025": lambda: strided(1025, 1),
    "path_4097": lambda: strided(4097, 1),
    "path_700000": lambda: strided(700000, 1),   # more tiles than workgroups
    "strided_2": lambda: strided(5001, 2),
    "strided_1023": lambda: strided(9000, 1023),
    "strided_1024": lambda: strided(9000, 1024),
    "comb_2": lambda: comb(6000, 2),
    "comb_30": lambda: comb(6000, 30),
    "ring_2049": lambda: ring(2049),
}


@pytest.mark.parametrize("name", CASES)
def test_cc_chains(blest, oracle, name):
    progress(f"case cc chains {name}")
    n, src, dst = CASES[name]()
    for label, ids in (("ascending", np.arange(n)), ("descending", np.arange(n)[::-1])):
        g = blest.CSC.from_edges(n, ids[src], ids[dst])
        want, comps = oracle.cc(n, *g.arrays())
        for opts in ({}, {"bu_probe": -1}):
            k = blest.BVSSCCKernel(blest.DeviceGraph(blest.BVSS().construct_from_csc(g), g, None, **opts))
            res = k.run()
            np.testing.assert_array_equal(res.components, want, err_msg=f"{label} {opts}")
            assert res.no_components == comps


TIMED = {
    "path": lambda B: B.CSC.from_edges(*strided(1 << 20, 1)),   # a chain over all vertices took four times as long
    "random": lambda B: B.CSC.erdos_renyi(100000, 5.0, seed=3),  # swaps that met at one root: 1.7 times
}


@pytest.mark.parametrize("name", TIMED)
def test_lists_are_no_slower_than_slices(blest, name):
    """With the lists resident, components take no longer than with every slice's edges hooked."""
    progress(f"case cc time {name}")
    g = TIMED[name](blest)
    bv = blest.BVSS().construct_from_csc(g)
    st = blest._lib.CcStats()
    ms = {}
    for label, opts in (("lists", {}), ("slices", {"keep_csr": 0, "direction": 1})):
        k = blest.BVSSCCKernel(blest.DeviceGraph(bv, g, None, **opts))
        times = []
        for _ in range(15):
            blest.check(blest._lib.load().blest_cc(k.q._h, 0, None, C.byref(st)))
            times.append(st.kernel_ms)
        ms[label] = np.median(times)
    assert ms["lists"] <= ms["slices"], ms
