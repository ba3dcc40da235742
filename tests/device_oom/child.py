"""Runs one group of calls of the library with each of their device allocations failing in
turn (fail_malloc.cpp, loaded first so that the library's hipMalloc binds to it): the call
either does without that memory or reports that there was none, and the handles it worked
on give the oracle's results afterwards.

child.py FAIL_MALLOC_LIBRARY GROUP"""
import ctypes as C
import sys
from pathlib import Path

sys.path.insert(0, str(Path(__file__).resolve().parents[2]))
fail = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library is loaded
fail.oom_arm.argtypes = [C.c_long, C.c_long]
fail.oom_calls.restype = C.c_long

import numpy as np  # noqa: E402

import blest_amd as B  # noqa: E402
import oracle  # noqa: E402

OUT_OF_DEVICE_MEMORY = 6


def attempts(name, call, needed=None):
    """call() returns after its allocations; each one in turn finds no memory.  Yields after
    every try, armed no longer, with whether the call went through.  needed: how many
    allocations the call may not do without."""
    fail.oom_arm(-1, 0)
    call()
    total = fail.oom_calls()
    assert total > 0, "the library's hipMalloc is not the counting one"
    refused = 0
    for k in range(total):
        fail.oom_arm(k, 1)
        try:
            call()
            ok = True
        except B.BlestError as e:
            assert e.status == OUT_OF_DEVICE_MEMORY, (name, k, e)
            ok = False
            refused += 1
        fail.oom_arm(-1, 0)
        yield ok
    print(f"{name}: {total} allocations, {refused} needed", flush=True)
    if needed is not None:
        assert refused == needed, (name, refused, needed)


def resident(g, **opts):
    return B.DeviceGraph(B.BVSS().construct_from_csc(g), g, None, **opts)


def labels_of(g):
    cp, rows = g.arrays()
    return oracle.cc(g.n, cp, rows)[0]


def mbfs(q, srcs, n):
    lv = np.empty((len(srcs), n), dtype=np.int32)
    o, st = B._lib.MbfsOpts(0, 128 if len(srcs) > 64 else 64), B._lib.BfsStats()
    s = np.ascontiguousarray(srcs, dtype=np.uint32)
    B.check(B._lib.load().blest_mbfs(q._h, s.ctypes.data_as(B._lib.U32P), len(s), lv.ctypes.data_as(B._lib.I32P),
                                     C.byref(o), C.byref(st)))
    return lv


def query_state():
    """State made by a query's first components call and by a multi-source call that needs
    more words a vertex than the one before."""
    g = B.CSC.rmat(11, 8, seed=4)
    cp, rows = g.arrays()
    dg, want = resident(g), labels_of(g)
    few, many = g.pick_roots(20, seed=1), g.pick_roots(90, seed=2)
    lv = {int(r): oracle.bfs(g.n, cp, rows, int(r)) for r in [*few, *many]}
    held = {}

    def components():
        held["k"] = B.BVSSCCKernel(dg)
        held["k"].run()

    for _ in attempts("components", components):
        np.testing.assert_array_equal(held["k"].run().components, want)  # the query of the refused call

    def check(q, srcs):
        for row, r in zip(mbfs(q, srcs, g.n), srcs):
            np.testing.assert_array_equal(row, lv[int(r)])

    def more_words():
        held["q"] = B._Query(dg, 128)
        check(held["q"], few)
        check(held["q"], many)

    for _ in attempts("multi-source", more_words):
        check(held["q"], few)  # one word a vertex again, after the wider state was refused
        check(held["q"], many)


def creation():
    """Graphs and queries: what only makes them faster (the device sort's scratch, the shares of
    long lists, vertex queues) is done without.  The eleven allocations that a graph needs are
    its segment bases, chunk bases, slices (five arrays), lists (two), probes and empty-list
    marks; a query needs its state and its level array."""
    rng = np.random.default_rng(3)
    graphs = {"hubs": (B.CSC.rmat(11, 16, seed=4), 2), "short lists": (B.CSC.grid(60, 0.9, 0.01, 3), 1),
              "directed": (B.CSC.from_edges(3000, rng.integers(0, 40, 20000), rng.integers(0, 3000, 20000),
                                            undirected=False), 2)}
    for name, (g, query_needs) in graphs.items():
        cp, rows = g.arrays()
        bv = B.BVSS().construct_from_csc(g)
        roots = [int(r) for r in g.pick_roots(3, seed=1)]
        want = {r: oracle.bfs(g.n, cp, rows, r) for r in roots}
        held = {}

        def check(dg):
            for direction in (0, 2):
                dg.set_thresholds(15, 18, direction)
                k = B.BVSSBFSKernel(dg)
                for r in roots:
                    np.testing.assert_array_equal(k.run(r).levels, want[r])
                for row, r in zip(mbfs(B._Query(dg, 64), roots, g.n), roots):
                    np.testing.assert_array_equal(row, want[r])
            dg.set_thresholds(15, 18, 0)

        def graph():
            held["dg"] = B.DeviceGraph(bv, g, None)

        for ok in attempts(f"{name}: graph", graph, needed=11):
            if ok:
                check(held["dg"])

        def query():
            held["q"] = B.BVSSBFSKernel(held["dg"])

        for ok in attempts(f"{name}: query", query, needed=query_needs):
            if ok:
                for r in roots:
                    np.testing.assert_array_equal(held["q"].run(r).levels, want[r])


def construction():
    """The bit matrix built on the device needs all of its 24 arrays."""
    g = B.CSC.rmat(11, 16, seed=4)
    want = B.BVSS().construct_from_csc(g).arrays()
    held = {}

    def build():
        held["b"] = B.BVSS().construct_on_device(g)

    for ok in attempts("device construction", build, needed=24):
        got = B.BVSS().construct_on_device(g).arrays()
        for k in want:
            np.testing.assert_array_equal(got[k], want[k])


GROUPS = {f.__name__: f for f in (query_state, creation, construction)}

if __name__ == "__main__":
    GROUPS[sys.argv[2]]()
    print("OOM GROUP OK", flush=True)
