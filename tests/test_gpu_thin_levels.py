"""The vertex-queue BFS of graphs with short lists against the oracle and the bit-matrix
levels (fuse_quads < 0) on the same graphs: frontiers around the one-workgroup kernel's
bounds, growing and shrinking through them, many components, list lengths at the path's
limit, replayed chunks, permutations, and the allocation-free call."""
import ctypes as C

import numpy as np
import pytest
from conftest import progress
from test_gpu_result_ranges import DeviceBuffer

pytestmark = pytest.mark.gpu


def tree(B, n, arity):
    """Complete arity-ary tree: levels grow arity-fold to the last, widest one."""
    v = np.arange(1, n)
    return B.CSC.from_edges(n, (v - 1) // arity, v)


def lens(B, width, steps):
    """Frontiers that jump from 1 to `width` vertices, stay, and shrink to 1: a ladder of `steps`
    ranks of `width` vertices, the first rank hung under a tree, the last one joined by one."""
    root, _ = 0, None
    t = np.arange(1, 2 * width)
    src, dst = [(t - 1) // 2], [t]                        # a binary tree, its last `width` vertices the first rank
    first = width
    base = 2 * width
    ranks = [np.arange(first, first + width)] + [base + np.arange(k * width, (k + 1) * width) for k in range(steps)]
    for a, b in zip(ranks, ranks[1:]):
        src.append(a)
        dst.append(b)
    return B.CSC.from_edges(base + steps * width, np.concatenate(src), np.concatenate(dst))


def ring_chords(B, n):
    """A ring and a random perfect matching: three neighbours each, about log2(n) levels."""
    v = np.arange(n)
    half = np.random.default_rng(1).permutation(n)
    return B.CSC.from_edges(n, np.concatenate([v, half[:n // 2]]), np.concatenate([(v + 1) % n, half[n // 2:]]))


def hub(B, n, degree):
    """A grid-like chain graph with one vertex of the given degree."""
    v = np.arange(n - 1)
    extra = np.linspace(10, n - 1, degree - 1, dtype=np.int64)
    return B.CSC.from_edges(n, np.concatenate([v, np.zeros(degree - 1, dtype=np.int64)]), np.concatenate([v + 1, extra]))


GRAPHS = {
    "grid300": lambda B: B.CSC.grid(300, 0.9, 0.01, 3),
    "grid700": lambda B: B.CSC.grid(700, 0.9, 0.01, 4),
    "grid_parts": lambda B: B.CSC.grid(420, 0.6, 0.0, 5),           # thousands of components
    "ring_chords": lambda B: ring_chords(B, 1500002),               # few, wide levels: the second run leaves the path
    "tree2": lambda B: tree(B, 300001, 2),
    "tree7": lambda B: tree(B, 250000, 7),                          # lists of 8 entries: the last length taken
    "lens2048": lambda B: lens(B, 2048, 70),                        # the growing frontier's bound
    "lens2049": lambda B: lens(B, 2049, 70),
    "lens4097": lambda B: lens(B, 4097, 40),                        # past the LDS queue
    "er4_from": lambda B: B.CSC.erdos_renyi(8193, 4.0, seed=8),     # medium lists, at both ends of their range
    "er4_edges": lambda B: B.CSC.erdos_renyi(343000, 4.0, seed=9),
    "hub32": lambda B: hub(B, 140000, 32),
    "hub33": lambda B: hub(B, 140000, 33),                          # one list too long: not on this path
    "hub9": lambda B: hub(B, 140000, 9),                            # a medium list among short ones
}


@pytest.mark.parametrize("name", GRAPHS)
def test_thin_levels(blest, oracle, name):
    progress(f"case thin levels {name}")
    lib = blest._lib.load()
    g = GRAPHS[name](blest)
    cp, rows = g.arrays()
    n = g.n
    degrees = np.diff(cp.astype(np.int64))
    perm = np.random.default_rng(3).permutation(n).astype(np.uint32)
    mixed = blest.CSC.from_arrays(n, cp, rows)
    mixed.apply_permutation(perm)
    bv, bvp = blest.BVSS().construct_from_csc(g), blest.BVSS().construct_from_csc(mixed)
    roots = [0, n // 2] if not name.startswith("hub") else [0]
    buf = DeviceBuffer(4 * n)
    st = blest._lib.BfsStats()
    for label, args, opts in (("natural", (bv, g, None), {}), ("permuted", (bvp, mixed, perm), {"use_graphs": 2}),
                              ("replayed", (bv, g, None), {"use_graphs": 1})):
        dg = blest.DeviceGraph(*args, **opts)
        k = blest.BVSSBFSKernel(dg)
        for r in roots:
            want = oracle.bfs(n, cp, rows, r)
            for fuse in ((0, -1) if label == "natural" else (0,)):
                dg.set_fuse(fuse)
                for rep in range(2):  # the second run starts from the first one's level hint
                    res = k.run(r)
                    np.testing.assert_array_equal(res.levels, want, err_msg=f"{label} root {r} fuse {fuse} rep {rep}")
                    assert res.total_levels == want.max() + 1 and res.no_visited == (want >= 0).sum()
                    assert res.edges_in_component == degrees[want >= 0].sum() // 2
                    assert res.td_levels + res.bu_levels == res.total_levels
            blest.check(lib.blest_bfs(k.q._h, r, buf.i32(), C.byref(st)))
            np.testing.assert_array_equal(buf.numpy(np.int32, n), want)
            blest.check(lib.blest_bfs_noalloc(dg._h, r, buf.i32(), C.byref(st), None))
            np.testing.assert_array_equal(buf.numpy(np.int32, n), want)
            assert st.total_levels == want.max() + 1 and st.no_visited == (want >= 0).sum()
