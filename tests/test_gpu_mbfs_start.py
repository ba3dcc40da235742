"""What a multi-source launch starts from: roots at both ends of every segment, many in one
segment or word, the same vertex many times, graphs of one word; one and two root words; rows
against the oracle."""
import numpy as np
import pytest
from conftest import progress

pytestmark = pytest.mark.gpu

GRAPHS = {
    "one": lambda B: B.CSC.from_edges(1, [], []),
    "path64": lambda B: B.CSC.from_edges(64, np.arange(63), np.arange(1, 64)),
    "path65": lambda B: B.CSC.from_edges(65, np.arange(64), np.arange(1, 65)),
    "rmat12": lambda B: B.CSC.rmat(12, 8, seed=3),
    "grid600": lambda B: B.CSC.grid(600, 0.9, 0.01, 5),  # several words a segment, a short last one
}


@pytest.mark.parametrize("name", GRAPHS)
@pytest.mark.parametrize("k", [1, 64, 65, 128])
def test_mbfs_roots(blest, oracle, name, k):
    progress(f"case mbfs start {name} k={k}")
    g = GRAPHS[name](blest)
    cp, rows = g.arrays()
    n = g.n
    run = blest.BVSSMBFSKernel(blest.DeviceGraph(blest.BVSS().construct_from_csc(g), g, None, use_graphs=2), batch=k)
    spread = np.linspace(0, n - 1, k).astype(np.int64) // 64 * 64 + np.tile([0, 63], k)[:k]  # first and last of words
    packed = n // 2 + np.arange(k) % max(1, min(70, n - n // 2))
    for roots in (np.minimum(spread, n - 1), packed, np.full(k, n - 1)):
        levels = np.asarray(run.host_code(np.asarray(roots, dtype=np.uint32)).level_arrays).reshape(k, n)
        for r in sorted({int(x) for x in roots}):
            want = oracle.bfs(n, cp, rows, r)
            for j in np.flatnonzero(roots == r):
                np.testing.assert_array_equal(levels[j], want, err_msg=f"row {j} root {r}")
