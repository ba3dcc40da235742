"""The single-source level kernels under the optimizing schedule at the ends of their knobs, on
graphs too large or too dense for the one-workgroup BFS and with lists too long for the vertex
queues (tests/test_paths.py holds the bounds)."""
import numpy as np
import pytest
from conftest import progress

pytestmark = pytest.mark.gpu


def cliques(B, count, size):
    """A chain of cliques: hundreds of levels, all small."""
    a, b = np.triu_indices(size, 1)
    first = np.arange(count)[:, None] * size
    link = np.arange(count - 1) * size
    return B.CSC.from_edges(count * size, np.concatenate([(first + a).ravel(), link + size - 1]),
                            np.concatenate([(first + b).ravel(), link + size]))


GRAPHS = {
    "rmat15": lambda B: B.CSC.rmat(15, 8, seed=8),            # 32,768 vertices
    "dense14": lambda B: B.CSC.erdos_renyi(16384, 16.5, 3),   # 16,384 vertices, more than 2^18 entries
    "er20k": lambda B: B.CSC.erdos_renyi(20000, 8.0, 2),
    "cliques": lambda B: cliques(B, 1100, 16),                # about 1,100 levels
}
KNOBS = {
    "alpha1_beta1": {"alpha": 1.0, "beta": 1.0},
    "alpha1000_beta1000": {"alpha": 1000.0, "beta": 1000.0},
    "alpha1000_beta1": {"alpha": 1000.0, "beta": 1.0},
    **{f"tiles_{t}_{b}": {"td_quads": t, "bu_group": b} for t in (1, 2, 4) for b in (4, 8)},
    "probe_off": {"bu_probe": -1},
    "never_fused": {"fuse_quads": -1},
    "fuse_32": {"fuse_quads": 32},
    "fuse_65536": {"fuse_quads": 65536},
    "replayed": {"use_graphs": 1},
    "one_workgroup_a_cu": {"blocks_per_cu": 1},
}


@pytest.fixture(scope="module")
def prepared(blest, oracle):
    out = {}
    for name, make in GRAPHS.items():
        g = make(blest)
        cp, rows = g.arrays()
        degrees = np.diff(cp.astype(np.int64))
        assert g.nnz > 5 * g.n and (g.n > 16384 or g.nnz > 1 << 18)  # not on the other paths
        roots = [int(r) for r in g.pick_roots(2, seed=1)] + [0]
        perm = np.random.default_rng(3).permutation(g.n).astype(np.uint32)
        mixed = blest.CSC.from_arrays(g.n, cp, rows)
        mixed.apply_permutation(perm)
        out[name] = (degrees, {r: oracle.bfs(g.n, cp, rows, r) for r in roots},
                     [(blest.BVSS().construct_from_csc(g), g, None),
                      (blest.BVSS().construct_from_csc(mixed), mixed, perm)])
    return out


@pytest.mark.parametrize("knobs", KNOBS)
@pytest.mark.parametrize("name", GRAPHS)
def test_level_kernels(blest, prepared, name, knobs):
    progress(f"case level kernels {name} {knobs}")
    degrees, want, forms = prepared[name]
    for args in forms:
        k = blest.BVSSBFSKernel(blest.DeviceGraph(*args, **KNOBS[knobs]))
        for rep in range(2):  # the second round starts from the first one's level hint
            for r, levels in want.items():
                res = k.run(r)
                np.testing.assert_array_equal(res.levels, levels, err_msg=f"root {r} rep {rep}")
                assert res.total_levels == levels.max() + 1 and res.no_visited == (levels >= 0).sum()
                assert res.edges_in_component == degrees[levels >= 0].sum() // 2
                assert res.td_levels + res.bu_levels == res.total_levels
