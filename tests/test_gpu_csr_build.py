"""The resident CSR prepared on the GPU: symmetric and nearly symmetric graphs told apart at
every place an edge can be missing (tile and list ends, hubs), list order by degree, and the
traversals that read it, against the host's check and the oracle."""
import numpy as np
import pytest
from conftest import progress

pytestmark = pytest.mark.gpu


def drop_edge(blest, n, cp, rows, p):
    """The pattern without its p-th stored entry (its reverse stays)."""
    cp = cp.copy()
    col = int(np.searchsorted(cp, p, side="right") - 1)
    cp[col + 1:] -= 1
    return blest.CSC.from_arrays(n, cp, np.delete(rows, p))


GRAPHS = {
    "rmat12": lambda B: B.CSC.rmat(12, 16, seed=2),          # hub lists, empty columns
    "grid60": lambda B: B.CSC.grid(60, 0.8, 0.01, 3),
    "star9000": lambda B: B.CSC.from_edges(9100, np.zeros(9000, dtype=np.int64), np.arange(1, 9001)),  # a list over tiles
    "pair": lambda B: B.CSC.from_edges(70, [3], [69]),
}


@pytest.mark.parametrize("name", GRAPHS)
def test_symmetry_on_device(blest, oracle, name):
    progress(f"case csr symmetry {name}")
    g = GRAPHS[name](blest)
    cp, rows = g.arrays()
    n, nnz = g.n, len(rows)
    bv = blest.BVSS().construct_from_csc(g)
    assert blest.DeviceGraph(bv, g, None).info()["symmetric"] == 1
    picks = sorted({0, 1, nnz // 2, 4095, 4096, 4097, nnz - 1} & set(range(nnz)))
    for p in picks:
        h = drop_edge(blest, n, cp, rows, p)
        assert not h.check_symmetry()
        dg = blest.DeviceGraph(blest.BVSS().construct_from_csc(h), h, None)
        assert dg.info()["symmetric"] == 0, f"entry {p}"
        src = int(g.pick_roots(1, seed=p)[0])
        hcp, hrows = h.arrays()
        for direction in (0, 2):  # bottom-up sweeps read the transpose's lists
            dg.set_thresholds(15, 18, direction)
            np.testing.assert_array_equal(blest.BVSSBFSKernel(dg).run(src).levels, oracle.bfs(n, hcp, hrows, src))


@pytest.mark.parametrize("name", GRAPHS)
def test_symmetry_balanced_and_repeated(blest, name):
    """One edge short in each direction (as many entries look up their reverse as do not),
    and lists with an entry twice: the host's answer."""
    progress(f"case csr symmetry balanced {name}")
    g = GRAPHS[name](blest)
    cp, rows = g.arrays()
    n, nnz = g.n, len(rows)
    rng = np.random.default_rng(3)
    for _ in range(6):
        h = drop_edge(blest, n, cp, rows, int(rng.integers(nnz)))
        hcp, hrows = h.arrays()
        h = drop_edge(blest, n, hcp, hrows, int(rng.integers(nnz - 1)))
        dg = blest.DeviceGraph(blest.BVSS().construct_from_csc(h), h, None)
        assert dg.info()["symmetric"] == int(h.check_symmetry())
    for p in sorted({0, nnz // 2, nnz - 1}):
        tcp = cp.copy()
        tcp[int(np.searchsorted(cp, p, side="right")):] += 1
        h = blest.CSC.from_arrays(n, tcp, np.insert(rows, p, rows[p]))
        dg = blest.DeviceGraph(blest.BVSS().construct_from_csc(g), h, None)
        assert dg.info()["symmetric"] == int(h.check_symmetry())


@pytest.mark.parametrize("n,src,dst", [(1, [], []), (64, [], []), (65, [0], [64]), (300, [0] * 299, list(range(1, 300)))])
@pytest.mark.parametrize("bu_probe", [0, -1])
def test_small_lists(blest, oracle, n, src, dst, bu_probe):
    progress(f"case csr lists n={n} bu_probe={bu_probe}")
    for undirected in (True, False):
        g = blest.CSC.from_edges(n, src, dst, undirected=undirected)
        cp, rows = g.arrays()
        k = blest.BVSSBFSKernel(blest.BVSS().construct_from_csc(g), g, direction=2, bu_probe=bu_probe)
        for s in sorted({0, n - 1}):
            np.testing.assert_array_equal(k.run(s).levels, oracle.bfs(n, cp, rows, s))


COUNTS = ("no_slices", "no_unpadded_slices", "no_padded_slices", "edges_check", "min_slices_per_set",
          "max_slices_per_set", "compression_ratio")


def test_device_counts_match_host(blest):
    """The slices and edges that the device build counts are those of the host's pass over the masks."""
    progress("case bvss counts")
    for g in (blest.CSC.rmat(13, 16, seed=5), blest.CSC.grid(100, 0.9, 0.01, 6), blest.CSC.from_edges(5, [], [])):
        for fp in (False, True):
            host = blest.BVSS().construct_from_csc(g, full_padding=fp).info()
            device = blest.BVSS().construct_on_device(g, full_padding=fp).info()
            assert {k: device[k] for k in COUNTS} == {k: host[k] for k in COUNTS}


def test_rejects_rows_out_of_range(blest, tmp_path):
    """A binary cache is not checked when it is read; its lists are before they are searched."""
    progress("case csr out of range")
    g = blest.CSC.rmat(8, 8, seed=1)
    cp, rows = g.arrays()
    bad = rows.copy()
    bad[len(bad) // 2] = g.n + 5
    path = tmp_path / "g.bin"
    with open(path, "wb") as f:
        f.write(np.array([g.n, len(rows)], dtype=np.uint32).tobytes() + bytes([0]))
        f.write(cp.tobytes() + bad.tobytes())
    h = blest.CSC.load_binary(str(path))
    with pytest.raises(blest.BlestError):
        blest.DeviceGraph(blest.BVSS().construct_from_csc(g), h, None)
