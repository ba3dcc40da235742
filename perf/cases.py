"""Performance cases of the traversal library: what its users run, over the sizes they run it at.

A case is a dict of plain values; `prepare` makes what a program holds before the call
(resident graph, query, roots, result buffers), `run` is one pass through the public
entry points.  Results are whole numbers (hop distances, component labels, counts).

Graphs that a program loads once and queries many times (BFS, multi-source BFS, the
batch of small graphs) are a property of the case and stay resident; the seed picks the
roots.  Where the graph itself is the input (components, loading), the seed makes it.
Results go to device arrays through the C ABI, as a GPU pipeline takes them, or to host
arrays through the Python classes (`"host": True`), as a script does.
"""
import ctypes
import functools
import math

import numpy as np
import torch

import blest_amd as B


def listed():
    return [
        # The smallest query: one BFS on a graph of a couple of thousand vertices, where
        # the call's latency is all there is (interactive use, the small end of a service).
        {"name": "bfs_er_2k", "do": "bfs", "graph": "er", "n": 2003, "degree": 8.0, "order": "natural", "roots": 1,
         "host": False},
        # The small R-MAT benchmark graph, 16 roots one after another, levels as numpy arrays.
        {"name": "bfs_rmat16_host", "do": "bfs", "graph": "rmat", "scale": 16, "order": "natural", "roots": 16,
         "host": True},
        # An ordinary social graph in the order the library picks for it (Jaccard windows);
        # results are mapped back to the caller's vertex numbers.
        {"name": "bfs_rmat18_jaccard", "do": "bfs", "graph": "rmat", "scale": 18, "order": "auto", "roots": 8,
         "host": False},
        # The large single-source graph: scale 22, vertices in arrival order.
        {"name": "bfs_rmat22", "do": "bfs", "graph": "rmat", "scale": 22, "order": "natural", "roots": 4,
         "host": False},
        # The same graph, 128 roots in one launch (all-pairs style analytics, sampling).
        {"name": "mbfs_rmat22_128", "do": "mbfs", "graph": "rmat", "scale": 22, "order": "natural", "roots": 128,
         "host": False},
        # A small multi-source query with a ragged number of roots, through the Python class.
        {"name": "mbfs_rmat14_37_host", "do": "mbfs", "graph": "rmat", "scale": 14, "order": "natural", "roots": 37,
         "host": True},
        # A road-like graph: a perturbed grid in RCM order, dozens of thin levels.
        {"name": "bfs_grid2047_rcm", "do": "bfs", "graph": "grid", "side": 2047, "order": "auto", "roots": 2,
         "host": False},
        # A directed graph of an odd size (links, citations): in-neighbours differ from out-neighbours.
        {"name": "bfs_directed_200k", "do": "bfs", "graph": "directed", "n": 200003, "degree": 8.0,
         "order": "natural", "roots": 4, "host": False},
        # Many small graphs, a root each, in one launch (molecules, ego networks, test beds).
        {"name": "batch_er_512", "do": "batch", "count": 512, "lo": 1024, "hi": 65536, "degree": 8.0},
        # Components of a social graph that has just been loaded.
        {"name": "cc_rmat20", "do": "cc", "graph": "rmat", "scale": 20, "order": "natural", "host": False},
        # Components of a road-like graph in RCM order, labels as a numpy array.
        {"name": "cc_grid1023_host", "do": "cc", "graph": "grid", "side": 1023, "order": "auto", "host": True},
        # A graph arriving in host memory: build its bit matrix on the GPU, make it
        # resident, answer the first query.
        {"name": "load_rmat18", "do": "load", "graph": "rmat", "scale": 18, "order": "natural"},
    ]


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["bfs", "bfs", "bfs", "mbfs", "batch", "cc", "load"])
    if do == "batch":
        lo = _log_between(rng, 100, 4000)
        return {"do": "batch", "count": _log_between(rng, 16, 512), "lo": lo, "hi": _log_between(rng, lo + 1, 65536),
                "degree": round(rng.uniform(2.0, 10.0), 2)}
    kinds = ["rmat", "grid", "er"] + (["directed"] if do == "bfs" else [])
    kind = rng.choice(kinds)
    case = {"do": do, "graph": kind}
    if kind == "rmat":
        case["scale"] = rng.randint(10, 18 if do == "load" else 20)
    elif kind == "grid":
        case["side"] = _log_between(rng, 40, 400 if do in ("mbfs", "load") else 1400)
    else:
        case["n"] = _log_between(rng, 1000, 200000 if do in ("mbfs", "load") or kind == "directed" else 800000)
        # components are of interest where there are several
        case["degree"] = round(rng.uniform(0.8, 4.0) if do == "cc" else rng.uniform(3.0, 16.0), 2)
    small = kind == "rmat" and case["scale"] <= 16 or kind == "grid"
    case["order"] = rng.choice(["natural", "auto"]) if small and do != "load" else "natural"
    if do == "bfs":
        case["roots"] = _log_between(rng, 1, 16)
    elif do == "mbfs":
        case["roots"] = rng.randint(2, 128)
    if do != "load":
        case["host"] = rng.random() < 0.3 and case.get("roots", 1) <= 60
    return case


# ----------------------------------------------------------------------------- graphs
def _csc(case, seed):
    kind = case["graph"]
    if kind == "rmat":
        return B.CSC.rmat(case["scale"], 16, 0.57, 0.19, 0.19, seed=1 + seed, permute=True)
    if kind == "grid":
        return B.CSC.grid(case["side"], 0.9, 0.01, seed=1 + seed)
    if kind == "er":
        return B.CSC.erdos_renyi(case["n"], case["degree"], seed=1 + seed)
    # directed: `degree` out-links per vertex on average, uniform targets
    n = case["n"]
    gen = np.random.default_rng(seed)
    ends = gen.integers(0, n, size=(2, int(n * case["degree"])), dtype=np.int64)
    return B.CSC.from_edges(n, ends[0], ends[1], undirected=False)


def _resident(case, seed, pool=0):
    """(device graph, some vertices of degree >= 1 in the caller's numbering)."""
    g = _csc(case, seed)
    roots = g.pick_roots(pool, seed=7) if pool else None
    social = g.is_social_network()
    # the reference harness's pipeline: order, pad unless social, build, upload
    inv = g.reorder(B.Reorder.AUTO, window=65536) if case["order"] == "auto" else None
    return B.DeviceGraph(B.BVSS(8, 4).construct_on_device(g, full_padding=not social), g, inv), roots


@functools.lru_cache(maxsize=16)
def _graph(key):
    return _resident(dict(key), 0, pool=256)


@functools.lru_cache(maxsize=4)
def _batch(count, lo, hi, degree):
    sizes = np.random.default_rng(3).integers(lo, hi + 1, size=count)
    return B.GraphBatch([B.CSC.erdos_renyi(int(n), degree, seed=10_000 + i) for i, n in enumerate(sizes)]), sizes


def _key(case):
    return tuple(sorted((k, v) for k, v in case.items() if k in ("graph", "scale", "side", "n", "degree", "order")))


def _device_i32(*shape):
    return torch.empty(shape, dtype=torch.int32, device="cuda")


def _out(t):
    return ctypes.cast(ctypes.c_void_p(t.data_ptr()), B._lib.I32P)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    if case["do"] == "batch":
        batch, sizes = _batch(case["count"], case["lo"], case["hi"], case["degree"])
        roots = (rng.random(len(sizes)) * sizes).astype(np.uint32)
        return {"do": "batch", "batch": batch, "roots": roots, "levels": _device_i32(int(sizes.sum()))}
    if case["do"] == "load":
        g = _csc(case, seed)
        return {"do": "load", "csc": g, "root": int(g.pick_roots(1, seed=seed)[0])}
    if case["do"] == "cc":
        dg, _ = _resident(case, seed)
        state = {"do": "cc", "kernel": B.BVSSCCKernel(dg), "host": case["host"]}
        if not case["host"]:
            state["labels"] = _device_i32(dg.n)
        return state
    dg, pool = _graph(_key(case))
    k = case["roots"]
    roots = rng.choice(pool, size=k, replace=False).astype(np.uint32)
    state = {"do": case["do"], "roots": roots, "host": case["host"]}
    if case["do"] == "bfs":
        state["kernel"] = B.BVSSBFSKernel(dg)
    else:
        state["kernel"] = B.BVSSMBFSKernel(dg, batch=128 if k > 64 else 64)
    if not case["host"]:
        state["levels"] = _device_i32(k, dg.n)
    return state


# ------------------------------------------------------------------------------ passes
def _run_bfs(state):
    kernel = state["kernel"]
    if state["host"]:
        res = [kernel.run(int(r)) for r in state["roots"]]
        return ([x.levels for x in res],
                np.array([(x.total_levels, x.no_visited, x.edges_in_component) for x in res], dtype=np.int64))
    lib, st, counts = B._lib.load(), B._lib.BfsStats(), []
    for row, root in zip(state["levels"], state["roots"]):
        B.check(lib.blest_bfs(kernel.q._h, int(root), _out(row), ctypes.byref(st)))
        counts.append((st.total_levels, st.no_visited, st.edges_traversed_component))
    return state["levels"], np.array(counts, dtype=np.int64)


def _run_mbfs(state):
    kernel, roots = state["kernel"], state["roots"]
    if state["host"]:
        return kernel.run(roots).level_arrays
    lib, st = B._lib.load(), B._lib.BfsStats()
    opts = B._lib.MbfsOpts(0, kernel.batch)
    B.check(lib.blest_mbfs(kernel.q._h, roots.ctypes.data_as(B._lib.U32P), len(roots), _out(state["levels"]),
                           ctypes.byref(opts), ctypes.byref(st)))
    return state["levels"], st.total_levels, st.no_visited


def _run_batch(state):
    ms = ctypes.c_double()
    B.check(B._lib.load().blest_graph_batch_bfs(state["batch"]._h, state["roots"].ctypes.data_as(B._lib.U32P),
                                                _out(state["levels"]), ctypes.byref(ms)))
    return state["levels"]


def _run_cc(state):
    kernel = state["kernel"]
    if state["host"]:
        res = kernel.run()
        return res.components, res.no_components
    st = B._lib.CcStats()
    labels = ctypes.cast(ctypes.c_void_p(state["labels"].data_ptr()), B._lib.U32P)
    B.check(B._lib.load().blest_cc(kernel.q._h, kernel.algo, labels, ctypes.byref(st)))
    return state["labels"], st.no_components


def _run_load(state):
    g = state["csc"]
    dg = B.DeviceGraph(B.BVSS(8, 4).construct_on_device(g, full_padding=not g.is_social_network()), g)
    info = dg.info()
    res = B.BVSSBFSKernel(dg).run(state["root"])
    return (res.levels, res.total_levels, res.no_visited, res.edges_in_component, info["vsets"], info["slices"],
            info["nnz"], info["stream_quads"])


def run(state):
    return {"bfs": _run_bfs, "mbfs": _run_mbfs, "batch": _run_batch, "cc": _run_cc, "load": _run_load}[state["do"]](state)


# -------------------------------------------------------------------------------- work
def _size(case):
    """Vertices and directed edges, to a few per cent."""
    kind = case["graph"]
    if kind == "rmat":
        n = 1 << case["scale"]
        return n, 29 * n
    if kind == "grid":
        n = case["side"] ** 2
        return n, 3.62 * n
    return case["n"], case["degree"] * case["n"]


def work(case):
    """Bytes: the adjacency (4 bytes an edge, 4 a vertex) once per traversal, the result
    written once; a multi-source launch reads the adjacency once for all of its roots.
    Loading reads the adjacency and writes it in both resident forms (bit matrix, CSR)."""
    if case["do"] == "batch":
        n = case["count"] * (case["lo"] + case["hi"]) / 2
        return {"bytes": n * (4 + 4 * case["degree"] + 4), "flops": 0}
    n, m = _size(case)
    graph, result = 4 * (n + m), 4 * n
    if case["do"] == "bfs":
        return {"bytes": case["roots"] * (graph + result), "flops": 0}
    if case["do"] == "mbfs":
        return {"bytes": graph + case["roots"] * result, "flops": 0}
    if case["do"] == "load":
        return {"bytes": graph + 5 * m + graph + graph + result, "flops": 0}
    return {"bytes": graph + result, "flops": 0}
