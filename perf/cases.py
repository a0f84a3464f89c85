"""What the walk engine is timed on: one pass is one call of a public walk entry point on inputs that are in place.

A case names a synthetic graph (R-MAT from the library's generator, or a small uniform graph uploaded from the host), an
application, the number and kind of start vertices, the walk length, the application's parameters and the entry point:
`device` (fw_walk_device: start vertices and path matrix in device memory), `noalloc` (fw_walk_device_noalloc, the call for
serving loops) or `batch` (fw_walk_batch: start vertices and path matrix in pinned host memory).  A pass returns the whole
path matrix and the two workload counters.  Walks are a function of (seed, walker id, graph, parameters), so every output
is compared exactly.
"""
import ctypes as C
import importlib
import math

import numpy as np
import torch

fw = importlib.import_module("flowwalker-artifact_amd")

APPS = {"deepwalk": fw.APP_DEEPWALK, "ppr": fw.APP_PPR, "node2vec": fw.APP_NODE2VEC, "metapath": fw.APP_METAPATH}
N_LABELS = 5

# What a case leaves out.
COMMON = {"entry": "device", "graph": "rmat", "scale": 0, "vertices": 0, "edges": 0, "edge_factor": 16, "skewed": True,
          "symmetrise": False, "w_hi": 100.0, "starts": "all", "length": 80, "tp": 0.2, "p": 2.0, "q": 0.5, "hub_threshold": 16384,
          "wg_threads": 512, "batch_size": 0}

LISTED = [
    # the reference's CPU-runnable size: one user asks for a hundred walks on a graph of seven thousand vertices
    {"name": "deepwalk_100_small_graph", "app": "deepwalk", "graph": "uniform", "vertices": 7115, "edges": 103689, "w_hi": 5.0,
     "starts": "random", "queries": 100},
    # a serving loop that must stay off the allocator: a few thousand short walks a call
    {"name": "deepwalk_serving_3001", "app": "deepwalk", "entry": "noalloc", "scale": 18, "symmetrise": True, "starts": "random",
     "queries": 3001, "length": 40},
    # few walkers, long lists: neighbourhoods of the best-connected vertices
    {"name": "deepwalk_1000_from_hubs", "app": "deepwalk", "scale": 20, "symmetrise": True, "starts": "hubs", "queries": 1000},
    # an ordinary batch: a minibatch of training walks, odd size and length
    {"name": "node2vec_50021_minibatch", "app": "node2vec", "scale": 20, "symmetrise": True, "starts": "random", "queries": 50021,
     "length": 41},
    # personalised PageRank as the reference's command line runs it: every query from the vertex of largest degree
    {"name": "ppr_1m_from_max_degree", "app": "ppr", "scale": 21, "starts": "max_degree", "queries": 1000003, "tp": 0.15},
    # one query per vertex with p and q at which proposals are turned down often (a local, depth-averse walk)
    {"name": "node2vec_all_rmat20_q4", "app": "node2vec", "scale": 20, "symmetrise": True, "queries": 1 << 20, "length": 40,
     "p": 0.25, "q": 4.0},
    # the benchmark's configurations: DeepWalk and PPR on a directed graph, one query per vertex
    {"name": "deepwalk_all_rmat22", "app": "deepwalk", "scale": 22, "queries": 1 << 22},
    {"name": "ppr_all_rmat22", "app": "ppr", "scale": 22, "queries": 1 << 22},
    # the same walks host to host, as the command line tool runs them (library's batch size)
    {"name": "deepwalk_all_rmat22_host", "app": "deepwalk", "entry": "batch", "scale": 22, "queries": 1 << 22},
    # MetaPath on the largest graph, random starts
    {"name": "metapath_10m_rmat26", "app": "metapath", "scale": 26, "starts": "random", "queries": 10000000, "length": 5},
    # the largest: the headline and node2vec on its graph
    {"name": "node2vec_all_rmat24_sym", "app": "node2vec", "scale": 24, "symmetrise": True, "queries": 1 << 24},
    {"name": "deepwalk_all_rmat24_sym", "app": "deepwalk", "scale": 24, "symmetrise": True, "queries": 1 << 24},
]


def listed():
    return [dict(COMMON, **c) for c in LISTED]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges: any application through any entry point, graphs from thousands of vertices to
    2^24, from 50 queries to some millions, walks of 3 to 100 steps."""
    c = dict(COMMON)
    c["app"] = rng.choice(["deepwalk", "deepwalk", "ppr", "node2vec", "metapath"])
    c["entry"] = rng.choice(["device", "device", "device", "batch", "noalloc"])
    if rng.random() < 0.2:
        c["graph"] = "uniform"
        c["vertices"] = _log_int(rng, 500, 50000)
        c["edges"] = c["vertices"] * rng.randint(4, 24) + rng.randint(0, 99)
    else:
        c["scale"] = rng.randint(12, 24)
        c["edge_factor"] = rng.choice([4, 8, 16, 16, 24])
        c["skewed"] = rng.random() < 0.8
        c["symmetrise"] = rng.random() < 0.5
    c["w_hi"] = rng.choice([5.0, 100.0, 100.0])
    c["starts"] = rng.choice(["random", "random", "all", "hubs", "max_degree"])
    c["length"] = rng.choice([80, _log_int(rng, 3, 100)])
    c["tp"] = round(rng.uniform(0.05, 0.5), 3)
    c["p"] = rng.choice([0.25, 0.5, 1.0, 2.0, 4.0])
    c["q"] = rng.choice([0.25, 0.5, 1.0, 2.0, 4.0])
    c["hub_threshold"] = rng.choice([16384, 16384, 16384, 1024])
    c["wg_threads"] = rng.choice([512, 512, 512, 256, 1024])
    c["queries"] = _log_int(rng, 50, 60000 if c["entry"] == "noalloc" else 4000000)
    if c["app"] == "node2vec":  # a step takes about max(1, q) trials
        c["queries"] = min(c["queries"], int(4000000 / max(1.0, c["q"])))
    if c["entry"] == "batch" and rng.random() < 0.5:
        c["batch_size"] = max(1, c["queries"] // rng.randint(1, 5))
    return c


def _uniform_graph(case, seed):
    """A directed graph of distinct random edges without loops, lists in ascending order."""
    rng = np.random.RandomState(seed % (1 << 31))
    V, E = case["vertices"], case["edges"]
    keys = np.empty(0, dtype=np.int64)
    while len(keys) < E:
        s = rng.randint(0, V, size=2 * E).astype(np.int64)
        d = rng.randint(0, V, size=2 * E).astype(np.int64)
        keys = np.unique(np.concatenate([keys, (s * V + d)[s != d]]))
    keys = np.sort(rng.choice(keys, size=E, replace=False))
    xadj = np.zeros(V + 1, dtype=np.uint32)
    np.cumsum(np.bincount(keys // V, minlength=V), out=xadj[1:])
    weight = (1.0 + (case["w_hi"] - 1.0) * rng.random_sample(E)).astype(np.float32)
    label = rng.randint(0, N_LABELS, size=E).astype(np.int32) if case["app"] == "metapath" else None
    return fw.Graph.from_csr(xadj, (keys % V).astype(np.int32), weight, label)


def _graph(case, seed):
    if case["graph"] == "uniform":
        return _uniform_graph(case, seed)
    a, b, c = (0.57, 0.19, 0.19) if case["skewed"] else (0.25, 0.25, 0.25)
    metapath = case["app"] == "metapath"
    return fw.Graph.rmat(case["scale"], case["edge_factor"], a, b, c, symmetrise=case["symmetrise"], w_lo=1.0, w_hi=case["w_hi"],
                         n_labels=N_LABELS if metapath else 0, make_weights=not metapath, seed=1 + seed)


def _starts(case, g, seed):
    n = case["queries"]
    rng = np.random.RandomState((seed + 77) % (1 << 31))
    if case["starts"] == "all":
        return (np.arange(n, dtype=np.int64) % g.V).astype(np.int32)
    if case["starts"] == "max_degree":
        return np.full(n, g.max_degree()[1], dtype=np.int32)
    if case["starts"] == "hubs":  # the 2,048 best-connected vertices
        deg = np.diff(g.download_xadj().astype(np.int64))
        return np.argsort(-deg, kind="stable")[:2048].astype(np.int32)[rng.randint(0, min(2048, g.V), size=n)]
    return rng.randint(0, g.V, size=n).astype(np.int32)


class _Device:
    """A torch tensor where the binding wants an object with a device pointer."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.ptr = C.c_void_p(tensor.data_ptr())


def prepare(case, seed):
    """The graph handle, the parameters, the start vertices and the (empty) path matrix."""
    g = _graph(case, seed)
    starts = torch.from_numpy(_starts(case, g, seed))
    n, depth = case["queries"], case["length"] + 1
    params = fw.default_params(app=APPS[case["app"]], max_depth=depth, seed=1337 + seed, tp=case["tp"], p=case["p"], q=case["q"],
                               schema=range(N_LABELS), hub_threshold=case["hub_threshold"], wg_threads=case["wg_threads"])
    state = {"entry": case["entry"], "graph": g, "params": params, "n": n, "batch_size": case["batch_size"]}
    if case["entry"] == "batch":
        state["starts"] = starts.pin_memory()
        state["paths"] = torch.empty((n, depth), dtype=torch.int32, pin_memory=True)
    else:
        state["starts"] = _Device(starts.cuda())
        state["paths"] = _Device(torch.empty((n, depth), dtype=torch.int32, device="cuda"))
    if case["app"] == "node2vec":
        g.is_sorted()  # a user finds out once whether the lists have to be sorted
    torch.cuda.synchronize()
    return state


def run(state):
    """One call: every query walks."""
    g, params, n = state["graph"], state["params"], state["n"]
    if state["entry"] == "batch":
        st = fw.WalkStats()
        paths = state["paths"]
        fw.check(fw.lib().fw_walk_batch(g.handle, C.byref(params), C.c_void_p(state["starts"].data_ptr()), n,
                                        state["batch_size"], 0, C.c_void_p(paths.data_ptr()), C.byref(st)))
    else:
        call = g.walk_device_noalloc if state["entry"] == "noalloc" else g.walk_device
        st = call(params, state["starts"], n, state["paths"])
        paths = state["paths"].tensor
    return {"paths": paths, "steps": int(st.steps), "sampled_edges": int(st.sampled_edges)}


def work(case):
    """Start vertices in, path matrix out, and of the graph what the walks cannot do without: each of its arrays once, or
    16 bytes a step (the vertex's range, the chosen edge's vertex and bias) where the steps are too few to touch it all."""
    n, length = case["queries"], case["length"]
    if case["graph"] == "uniform":
        V, E = case["vertices"], case["edges"]
    else:
        V = 1 << case["scale"]
        E = V * case["edge_factor"] * (2 if case["symmetrise"] else 1)
    steps = n * (min(length, 1.0 / case["tp"]) if case["app"] == "ppr" else length)
    return {"bytes": 4.0 * n + 4.0 * n * (length + 1) + min(8.0 * E + 4.0 * (V + 1), 16.0 * steps), "flops": 0.0}


def tolerance(case):
    return "exact"
