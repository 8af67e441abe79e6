"""Performance cases of the library: what its users' programs have it do.

Three groups, each through the Python entry points:

* searches — one Reset + EnactSearch on a device-resident graph, per strategy:
  RMAT graphs (small diameter, skewed degrees) from scale 10, where launches
  and latency count, to scale 22, and 3-D lattices (hundreds of narrow
  levels).  The batched engine answers many queries over a pool of graphs.
* the CSR build — radix sort of packed edges or of (row, column) pairs,
  consecutive removal, prefix scan, and the whole COO -> CSR call.
* the same primitives at a few thousand elements, as they are called for
  small graphs.

A search's predecessors are any valid parent: which one is decided by a race
on the device.  A pass therefore returns every vertex's depth and the depth
of its predecessor, which the graph alone determines.  Sorted keys are
returned as whole numbers (the bits of floating-point keys).
"""
import math

import numpy as np
import torch

from back40computing_amd import _lib, autotune, bfs, primitives, radix_sort
from back40computing_amd._lib import check, lib, ptr
from back40computing_amd.batch import MultiGraph, MultiSourceBFS
from back40computing_amd.sources import pick_sources

STRATEGIES = {
    "expand_contract": _lib.EXPAND_CONTRACT,
    "contract_expand": _lib.CONTRACT_EXPAND,
    "two_phase": _lib.TWO_PHASE,
    "hybrid": _lib.HYBRID,
    "direction_optimizing": _lib.DIRECTION_OPTIMIZING,
}
KEY_TYPES = {"u32": np.uint32, "i32": np.int32, "f32": np.float32, "u64": np.uint64, "i64": np.int64, "f64": np.float64}


def listed():
    return [
        # One search on the served pool's smaller graphs: launches and latency.
        {"name": "search_do_rmat12", "kind": "search", "strategy": "direction_optimizing", "graph": "rmat", "size": 12,
         "edge_factor": 16},
        # The headline search: scale 22, edge factor 16.
        {"name": "search_do_rmat22", "kind": "search", "strategy": "direction_optimizing", "graph": "rmat", "size": 22,
         "edge_factor": 16},
        # The reference's expand-contract in its default (single launch) form on a mid-sized graph.
        {"name": "search_ec_rmat20", "kind": "search", "strategy": "expand_contract", "graph": "rmat", "size": 20,
         "edge_factor": 16},
        # The reference's hybrid: edge frontiers, narrow levels fused, wide ones in three launches.
        {"name": "search_hybrid_rmat20", "kind": "search", "strategy": "hybrid", "graph": "rmat", "size": 20,
         "edge_factor": 16},
        # High diameter: about 450 narrow levels.
        {"name": "search_ec_lattice200", "kind": "search", "strategy": "expand_contract", "graph": "lattice",
         "size": 200, "edge_factor": 6},
        # A batch of queries over a resident pool of small and ordinary graphs, labels taken to the host.
        {"name": "batch_64_graphs", "kind": "batch", "graphs": 64, "per_graph": 4, "scale_lo": 10, "scale_hi": 15},
        # Loading a graph: host edge list to a deduplicated, symmetrized device CSR.
        {"name": "build_coo_1m", "kind": "build", "scale": 16, "edges": 1000003, "symmetrize": True},
        # The CSR build's sort at large size: full-width random keys.
        {"name": "sort_u64_64m", "kind": "sort", "key": "u64", "values": False, "n": 1 << 26, "bits": 64,
         "dist": "uniform"},
        # COO rows with their columns: power-law row ids, only the id's bits sorted.
        {"name": "sort_pairs_u32_1m", "kind": "sort", "key": "u32", "values": True, "n": 1300021, "bits": 20,
         "dist": "ids"},
        # A small sort with values: every launch counts.
        {"name": "sort_pairs_f32_6k", "kind": "sort", "key": "f32", "values": True, "n": 6001, "bits": 32,
         "dist": "uniform"},
        # Duplicate removal of sorted packed edges with their values.
        {"name": "trim_pairs_32m", "kind": "trim", "values": True, "n": (1 << 25) + 7, "run": 2},
        # Row lengths to row offsets of a large graph.
        {"name": "scan_64m", "kind": "scan", "n": (1 << 26) + 4, "exclusive": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search", "search", "search", "search", "batch", "build", "sort", "sort", "trim", "scan"])
    if kind == "search":
        strategy = rng.choice(sorted(STRATEGIES))
        if rng.random() < 0.3:
            return {"kind": kind, "strategy": strategy, "graph": "lattice", "size": _log_int(rng, 9, 150),
                    "edge_factor": 6}
        top = 22 if strategy == "direction_optimizing" else 20
        return {"kind": kind, "strategy": strategy, "graph": "rmat", "size": rng.randint(10, top),
                "edge_factor": rng.randint(5, 16)}
    if kind == "batch":
        lo = rng.randint(8, 12)
        return {"kind": kind, "graphs": _log_int(rng, 6, 64), "per_graph": rng.randint(1, 4), "scale_lo": lo,
                "scale_hi": lo + rng.randint(1, 3)}
    if kind == "build":
        m = _log_int(rng, 1000, 1000000)
        return {"kind": kind, "scale": max(7, int(math.log2(m)) - rng.randint(2, 4)), "edges": m,
                "symmetrize": rng.random() < 0.5}
    if kind == "sort":
        key = rng.choice(sorted(KEY_TYPES))
        full = 8 * np.dtype(KEY_TYPES[key]).itemsize
        ids = key in ("u32", "u64") and rng.random() < 0.5
        return {"kind": kind, "key": key, "values": rng.random() < 0.5, "n": _log_int(rng, 1000, 40000000),
                "bits": rng.randint(11, full * 3 // 4) if ids else full, "dist": "ids" if ids else "uniform"}
    if kind == "trim":
        return {"kind": kind, "values": rng.random() < 0.5, "n": _log_int(rng, 1000, 30000000),
                "run": rng.randint(1, 9)}
    return {"kind": kind, "n": _log_int(rng, 1000, 60000000), "exclusive": rng.random() < 0.5}


class _View:
    """Device memory of the library as torch sees it; `owner` is the object
    that frees it, kept for as long as a tensor over it lives."""

    def __init__(self, owner, address, count, dtype):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": dtype, "data": (address, False), "version": 2}


def _tensor(owner, address, count, itemsize):
    return torch.as_tensor(_View(owner, address, count, "<i4" if itemsize == 4 else "<i8"), device="cuda")


def _array(a, count, itemsize):
    return _tensor(a, a.ptr.value, count, itemsize)


def _offsets(graph):
    off = np.empty(graph.nodes + 1, np.int32)
    check(lib().b40c_graph_copy_to_host(graph.handle, ptr(off), None))
    return off


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _ids(n, bits, gen):
    """Power-law ids in [0, 2^bits): a few ids repeat often, as hub rows do."""
    u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
    low = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
    return ((u * u * u * (0.5 + 0.5 * low)) * float(1 << bits)).to(torch.int64)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "search":
        if case["graph"] == "rmat":
            graph = bfs.Graph.rmat(case["size"], case["edge_factor"], seed=seed)
        else:
            graph = bfs.Graph.lattice3d(case["size"], seed=seed)
        strategy = STRATEGIES[case["strategy"]]
        problem = bfs.CsrProblem()
        check(problem.FromGraph(graph))
        enactor = bfs.ENACTORS[strategy]()
        tuning = autotune.lookup(bfs.device_info()["arch"], strategy, graph.nodes, graph.edges)
        if tuning:
            enactor.set_tuning(**tuning)
        frontier = enactor.GetFrontierType()
        check(problem.Reset(frontier))
        d, p = problem.device_labels()
        return {"kind": kind, "graph": graph, "problem": problem, "enactor": enactor, "frontier": frontier,
                "source": int(pick_sources(_offsets(graph), seed, 1)[0]),
                "stream": torch.cuda.ExternalStream(problem.stream()),
                "depth": _tensor(problem, d, graph.nodes, 4), "pred": _tensor(problem, p, graph.nodes, 4)}
    if kind == "batch":
        span = case["scale_hi"] - case["scale_lo"] + 1
        scales = [case["scale_lo"] + i % span for i in range(case["graphs"])]
        graphs = [bfs.Graph.rmat(int(s), 16, seed=seed + 1000 * i) for i, s in enumerate(scales)]
        queries = [(g, int(s)) for g, graph in enumerate(graphs)
                   for s in pick_sources(_offsets(graph), seed + g, case["per_graph"])]
        pack = MultiGraph(graphs)
        budget = int(sum(graphs[g].nodes for g, _ in queries) * 8 * 1.05) + (1 << 20)
        engine = MultiSourceBFS(pack, budget, len(queries) + 8)
        engine.set_levels_per_step(4)
        return {"kind": kind, "pack": pack, "engine": engine, "queries": queries}
    if kind == "build":
        gen = _generator(seed)
        rows = _ids(case["edges"], case["scale"], gen).to(torch.int32).cpu().numpy()
        cols = _ids(case["edges"], case["scale"], gen).to(torch.int32).cpu().numpy()
        # The caller's host CSR, with room for a graph without duplicates.
        most = case["edges"] * (2 if case["symmetrize"] else 1)
        return {"kind": kind, "nodes": 1 << case["scale"], "rows": rows, "cols": cols,
                "symmetrize": case["symmetrize"], "offsets": np.zeros((1 << case["scale"]) + 1, np.int32),
                "columns": np.zeros(most, np.int32)}
    gen = _generator(seed)
    n = case["n"]
    if kind == "sort":
        dtype = np.dtype(KEY_TYPES[case["key"]])
        word = torch.int32 if dtype.itemsize == 4 else torch.int64
        if case["dist"] == "ids":
            keys = _ids(n, case["bits"], gen).to(word)
        elif dtype.kind == "f":
            keys = torch.randn(n, generator=gen, device="cuda",
                               dtype=torch.float32 if dtype.itemsize == 4 else torch.float64).view(word)
        else:
            lim = torch.iinfo(word)
            keys = torch.randint(lim.min, lim.max, (n,), generator=gen, device="cuda", dtype=word)
        values = torch.arange(n, device="cuda", dtype=torch.int32) if case["values"] else None
        storage = radix_sort.DoubleBuffer(dtype, n, with_values=case["values"])
        return {"kind": kind, "keys": keys, "values": values, "storage": storage, "n": n, "bits": case["bits"],
                "enactor": radix_sort.Enactor(),
                "d_keys": [_array(a, n, dtype.itemsize) for a in storage.d_keys],
                "d_values": [_array(a, n, 4) for a in storage.d_values] if case["values"] else None}
    if kind == "trim":
        # Sorted packed edges: runs of 1 .. 2 * run - 1 equal keys.
        heads = torch.rand(n, generator=gen, device="cuda") * case["run"] < 1.0
        storage = radix_sort.DoubleBuffer(np.uint64, n, with_values=case["values"])
        keys = [_array(a, n, 8) for a in storage.d_keys]
        keys[0].copy_(torch.cumsum(heads, 0) * 2654435761)
        keys[1].zero_()  # the entries past the compacted count are never written
        values = [_array(a, n, 4) for a in storage.d_values] if case["values"] else None
        if values:
            values[0].copy_(torch.randint(0, 1 << 30, (n,), generator=gen, device="cuda", dtype=torch.int32))
            values[1].zero_()
        return {"kind": kind, "storage": storage, "n": n, "enactor": primitives.ConsecutiveRemoval(), "d_keys": keys,
                "d_values": values}
    src, dst = radix_sort.DeviceArray(4 * n), radix_sort.DeviceArray(4 * n)
    # Row lengths: mostly short, a few hubs.
    u = torch.rand(n, generator=gen, device="cuda")
    _array(src, n, 4).copy_((8.0 / (u + 1e-3)).to(torch.int32))
    return {"kind": kind, "src": src, "dst": dst, "n": n, "exclusive": case["exclusive"], "enactor": primitives.Scan(),
            "out": _array(dst, n, 4)}


def run(state):
    kind = state["kind"]
    if kind == "search":
        problem = state["problem"]
        check(problem.Reset(state["frontier"]))
        check(state["enactor"].EnactSearch(problem, state["source"]))
        with torch.cuda.stream(state["stream"]):
            parent_depth = torch.index_select(state["depth"], 0, state["pred"].clamp(min=0))
        return {"depth": state["depth"], "parent_depth": parent_depth}
    if kind == "batch":
        engine = state["engine"]
        ids = [engine.submit(g, s) for g, s in state["queries"]]
        engine.run()
        engine.poll()
        got = [engine.result(q, g, want_pred=False) for q, (g, _) in zip(ids, state["queries"])]
        return {"depth": np.concatenate([d for d, _, _ in got]), "levels": np.array([x for _, _, x in got], np.int32)}
    if kind == "build":
        graph = bfs.Graph.from_coo_unique(state["nodes"], state["rows"], state["cols"], drop_self_loops=True,
                                          symmetrize=state["symmetrize"])
        check(lib().b40c_graph_copy_to_host(graph.handle, ptr(state["offsets"]), ptr(state["columns"])))
        graph.close()
        return {"edges": graph.edges, "offsets": state["offsets"], "columns": state["columns"]}
    storage = state.get("storage")
    if kind == "sort":
        # The sort works in place on the double buffer, on the enactor's own
        # stream: the caller fills the buffer and waits for that first.
        state["d_keys"][0].copy_(state["keys"])
        if state["d_values"]:
            state["d_values"][0].copy_(state["values"])
        torch.cuda.current_stream().synchronize()
        storage.selector = 0
        check(state["enactor"].Sort(storage, state["n"], 0, state["bits"]))
        out = {"keys": state["d_keys"][storage.selector]}
        if state["d_values"]:
            out["values"] = state["d_values"][storage.selector]
        return out
    if kind == "trim":
        storage.selector = 0
        count = state["enactor"].Trim(storage, state["n"])
        out = {"count": count, "keys": state["d_keys"][1]}
        if state["d_values"]:
            out["values"] = state["d_values"][1]
        return out
    total = state["enactor"].Scan(state["dst"], state["src"], state["n"], state["exclusive"])
    return {"out": state["out"], "total": total}


def work(case):
    kind = case["kind"]
    if kind == "search":
        # Row offsets and columns read once, depth and predecessor written once.
        if case["graph"] == "rmat":
            v = 1 << case["size"]
            e = 2 * case["edge_factor"] * v * 0.93  # both directions, duplicates removed
        else:
            w = case["size"]
            v, e = w ** 3, 6 * (w ** 3 - w ** 2)
        return {"bytes": 4 * v + 4 * e + 8 * v, "flops": 0}
    if kind == "batch":
        # Every graph's CSR read once, each query's depth and predecessor written once.
        scales = range(case["scale_lo"], case["scale_hi"] + 1)
        v = case["graphs"] * sum(1 << s for s in scales) / len(scales)
        return {"bytes": 4 * v + 4 * 30 * v + 8 * v * case["per_graph"], "flops": 0}
    if kind == "build":
        e = case["edges"] * (2 if case["symmetrize"] else 1)
        return {"bytes": 8 * case["edges"] + 4 * e + (4 << case["scale"]), "flops": 0}
    n = case["n"]
    if kind == "sort":
        return {"bytes": 2 * n * (np.dtype(KEY_TYPES[case["key"]]).itemsize + (4 if case["values"] else 0)),
                "flops": 0}
    if kind == "trim":
        element = 8 + (4 if case["values"] else 0)
        return {"bytes": n * element * (1 + 1 / case["run"]), "flops": 0}
    return {"bytes": 8 * n, "flops": 0}


def exact(case, seed):
    """Every output is a whole number, compared for equality."""
    return None
