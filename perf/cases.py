"""Performance cases: the work users have this library do, timed through its public entry points.

listed() names the cases, draw() makes more of the same ranges.  Kinds:

search     one breadth-first search on a resident graph: CsrProblem.enact, the depth labels (or the
           predecessors) read where the program uses them: in device memory on large graphs (through
           bfs_problem_device_arrays), on the host on small ones
batch      queries over a pool of graphs in one Batch.enact, every query's depths read back
from_coo   host (source, destination) pairs -> device CSR, symmetrised, deduplicated, without loops
transpose  the in-neighbour CSR of a device CSR
scan       ScanEnactor.scan of uint32 words in device memory
copy_if    ScanEnactor.copy_if of uint32 words in device memory
"""
import ctypes
import math

import numpy as np
import torch

import back40computing_amd as b40c
from back40computing_amd import _native, primitives
from back40computing_amd.batch import Batch, GraphPool

STRATEGIES = {"expand_contract": b40c.EXPAND_CONTRACT, "contract_expand": b40c.CONTRACT_EXPAND,
              "two_phase": b40c.TWO_PHASE, "hybrid": b40c.HYBRID,
              "direction_optimizing": b40c.DIRECTION_OPTIMIZING}
HOST_RESULT_NODES = 1 << 17  # searches of at most this many vertices hand their labels to the host


def listed():
    return [
        # the smallest call: one interactive query on a small social graph, answer on the host
        {"name": "rmat10_do", "kind": "search", "graph": "rmat", "scale": 10, "ef": 16,
         "strategy": "direction_optimizing", "pred": False, "fused": True},
        # an ordinary directed graph of odd size (bottom-up levels read the in-neighbour CSR)
        {"name": "directed_100k_do", "kind": "search", "graph": "directed", "nodes": 100003, "edges": 1600033,
         "strategy": "direction_optimizing", "pred": False, "fused": True},
        # the headline workload: R-MAT scale 22, edge factor 16, direction-optimizing
        {"name": "rmat22_do", "kind": "search", "graph": "rmat", "scale": 22, "ef": 16,
         "strategy": "direction_optimizing", "pred": False, "fused": True},
        # the top-down search of the same family (graphs without an in-neighbour order worth having)
        {"name": "rmat20_ec", "kind": "search", "graph": "rmat", "scale": 20, "ef": 16,
         "strategy": "expand_contract", "pred": False, "fused": True},
        # the reference driver's default strategy: edge frontiers, persistent and per-level launches
        {"name": "rmat20_hybrid", "kind": "search", "graph": "rmat", "scale": 20, "ef": 16,
         "strategy": "hybrid", "pred": False, "fused": True},
        # predecessors: the parent array of a hierarchy (unique parents)
        {"name": "tree_1m_tp_pred", "kind": "search", "graph": "tree", "nodes": 1000003,
         "strategy": "two_phase", "pred": True, "fused": True},
        # high diameter: a road-like lattice, 1999 levels
        {"name": "grid2d_1000_ec", "kind": "search", "graph": "grid2d", "width": 1000,
         "strategy": "expand_contract", "pred": False, "fused": True},
        # high diameter, wide levels: a 3D mesh, 898 levels
        {"name": "grid3d_300_ce", "kind": "search", "graph": "grid3d", "width": 300,
         "strategy": "contract_expand", "pred": False, "fused": True},
        # many queries over a pool of resident graphs, answers on the host
        {"name": "batch_64q_16g", "kind": "batch", "graphs": 16, "queries": 64, "scale_lo": 14, "scale_hi": 17,
         "ef_lo": 8, "ef_hi": 32, "direction": True},
        # graph ingest: host pairs to a device CSR
        {"name": "from_coo_4m", "kind": "from_coo", "nodes": 1 << 18, "pairs": 4000037},
        # a resident graph's transpose (directed graphs entering a pool)
        {"name": "transpose_16m", "kind": "transpose", "nodes": 1 << 20, "pairs": 16000057},
        # the scan primitive on a large odd length
        {"name": "scan_67m", "kind": "scan", "n": (1 << 26) + 12345, "exclusive": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["search"] * 6 + ["batch", "from_coo", "transpose", "scan", "copy_if"])
    if kind == "search":
        c = {"kind": kind, "graph": rng.choice(["rmat", "rmat", "directed", "tree", "grid2d", "grid3d"])}
        if c["graph"] == "rmat":
            c["scale"] = rng.randint(9, 20)
            c["ef"] = rng.randint(4, 32)
        elif c["graph"] == "directed":
            c["nodes"] = _log_int(rng, 500, 2000000) | 1
            c["edges"] = int(c["nodes"] * rng.uniform(2.0, 24.0))
        elif c["graph"] == "tree":
            c["nodes"] = _log_int(rng, 500, 4000000)
        elif c["graph"] == "grid2d":
            c["width"] = _log_int(rng, 20, 1000)
        else:
            c["width"] = _log_int(rng, 10, 200)
        c["strategy"] = rng.choice(sorted(STRATEGIES))
        c["pred"] = c["graph"] == "tree"
        # searches with a launch per level, on graphs of few levels
        c["fused"] = c["graph"] in ("grid2d", "grid3d") or c["strategy"] == "hybrid" or rng.random() < 0.85
        return c
    if kind == "batch":
        lo = rng.randint(10, 16)
        return {"kind": kind, "graphs": rng.randint(1, 16), "queries": _log_int(rng, 1, 64), "scale_lo": lo,
                "scale_hi": rng.randint(lo, 17), "ef_lo": 8, "ef_hi": rng.randint(8, 32),
                "direction": rng.random() < 0.8}
    if kind == "from_coo":
        return {"kind": kind, "nodes": _log_int(rng, 1000, 1 << 21), "pairs": _log_int(rng, 1000, 8000000)}
    if kind == "transpose":
        return {"kind": kind, "nodes": _log_int(rng, 1000, 1 << 21), "pairs": _log_int(rng, 1000, 16000000)}
    if kind == "scan":
        return {"kind": kind, "n": _log_int(rng, 1, 1 << 26), "exclusive": rng.random() < 0.5}
    return {"kind": kind, "n": _log_int(rng, 1, 1 << 26), "keep": rng.choice([0.02, 0.5, 0.97])}


class _DeviceInts:
    """int32 device memory of the library, for torch.as_tensor (no copy); keeps its owner alive."""

    def __init__(self, ptr, n, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<i4", "data": (ptr, False), "version": 2}


def _view(ptr, n, owner):
    if n == 0:
        return torch.empty(0, dtype=torch.int32, device="cuda")
    return torch.as_tensor(_DeviceInts(ptr, n, owner), device="cuda")


def _rmat(scale, ef, seed):
    """Host CSR of an R-MAT graph, built on the device."""
    d = primitives.DeviceCsr.rmat(scale, ef, seed=seed)
    g = d.to_host()
    d.free()
    return g


def _tree(n, seed):
    """Random recursive tree: vertex v > 0 hangs below a vertex drawn from those before it."""
    rng = np.random.default_rng(seed)
    child = np.arange(1, n, dtype=np.int64)
    parent = (rng.random(n - 1) * child).astype(np.int64)
    label = rng.permutation(n)
    d = primitives.DeviceCsr.from_coo(n, label[child].astype(np.int32), label[parent].astype(np.int32),
                                      symmetrize=True)
    g = d.to_host()
    d.free()
    return g


def _host_graph(case, seed):
    if case["graph"] == "rmat":
        return _rmat(case["scale"], case["ef"], seed)
    if case["graph"] == "tree":
        return _tree(case["nodes"], seed)
    if case["graph"] == "grid2d":
        return b40c.CsrGraph.grid2d(case["width"])
    if case["graph"] == "grid3d":
        return b40c.CsrGraph.grid3d(case["width"])
    return b40c.CsrGraph.random(case["nodes"], case["edges"], seed=seed)


def _source(case, g, seed):
    """A source vertex: non-isolated, and on a lattice near a corner (the full diameter)."""
    if case["graph"] == "grid2d":
        w = case["width"]
        return (seed % 7) % w * w + (seed // 7 % 7) % w
    if case["graph"] == "grid3d":
        w = case["width"]
        return ((seed % 7) % w * w + (seed // 7 % 7) % w) * w
    return int(g.sample_sources(1, seed=seed)[0])


def _pairs(case, seed):
    """Host pairs with a heavy-tailed endpoint distribution (hubs, duplicates and some loops); the seed
    numbers the vertices, so every seed has as many distinct pairs."""
    n, m = case["nodes"], case["pairs"]
    rng = np.random.default_rng(n + m)
    src = np.minimum((n * rng.random(m) ** 3).astype(np.int32), n - 1)
    dst = np.minimum((n * rng.random(m) ** 2).astype(np.int32), n - 1)
    label = np.random.default_rng(seed).permutation(n).astype(np.int32)
    return label[src], label[dst]


def _words(n, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    return torch.randint(0, 1 << 16, (n,), dtype=torch.int32, device="cuda", generator=gen)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "search":
        g = _host_graph(case, seed)
        p = b40c.CsrProblem(mark_predecessors=case["pred"]).from_host_problem(g)
        strategy = STRATEGIES[case["strategy"]]
        p.reset(_native.load().bfs_strategy_frontier_type(strategy))
        state = {"case": case, "problem": p, "strategy": strategy, "src": _source(case, g, seed), "depths": None}
        if g.nodes > HOST_RESULT_NODES and not case["pred"]:
            ptr = ctypes.c_void_p()
            rc = _native.load().bfs_problem_device_arrays(p._h, None, None, None, None, ctypes.byref(ptr))
            assert rc == 0
            state["depths"] = _view(ptr.value, g.nodes, p)
        return state
    if kind == "batch":
        pool = GraphPool()
        src = []
        hosts = []
        scales = range(case["scale_lo"], case["scale_hi"] + 1)
        efs = range(case["ef_lo"], case["ef_hi"] + 1)
        for k in range(case["graphs"]):
            d = primitives.DeviceCsr.rmat(scales[k % len(scales)], efs[5 * k % len(efs)], seed=seed + k)
            pool.add_device(d)
            hosts.append(d.to_host())
            d.free()
        # the queries' graphs in an order that mixes large and small ones
        gids = (np.arange(case["queries"]) * 7 % case["graphs"]).astype(np.int32)
        for q, gid in enumerate(gids):
            src.append(hosts[gid].sample_sources(1, seed=seed + 1000 + q)[0])
        return {"case": case, "pool": pool, "batch": Batch(pool, max_queries=case["queries"]), "gids": gids,
                "src": np.array(src, np.int32)}
    if kind == "from_coo":
        src, dst = _pairs(case, seed)
        return {"case": case, "src": src, "dst": dst}
    if kind == "transpose":
        src, dst = _pairs(case, seed)
        return {"case": case, "graph": primitives.DeviceCsr.from_coo(case["nodes"], src, dst)}
    a = _words(case["n"], seed)
    return {"case": case, "scan": primitives.ScanEnactor(), "in": a, "out": torch.zeros_like(a)}


def _csr_out(d):
    return [_view(d._s.row_offsets, d.nodes + 1, d), _view(d._s.column_indices, d.edges, d)]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "search":
        p = state["problem"]
        st = p.enact(state["strategy"], state["src"], fused=case["fused"])
        labels = state["depths"] if state["depths"] is not None else p.extract_results()
        return [labels, st.search_depth]
    if kind == "batch":
        b = state["batch"]
        b.enact(state["gids"], state["src"], direction_optimizing=case["direction"])
        return [b.depths(q) for q in range(case["queries"])]
    if kind == "from_coo":
        return _csr_out(primitives.DeviceCsr.from_coo(case["nodes"], state["src"], state["dst"], symmetrize=True,
                                                      dedup=True, drop_self_loops=True))
    if kind == "transpose":
        return _csr_out(state["graph"].transpose())
    a, out = state["in"], state["out"]
    if kind == "scan":
        total = state["scan"].scan(a.data_ptr(), out.data_ptr(), case["n"], exclusive=case["exclusive"])
        return [out, total]
    kept = state["scan"].copy_if(a.data_ptr(), out.data_ptr(), case["n"], op=primitives.SELECT_LESS,
                                 comparand=int(case["keep"] * (1 << 16)))
    return [out, kept]


def work(case):
    """Bytes: the CSR read once and the labels written once; pairs read, CSR written; words read and written."""
    kind = case["kind"]
    if kind == "search":
        if case["graph"] == "rmat":
            v, e = 1 << case["scale"], 1.8 * case["ef"] * (1 << case["scale"])
        elif case["graph"] == "directed":
            v, e = case["nodes"], case["edges"]
        elif case["graph"] == "tree":
            v, e = case["nodes"], 2 * (case["nodes"] - 1)
        elif case["graph"] == "grid2d":
            v = case["width"] ** 2
            e = 4 * v
        else:
            v = case["width"] ** 3
            e = 6 * v
        return {"bytes": 4.0 * e + 8.0 * v, "flops": 0}
    if kind == "batch":
        v = 2.0 ** (0.5 * (case["scale_lo"] + case["scale_hi"]))
        e = 0.9 * (case["ef_lo"] + case["ef_hi"]) * v
        return {"bytes": case["queries"] * (4.0 * e + 8.0 * v), "flops": 0}
    if kind == "from_coo":
        return {"bytes": 8.0 * case["pairs"] + 4.0 * case["nodes"] + 8.0 * case["pairs"], "flops": 0}
    if kind == "transpose":
        return {"bytes": 8.0 * case["pairs"] + 8.0 * case["nodes"], "flops": 0}
    if kind == "scan":
        return {"bytes": 8.0 * case["n"], "flops": 0}
    return {"bytes": 4.0 * case["n"] * (1.0 + case["keep"]), "flops": 0}


def _exact_search(row, col, src, pred):
    """Level-synchronous search with torch operations over the whole edge list."""
    n = len(row) - 1
    row, col = (torch.from_numpy(np.array(x)).cuda().long() for x in (row, col))
    owner = torch.repeat_interleave(torch.arange(n, device="cuda"), row[1:] - row[:-1])
    depth = torch.full((n,), -1, dtype=torch.int64, device="cuda")
    depth[src] = 0
    level = 0
    while True:
        hit = col[depth[owner] == level]
        hit = hit[depth[hit] < 0]
        if hit.numel() == 0:
            break
        level += 1
        depth[hit] = level
    if not pred:
        return [depth.int(), level + 1]
    parent = torch.full((n,), -1, dtype=torch.int64, device="cuda")
    up = (depth[owner] >= 0) & (depth[col] == depth[owner] + 1)
    parent[col[up]] = owner[up]
    parent[src] = -2
    return [parent.int(), level + 1]


def _exact_csr(n, row, col, dedup):
    key = row.long() * n + col.long()
    key = torch.unique(key) if dedup else torch.sort(key).values
    out = torch.zeros(n + 1, dtype=torch.int64, device=key.device)
    out[1:] = torch.cumsum(torch.bincount(key // n, minlength=n), 0)
    return [out.int(), (key % n).int()]


def exact(case, seed):
    """The outputs (all whole numbers) by plain torch; None where the repeated passes over the edge list
    would take long (a mesh has hundreds of levels, a batch many graphs)."""
    kind = case["kind"]
    if kind == "search":
        if case["graph"] in ("grid2d", "grid3d"):
            return None
        g = _host_graph(case, seed)
        return _exact_search(g.row_offsets, g.column_indices, _source(case, g, seed), case["pred"])
    if kind == "batch":
        return None
    if kind == "from_coo":
        src, dst = (torch.from_numpy(x).cuda() for x in _pairs(case, seed))
        keep = src != dst
        src, dst = src[keep], dst[keep]
        return _exact_csr(case["nodes"], torch.cat([src, dst]), torch.cat([dst, src]), True)
    if kind == "transpose":
        src, dst = (torch.from_numpy(x).cuda() for x in _pairs(case, seed))
        return _exact_csr(case["nodes"], dst, src, False)
    a = _words(case["n"], seed)
    out = torch.zeros_like(a)
    if kind == "copy_if":
        kept = a[a < int(case["keep"] * (1 << 16))]
        out[: kept.numel()] = kept
        return [out, kept.numel()]
    sums = torch.cumsum(a.long(), 0)
    out64 = sums - a.long() if case["exclusive"] else sums
    out64 = out64 & 0xFFFFFFFF
    return [torch.where(out64 >= 1 << 31, out64 - (1 << 32), out64).int(), int(sums[-1]) & 0xFFFFFFFF]
