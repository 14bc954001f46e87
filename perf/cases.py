"""Timed cases of the frontier engine, through its public entry points.

A case names an operation and its sizes:

  bfs            single-source hop distances (Graph.bfs)
  build_bfs      edge list on the device -> graph, one traversal, graph freed
  sssp           single-source int32 min-plus distances (Graph.sssp)
  mssp           multi-source distance rows and sums (Graph.mssp), unweighted
                 or int32-weighted
  apsp           a block of consecutive sources (dawn_apsp_block)
  closeness      sums and closeness of a set of vertices, no rows (Graph.closeness)
  batch          many graphs of uneven size in one call (dawn_batch_mssp)

Graphs are the families the engine's workloads use: Erdos-Renyi, RMAT
(.57, .19, .19, .05), and 4-neighbour grids with 1% random long-range edges;
undirected ones hold both directions of every pair, directed ones the pairs as
drawn; duplicates and self-loops are dropped; weights are uniform in [1, 1000].
Edge lists and sources are drawn from the seed with torch and numpy.  Distance
rows stay in device memory, where the next stage of a program reads them.
"""
import ctypes
import importlib.util
import json
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "gal-dawn_amd")
WMAX = 1000


def _package():
    """gal-dawn_amd/ as module gal_dawn_amd, with the shipped launch knobs and
    scheduler networks installed, as the benchmark installs them."""
    if "gal_dawn_amd" in sys.modules:
        return sys.modules["gal_dawn_amd"]
    spec = importlib.util.spec_from_file_location(
        "gal_dawn_amd", os.path.join(PKG, "__init__.py"), submodule_search_locations=[PKG])
    mod = importlib.util.module_from_spec(spec)
    sys.modules["gal_dawn_amd"] = mod
    spec.loader.exec_module(mod)
    mod.tune_load(os.path.join(PKG, "tune_cache.txt"))
    for name, single in (("sched_mlp.json", False), ("sched_mlp_single.json", True)):
        with open(os.path.join(PKG, name)) as f:
            w = json.load(f)
        mod.sched_set_mlp(np.array(w["params"], np.float32), np.array(w["mean"], np.float32),
                          np.array(w["inv_std"], np.float32), single=single)
    return mod


# ---- cases -------------------------------------------------------------------

def listed():
    return [
        # A query on a small graph: a handful of short steps, launches count.
        {"name": "bfs_er65k", "op": "bfs", "family": "er", "size": 65536, "degree": 8,
         "weighted": False, "directed": False, "policy": "fixed"},
        # A query on a large skewed graph, the trained step scheduler choosing.
        {"name": "bfs_rmat22", "op": "bfs", "family": "rmat", "size": 22, "degree": 16,
         "weighted": False, "directed": False, "policy": "learned"},
        # A program that gets an edge list, builds the graph and asks once.
        {"name": "build_bfs_rmat20", "op": "build_bfs", "family": "rmat", "size": 20, "degree": 16,
         "weighted": False, "directed": False, "policy": "fixed"},
        # Weighted road-like network: high diameter, many dependent steps.
        {"name": "sssp_grid2048", "op": "sssp", "family": "grid", "size": 2048, "degree": 4,
         "weighted": True, "directed": False, "policy": "fixed"},
        # A small multi-source request: source 0 and 64 more, one narrow batch.
        {"name": "mssp_er65k", "op": "mssp", "family": "er", "size": 65536, "degree": 8,
         "weighted": False, "directed": False, "policy": "fixed", "sources": 65},
        # The ordinary bulk job: 4096 uniform sources of a social-network-like graph.
        {"name": "mssp_rmat20", "op": "mssp", "family": "rmat", "size": 20, "degree": 16,
         "weighted": False, "directed": False, "policy": "learned", "sources": 4096},
        # The largest: 34 GB of distance rows over a graph of about 130 M edges.
        {"name": "mssp_rmat22", "op": "mssp", "family": "rmat", "size": 22, "degree": 16,
         "weighted": False, "directed": False, "policy": "learned", "sources": 2048},
        # Centrality of a block of vertices: sums only.
        {"name": "closeness_rmat20", "op": "closeness", "family": "rmat", "size": 20, "degree": 16,
         "weighted": False, "directed": False, "policy": "fixed", "sources": 4096},
        # Several weighted queries at once on the road-like network.
        {"name": "mssp_grid2048_weighted", "op": "mssp", "family": "grid", "size": 2048, "degree": 4,
         "weighted": True, "directed": False, "policy": "fixed", "sources": 16},
        # A block of weighted all-pairs on a small graph: batches of 64 sources.
        {"name": "apsp_er16k_weighted", "op": "apsp", "family": "er", "size": 16384, "degree": 8,
         "weighted": True, "directed": False, "policy": "fixed", "sources": 256},
        # Many small and middling graphs served in one call, hop counts.
        {"name": "batch512", "op": "batch", "weighted": False, "graphs": 512, "sources": 8,
         "nmax": 130000},
        # The same with weights.
        {"name": "batch512_weighted", "op": "batch", "weighted": True, "graphs": 512, "sources": 8,
         "nmax": 130000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges: any operation, family, direction,
    policy; sizes spread over their logarithm, odd ones among them."""
    op = rng.choice(["bfs", "bfs", "build_bfs", "sssp", "mssp", "mssp", "wmssp", "apsp", "closeness",
                     "batch", "wbatch"])
    if op in ("batch", "wbatch"):
        return {"op": "batch", "weighted": op == "wbatch", "graphs": _log_int(rng, 8, 400),
                "sources": rng.choice([1, 3, 4, 8, 8, 11, 16]) if op == "batch" else rng.choice([1, 3, 5, 8]),
                "nmax": _log_int(rng, 5000, 130000)}
    family = rng.choice(["er", "rmat", "grid"])
    weighted = op in ("sssp", "wmssp") or (op in ("apsp", "build_bfs") and rng.random() < 0.5)
    if op in ("bfs", "build_bfs", "sssp"):
        nmax, sources = (1 << 21 if op == "build_bfs" else 1 << 22), 1
    elif weighted:
        sources = _log_int(rng, 2, 100)
        nmax = min(1 << 20, (1 << 26) // sources)
    else:
        sources = _log_int(rng, 2, 4096)
        nmax = min(1 << 21, (1 << 31) // sources)
    n = _log_int(rng, 1500, nmax)
    if op == "apsp":
        sources = min(sources, n)
    if family == "rmat":
        size, degree = max(10, int(math.log2(n))), rng.choice([8, 16])
    elif family == "grid":
        size, degree = max(32, int(math.sqrt(n))), 4
    else:
        size, degree = n, rng.randint(4, 16)
    case = {"op": "mssp" if op == "wmssp" else op, "family": family, "size": size, "degree": degree,
            "weighted": weighted, "directed": rng.random() < 0.25,
            "policy": rng.choice(["fixed", "fixed", "learned"])}
    if sources > 1:
        case["sources"] = sources
    return case


def _vertices(case):
    size = case["size"]
    return {"er": size, "rmat": 1 << size, "grid": size * size}[case["family"]]


def _pairs_count(family, size, degree):
    """Pairs drawn before duplicates and self-loops are dropped."""
    if family == "er":
        return int(round(size * degree / 2.0))
    if family == "rmat":
        return degree << size
    edges = 2 * size * (size - 1)
    return edges + int(round(0.01 * edges))


# ---- inputs ------------------------------------------------------------------

def _pairs(family, size, degree, gen):
    """(u, v) of a graph family as int32 device tensors."""
    dev = "cuda"
    if family == "er":
        count = _pairs_count(family, size, degree)
        uv = torch.randint(0, size, (2, count), generator=gen, device=dev, dtype=torch.int32)
        return uv[0].contiguous(), uv[1].contiguous()
    if family == "rmat":
        count = _pairs_count(family, size, degree)
        u = torch.zeros(count, dtype=torch.int32, device=dev)
        v = torch.zeros(count, dtype=torch.int32, device=dev)
        for _ in range(size):  # quadrants a, b, c, d with .57, .19, .19, .05
            x = torch.rand(count, generator=gen, device=dev)
            down = x >= 0.76
            u.mul_(2).add_(down)
            v.mul_(2).add_(((x >= 0.57) & ~down) | (x >= 0.95))
        return u, v
    ids = torch.arange(size * size, dtype=torch.int32, device=dev).reshape(size, size)
    extra = _pairs_count(family, size, degree) - 2 * size * (size - 1)
    far = torch.randint(0, size * size, (2, extra), generator=gen, device=dev, dtype=torch.int32)
    u = torch.cat([ids[:, :-1].reshape(-1), ids[:-1].reshape(-1), far[0]])
    v = torch.cat([ids[:, 1:].reshape(-1), ids[1:].reshape(-1), far[1]])
    return u, v


def _edges(case, seed):
    """Edge list and sources of a one-graph case, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 1000003 + 17)
    n = _vertices(case)
    u, v = _pairs(case["family"], case["size"], case["degree"], gen)
    w = None
    if case["weighted"]:
        w = torch.randint(1, WMAX + 1, (u.numel(),), generator=gen, device="cuda", dtype=torch.int32)
    rng = np.random.default_rng([int(seed), 5])
    count = case.get("sources", 1)
    if case["op"] == "apsp":  # a block of consecutive vertices
        first = int(rng.integers(n - count + 1))
        sources = np.arange(first, first + count, dtype=np.int32)
    elif count > 1:           # uniform vertices, isolated ones among them
        sources = rng.integers(0, n, count).astype(np.int32)
    else:                     # a vertex with an out-edge
        live = torch.nonzero(u != v).reshape(-1)
        sources = np.array([int(u[live[int(rng.integers(live.numel()))]])], np.int32)
    return n, u, v, w, sources


def _device_array(dawn, t):
    a = dawn.DeviceArray(t.numel(), np.int32)
    if dawn.lib().dawn_memcpy(ctypes.c_void_p(a.data_ptr()), ctypes.c_void_p(t.data_ptr()), a.nbytes):
        raise RuntimeError("dawn_memcpy")
    torch.cuda.synchronize()  # a device-to-device copy may return before it is done
    return a


def _graph(dawn, n, u, v, w, directed):
    return dawn.Graph.from_edges_device(n, _device_array(dawn, u), _device_array(dawn, v),
                                        None if w is None else _device_array(dawn, w),
                                        symmetrize=not directed, dedup=True)


def _batch_plan(case):
    """Families and sizes of a batch: vertex counts log-uniform in
    [1000, nmax], ER of average degree 4-32, RMAT of scale 10-17 with 16
    pairs per vertex, grids of side 64-362.  The edges and sources come from
    the seed, the sizes from the case."""
    rng = np.random.default_rng([case["graphs"], case["nmax"], 4])
    plan = []
    for _ in range(case["graphs"]):
        n = math.exp(rng.uniform(math.log(1000), math.log(case["nmax"])))
        family = int(rng.integers(3))
        degree = int(rng.integers(4, 33))
        if family == 0:
            plan.append(("er", int(round(n)), degree))
        elif family == 1:
            plan.append(("rmat", int(min(17, max(10, round(math.log2(n))))), 16))
        else:
            plan.append(("grid", int(min(362, max(64, round(math.sqrt(n))))), 4))
    return plan


def _prepare_batch(dawn, case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed) * 1000003 + 29)
    rng = np.random.default_rng([int(seed), 7])
    graphs, sources = [], []
    for family, size, degree in _batch_plan(case):
        u, v = _pairs(family, size, degree, gen)
        n = _vertices({"family": family, "size": size})
        w = None
        if case["weighted"]:
            w = torch.randint(1, WMAX + 1, (u.numel(),), generator=gen, device="cuda", dtype=torch.int32)
        graphs.append(_graph(dawn, n, u, v, w, False))
        sources.append(rng.integers(0, n, case["sources"]))
    sizes = np.array([g.n * case["sources"] for g in graphs], np.int64)
    offsets = np.zeros(len(graphs), np.int64)
    offsets[1:] = np.cumsum(sizes)[:-1]
    return {"op": "batch", "dawn": dawn, "graphs": graphs,
            "handles": (ctypes.c_void_p * len(graphs))(*[g.handle.value for g in graphs]),
            "sources": np.concatenate(sources).astype(np.int32), "count": case["sources"],
            "offsets": offsets, "out": torch.empty(int(sizes.sum()), dtype=torch.int32, device="cuda")}


def prepare(case, seed):
    dawn = _package()
    if case["op"] == "batch":
        return _prepare_batch(dawn, case, seed)
    n, u, v, w, sources = _edges(case, seed)
    state = {"op": case["op"], "dawn": dawn, "n": n, "sources": sources, "policy": case["policy"],
             "weighted": case["weighted"], "directed": case["directed"]}
    if case["op"] == "build_bfs":
        state["u"], state["v"] = _device_array(dawn, u), _device_array(dawn, v)
        state["w"] = None if w is None else _device_array(dawn, w)
        state["out"] = torch.empty(n, dtype=torch.int32, device="cuda")
        return state
    state["graph"] = _graph(dawn, n, u, v, w, case["directed"])
    del u, v, w
    torch.cuda.empty_cache()
    if case["op"] in ("bfs", "sssp"):
        state["out"] = torch.empty(n, dtype=torch.int32, device="cuda")
    elif case["op"] != "closeness":
        state["out"] = torch.empty((len(sources), n), dtype=torch.int32, device="cuda")
    return state


# ---- one pass ----------------------------------------------------------------

def _i32p(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int32))


def _i64p(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_int64))


def run(state):
    op, dawn = state["op"], state["dawn"]
    if op == "bfs":
        return state["graph"].bfs(int(state["sources"][0]), policy=state["policy"], out=state["out"])
    if op == "sssp":
        return state["graph"].sssp(int(state["sources"][0]), policy=state["policy"], out=state["out"])
    if op == "build_bfs":
        g = dawn.Graph.from_edges_device(state["n"], state["u"], state["v"], state["w"],
                                         symmetrize=not state["directed"], dedup=True)
        d, st = g.bfs(int(state["sources"][0]), policy=state["policy"], out=state["out"], stats=True)
        g.close()
        return d, g.m, st["vertices_reached"], st["edges_reached"]
    if op == "mssp":
        return state["graph"].mssp(state["sources"], policy=state["policy"], out=state["out"])
    if op == "apsp":
        # Rows into device memory: the C entry point (the Python method returns host rows).
        src = state["sources"]
        sums = np.zeros(len(src), np.int64)
        rc = dawn.lib().dawn_apsp_block(state["graph"].handle, int(src[0]), len(src),
                                        ctypes.c_void_p(state["out"].data_ptr()), _i64p(sums),
                                        dawn.POLICIES[state["policy"]], None)
        if rc:
            raise RuntimeError("dawn_apsp_block: %d" % rc)
        return state["out"], sums
    if op == "closeness":
        return state["graph"].closeness(state["sources"], policy=state["policy"])
    st = dawn.Stats()
    rc = dawn.lib().dawn_batch_mssp(state["handles"], len(state["graphs"]), _i32p(state["sources"]),
                                    state["count"], ctypes.c_void_p(state["out"].data_ptr()),
                                    _i64p(state["offsets"]), ctypes.byref(st))
    if rc:
        raise RuntimeError("dawn_batch_mssp: %d" % rc)
    return state["out"], int(st.skipped_sources)


# ---- what a pass cannot do without -------------------------------------------

def work(case):
    """Bytes: offsets, columns and weights once, every distance and sum once
    (edge counts before duplicates are dropped); a build also reads the pairs
    and writes the arrays.  The path computes no products: no flops."""
    if case["op"] == "batch":
        total = 0
        for family, size, degree in _batch_plan(case):
            n = _vertices({"family": family, "size": size})
            m = 2 * _pairs_count(family, size, degree)
            total += 4 * (n + 1) + (8 if case["weighted"] else 4) * m + 4 * n * case["sources"]
        return {"bytes": total, "flops": 0}
    n = _vertices(case)
    pairs = _pairs_count(case["family"], case["size"], case["degree"])
    m = pairs * (1 if case["directed"] else 2)
    graph = 4 * (n + 1) + (8 if case["weighted"] else 4) * m
    count = case.get("sources", 1)
    if case["op"] == "closeness":
        return {"bytes": graph + 24 * count, "flops": 0}
    rows = 4 * n * count + (8 * count if count > 1 else 0)
    build = (12 if case["weighted"] else 8) * pairs + graph if case["op"] == "build_bfs" else 0
    return {"bytes": graph + rows + build, "flops": 0}


# ---- the same numbers in 64 bits ---------------------------------------------

def exact(case, seed):
    """Closeness (n - 1) / sum of hop distances by plain level-synchronous
    search; every other output is a whole number.  Large cases: None."""
    if case["op"] != "closeness":
        return None
    n, u, v, _, sources = _edges(case, seed)
    if (u.numel() * 2) * len(sources) > 400_000_000:
        return None
    keep = u != v
    u, v = u[keep].long(), v[keep].long()
    if not case["directed"]:
        u, v = torch.cat([u, v]), torch.cat([v, u])
    has_out = torch.zeros(n, dtype=torch.bool, device="cuda")
    has_out[u] = True
    sums = torch.zeros(len(sources), dtype=torch.int64, device="cuda")
    for at in range(0, len(sources), 32):
        src = torch.from_numpy(sources[at:at + 32].astype(np.int64)).cuda()
        lanes = torch.arange(len(src), device="cuda")
        front = torch.zeros((n, len(src)), dtype=torch.float32, device="cuda")
        front[src, lanes] = 1
        seen, level = front > 0, 0
        while bool(front.any()):
            level += 1
            front = torch.zeros_like(front).index_add_(0, v, front[u])
            new = (front > 0) & ~seen
            seen |= new
            sums[at:at + 32] += level * new.sum(0)
            front = new.float()
        sums[at:at + 32][~has_out[src]] = 0
    s = sums.cpu().numpy()
    cc = np.where(s > 0, (n - 1) / np.maximum(s, 1).astype(np.float64), 0.0)
    ref = np.where(s != 0, (n - 1) // np.maximum(s, 1), 0).astype(np.float64)
    return cc, s, ref
