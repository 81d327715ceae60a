"""Timed cases of the graph engine: what its users run, over the range of sizes.

A program that uses this library holds one graph in HBM and asks questions of
it (ranks at some damping, components from labels it has, searches from
roots), or takes a new edge list through the whole way: ingress, run, results.
Both kinds are here.

  "ask"   the graph is loaded already, as weights are for a model: it belongs
          to the case (graph_seed); the question comes from the state's seed
          (damping, starting labels, roots).  Results stay on the device, in
          the device's numbering, where the program's next step reads them.
  "load"  the edges come from the state's seed; one pass is the ingress, the
          run and the result in host memory.

The library keeps one graph at a time, so states of one "ask" case share it,
and a pass whose graph is no longer the loaded one loads it first.
"""
from __future__ import annotations

import ctypes as C
import json
import math
import os
import sys
import warnings

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "grazelle-ppopp18_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)
import grazelle as gz  # noqa: E402

gz.lib.gz_device_copy.restype, gz.lib.gz_device_copy.argtypes = None, [C.c_void_p, C.c_void_p, C.c_size_t]

FULL = {"scale": 26, "vertices": gz.FULL_VERTICES, "edges": gz.FULL_RAW_EDGES, "graph_seed": 1,
        "slices_log2": 20, "tiers": 2, "blocks": 5}
SLICED_CHUNK, PLAIN_CHUNK = 2048, 512  # vectors per chunk the library's documents give for the two pulls
HOT_CACHE = 20480


def listed():
    return [
        # PageRank over the reference's own graph size, asked again at another
        # damping: 20 iterations of a few microseconds each, bound by launches.
        {"name": "pr-s16", "kind": "ask", "what": "pr", "iterations": 20, "scale": 16, "vertices": 0,
         "edges": 16 << 16, "graph_seed": 1, "slices_log2": 0, "tiers": 1, "blocks": 0},
        # The ordinary (unsliced, not renumbered) pull on a mid-sized graph with an odd
        # vertex count: what a caller gets who loads a graph and changes nothing.
        {"name": "pr-1.5m", "kind": "ask", "what": "pr", "iterations": 20, "scale": 21, "vertices": 1500007,
         "edges": 24000000, "graph_seed": 1, "slices_log2": 0, "tiers": 1, "blocks": 0},
        # The headline graph with the source-sliced pull: a long-lived rank service.
        {"name": "pr-full", "kind": "ask", "what": "pr", "iterations": 10, **FULL},
        # Components of a small symmetrised graph with planted trees, propagated
        # from labels the program has: a few small iterations, bound by latency.
        {"name": "cc-s16", "kind": "ask", "what": "cc", "scale": 16, "vertices": 0, "edges": 16 << 16, "trees": 64,
         "tree_size": 100, "graph_seed": 1, "slices_log2": 0, "tiers": 1, "blocks": 0},
        # The components configuration of the benchmark with its fast layout.
        {"name": "cc-s22", "kind": "ask", "what": "cc", "scale": 22, "vertices": 0, "edges": 16 << 22, "trees": 64,
         "tree_size": 1000, "graph_seed": 1, "slices_log2": 19, "tiers": 1, "blocks": 0},
        # Searches from roots that arrive one by one, fixed engine threshold:
        # the benchmark's search graph.
        {"name": "bfs-s24", "kind": "ask", "what": "bfs", "engine": "hybrid", "roots": 4, "scale": 24, "vertices": 0,
         "edges": 16 << 24, "graph_seed": 1, "slices_log2": 0, "tiers": 1, "blocks": 0},
        # The same on a small graph, where a level is a few launches.
        {"name": "bfs-s17", "kind": "ask", "what": "bfs", "engine": "hybrid", "roots": 4, "scale": 17, "vertices": 0,
         "edges": 16 << 17, "graph_seed": 1, "slices_log2": 0, "tiers": 1, "blocks": 0},
        # Searches on the headline graph with the learned engine choice.
        {"name": "bfs-full", "kind": "ask", "what": "bfs", "engine": "learned", "roots": 2, **FULL},
        # A new small edge list through the whole way, as the first program a
        # user writes: host pairs in, ranks out.
        {"name": "load-pr-20k", "kind": "load", "what": "pr", "iterations": 20, "scale": 15, "vertices": 20011,
         "edges": 200000, "from": "pairs", "slices_log2": 0, "tiers": 1, "blocks": 0},
        # A mid-sized undirected edge list: symmetrised ingress, components, labels out.
        {"name": "load-cc-300k", "kind": "load", "what": "cc", "scale": 19, "vertices": 300007, "edges": 3000000,
         "from": "pairs", "slices_log2": 0, "tiers": 1, "blocks": 0},
        # A large generated graph renumbered and sliced for the fast pull, then ranked once.
        {"name": "load-pr-4m", "kind": "load", "what": "pr", "iterations": 20, "scale": 22, "vertices": 0,
         "edges": 16 << 22, "from": "rmat", "slices_log2": 18, "tiers": 1, "blocks": 3},
        # Many small graphs ingested and ranked as one batch.
        {"name": "load-batch-128", "kind": "load", "what": "batch", "iterations": 10, "graphs": 128},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    pick = rng.random()
    if pick < 0.1:
        return {"kind": "load", "what": "batch", "iterations": rng.randint(5, 10), "graphs": _log_int(rng, 12, 128)}
    kind, what = ("ask", rng.choice(["pr", "cc", "bfs"])) if pick < 0.6 else ("load", rng.choice(["pr", "cc"]))
    rmat = kind == "ask" or rng.random() < 0.5
    top = 14 << 20 if what == "bfs" else 4 << 20 if rmat else 1 << 20
    v = _log_int(rng, 1 << 14, top)
    c = {"kind": kind, "what": what, "scale": max(2, (v - 1).bit_length()), "vertices": v,
         "edges": int(v * rng.uniform(4, 16)), "slices_log2": 0, "tiers": 1, "blocks": 0}
    if kind == "ask":
        c["graph_seed"] = rng.randint(1, 1 << 20)
    else:
        c["from"] = "rmat" if rmat else "pairs"
    if what == "pr":
        c["iterations"] = rng.randint(5, 20)
    if what == "cc" and kind == "ask":
        c.update(trees=rng.randint(1, 64), tree_size=rng.randint(50, 1000))
    if what == "bfs":
        c.update(engine=rng.choice(["hybrid", "learned"]), roots=rng.randint(1, 4))
    elif rmat and v > 1 << 19 and rng.random() < 0.6:
        c.update(slices_log2=rng.randint(15, 18), tiers=rng.randint(1, 2), blocks=rng.choice([0, 2, 3, 5]))
    return c


# ---- the loaded graph ---------------------------------------------------------

_loaded = None


def _layout(case):
    """Ingress arguments and settings of the layout the case asks for."""
    sliced = case["slices_log2"] > 0
    gz.set_chunk_vectors(SLICED_CHUNK if sliced else PLAIN_CHUNK)
    gz.slices_set_hot_cache(HOT_CACHE if sliced else 0)
    return {"relabel": sliced, "slices_log2": case["slices_log2"], "slice_tiers": case["tiers"],
            "slice_blocks": case["blocks"]}


def _load(case):
    """Make the case's graph the loaded one."""
    global _loaded
    layout = _layout(case)
    spec = json.dumps([case["what"] == "cc", case.get("trees", 0), case.get("tree_size", 0), layout]
                      + [case[k] for k in ("scale", "vertices", "edges", "graph_seed")])
    if spec == _loaded:
        return
    n = case["vertices"] or 1 << case["scale"]
    extra = None
    if case.get("trees"):
        extra = gz.planted_trees(n, case["trees"], case["tree_size"], case["graph_seed"] + 1000)
    gz.load_rmat_device(case["scale"], case["edges"], case["graph_seed"], symmetrize=case["what"] == "cc",
                        num_vertices=n + case.get("trees", 0) * case.get("tree_size", 0), extra=extra,
                        rmat_vertices=case["vertices"], **layout)
    _loaded = spec


def _pull_variant(case):
    return "source_sliced" if case["slices_log2"] else "sched_aware"


class _DeviceWords:
    """The loaded graph's vertex words as they lie in HBM."""

    def __init__(self, typestr):
        self.__cuda_array_interface__ = {"shape": (gz.num_vertices(),), "typestr": typestr, "version": 2,
                                         "data": (gz.phase_graph.vertex_props, False), "strides": None}


def _props(typestr):
    return torch.as_tensor(_DeviceWords(typestr), device="cuda")


def _damping(rng):
    return float(rng.uniform(0.8, 0.9))


def _batch(case, seed):
    """Scale, edge factor and edge seed of each graph; the sizes belong to the case."""
    return [(scale, factor, seed + i) for i, (scale, factor, _) in enumerate(gz.batch_specs(case["graphs"]))]


# ---- states and passes ---------------------------------------------------------

def prepare(case, seed):
    rng = np.random.default_rng(seed)
    s = {"case": case}
    if case["kind"] == "load":
        s["damping"], s["graph_seed"] = _damping(rng), int(rng.integers(1, 1 << 30))
        if case["what"] == "batch":
            s["specs"] = _batch(case, s["graph_seed"])
        elif case["from"] == "pairs":
            s["pairs"] = gz.rmat_edges(case["scale"], case["edges"], s["graph_seed"],
                                       num_vertices=case["vertices"])
        gz.init()
        return s
    _load(case)
    if case["what"] == "pr":
        s["options"] = gz.options("pr", iterations=case["iterations"], damping=_damping(rng),
                                  pull_variant=_pull_variant(case))
    elif case["what"] == "cc":
        s["options"] = gz.options("cc", pull_variant=_pull_variant(case))
        g = torch.Generator("cuda").manual_seed(int(rng.integers(1 << 40)))
        s["labels"] = torch.randperm(gz.num_vertices(), generator=g, device="cuda")
        torch.cuda.synchronize()
    else:
        gz.selector_load(os.path.join(_PKG, "selector_bfs.bin"))
        # roots with out-edges, as the benchmark draws them
        deg = gz.outdegrees()
        roots = []
        while len(roots) < case["roots"]:
            v = int(rng.integers(deg.shape[0]))
            if deg[v] > 0:
                roots.append(v)
        if case["slices_log2"]:
            original = gz.original_ids()
            roots = [int(original[v]) for v in roots]
        s["options"] = [gz.options("bfs", engine=case["engine"], root=r) for r in roots]
        s["found"] = [torch.empty(gz.num_vertices(), dtype=torch.int64, device="cuda") for _ in roots]
    return s


def run(state):
    case = state["case"]
    if case["kind"] == "load":
        return _run_load(state)
    _load(case)
    if case["what"] == "pr":
        gz.run(state["options"])
        return _props("<f8")
    if case["what"] == "cc":
        # labels spread from the ones the program has (gz_execution_prepare
        # starts every vertex at its own id)
        o, r = state["options"], gz.RunResult()
        gz.lib.gz_execution_prepare(C.byref(o))
        gz.lib.gz_device_copy(gz.phase_graph.vertex_props, state["labels"].data_ptr(), 8 * gz.num_vertices())
        gz.lib.gz_execution_run(C.byref(o), C.byref(r))
        return _props("<i8")
    for o, out in zip(state["options"], state["found"]):
        gz.run(o)
        if case["engine"] == "learned":
            # depths alone: of several parents one level up, the engine that ran
            # the level picks, and the learned choice goes by measured times
            torch.bitwise_right_shift(_props("<i8"), 48, out=out)
            torch.cuda.current_stream().synchronize()
        else:
            gz.lib.gz_device_copy(out.data_ptr(), gz.phase_graph.vertex_props, 8 * gz.num_vertices())
    gz.lib.gz_synchronize()
    return state["found"]


def _run_load(state):
    global _loaded
    case, _loaded = state["case"], None
    if case["what"] == "batch":
        gz.load_batch_device(state["specs"])
        gz.batch_pr(case["iterations"], damping=state["damping"])
        return gz.batch_pr_ranks()
    layout, symmetrize = _layout(case), case["what"] == "cc"
    if case["from"] == "pairs":
        gz.load_pairs_device(case["vertices"], state["pairs"], symmetrize=symmetrize, **layout)
    else:
        gz.load_rmat_device(case["scale"], case["edges"], state["graph_seed"], symmetrize=symmetrize,
                            rmat_vertices=case["vertices"], **layout)
    if case["what"] == "cc":
        gz.run(gz.options("cc", pull_variant=_pull_variant(case)))
        return gz.cc_labels().view(np.int64)
    gz.run(gz.options("pr", iterations=case["iterations"], damping=state["damping"],
                      pull_variant=_pull_variant(case)))
    return gz.pr_ranks()


# ---- what a pass cannot do without ----------------------------------------------

def work(case):
    """An iteration of PageRank reads a 4-byte source per edge and three FP64
    words per vertex (rank, out-degree, new rank); components read every edge
    once; a search reads an edge for, and writes a word of, every vertex; a
    load reads the pairs."""
    if case["what"] == "batch":
        specs = _batch(case, 1)
        v, e = sum(1 << s for s, _, _ in specs), sum(f << s for s, f, _ in specs)
    else:
        v, e = case["vertices"] or 1 << case["scale"], case["edges"]
    if case["what"] == "cc":
        v, e = v + case.get("trees", 0) * case.get("tree_size", 0), 2 * (e + case.get("trees", 0) * case.get("tree_size", 0))
        size, ops = 4 * e + 16 * v, e
    elif case["what"] == "bfs":
        size, ops = case["roots"] * 12 * v, case["roots"] * v
    else:
        size, ops = case["iterations"] * (4 * e + 24 * v), case["iterations"] * (e + 5 * v)
    if case["kind"] == "load":
        size += 16 * e + 8 * v
    return {"bytes": size, "flops": ops}


# ---- the same in plain torch, 64 bits --------------------------------------------

def _i64(x):
    return x - (1 << 64) if x >= 1 << 63 else x


def _mix(x):
    x = x + _i64(0x9e3779b97f4a7c15)
    x = (x ^ ((x >> 30) & ((1 << 34) - 1))) * _i64(0xbf58476d1ce4e5b9)
    x = (x ^ ((x >> 27) & ((1 << 37) - 1))) * _i64(0x94d049bb133111eb)
    return x ^ ((x >> 31) & ((1 << 33) - 1))


def _rmat(scale, vertices, edges, seed):
    """The edges (source, destination) of the seeded R-MAT stream."""
    a, b, c = 0.57, 0.19, 0.19
    ta, tb, tc = int(a * 65536), int((a + b) * 65536), int((a + b + c) * 65536)
    src = torch.empty(edges, dtype=torch.int64, device="cuda")
    dst = torch.empty_like(src)
    for lo in range(0, edges, 1 << 26):
        x = _mix(torch.arange(lo, min(edges, lo + (1 << 26)), device="cuda"))
        x = _mix(seed ^ x)
        s, d = torch.zeros_like(x), torch.zeros_like(x)
        for level in range(scale):
            if level and level % 4 == 0:
                x = _mix(x)
            u = (x >> (16 * (level % 4))) & 0xffff
            s = 2 * s + (u >= tb).to(torch.int64)
            d = 2 * d + (((u >= ta) & (u < tb)) | (u >= tc)).to(torch.int64)
        src[lo:lo + (1 << 26)], dst[lo:lo + (1 << 26)] = s, d
    if vertices:
        src.remainder_(vertices)
        dst.remainder_(vertices)
    return src, dst


def _ranks(src, dst, v, base, iterations, damping):
    """props = rank / out-degree after the iterations, and out-degree (the
    graph's vertex count for sinks), per vertex; `base`: first vertex of each
    graph of a union."""
    keys = torch.sort((dst << 32) | src).values
    keep = torch.ones_like(keys, dtype=torch.bool)
    keep[1:] = keys[1:] != keys[:-1]
    keys = keys[keep]
    del keep
    dst, src = keys >> 32, keys & 0xffffffff
    del keys
    keep = src != dst
    src, dst = src[keep], dst[keep]
    sizes = torch.tensor(np.diff(base), device="cuda")
    graph = torch.repeat_interleave(torch.arange(len(sizes), device="cuda"), sizes)
    nv = sizes.double()[graph]
    deg = torch.bincount(src, minlength=v).double()
    deg = torch.where(deg == 0, nv, deg)
    first = torch.zeros(v + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(torch.bincount(dst, minlength=v), 0, out=first[1:])
    warnings.filterwarnings("ignore", message="Sparse CSR tensor support")
    pull = torch.sparse_csr_tensor(first.int(), src.int(), torch.ones(src.numel(), dtype=torch.float64, device="cuda"),
                                   size=(v, v), check_invariants=False)
    del src, dst, first
    props = 1 / nv / deg
    for _ in range(iterations):
        acc = pull.matmul(props)
        total = torch.stack([acc[lo:hi].sum() for lo, hi in zip(base, base[1:])])
        props = ((acc + (1 - total[graph]) / nv) * damping + (1 - damping) / nv) / deg
    return props, deg


def _device_order(src, v, slice_vertices, tiers):
    """Original id of each device vertex of a graph renumbered by out-degree
    (duplicates and self-loops counted, ties by id), each run of 8 S ranks
    dealt round robin into eight windows of S."""
    order = torch.sort(torch.bincount(src, minlength=v), descending=True, stable=True).indices
    rank = torch.arange(v, device="cuda")
    s = min(slice_vertices, v // (8 * tiers), 1 << 23)
    t, q = rank // (8 * s), rank % (8 * s)
    place = torch.where(rank < 8 * s * tiers, t * 8 * s + (q % 8) * s + q // 8, rank)
    out = torch.empty_like(order)
    out[place] = order
    return out


def exact(case, seed):
    if case["what"] not in ("pr", "batch"):
        return None
    rng = np.random.default_rng(seed)
    damping, graph_seed = _damping(rng), case.get("graph_seed") or int(rng.integers(1, 1 << 30))
    if case["what"] == "batch":
        specs, base, parts = _batch(case, graph_seed), [0], []
        for scale, factor, g in specs:
            s, d = _rmat(scale, 0, factor << scale, g)
            parts.append((s + base[-1], d + base[-1]))
            base.append(base[-1] + (1 << scale))
        src, dst = torch.cat([p[0] for p in parts]), torch.cat([p[1] for p in parts])
        del parts
    else:
        src, dst = _rmat(case["scale"], case["vertices"], case["edges"], graph_seed)
        base = [0, case["vertices"] or 1 << case["scale"]]
    place = None
    if case["kind"] == "ask" and case["slices_log2"]:
        place = _device_order(src, base[-1], 1 << case["slices_log2"], case["tiers"])
    props, deg = _ranks(src, dst, base[-1], base, case["iterations"], damping)
    if case["kind"] == "load":
        return (props * deg).cpu().numpy()
    return props if place is None else props[place]
