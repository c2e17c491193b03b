"""Performance cases: what a program that uses this library has it do.

Twelve listed cases cover the graph operations behind the reference's
applications, each through the binding a program calls (graphchi-cpp_amd/gchi.py
over include/gchi.h): PageRank sweeps in both engine modes, many graphs and many
personalized queries at once, the set-up from an edge list, shard files in both
directions, components, triangles and edge-list text.  draw() gives more sizes
of the same ranges.

Inputs are made on the GPU from the seed alone: R-MAT pairs of the benchmark's
quadrant probabilities (skewed degrees, hubs) or equal ones (no hubs),
duplicates kept, no self-loops, over 2^scale vertices.
"""
import ctypes
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "graphchi-cpp_amd"))
import gchi  # noqa: E402

SKEWED = (0.57, 0.19, 0.19, 0.05)
EVEN = (0.25, 0.25, 0.25, 0.25)

# The shape the functional engine gives its synchronous sweeps (rank-space tiles).
ENGINE_SHAPE = {"edges_per_block": 512, "short_row_max": 0, "persistent": 4, "hot_vertices": 1 << 20}
TELEPORT, DAMPING = 0.15, 0.85
INDEX_ENTRIES = 4096  # .adjidx entries of one shard, at most


def listed():
    return [
        # a small graph iterated: launches and latency, hardly any data
        {"name": "pagerank_small", "kind": "pagerank", "scale": 12, "edges": 65521, "skewed": True, "sweeps": 20},
        # the benchmark's graph and sweep count
        {"name": "pagerank_rmat22", "kind": "pagerank", "scale": 22, "edges": 16 << 22, "skewed": True, "sweeps": 20},
        # a graph without hubs, ragged size: every source is as cold as the next
        {"name": "pagerank_even", "kind": "pagerank", "scale": 20, "edges": 11534339, "skewed": False, "sweeps": 10},
        # the functional engine's default mode over several sub-intervals
        {"name": "semisync", "kind": "semisync", "scale": 19, "edges": 8388593, "skewed": True, "blocks": 7,
         "sweeps": 4},
        # many uneven graphs in one batch plan
        {"name": "many_graphs", "kind": "graphs", "graphs": 300, "low": 10, "high": 17, "factor": 16, "sweeps": 10},
        # personalized queries, three query blocks, the last one ragged
        {"name": "ppr", "kind": "ppr", "scale": 17, "edges": 2097143, "skewed": True, "queries": 130},
        # a program's whole run: edge list in HBM -> CSC -> plan -> ranks
        {"name": "edges_to_ranks", "kind": "whole", "scale": 21, "edges": 33554393, "skewed": True, "sweeps": 4},
        # the sharder: intervals, order and the .adj bytes of every shard on the host
        {"name": "shard_encode", "kind": "encode", "scale": 18, "edges": 4194301, "skewed": True, "shards": 3},
        # an engine's load: every shard's bytes decoded into edge lists
        {"name": "shard_decode", "kind": "decode", "scale": 21, "edges": 33554393, "skewed": True, "shards": 4},
        # connected components as the engine runs them, under the scheduler
        {"name": "components", "kind": "components", "scale": 22, "edges": 33554393, "skewed": True},
        # triangle counting from a simple undirected edge list: order, orient, count
        {"name": "triangles", "kind": "triangles", "scale": 19, "edges": 8388593, "skewed": True},
        # an edge-list file's text
        {"name": "edge_text", "kind": "text", "scale": 20, "edges": 3000017, "skewed": True},
    ]


def _log(rng, low, high):
    """Log-uniform integer of [low, high]."""
    return int(round(low * (high / low) ** rng.random()))


def draw(rng):
    kind = rng.choice(["pagerank", "pagerank", "semisync", "graphs", "ppr", "whole", "encode", "decode",
                       "components", "triangles", "text"])
    skewed = rng.random() < 0.75
    if kind == "graphs":
        low = rng.randint(10, 13)
        return {"kind": kind, "graphs": _log(rng, 20, 300), "low": low, "high": rng.randint(low, 17),
                "factor": rng.randint(8, 16), "sweeps": rng.randint(4, 10)}
    top = {"pagerank": 22, "semisync": 20, "ppr": 17, "whole": 21, "encode": 18, "decode": 21, "components": 22,
           "triangles": 19, "text": 20}[kind]
    scale = rng.randint(12, top)
    most = min(16 << scale, {"ppr": 2 << 20, "text": 3 << 20, "encode": 4 << 20, "decode": 32 << 20, "whole": 32 << 20,
                             "components": 32 << 20, "triangles": 8 << 20}.get(kind, 64 << 20))
    case = {"kind": kind, "scale": scale, "edges": _log(rng, max(4 << scale, 30000) // 2, most) | 1, "skewed": skewed}
    if kind == "pagerank":
        case["sweeps"] = rng.randint(5, 20)
    elif kind == "semisync":
        case.update(blocks=rng.randint(1, 19), sweeps=rng.randint(2, 4))
    elif kind == "ppr":
        case["queries"] = _log(rng, 1, 130)
    elif kind == "whole":
        case["sweeps"] = rng.randint(1, 10)
    elif kind in ("encode", "decode"):
        case["shards"] = rng.randint(1, 7)
    return case


# ------------------------------------------------------------------ inputs
def _pairs(scale, count, skewed, gen, levels=None):
    """`count` R-MAT pairs (int64); levels (a tensor) gives each pair its own scale."""
    a, b, c, _ = SKEWED if skewed else EVEN
    src = torch.zeros(count, dtype=torch.int64, device="cuda")
    dst = torch.zeros(count, dtype=torch.int64, device="cuda")
    for k in range(scale):
        u = torch.rand(count, device="cuda", generator=gen)
        bits = torch.stack([u >= a + b, ((u >= a) & (u < a + b)) | (u >= a + b + c)]).long()
        if levels is None:
            src.mul_(2).add_(bits[0])
            dst.mul_(2).add_(bits[1])
        else:
            src = torch.where(levels > k, 2 * src + bits[0], src)
            dst = torch.where(levels > k, 2 * dst + bits[1], dst)
    return src, dst


def _no_loops(src, dst):
    """A self-loop's head becomes its neighbour in id."""
    return src.int(), torch.where(src == dst, dst ^ 1, dst).int()


def _edges(case, seed):
    """(src, dst, N): int32 pairs without self-loops."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    src, dst = _pairs(case["scale"], case["edges"], case["skewed"], gen)
    return (*_no_loops(src, dst), 1 << case["scale"])


def _many(case, seed):
    """Uneven graphs: [(src, dst, N)], each with ids of its own."""
    rng = np.random.default_rng(case["graphs"])
    scales = rng.integers(case["low"], case["high"] + 1, case["graphs"])
    counts = (case["factor"] << scales) - rng.integers(0, 1 << scales)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    levels = torch.from_numpy(np.repeat(scales, counts)).to("cuda")
    src, dst = _no_loops(*_pairs(case["high"], int(counts.sum()), True, gen, levels))
    ends = np.cumsum(counts)
    return [(src[e - c:e], dst[e - c:e], 1 << s) for s, c, e in zip(scales.tolist(), counts.tolist(), ends.tolist())]


def _queries(case, n, seed):
    """Restart sets of 1..64 distinct vertices."""
    return gchi.ppr_workload_queries(n, case["queries"], seed)


def _simple(src, dst):
    """One (min, max) record per undirected edge."""
    key = torch.unique((torch.minimum(src, dst).long() << 32) | torch.maximum(src, dst).long())
    return (key >> 32).int(), (key & 0xffffffff).int()


def _text(src, dst, seed):
    """The edge list as text: comment lines, then one 'from<sep>to' line an edge."""
    count, width = src.numel(), 7
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    line = torch.zeros((count, 2 * width + 2), dtype=torch.uint8, device="cuda")
    used = torch.ones((count, 2 * width + 2), dtype=torch.bool, device="cuda")
    for at, ids in ((0, src.long()), (width + 1, dst.long())):
        for k in range(width):
            p = 10 ** (width - 1 - k)
            line[:, at + k] = (ids // p % 10 + 48).to(torch.uint8)
            if p > 1:
                used[:, at + k] = ids >= p
    seps = torch.tensor([9, 9, 9, 32], dtype=torch.uint8, device="cuda")
    line[:, width] = seps[torch.randint(0, 4, (1,), device="cuda", generator=gen)]
    line[:, 2 * width + 1] = 10
    head = np.frombuffer(b"# Directed graph\n# FromNodeId\tToNodeId\n", np.uint8).copy()
    return torch.cat([torch.from_numpy(head).to("cuda"), line[used]])


def _bounds(n, blocks):
    """Equal vertex blocks (at most n of them)."""
    return np.unique(np.linspace(0, n, min(blocks, n) + 1).astype(np.uint32))


def prepare(case, seed):
    gchi.open_device(0)
    kind = case["kind"]
    state = {"kind": kind, "case": case}
    op = gchi.pr_op(TELEPORT, DAMPING)
    if kind == "graphs":
        made = [gchi.DeviceGraph(*g) for g in _many(case, seed)]
        tele = torch.tensor([TELEPORT / g.N for g in made], dtype=torch.float64, device="cuda")
        plan = gchi.PageRankPlan.batch(made, persistent=1)
        state["exec"] = gchi.PageRankExec(plan, gchi.pr_op(TELEPORT, DAMPING, graph_teleport=tele), 1.0,
                                          case["sweeps"])
        return state
    src, dst, n = _edges(case, seed)
    state["n"] = n
    if kind == "pagerank":
        plan = gchi.PageRankPlan(gchi.DeviceGraph(src, dst, n), **ENGINE_SHAPE)
        state["exec"] = gchi.PageRankExec(plan, op, 1.0, case["sweeps"])
    elif kind == "semisync":
        state["op"] = op
        state["blocked"] = gchi.PageRankBlocked(gchi.DeviceGraph(src, dst, n), _bounds(n, case["blocks"]))
    elif kind == "ppr":
        plan = gchi.PageRankPlan(gchi.DeviceGraph(src, dst, n), edges_per_block=2048, persistent=1)
        state["queries"] = _queries(case, n, seed)
        state["batch"] = gchi.PprBatch(plan, case["queries"])
    elif kind == "decode":
        shards = gchi.Shards(src, dst, n - 1, case["shards"])
        files = [np.frombuffer(shards.encode(p)[0], np.uint8).copy() for p in range(shards.nshards)]
        state["streams"] = [(torch.from_numpy(b).to("cuda"), b.size) for b in files]
        shards.close()
    elif kind == "encode":
        # pinned host memory that the .adj bytes and index entries are written to
        rows = min(case["edges"], n * case["shards"])
        state["edges"] = (src, dst)
        state["bytes"] = torch.zeros(4 * case["edges"] + 7 * rows + n * case["shards"] // 64 + 4096, dtype=torch.uint8,
                                     pin_memory=True)
        state["index"] = torch.zeros((case["shards"] + 1, 3 * INDEX_ENTRIES), dtype=torch.int64, pin_memory=True)
    elif kind == "components":
        state["graph"] = gchi.DeviceGraph(torch.cat([src, dst]), torch.cat([dst, src]), n)
    elif kind == "triangles":
        state["edges"] = _simple(src, dst)
    elif kind == "text":
        state["text"] = _text(src, dst, seed)
    else:
        state["edges"] = (src, dst)
    return state


# ------------------------------------------------------------------ one pass
def run(state):
    kind, case = state["kind"], state["case"]
    if kind in ("pagerank", "graphs"):
        ex = state["exec"]
        ex.launch()  # each sweep's residual and rank sum are sums over these vectors
        return {"ranks": ex.ranks(), "x": ex.x[case["sweeps"] & 1]}
    if kind == "semisync":
        return state["blocked"].run(state["op"], 1.0, case["sweeps"])[0]
    if kind == "ppr":
        batch = state["batch"]
        batch.run(state["queries"])
        return torch.stack([batch.ranks(q) for q in range(case["queries"])])
    if kind == "whole":
        graph = gchi.DeviceGraph(*state["edges"], state["n"])
        plan = gchi.PageRankPlan(graph, **ENGINE_SHAPE)
        ex = gchi.PageRankExec(plan, gchi.pr_op(TELEPORT, DAMPING), 1.0, case["sweeps"])
        ex.launch()
        return {"in_off": graph.in_off, "in_src": graph.in_src, "outdeg": graph.outdeg, "indeg": graph.indeg,
                "ranks": ex.ranks()}
    if kind == "encode":  # as the sharder: the size of each shard's stream, then its bytes
        lib, stream = gchi.lib(), gchi.stream()
        shards = gchi.Shards(*state["edges"], state["n"] - 1, case["shards"])
        ends, size, entries, at = np.zeros(case["shards"] + 1, np.int64), ctypes.c_uint64(), ctypes.c_uint32(), 0
        for p in range(shards.nshards):
            gchi.check(lib.gchi_shard_encode(shards.handle, p, None, ctypes.byref(size), None, 0, None, stream))
            gchi.check(lib.gchi_shard_encode(shards.handle, p, state["bytes"].data_ptr() + at, ctypes.byref(size),
                                             state["index"][p].data_ptr(), INDEX_ENTRIES, ctypes.byref(entries),
                                             stream))
            ends[p] = shards.ends[p]
            at += size.value
        shards.close()
        return {"ends": ends, "bytes": state["bytes"], "index": state["index"], "size": at}
    if kind == "decode":
        src, dst, counts, ends = gchi.shard_decode_many(state["streams"])
        return {"src": src, "dst": dst, "counts": counts, "ends": ends}
    if kind == "components":
        g = state["graph"]
        return gchi.cc_scheduled(g.in_off, g.in_src, g.N)[0]  # how often a vertex is evaluated is not fixed
    if kind == "triangles":
        prep = gchi.TrianglePrep(*state["edges"], state["n"])
        per_vertex, total, overflow = prep.count()
        return {"map": prep.vertexmap, "off": prep.off, "per_vertex": per_vertex, "total": total,
                "overflow": overflow}
    src, dst, _, maxid = gchi.parse_edgelist(state["text"])
    return {"src": src, "dst": dst, "maxid": maxid}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    kind = case["kind"]
    if kind == "graphs":
        each = [1 << s for s in range(case["low"], case["high"] + 1)]
        n = case["graphs"] * sum(each) // len(each)
        e = case["factor"] * n
    else:
        n, e = 1 << case["scale"], case["edges"]
    sweep = 4 * e + 20 * n  # source ids; offsets, out-degrees, x in, r in and r out (x out replaces x in)
    if kind in ("pagerank", "semisync", "graphs"):
        return {"bytes": case["sweeps"] * sweep, "flops": case["sweeps"] * 2 * e}
    if kind == "ppr":  # about 75 sweeps to the tolerance; each reads the ids and turns every query's vector over
        q = case["queries"]
        return {"bytes": 75 * (4 * e + 8 * n * q), "flops": 75 * 2 * e * q}
    if kind == "whole":
        return {"bytes": 12 * e + 12 * n + case["sweeps"] * sweep, "flops": case["sweeps"] * 2 * e}
    if kind == "encode":
        return {"bytes": 12 * e + 2 * n, "flops": 0}
    if kind == "decode":
        return {"bytes": 12 * e + 2 * n, "flops": 0}
    if kind == "components":
        return {"bytes": 8 * e + 8 * n, "flops": 0}
    if kind == "triangles":  # the wedges need at least one look at every oriented edge
        return {"bytes": 12 * e + 12 * n, "flops": 0}
    return {"bytes": 14 * e + 8 * e, "flops": 0}


# ------------------------------------------------------------------ the same in 64 bits, in plain torch
def _sweep64(src, dst, outdeg, r, teleport):
    x = torch.where(outdeg > 0, r / outdeg.clamp(min=1), torch.zeros_like(r))
    s = torch.zeros_like(r).index_add_(0, dst, x[src])
    return teleport + DAMPING * s


def _share64(r, outdeg):
    return torch.where(outdeg > 0, r / outdeg.clamp(min=1), torch.zeros_like(r))


def exact(case, seed):
    kind = case["kind"]
    if kind == "graphs":
        made = _many(case, seed)
        base = np.concatenate([[0], np.cumsum([g[2] for g in made])]).tolist()
        src = torch.cat([g[0].long() + b for g, b in zip(made, base)])
        dst = torch.cat([g[1].long() + b for g, b in zip(made, base)])
        n = base[-1]
        teleport = torch.cat([torch.full((g[2],), TELEPORT / g[2], dtype=torch.float64, device="cuda") for g in made])
    elif kind in ("pagerank", "semisync", "whole", "ppr"):
        src, dst, n = _edges(case, seed)
        src, dst = src.long(), dst.long()
        teleport = TELEPORT
    else:
        return None  # whole numbers and bytes
    outdeg = torch.bincount(src, minlength=n).double()
    if kind == "ppr":
        queries = _queries(case, n, seed)
        r0 = torch.zeros((n, len(queries)), dtype=torch.float64, device="cuda")
        for q, seeds in enumerate(queries):
            r0[torch.from_numpy(seeds.astype(np.int64)).to("cuda"), q] = (1.0 - DAMPING) / len(seeds)
        r, inv = r0.clone(), torch.where(outdeg > 0, 1.0 / outdeg.clamp(min=1), torch.zeros_like(outdeg))[:, None]
        for _ in range(170):
            x, s = r * inv, torch.zeros_like(r)
            for at in range(0, src.numel(), 1 << 19):
                s.index_add_(0, dst[at:at + (1 << 19)], x[src[at:at + (1 << 19)]])
            r = r0 + DAMPING * s
        return r.t().contiguous()
    r = torch.ones(n, dtype=torch.float64, device="cuda")
    if kind == "semisync":
        bounds = _bounds(n, case["blocks"]).tolist()
        order = torch.argsort(dst)
        src, dst = src[order], dst[order]
        cut = torch.searchsorted(dst, torch.tensor(bounds, device="cuda")).tolist()
        x = _share64(r, outdeg)
        for _ in range(case["sweeps"]):
            for j in range(len(bounds) - 1):
                lo, hi = bounds[j], bounds[j + 1]
                s = torch.zeros(hi - lo, dtype=torch.float64, device="cuda")
                s.index_add_(0, dst[cut[j]:cut[j + 1]] - lo, x[src[cut[j]:cut[j + 1]]])
                r[lo:hi] = teleport + DAMPING * s
                x[lo:hi] = _share64(r[lo:hi], outdeg[lo:hi])
        return r
    for _ in range(case["sweeps"]):
        r = _sweep64(src, dst, outdeg, r, teleport)
    if kind == "whole":
        return {"in_off": None, "in_src": None, "outdeg": None, "indeg": None, "ranks": r}
    return {"ranks": r, "x": _share64(r, outdeg)}
