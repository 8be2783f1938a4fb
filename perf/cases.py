"""The workloads the store's performance is measured on: streams of update
batches, bulk builds, groups of graphs, merged requests, reads, exports and
analytics, each through the package's public calls.

A case is a dict of plain values.  `listed()` gives the fixed ones, `draw()`
one more of the same ranges, `prepare()` what a program holds before the call,
`run()` one pass, `work()` the bytes a pass cannot do without and `exact()` the
floating results in 64 bits.

Graphs are R-MAT (a, b, c, d = 0.57, 0.19, 0.19, 0.05), as in the benchmark,
drawn with torch from the seed: `edges` distinct ones in random order.  Update
batches keep repeats, which the store drops.  The sizes of a case fix the
shapes of its outputs: graphs lie well inside one capacity, and neighbor reads
are chosen to return a fixed number of edges.
"""
import math

import numpy as np
import torch

import lpma_amd as L

RMAT = (0.57, 0.19, 0.19)

# density policies: (lower leaf, lower root, upper leaf, upper root); the
# first is the default of the store, the others are the autotuner's
DENSITY = {
    "flat": (0.42, 0.42, 1.0, 1.0),
    "low": (0.25, 0.25, 1.0, 1.0),
    "slack": (0.42, 0.42, 0.9, 0.9),
    "interpolated": (0.08, 0.30, 1.0, 0.75),
}


def listed():
    base = {"segment_slots": 32, "density": "flat"}
    big = {"vertices": 1 << 20, "edges": 1 << 23}
    return [
        # a small graph taking small batches: launches and latency only
        {"name": "stream_4k_b256", "kind": "stream", "vertices": 1 << 12, "edges": 40000, "batch": 256, **base},
        # the benchmark's power-law graph, fine-grained batches
        {"name": "stream_1m_b1e3", "kind": "stream", **big, "batch": 1000, **base},
        # the benchmark's headline batch, 1e5 edges in, 1e5 edges out, half way through its stream
        {"name": "stream_1m_b1e5", "kind": "stream", "vertices": 1 << 20, "edges": 12000000, "batch": 100000, **base},
        # a window moved by one large mixed batch
        {"name": "mixed_1m_b1e6", "kind": "mixed", **big, "batch": 1000000, **base},
        # write requests queued at a server, merged into one run (mean 1e4 keys each)
        {"name": "sequence_4m_r32", "kind": "sequence", "vertices": 1 << 22, "edges": 1 << 25, "requests": 32,
         "batch": 5000, **base},
        # many small graphs updated together, with the autotuner's usual choice
        {"name": "group_24_b5e3", "kind": "group", "graphs": 24, "edges_min": 10000, "edges_max": 1000000,
         "batch": 5000, "sizes": 3, "segment_slots": 64, "density": "interpolated"},
        # a graph built from its edge list
        {"name": "build_1m_8m", "kind": "build", **big, **base},
        # neighbor lists of as many vertices as one read request asks for
        {"name": "neighbors_1m_n512", "kind": "neighbors", **big, "queries": 512, **base},
        # membership of a million edges, half of them present
        {"name": "edge_query_1m_n1e6", "kind": "edge_query", **big, "queries": 1000000, **base},
        # the compacted edge list and CSR offsets of the live graph
        {"name": "export_1m_8m", "kind": "export", "form": "export", **big, **base},
        # a search and a ranking of a larger graph
        {"name": "bfs_4m_64m", "kind": "bfs", "form": "live", "vertices": 1 << 22, "edges": 1 << 26, **base},
        {"name": "pagerank_4m_64m", "kind": "pagerank", "vertices": 1 << 22, "edges": 1 << 26, **base},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _settled(edges, V, batch, case):
    """The number of edges nearest to `edges` that keeps a graph inside one capacity while batches go in and out."""
    _, _, _, upper = DENSITY[case["density"]]
    top = case["segment_slots"]
    while int(upper * top) < edges + V:
        top *= 2
    top = int(upper * top)
    return int(min(max(edges + V, 0.7 * top), 0.98 * top - 2 * batch)) - V


def draw(rng):
    kind = rng.choice(("stream", "stream", "stream", "mixed", "sequence", "group", "build", "neighbors", "edge_query",
                       "export", "bfs", "pagerank"))
    case = {"kind": kind, "segment_slots": rng.choice((32, 32, 32, 16, 64, 128)),
            "density": rng.choice(("flat", "flat", "low", "slack", "interpolated"))}
    if kind == "group":
        lo = _spread(rng, 3000, 30000)
        case.update(graphs=rng.randint(2, 32), edges_min=lo, edges_max=_spread(rng, lo, 1000000),
                    batch=_spread(rng, 100, 10000), sizes=rng.randrange(1 << 20))
        return case
    top = {"bfs": 1 << 25, "pagerank": 1 << 25, "sequence": 1 << 24}.get(kind, 1 << 23)
    case["edges"] = _spread(rng, 20000, top)
    # 8 to 32 edges for each vertex
    case["vertices"] = max(1000, int(case["edges"] / rng.uniform(8, 32)))
    if kind in ("stream", "mixed"):
        case["batch"] = _spread(rng, 50, min(1000000, case["edges"] // 8))
    elif kind == "sequence":
        case["requests"] = _spread(rng, 2, 64)
        case["batch"] = _spread(rng, 50, max(100, min(10000, case["edges"] // (8 * case["requests"]))))
    elif kind == "neighbors":
        case["queries"] = _spread(rng, 1, 50000)
    elif kind == "edge_query":
        case["queries"] = _spread(rng, 100, 2000000)
    elif kind == "export":
        case["form"] = rng.choice(("export", "to_csr", "get_data", "copy_view"))
    elif kind == "bfs":
        case["form"] = rng.choice(("live", "snapshot"))
    if kind in ("stream", "mixed", "sequence", "build", "export"):
        case["edges"] = _settled(case["edges"], case["vertices"], case.get("batch", 0) * case.get("requests", 1), case)
    return case


# ------------------------------------------------------------------ inputs


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 2654435761 % (1 << 62) + 1)
    return g


def _rmat(V, n, g):
    """n R-MAT edges on V vertices as int64 keys src << 32 | dst (repeats kept, no self loops)."""
    a, b, c = RMAT
    src = torch.zeros(n, dtype=torch.int64, device="cuda")
    dst = torch.zeros(n, dtype=torch.int64, device="cuda")
    for _ in range(max(1, (V - 1).bit_length())):
        r = torch.rand(n, generator=g, device="cuda")
        right = r >= a + b
        src.mul_(2).add_(right)
        dst.mul_(2).add_(((r >= a) & ~right) | (r >= a + b + c))
    if V & (V - 1):
        src.remainder_(V)
        dst.remainder_(V)
    dst = torch.where(src == dst, (dst + 1) % V, dst)
    return src.mul_(1 << 32).add_(dst)


def _graph_keys(V, n, g):
    """n distinct R-MAT edges in random order."""
    keys = torch.unique(_rmat(V, n + n // 8, g))
    while keys.numel() < n:
        keys = torch.unique(torch.cat([keys, _rmat(V, 2 * (n - keys.numel()) + 64, g)]))
    return keys[torch.randperm(keys.numel(), generator=g, device="cuda")[:n]]


def _vertices_with(keys, V, n, total, seed):
    """n vertices, drawn uniformly and then exchanged one by one until their rows hold `total` edges."""
    degree = torch.bincount(keys >> 32, minlength=V).cpu().numpy()
    rng = np.random.default_rng(seed)
    order = np.argsort(degree, kind="stable")
    by = degree[order]
    at = rng.integers(0, V, n)
    for i in range(n):
        over = int(degree[at].sum()) - total
        if over == 0:
            break
        k = min(int(np.searchsorted(by, max(0, int(degree[at[i]]) - over))), V - 1)
        at[i] = order[k]
    return torch.from_numpy(at.astype(np.int32)).to("cuda")


def _group_shapes(case):
    """(edges, vertices, batch) of every graph of a group; the sizes belong to the case, not to the seed."""
    rng = np.random.default_rng(case["sizes"])
    n = case["graphs"]
    shapes = []
    for e, b in zip(rng.uniform(math.log(case["edges_min"]), math.log(case["edges_max"]), n),
                    rng.lognormal(math.log(case["batch"]), 1.5, n)):
        edges = int(math.exp(e))
        V = max(128, edges // 16)
        batch = max(1, min(int(b), edges // 10))
        shapes.append((_settled(edges, V, batch, case), V, batch))
    return shapes


def _pma(case, V):
    ll, lr, ul, ur = DENSITY[case["density"]]
    return L.PMA(V, segment_slots=case["segment_slots"], density_lower=lr, density_upper=ur, density_lower_leaf=ll,
                 density_upper_leaf=ul)


class _Memory:
    """Device memory of a PMA's view, for torch: the tensor made from it keeps the PMA."""

    def __init__(self, pma, ptr, n, typestr):
        self.pma = pma
        self.__cuda_array_interface__ = {"shape": (int(n),), "typestr": typestr, "data": (int(ptr), False),
                                         "version": 2}


class _Graph:
    """A PMA and its gapped view as tensors, wrapped again only when its arrays move."""

    def __init__(self, pma):
        self.pma = pma
        self.at = None
        self.tensors = None

    def view(self):
        v = self.pma.view()
        at = (v.keys, v.capacity, v.row_offsets)
        if at != self.at:
            self.tensors = (torch.as_tensor(_Memory(self.pma, v.keys, v.capacity, "<i8"), device="cuda"),
                            torch.as_tensor(_Memory(self.pma, v.row_offsets, v.num_vertices + 1, "<i4"),
                                            device="cuda"))
            self.at = at
        return self.tensors


# Batches a streaming case goes round: a pass brings in the next one and takes
# out the one before, so the graph's size stays where it is.
ROUND = 6


def prepare(case, seed):
    kind = case["kind"]
    g = _generator(seed)
    state = {"kind": kind, "case": case, "at": 0}
    if kind == "group":
        members, rounds = [], [[] for _ in range(ROUND)]
        for e, V, b in _group_shapes(case):
            p = _pma(case, V)
            p.bulk_load(_graph_keys(V, e, g))
            keys = _rmat(V, ROUND * b, g)
            p.insert(keys[-b:])
            for r in range(ROUND):
                rounds[r].append(keys[r * b:(r + 1) * b].clone())
            members.append(p)
        state.update(group=L.Group(members), graphs=[_Graph(p) for p in members], rounds=rounds)
        return state
    V = case["vertices"]
    keys = _graph_keys(V, case["edges"], g)
    if kind == "build":
        state["keys"] = keys
        return state
    pma = _pma(case, V)
    pma.bulk_load(keys)
    state.update(pma=pma, graph=_Graph(pma))
    if kind in ("stream", "mixed"):
        state["batches"] = [_rmat(V, case["batch"], g) for _ in range(ROUND)]
        pma.insert(state["batches"][-1])
    elif kind == "sequence":
        state["batches"] = [[_rmat(V, case["batch"], g) for _ in range(case["requests"])] for _ in range(ROUND)]
        pma.insert(torch.cat(state["batches"][-1]))
    elif kind == "neighbors":
        n = case["queries"]
        state["srcs"] = _vertices_with(keys, V, n, round(n * case["edges"] / V), seed)
    elif kind == "edge_query":
        n = case["queries"]
        there = keys[torch.randint(0, keys.numel(), (n - n // 2,), generator=g, device="cuda")]
        both = torch.cat([there, _rmat(V, n // 2, g)]) if n > 1 else there
        state["queries"] = both[torch.randperm(both.numel(), generator=g, device="cuda")].contiguous()
    return state


# -------------------------------------------------------------------- pass


def run(state):
    kind = state["kind"]
    if kind in ("stream", "mixed", "sequence", "group"):
        at = state["at"]
        state["at"] = (at + 1) % ROUND
        if kind == "group":
            state["group"].update(state["rounds"][at], state["rounds"][at - 1])
            return [t for gr in state["graphs"] for t in gr.view()]
        new, old = state["batches"][at], state["batches"][at - 1]
        pma = state["pma"]
        if kind == "stream":
            pma.insert(new)
            pma.delete(old)
        elif kind == "mixed":
            pma.update_mixed(new, old)
        else:
            pma.update_sequence(list(zip(new, old)))
        return state["graph"].view()
    if kind == "build":
        case = state["case"]
        pma = _pma(case, case["vertices"])
        pma.bulk_load(state["keys"])
        return _Graph(pma).view()
    pma = state["pma"]
    if kind == "neighbors":
        return pma.neighbors(state["srcs"])
    if kind == "edge_query":
        return pma.edge_query(state["queries"])
    if kind == "export":
        return getattr(pma, state["case"]["form"])()
    if kind == "bfs":
        if state["case"]["form"] == "live":
            return pma.bfs(0)
        snap = L.Snapshot(pma)
        out = snap.bfs(0)
        snap.close()
        return out
    rank, iterations, _ = pma.pagerank(0.85, 1e-6, 50)
    return rank, iterations


# -------------------------------------------------------------------- work


def _update_bytes(batch, live, V, S):
    """Bytes of one batch: its keys, and the live keys of the segments it lands in, read and written."""
    nseg = 1 << max(0, math.ceil(math.log2(max(1.0, (live + V) / S))))
    hit = nseg * -math.expm1(-batch / nseg)
    return 8 * batch + 16 * hit * (live + V) / nseg


# edges of an R-MAT graph's rows and reach of a search are taken at their
# means: a row holds E / V edges, a search meets every edge
def work(case):
    kind, S = case["kind"], case["segment_slots"]
    if kind == "group":
        return {"bytes": sum(_update_bytes(2 * b, e, V, S) for e, V, b in _group_shapes(case)), "flops": 0}
    E, V = case["edges"], case["vertices"]
    if kind == "stream":
        n = 2 * _update_bytes(case["batch"], E, V, S)
    elif kind == "mixed":
        n = _update_bytes(2 * case["batch"], E, V, S)
    elif kind == "sequence":
        n = _update_bytes(2 * case["requests"] * case["batch"], E, V, S)
    elif kind == "build":
        n = 16 * E + 8 * V + 4 * V
    elif kind == "neighbors":
        n = case["queries"] * (4 + 4 + 12 * E / V)
    elif kind == "edge_query":
        n = case["queries"] * (8 + 4 + 8)
    elif kind == "export":
        written = {"export": 8 * E + 4 * V, "to_csr": 4 * (E + V) + 4 * V, "get_data": 8 * (E + V),
                   "copy_view": 8 * (E + V) + 4 * V}[case["form"]]
        n = 8 * (E + V) + written
    elif kind == "bfs":
        n = 8 * (E + V) + 4 * V + (16 * (E + V) if case["form"] == "snapshot" else 0)
    else:  # pagerank: about 20 iterations, each edge's source and destination and each vertex's rank
        return {"bytes": 20.0 * (8 * E + 12 * V), "flops": 20.0 * 2 * E}
    return {"bytes": float(n), "flops": 0}


# ------------------------------------------------------------------- exact


def exact(case, seed):
    """PageRank in 64 bits by plain torch; the other kinds compute no floating values."""
    if case["kind"] != "pagerank":
        return None
    V = case["vertices"]
    keys = _graph_keys(V, case["edges"], _generator(seed))
    src, dst = keys >> 32, keys & 0xFFFFFFFF
    del keys
    deg = torch.bincount(src, minlength=V).double()
    # edges by destination: a vertex's sum is a difference of running sums
    order = torch.sort(dst, stable=True).indices
    src = src[order]
    ends = torch.cumsum(torch.bincount(dst, minlength=V), 0)
    del dst, order
    alpha = 0.85
    rank = torch.full((V,), 1.0 / V, dtype=torch.float64, device="cuda")
    for _ in range(50):
        share = torch.where(deg > 0, rank / deg.clamp(min=1), torch.zeros_like(rank))
        run_sum = torch.cat([torch.zeros(1, dtype=torch.float64, device="cuda"), torch.cumsum(share[src], 0)])
        into = run_sum[ends]
        into = into - torch.cat([run_sum[:1], into[:-1]])
        lost = rank[deg == 0].sum()
        new = alpha * into + (alpha * lost + (1 - alpha) * rank.sum()) / V
        change = (new - rank).abs().sum()
        rank = new
        if change < 1e-6:
            break
    return rank / rank.abs().sum(), None
