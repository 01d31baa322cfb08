"""Measured workloads: what users of the library run, through its public Python API.

A case names a graph (R-MAT, Erdos-Renyi or a road-like grid; V need not be a
power of two), the algorithm run on it and the options in use.  Graphs are
drawn on the GPU by plain torch code from the seed alone and handed to the
library as host arrays (Context.borrow_arrays), the form a program that reads
its own files holds them in.  A program keeps the Context and the Graph (and
the Server) open and asks one query after another, so these are prepared once;
a pass is one query, its result array included.
"""
import math

import numpy as np
import torch

import ascetic_amd as A
from ascetic_amd import _abi

RMAT = (0.57, 0.19, 0.19, 0.05)     # quadrant probabilities of every R-MAT workload of this repository
PR_ITERATIONS = 20
DAMPING = 0.85
PR_THRESHOLD = 0.001


def listed():
    return [
        # one query of a small graph inside a larger program: launches and round trips are all of it
        dict(name="bfs_rmat12", algo="bfs", graph="rmat", v=1 << 12, ef=16, offset_bytes=4, source="random"),
        # BFS on R-MAT scale 20 from its hub with 4-byte offsets: the benchmark's per-algorithm BFS line
        dict(name="bfs_rmat20", algo="bfs", graph="rmat", v=1 << 20, ef=16, offset_bytes=4, source="hub"),
        # directed web-like graph, odd V, zero-based levels: no bottom-up steps, every level top-down
        dict(name="bfs_directed_rmat22", algo="bfs", graph="rmat", v=4_000_003, ef=16, directed=True, offset_bytes=8,
             source="hub", zero_based=True),
        # BFS beyond the device budget: edge factor 32, weights to 255 in the 5-byte split record form,
        # about a third resident (the shape of the benchmark's scale-30 run)
        dict(name="bfs_stream_rmat21", algo="bfs", graph="rmat", v=1 << 21, ef=32, wmax=255, offset_bytes=8,
             source="hub", resident=0.355, stream_pack=2),
        # SSSP on a fully resident social-network-like graph
        dict(name="sssp_rmat22", algo="sssp", graph="rmat", v=1 << 22, ef=16, wmax=64, offset_bytes=8, source="hub"),
        # shortest paths on a road-like mesh: thousands of small frontiers
        dict(name="sssp_grid", algo="sssp", graph="grid", v=1201 * 1033, rows=1201, wmax=255, offset_bytes=4,
             source="random"),
        # the headline: SSSP with a device edge budget of 40%, the rest streamed from host memory
        dict(name="sssp_stream_rmat23", algo="sssp", graph="rmat", v=1 << 23, ef=16, wmax=64, offset_bytes=8,
             source="hub", resident=0.4),
        # connected components: one giant component and many small ones, odd V
        dict(name="cc_rmat22", algo="cc", graph="rmat", v=4_000_037, ef=16, offset_bytes=8),
        # normalised PageRank, 20 iterations, on the benchmark's kind of graph (2^28 in-edges)
        dict(name="pr_er23", algo="pr", graph="er", v=1 << 23, ef=16, offset_bytes=8),
        # normalised PageRank on a graph whose ranks fit the caches
        dict(name="pr_rmat18", algo="pr", graph="rmat", v=1 << 18, ef=16, offset_bytes=4),
        # the drop-in PageRank form: FP64, active set, run to convergence
        dict(name="pr_reference_rmat20", algo="pr_reference", graph="rmat", v=1 << 20, ef=16, offset_bytes=8),
        # a batch of 64 queries, 70% BFS and 30% SSSP, submitted to an open server and waited for
        dict(name="serve_rmat19", algo="serve", graph="rmat", v=1 << 19, ef=16, wmax=64, offset_bytes=8, queries=64,
             lanes=64),
    ]


# algorithm -> (smallest V, largest V, most directed edges) of a drawn case
RANGES = {
    "bfs": (1 << 10, 4_200_000, 1 << 27),
    "sssp": (1 << 10, 4_200_000, 1 << 27),
    "cc": (1 << 10, 4_200_000, 1 << 27),
    "pr": (1 << 12, 1 << 23, 1 << 28),
    "pr_reference": (1 << 12, 1 << 20, 1 << 25),
    "serve": (1 << 12, 1 << 19, 1 << 24),
}


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    algo = rng.choice(["bfs", "bfs", "sssp", "sssp", "cc", "pr", "pr_reference", "serve"])
    lo, hi, most = RANGES[algo]
    v = _log_uniform(rng, lo, hi)
    if rng.random() < 0.4:
        v = 1 << (v.bit_length() - 1)   # a power of two, as the generators make them
    else:
        v |= 1
    ef = max(2, min(_log_uniform(rng, 4, 32), most // (2 * v)))
    graph = "rmat" if rng.random() < 0.6 else "er"
    case = dict(algo=algo, graph=graph, v=v, ef=ef, offset_bytes=rng.choice([4, 8]))
    if algo == "pr":
        case["directed"] = rng.random() < 0.25
        return case
    if algo == "pr_reference":
        return case
    if algo == "cc":
        case["directed"] = rng.random() < 0.25
        if graph == "er":
            case["ef"] = rng.randint(1, 3)   # sparse: several components at every V
        if rng.random() < 0.3:
            case["wmax"] = 64
        return case
    if algo == "serve":
        case.update(wmax=64, queries=rng.randint(8, 64), lanes=64)
        return case
    # bfs / sssp: one source
    case.update(source=rng.choice(["hub", "random"]), zero_based=rng.random() < 0.3)
    if algo == "sssp" or rng.random() < 0.4:
        case["wmax"] = rng.choice([8, 64, 255, 1000])
    form = rng.random()
    if form < 0.25 and v >= 1 << 16 and (algo == "bfs" or v * ef * 2 <= 1 << 26):
        case["resident"] = round(rng.uniform(0.2, 0.8), 3)
    elif form < 0.45:
        case["directed"] = True
    elif form < 0.6 and v >= 1 << 14:
        rows = int(round(math.sqrt(min(v, 1_200_000)) * rng.uniform(0.6, 1.4)))
        case.update(graph="grid", rows=rows, v=rows * (min(v, 1_200_000) // rows))
        case.pop("ef")
    return case


def _device():
    return torch.device("cuda") if torch.cuda.is_available() else torch.device("cpu")


def _sampled_pairs(case, seed):
    """The undirected (or directed) vertex pairs of a case, duplicates and self-loops included."""
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    V = case["v"]
    if case["graph"] == "grid":
        # rows x cols mesh; one street in ten is missing
        rows = case["rows"]
        cols = V // rows
        at = torch.arange(rows * cols, device=dev).reshape(rows, cols)
        u = torch.cat([at[:, :-1].reshape(-1), at[:-1, :].reshape(-1)])
        v = torch.cat([at[:, 1:].reshape(-1), at[1:, :].reshape(-1)])
        keep = torch.rand(u.numel(), device=dev, generator=gen) < 0.9
        return u[keep], v[keep]
    n = V * case["ef"]
    if case["graph"] == "er":
        return (torch.randint(0, V, (n,), device=dev, generator=gen),
                torch.randint(0, V, (n,), device=dev, generator=gen))
    a, b, c, _ = RMAT
    u = torch.zeros(n, dtype=torch.int32, device=dev)
    v = torch.zeros(n, dtype=torch.int32, device=dev)
    for _ in range((V - 1).bit_length()):
        r = torch.rand(n, device=dev, generator=gen)
        u = (u << 1) | (r >= a + b)
        v = (v << 1) | (((r >= a) & (r < a + b)) | (r >= a + b + c))
    inside = (u < V) & (v < V)
    return u[inside].long(), v[inside].long()


def _graph(case, seed):
    """CSR arrays of a case: offsets (V + 1), sorted neighbour ids or {dst, w} records, and for
    PageRank (an in-CSR) the out-degrees."""
    V = case["v"]
    in_csr = case["algo"].startswith("pr")
    u, v = _sampled_pairs(case, seed)
    loop = u == v
    u, v = u[~loop], v[~loop]
    if not case.get("directed"):
        u, v = torch.cat([u, v]), torch.cat([v, u])
    key = torch.unique(v * V + u if in_csr else u * V + v)
    del u, v
    rows = torch.arange(V + 1, device=key.device) * V
    off = torch.searchsorted(key, rows)
    out_degree = None
    row, dst = torch.div(key, V, rounding_mode="floor"), key % V
    del key
    if in_csr:
        out_degree = torch.bincount(dst, minlength=V) if case.get("directed") else off[1:] - off[:-1]
        out_degree = out_degree.to(torch.int32).cpu().numpy().view(np.uint32)
    if case.get("wmax"):
        # one weight per unordered pair, uniform in [1, wmax]
        lo, hi = torch.minimum(row, dst), torch.maximum(row, dst)
        h = (lo * 0x9E3779B97F4A7C1 + hi * 0x5851F42D4C957F2D) ^ (seed * 0x2545F4914F6CDD1D & 0x7FFFFFFFFFFFFFFF)
        h = (h ^ (h >> 29)) * 0x369DEA0F31A53F85
        w = ((h >> 32) & 0x7FFFFFFF) % case["wmax"] + 1
        edges = torch.stack([dst.to(torch.int32), w.to(torch.int32)], dim=1)
    else:
        edges = dst.to(torch.int32)
    edges = edges.cpu().numpy().view(np.uint32)
    off = off.cpu().numpy().astype(np.uint32 if case["offset_bytes"] == 4 else np.uint64)
    return off, edges, out_degree


class State:
    """What a program keeps open between queries; closed with its last reference."""

    def __init__(self, case, seed):
        self.case, self.server, self.graph, self.ctx = case, None, None, None
        off, edges, out_degree = _graph(case, seed)
        if _device().type == "cuda":
            torch.cuda.empty_cache()   # the library allocates beside torch
        options = {}
        if case.get("resident"):
            options["edge_budget_bytes"] = int(case["resident"] * edges.nbytes)
        if case.get("zero_based"):
            options["value_convention"] = _abi.VALUES_ZERO_BASED
        if case.get("stream_pack"):
            options["stream_pack"] = case["stream_pack"]
        self.ctx = A.Context(**options)
        self.graph = self.ctx.borrow_arrays(off, edges, out_degree=out_degree)
        degree = np.diff(off.astype(np.int64))
        rng = np.random.default_rng(seed)
        reach = np.flatnonzero(degree)
        self.source = 0
        if case.get("source") == "hub":
            self.source = int(np.argmax(degree))
        elif case.get("source") == "random":
            self.source = int(rng.choice(reach))
        if case["algo"] == "serve":
            self.server = A.Server(self.graph, lanes=case["lanes"])
            kinds = np.where(rng.random(case["queries"]) < 0.7, A.Server.BFS, A.Server.SSSP)
            sources = rng.choice(reach, case["queries"])
            self.queries = [(int(k), int(s), np.empty(case["v"], np.uint32)) for k, s in zip(kinds, sources)]

    def close(self):
        for part in (self.server, self.graph, self.ctx):
            if part is not None:
                part.close()
        self.server = self.graph = self.ctx = None

    def __del__(self):
        self.close()


def prepare(case, seed):
    return State(case, seed)


def run(state):
    algo, g = state.case["algo"], state.graph
    if algo == "bfs":
        return g.bfs(state.source)[0]
    if algo == "sssp":
        return g.sssp(state.source)[0]
    if algo == "cc":
        return g.cc()[0]
    if algo == "pr":
        return g.pagerank(damping=DAMPING, iterations=PR_ITERATIONS)[0]
    if algo == "pr_reference":
        return g.pagerank(mode=_abi.PR_REFERENCE, damping=DAMPING, threshold=PR_THRESHOLD)[0]
    tickets = [state.server.submit(kind, source, out) for kind, source, out in state.queries]
    for t in tickets:
        state.server.wait(t)
    return [out for _, _, out in state.queries]


def _edges(case):
    """Directed edges, duplicates not taken off."""
    if case["graph"] == "grid":
        return int(0.9 * 4 * case["v"])
    return case["v"] * case["ef"] * (1 if case.get("directed") else 2)


def work(case):
    """The graph read and the values written once; PageRank once per iteration (its in-edges, ranks and
    contributions do not stay on the chip); a served batch reads the graph once per kind of query."""
    V, E = case["v"], _edges(case)
    record = 8 if case.get("wmax") else 4
    graph = E * record + V * case["offset_bytes"]
    if case["algo"] == "pr":
        return {"bytes": PR_ITERATIONS * (graph + 16 * V), "flops": PR_ITERATIONS * 2 * E}
    if case["algo"] == "pr_reference":
        # about 20 sweeps to the threshold, FP64 contributions
        return {"bytes": 20 * (graph + 16 * V) + 8 * V, "flops": 20 * 2 * E}
    if case["algo"] == "serve":
        return {"bytes": 2 * graph + 4 * V * case["queries"], "flops": 0}
    return {"bytes": graph + 4 * V, "flops": 0}


def exact(case, seed):
    """PageRank in FP64 by torch; the other algorithms return whole numbers."""
    if not case["algo"].startswith("pr"):
        return None
    off, src, out_degree = _graph(case, seed)
    dev, V = _device(), case["v"]
    off = torch.from_numpy(off.astype(np.int64)).to(dev)
    src = torch.from_numpy(src.view(np.int32)).to(dev).long()
    out = torch.from_numpy(out_degree.view(np.int32)).to(dev).double()
    rank = torch.full((V,), 1.0 / V, dtype=torch.float64, device=dev)

    def pulled(r):
        share = torch.where(out > 0, r / out.clamp(min=1), torch.zeros_like(r))
        return torch.segment_reduce(share[src], "sum", offsets=off, initial=0.0)

    if case["algo"] == "pr":
        for _ in range(PR_ITERATIONS):
            lost = rank[out == 0].sum()
            rank = (1 - DAMPING) / V + DAMPING * (pulled(rank) + lost / V)
        return rank.cpu()
    # active-set form: a vertex that moves by no more than the threshold keeps its value and stops
    active = torch.ones(V, dtype=torch.bool, device=dev)
    while bool(active.any()):
        new = 0.15 + DAMPING * pulled(rank)
        moved = active & ((new - rank).abs() > PR_THRESHOLD)
        rank = torch.where(moved, new, rank)
        active = moved
    return rank.cpu()
