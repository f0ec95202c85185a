"""The graph queries that this library is timed on.

Every case is one query on a graph that is already resident in HBM, issued
through the public Python binding or, where a device result is wanted that
the binding would copy to the host, through the C ABI under it: the way
bench.py and the server use the library.  Graphs are the two families of the
benchmark: Kronecker (RMAT .57/.19/.19, vertices in order of falling degree)
and uniform random, symmetrised, without self-loops and duplicates, integer
weights uniform in [1, 255].  They are built on the GPU with torch, from the
seed alone, and handed over as a host CSR, because that is what the library
takes.
"""
import ctypes
import importlib
import math

import numpy as np
import torch

hc = importlib.import_module("hetero-compute_amd")

INF = hc.INF_DIST
WIDTH = hc.MULTI_WIDTH

# Largest vertices * edge factor of a drawn case per query kind (the listed
# cases' largest), and its vertex range.
_LIMITS = {
    "bfs": (1 << 12, 1 << 23, 1 << 27),
    "sssp": (1 << 12, 1 << 23, 1 << 27),
    "sssp_pull": (1 << 14, 1 << 20, 1 << 24),
    "pagerank": (1 << 14, 1 << 24, 1 << 28),
    "sssp_multi": (1 << 14, 1 << 22, 1 << 24),
    "bfs_multi": (1 << 14, 1 << 22, 1 << 26),
}


def listed():
    return [
        # The smallest single queries: a serving request on a small graph,
        # the result wanted on the host.  Launches and latency decide.
        dict(name="bfs_kron_4k", algo="bfs", graph="kron", n=1 << 12, degree=16, sources=1, fetch=True),
        dict(name="sssp_kron_64k", algo="sssp", graph="kron", n=1 << 16, degree=16, sources=1, fetch=True),
        # The headline: direction-optimizing BFS and SSSP on a skewed graph
        # of 2^23 vertices and about 259 M directed edges.
        dict(name="bfs_kron_8m", algo="bfs", graph="kron", n=1 << 23, degree=16, sources=1, fetch=False),
        dict(name="sssp_kron_8m", algo="sssp", graph="kron", n=1 << 23, degree=16, sources=1, fetch=False),
        # The same queries on a graph without hubs (many light levels and
        # buckets), of a ragged size for BFS.
        dict(name="bfs_uniform_5m", algo="bfs", graph="uniform", n=5_000_011, degree=16, sources=1, fetch=False),
        dict(name="sssp_uniform_8m", algo="sssp", graph="uniform", n=1 << 23, degree=16, sources=1, fetch=False),
        # The pull-only driver of the reference (initial distances in, no
        # direction switch), ragged and of another edge factor.
        dict(name="sssp_pull_kron_900k", algo="sssp_pull", graph="kron", n=900_001, degree=12, sources=1, fetch=False),
        # PageRank to an L1 residual of 1e-4: the benchmark's graph, and an
        # ordinary flat one.
        dict(name="pagerank_kron_16m", algo="pagerank", graph="kron", n=1 << 24, degree=16, sources=0, fetch=False),
        dict(name="pagerank_uniform_1m", algo="pagerank", graph="uniform", n=1_000_003, degree=10, sources=0,
             fetch=False),
        # Batched queries: 64 sources of one graph in one sweep.
        dict(name="sssp_multi_kron_1m", algo="sssp_multi", graph="kron", n=1 << 20, degree=16, sources=64, fetch=False),
        dict(name="bfs_multi_kron_4m", algo="bfs_multi", graph="kron", n=1 << 22, degree=16, sources=64, fetch=False),
        # 512 small graphs of uneven size (scale 10 to 16, edge factor 8 to
        # 32), one BFS each, in one launch.
        dict(name="bfs_many_512", algo="bfs_many", graph="kron", n=1 << 16, degree=32, sources=512, fetch=False),
    ]


def draw(rng):
    algo = rng.choice(["bfs", "bfs", "sssp", "sssp", "sssp_pull", "pagerank", "sssp_multi", "bfs_multi", "bfs_many"])
    if algo == "bfs_many":
        # n and degree are the largest graph's.
        return dict(algo=algo, graph="kron", n=int(2 ** rng.uniform(11, 16)), degree=rng.randint(9, 32),
                    sources=rng.randint(32, 512), fetch=False)
    low, high, edges = _LIMITS[algo]
    n = int(2 ** rng.uniform(math.log2(low), math.log2(high))) | 1
    degree = min(rng.randint(4, 32), max(4, edges // n))
    return dict(
        algo=algo,
        graph=rng.choice(["kron", "uniform"]),
        n=min(n, edges // degree),
        degree=degree,
        sources={"pagerank": 0, "sssp_multi": rng.randint(33, 64), "bfs_multi": rng.randint(33, 64)}.get(algo, 1),
        fetch=n < 1 << 18 and algo in ("bfs", "sssp"),
    )


# ---------------------------------------------------------------------------
# Graphs
# ---------------------------------------------------------------------------

def _random_edges(kind, n, degree, gen):
    """Endpoints of n * degree random edges (loops and repeats among them)."""
    count = n * degree
    if kind == "uniform":
        u = torch.randint(0, n, (count,), device="cuda", generator=gen, dtype=torch.int32)
        v = torch.randint(0, n, (count,), device="cuda", generator=gen, dtype=torch.int32)
        return u, v
    u = torch.zeros(count, device="cuda", dtype=torch.int32)
    v = torch.zeros(count, device="cuda", dtype=torch.int32)
    for _ in range(max(1, (n - 1).bit_length())):
        r = torch.rand(count, device="cuda", generator=gen)
        low = r > 0.76
        u.mul_(2).add_(low)
        v.mul_(2).add_(((r > 0.57) & ~low) | (r > 0.95))
    if n & (n - 1):
        u %= n
        v %= n
    # Vertex ids carry no order of their own.
    perm = torch.randperm(n, device="cuda", generator=gen, dtype=torch.int32)
    return perm[u], perm[v]


def _symmetric_keys(u, v, n):
    """Sorted distinct u * n + v of the edges in both directions."""
    keep = u != v
    u, v = u[keep].long(), v[keep].long()
    key = torch.cat([u * n + v, v * n + u])
    del u, v
    return torch.unique_consecutive(key.sort().values)


def _csr(kind, n, degree, gen):
    """(offsets int64[n + 1], neighbours int32[m]) on the GPU, neighbours in
    rising order, vertices in order of falling degree."""
    key = _symmetric_keys(*_random_edges(kind, n, degree, gen), n)
    row = torch.div(key, n, rounding_mode="floor")
    deg = torch.bincount(row, minlength=n)
    rank = torch.empty(n, device="cuda", dtype=torch.int64)
    rank[deg.sort(descending=True, stable=True).indices] = torch.arange(n, device="cuda")
    key = rank[row] * n + rank[key - row * n]
    del row
    key = key.sort().values
    row = torch.div(key, n, rounding_mode="floor")
    off = torch.zeros(n + 1, device="cuda", dtype=torch.int64)
    torch.cumsum(torch.bincount(row, minlength=n), 0, out=off[1:])
    return off, (key - row * n).int()


def _rows(off):
    return torch.repeat_interleave(torch.arange(off.numel() - 1, device="cuda"), off.diff())


def _weights(off, adj, seed):
    """int32 weights in [1, 255], the same in both directions of an edge."""
    u, v = _rows(off), adj.long()
    x = torch.minimum(u, v) * 0x5851F42D + torch.maximum(u, v) * 0x14057B7E + seed * 0x2545F491
    del u, v
    x = (x ^ (x >> 29)) * 0x3C79AC49
    x = (x ^ (x >> 31)) * 0x1CE4E5B9
    return ((x >> 24) % 255 + 1).int()


def _host(off, adj, wt=None):
    return hc.HostGraph.from_csr(off.cpu().numpy(), adj.cpu().numpy(), None if wt is None else wt.cpu().numpy())


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _sources(off, count, seed):
    """`count` random vertices that have neighbours."""
    have = torch.nonzero(off.diff()).flatten()
    at = torch.randint(0, have.numel(), (count,), device="cuda", generator=_generator(seed + 7))
    return [int(v) for v in have[at].cpu()]


def _graph(case, seed):
    """(offsets, neighbours, weights or None) of a one-graph case."""
    off, adj = _csr(case["graph"], case["n"], case["degree"], _generator(seed))
    return off, adj, _weights(off, adj, seed) if case["algo"].startswith("sssp") else None


def _many_sizes(case):
    """(vertices, edge factor) of each graph of a many-graph case: scales
    from 10 to the largest, edge factors from 8 to the largest, at random."""
    rng = np.random.default_rng([case["n"], case["degree"], case["sources"]])
    top = math.log2(case["n"])
    sizes = [(int(round(2 ** rng.uniform(10, top))), int(rng.integers(8, case["degree"] + 1)))
             for _ in range(case["sources"])]
    return sizes[:-1] + [(case["n"], case["degree"])]


def _many(case, seed):
    """(offsets, neighbours) of each graph of a many-graph case on the host,
    and one source per graph."""
    rng = np.random.default_rng(seed)
    gen = _generator(seed)
    graphs, sources = [], []
    for n, degree in _many_sizes(case):
        off, adj = (x.cpu().numpy() for x in _csr("kron", n, degree, gen))
        graphs.append((off, adj))
        have = np.flatnonzero(np.diff(off))
        sources.append(int(have[rng.integers(0, have.size)]))
    return graphs, sources


# ---------------------------------------------------------------------------
# Queries
# ---------------------------------------------------------------------------

class _Out:
    """A torch tensor where the binding takes a device array."""

    def __init__(self, shape, dtype):
        self.tensor = torch.empty(shape, device="cuda", dtype=dtype)
        self.ptr = ctypes.c_void_p(self.tensor.data_ptr())


def prepare(case, seed):
    state = dict(case)
    n, algo = case["n"], case["algo"]
    if algo == "bfs_many":
        graphs, state["sources"] = _many(case, seed)
        state["batch"] = hc.GraphBatch([hc.HostGraph.from_csr(*g) for g in graphs])
        state["out"] = _Out(state["batch"].total_nodes, torch.int32)
        return state
    off, adj, wt = _graph(case, seed)
    state["graph"] = hc.DeviceGraph(_host(off, adj, wt))
    state["sources"] = _sources(off, case["sources"], seed)
    del off, adj, wt
    torch.cuda.empty_cache()
    if algo == "pagerank":
        state["out"] = _Out(n, torch.float32)
    elif algo.endswith("_multi"):
        state["out"] = _Out((n, WIDTH), torch.int32)
    elif not case["fetch"]:
        state["out"] = _Out(n, torch.int32)
    if algo == "sssp_pull":
        state["init"] = torch.full((n,), INF, device="cuda", dtype=torch.int32)
        state["init"][state["sources"][0]] = 0
    return state


def run(state):
    algo, out = state["algo"], state.get("out")
    if algo == "bfs_many":
        state["batch"].bfs(state["sources"], want_parents=False, depth=out, fetch=False)
        return out.tensor
    g = state["graph"]
    if algo == "bfs":
        r = hc.bfs(g, state["sources"][0], want_parents=False, depth_out=out, fetch=state["fetch"])
        return r.values if state["fetch"] else out.tensor
    if algo == "sssp":
        r = hc.sssp(g, state["sources"][0], out=out, fetch=state["fetch"])
        return r.values if state["fetch"] else out.tensor
    if algo == "sssp_multi":
        hc.sssp_multi(g, state["sources"], out=out, fetch=False)
    elif algo == "bfs_multi":
        hc.bfs_multi(g, state["sources"], out=out, fetch=False)
    elif algo == "sssp_pull":
        # sssp_pull and pagerank leave their result on the device through the
        # C ABI only.
        hc.check(hc.lib().hc_sssp_pull(g.h, hc.MAP_BUCKETED, state["init"].data_ptr(), out.ptr, 0, 0,
                                       ctypes.byref(hc.RunStats()), None))
    else:
        opts = hc.PrOpts(0.85, 1e-4, 20, 0)
        hc.check(hc.lib().hc_pagerank(g.h, out.ptr, ctypes.byref(opts), ctypes.byref(hc.RunStats()), None))
    return out.tensor


# ---------------------------------------------------------------------------
# What a pass needs, and what it should say
# ---------------------------------------------------------------------------

def work(case):
    """Bytes of one pass, every input read once and every result written once,
    with 2 * n * degree directed edges (a little more than remain after
    duplicates go).  BFS need not look at every edge: offsets, one neighbour
    and the depth of every vertex; the single-source runs read ids and
    weights of all edges, PageRank ids and scores once per iteration, of
    which it takes about seven."""
    n, m = case["n"], 2 * case["n"] * case["degree"]
    if case["algo"] == "bfs":
        return {"bytes": 12 * n, "flops": 0}
    if case["algo"] == "bfs_many":
        return {"bytes": 12 * sum(size for size, _ in _many_sizes(case)), "flops": 0}
    if case["algo"] == "bfs_multi":
        return {"bytes": 4 * m + 4 * n + 4 * n * WIDTH, "flops": 0}
    if case["algo"] == "sssp_multi":
        return {"bytes": 8 * m + 4 * n + 4 * n * WIDTH, "flops": m * case["sources"]}
    if case["algo"] == "pagerank":
        return {"bytes": 7 * (4 * m + 16 * n), "flops": 7 * m}
    return {"bytes": 8 * m + 8 * n, "flops": m}


def tolerance(case):
    if case["algo"] == "pagerank":
        # FP32 scores from compensated sums: 3e-8 off the 64-bit iteration.
        return {"rel": 2e-7, "max": 2e-6}
    return "exact"


def _relax(off, adj, wt, sources):
    """Distances (weights; hops without them) from `sources` by rounds of
    relaxing every edge, as plain torch says it; -1 where none leads."""
    n = off.numel() - 1
    row = _rows(off)
    dist = torch.full((n,), 1 << 40, device="cuda", dtype=torch.int64)
    dist[torch.tensor(sources, device="cuda")] = 0
    step = 1 << 26
    while True:
        new = dist.clone()
        for i in range(0, adj.numel(), step):
            cand = dist[adj[i:i + step].long()] + (1 if wt is None else wt[i:i + step])
            new.scatter_reduce_(0, row[i:i + step], cand, "amin")
        if torch.equal(new, dist):
            return torch.where(dist < 1 << 40, dist, -1)
        dist = new


def _pagerank(off, adj):
    """Scores after the iteration whose L1 change is below 1e-4, in float64."""
    n = off.numel() - 1
    deg = off.diff().double()
    inv = torch.where(deg > 0, 1 / deg.clamp(min=1), 0.0)
    score = torch.full((n,), 1 / n, device="cuda", dtype=torch.float64)
    for _ in range(20):
        contrib = score * inv
        total = torch.empty_like(score)
        step = max(1, n // 8)
        for a in range(0, n, step):
            b = min(n, a + step)
            lo, hi = int(off[a]), int(off[b])
            total[a:b] = torch.segment_reduce(contrib[adj[lo:hi].long()], "sum", offsets=off[a:b + 1] - lo, initial=0.0)
        new = 0.15 / n + 0.85 * total
        change = float((new - score).abs().sum())
        score = new
        if change < 1e-4:
            break
    return score


def exact(case, seed):
    algo = case["algo"]
    if algo == "bfs_many":
        graphs, sources = _many(case, seed)
        base = np.cumsum([0] + [g[0].size - 1 for g in graphs])
        ends = np.cumsum([0] + [int(g[0][-1]) for g in graphs])
        off = np.concatenate([g[0][:-1] + e for g, e in zip(graphs, ends)] + [ends[-1:]])
        adj = np.concatenate([g[1] + b for g, b in zip(graphs, base)])
        return _relax(torch.from_numpy(off).cuda(), torch.from_numpy(adj).cuda(), None,
                      [s + int(b) for s, b in zip(sources, base)])
    off, adj, wt = _graph(case, seed)
    if algo == "pagerank":
        return _pagerank(off, adj)
    if algo.endswith("_multi"):
        if case["n"] * case["degree"] * case["sources"] > 1 << 27:
            return None  # one relaxation per source would take too long
        cols = [_relax(off, adj, wt, [s]) for s in _sources(off, case["sources"], seed)]
        out = torch.full((case["n"], WIDTH), -1, device="cuda", dtype=torch.int64)
        out[:, :len(cols)] = torch.stack(cols, 1)
        return torch.where(out < 0, INF, out).int()
    dist = _relax(off, adj, wt, _sources(off, 1, seed))
    return dist.int() if algo == "bfs" else torch.where(dist < 0, INF, dist).int()
