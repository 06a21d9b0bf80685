"""Timed cases of the graph runtime: what a program that uses it calls, from the smallest traversal to the largest.

A case is one pass through a public entry point (DeviceGraph.bfs / .sssp / .sssp_minplus / .color / .mis / .pagerank /
.bc, wgm_bfs_noalloc, Batch.run, Server) on a graph that stays resident, with its results in the caller's hands. The
graphs are the framework's workloads: Erdos-Renyi (latency-bound, configured at n = 2^16, average degree 8), RMAT (a, b,
c) = (.57, .19, .19) with edge factor 16 (skewed degrees; configured at scale 20), 4-neighbour grids with one link in
a hundred blocked (road-like: many narrow levels for the traversals; configured at 2048 x 2048 for the topology-driven
apps), weights in [1, 255]. Launch shapes are the benchmark's: 1024-thread workgroups at the discovered occupancy
(num_wgs 0) or 64 of them, 64 of 512, and 1024 of 256 for betweenness (one source each). Graphs are drawn on the GPU
from the seed.
"""
import ctypes

import numpy as np
import torch

from gpu_workgroup_managment_amd import _lib as L
from gpu_workgroup_managment_amd import batched as B
from gpu_workgroup_managment_amd import graphs as G
from gpu_workgroup_managment_amd import runtime as R
from gpu_workgroup_managment_amd import serving as S

INF = 1_000_000_000
# the benchmark's launch shape of a batch
BATCH = dict(wg_size=1024, wgs_per_cu=2, chunk=256, team_edges=1 << 20, max_team=16, delta=512, delta_high_degree=12,
             far_flags_lds=1, low_ell=2, sssp_team_edges=786432)

_runtime = None


def _rt():
    """The program's one runtime on the GPU."""
    global _runtime
    if _runtime is None:
        _runtime = R.Runtime(0)
    return _runtime


def listed():
    return [
        # a small query on device buffers, as a serving loop or a captured program makes it: latency alone
        dict(name="bfs_device_er_4k", app="bfs_device", graph="er", n=4096, degree=8, wg=256, wgs=64),
        # the configured BFS: nine short levels on a graph that fits the caches
        dict(name="bfs_er_64k", app="bfs", graph="er", n=1 << 16, degree=8, wg=512, wgs=64),
        # a large skewed graph from one source: a social or web graph's hop distances
        dict(name="bfs_rmat_20", app="bfs", graph="rmat", n=1 << 20, degree=16, wg=1024, wgs=0),
        # the configured SSSP (the pull direction on this graph)
        dict(name="sssp_rmat_20", app="sssp", graph="rmat", n=1 << 20, degree=16, wg=1024, wgs=0),
        # road-like traversals (here SSSP: push, near-far bands): hundreds of narrow levels, ragged sides
        dict(name="sssp_grid_361x415", app="sssp", graph="grid", rows=361, cols=415, wg=1024, wgs=64),
        # the configured colouring of a mesh
        dict(name="color_grid_2048", app="color", graph="grid", rows=2048, cols=2048, wg=1024, wgs=0),
        # an independent set of a skewed undirected graph: rows from one edge to thousands
        dict(name="mis_rmat_17", app="mis", graph="rmat_sym", n=1 << 17, degree=16, wg=1024, wgs=0),
        # the configured PageRank
        dict(name="pagerank_grid_2048", app="pagerank", graph="grid", rows=2048, cols=2048, iterations=50, wg=1024,
             wgs=0),
        # PageRank of a skewed undirected graph, as of links between pages or people
        dict(name="pagerank_rmat_17", app="pagerank", graph="rmat_sym", n=1 << 17, degree=16, iterations=50, wg=1024,
             wgs=0),
        # betweenness of every vertex of a small skewed graph, the size its configuration names
        dict(name="bc_rmat_12", app="bc", graph="rmat", n=1 << 12, degree=8, sources=1 << 12, wg=256, wgs=1024),
        # many graphs of mixed size and kind in one launch
        dict(name="batch_60", app="batch", count=60, lo=10, hi=18, spec=5),
        # a query server's session: start, a burst of queries with tasks between them, drain, stop
        dict(name="serve_192", app="serve", count=64, lo=10, hi=15, spec=7, requests=192, tasks=6),
    ]


def _size(rng, lo, hi):
    """An odd size, log-uniform in [lo, hi]."""
    return int(round(lo * (hi / lo) ** rng.random())) | 1


def draw(rng):
    app = rng.choice(["bfs_device", "bfs", "bfs", "bfs", "sssp", "sssp", "sssp_minplus", "color", "mis", "pagerank",
                      "bc", "batch", "serve"])
    wg, wgs = rng.choice([(1024, 0), (1024, 0), (1024, 64), (512, 64)])
    if app == "batch":
        return dict(app=app, count=rng.randrange(12, 61), lo=rng.randrange(8, 12), hi=rng.randrange(14, 19),
                    spec=rng.randrange(1, 1 << 20))
    if app == "serve":
        return dict(app=app, count=rng.randrange(8, 65), lo=rng.randrange(8, 11), hi=rng.randrange(12, 16),
                    spec=rng.randrange(1, 1 << 20), requests=rng.randrange(32, 193), tasks=rng.randrange(0, 7))
    if app == "bc":
        n = _size(rng, 500, 4096)
        return dict(app=app, graph=rng.choice(["rmat", "er", "grid"]), n=n, rows=int(n ** 0.5), cols=int(n ** 0.5) + 3,
                    degree=8, sources=rng.randrange(max(1, n // 8), n // 2), wg=256, wgs=1024)
    kinds = {"bfs_device": ["er", "rmat"], "bfs": ["er", "rmat", "grid"], "sssp": ["er", "rmat", "grid"],
             "sssp_minplus": ["er", "rmat"], "color": ["grid", "er", "rmat_sym"], "mis": ["grid", "er", "rmat_sym"],
             "pagerank": ["grid", "er", "rmat_sym"]}[app]
    graph = rng.choice(kinds)
    case = dict(app=app, graph=graph, wg=wg, wgs=wgs)
    if graph == "grid":  # a traversal's levels grow with the sides; the topology-driven apps take whole meshes
        top = 512 if app in ("bfs", "sssp") else 2047
        case["rows"], case["cols"] = _size(rng, 65, top), _size(rng, 65, top)
    elif graph == "er":
        case["n"], case["degree"] = _size(rng, 1 << 12, 1 << 18), rng.choice([4, 8, 16])
    elif graph == "rmat":
        case["n"], case["degree"] = _size(rng, 1 << 13, 1 << 19), rng.choice([8, 16])
    else:
        case["n"], case["degree"] = _size(rng, 1 << 12, 1 << 17), rng.choice([8, 16])
    if app == "pagerank":
        case["iterations"] = rng.randrange(10, 51)
    return case


# ------------------------------------------------------------------ inputs
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _csr_from_keys(n, key):
    """row_ptr and col (int32, rows ascending) of the sorted distinct keys src * n + dst."""
    src, dst = torch.div(key, n, rounding_mode="floor"), key % n
    row = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    row[1:] = torch.cumsum(torch.bincount(src, minlength=n), 0)
    return row.to(torch.int32), dst.to(torch.int32)


def _pairs(case, seed):
    """Distinct non-loop arcs of a random graph, as sorted keys src * n + dst."""
    n, gen = case["n"], _gen(seed)
    m = n * case["degree"]
    if case["graph"] == "er":  # undirected pairs, both arcs
        a = torch.randint(n, (m // 2,), device="cuda", generator=gen)
        b = torch.randint(n, (m // 2,), device="cuda", generator=gen)
        a, b = torch.cat([a, b]), torch.cat([b, a])
    else:
        a = torch.zeros(m, dtype=torch.int64, device="cuda")
        b = torch.zeros(m, dtype=torch.int64, device="cuda")
        for _ in range((n - 1).bit_length()):  # (.57, .19, .19, .05), one quadrant per bit
            r = torch.rand(m, device="cuda", generator=gen)
            a = 2 * a + (r >= 0.76)
            b = 2 * b + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        if case["graph"] == "rmat_sym":
            a, b = torch.cat([a, b]), torch.cat([b, a])
    keep = (a != b) & (a < n) & (b < n)
    return torch.unique(a[keep] * n + b[keep])


def _links(rows, cols, seed):
    """Arcs of a rows x cols 4-neighbour grid (id = r * cols + c) with one link in a hundred blocked, as sorted keys."""
    n, gen = rows * cols, _gen(seed)
    ids = torch.arange(n, device="cuda").view(rows, cols)
    a = torch.cat([ids[:, :-1].reshape(-1), ids[:-1, :].reshape(-1)])
    b = torch.cat([ids[:, 1:].reshape(-1), ids[1:, :].reshape(-1)])
    keep = torch.rand(len(a), device="cuda", generator=gen) >= 0.01
    a, b = a[keep], b[keep]
    return torch.sort(torch.cat([a * n + b, b * n + a])).values


def _graph(case, seed):
    """(row_ptr, col) of a case as int32 numpy arrays."""
    if case["graph"] == "grid":
        n = case["rows"] * case["cols"]
        key = _links(case["rows"], case["cols"], seed)
    else:
        n, key = case["n"], _pairs(case, seed)
    row, col = _csr_from_keys(n, key)
    return row.cpu().numpy(), col.cpu().numpy()


def _source(case, row, seed):
    """A vertex that has edges (a user asks about a vertex of the graph's body); a mesh's first row."""
    deg = np.diff(row)
    rng = np.random.default_rng(seed)
    if case["graph"] == "grid":
        return int(rng.choice(np.flatnonzero(deg[: case["cols"]] > 0)))
    return int(rng.choice(np.flatnonzero(deg >= max(1, int(deg.mean())))))


def _inputs(case, seed):
    row, col = _graph(case, seed)
    g = G.CSR(row, col)
    if case["app"] in ("sssp", "sssp_minplus"):
        g.wt = np.random.default_rng(seed + 1).integers(1, 256, g.m).astype(np.int32)
    if case["app"] in ("color", "mis"):
        g.prio = np.random.default_rng(seed + 2).permutation(g.n).astype(np.uint32)
    return g, _source(case, row, seed + 3)


def _batch_graphs(case, seed):
    """Graphs and queries of a mixed batch: sizes, kinds and queries from the batch spec, contents from the seed."""
    graphs, queries = [], []
    for k, it in enumerate(G.batch_spec(case["count"], case["spec"], case["lo"], case["hi"])):
        kind = "grid" if it.kind == L.GRAPH_GRID else "rmat"
        g = G.CSR(*_graph(dict(graph=kind, rows=it.rows, cols=it.cols, n=it.n, degree=16), seed * 1000 + k))
        g.wt = np.random.default_rng(seed * 1000 + k).integers(1, 256, g.m, dtype=np.int32)
        graphs.append(g)
        queries.append(it.query)
    return graphs, np.array(queries, np.int32)


def prepare(case, seed):
    rt = _rt()
    app = case["app"]
    if app in ("batch", "serve"):
        graphs, queries = _batch_graphs(case, seed)
        if app == "batch":
            return dict(app=app, batch=B.Batch(rt, graphs, queries), cfg=B.config(use_graph=True, **BATCH))
        rng = np.random.default_rng(seed)
        asked = [(i, int(queries[i]), int(rng.integers(0, graphs[i].n)))
                 for i in rng.integers(0, len(graphs), case["requests"]).tolist()]
        server = S.Server(rt, graphs, S.config(wg_size=1024, max_inflight=256, reserve=16, budget_bytes=8 << 30))
        return dict(app=app, server=server, asked=asked, tasks=case["tasks"])
    g, src = _inputs(case, seed)
    st = dict(app=app, src=src, shape=dict(wg_size=case["wg"], num_wgs=case["wgs"]), case=case)
    if app == "bfs_device":
        st["row"], st["col"] = torch.from_numpy(g.row_ptr).cuda(), torch.from_numpy(g.col).cuda()
        st["dist"] = torch.empty(g.n, dtype=torch.int32, device="cuda")
        st["n"], st["m"], st["rt"] = g.n, g.m, rt
        torch.cuda.synchronize()
    else:
        st["graph"] = rt.graph(g)
    return st


def run(st):
    app = st["app"]
    if app == "bfs_device":
        lc, stats = L.Launch(), L.RunStats()
        lc.wg_size, lc.num_wgs = st["shape"]["wg_size"], st["shape"]["num_wgs"]
        L.check(L.lib().wgm_bfs_noalloc(st["rt"].handle, st["row"].data_ptr(), st["col"].data_ptr(), st["n"], st["m"],
                                        st["src"], ctypes.byref(lc), st["dist"].data_ptr(), ctypes.byref(stats)),
                st["rt"].handle)
        return st["dist"], int(stats.iterations), int(stats.edges_scanned)
    if app == "batch":
        batch = st["batch"]
        stats = batch.run(st["cfg"])
        return [batch.result(i)[0] for i in range(len(batch.graphs))], int(stats["edges_scanned"])
    if app == "serve":
        server, asked, done = st["server"], st["asked"], []
        server.start()
        per = len(asked) // (st["tasks"] + 1) + 1
        first, oks = None, []
        for k, (graph, query, src) in enumerate(asked):
            i = server.submit(graph, query, src)
            first = i if first is None else first
            if k % per == per - 1:
                kind = S.NP_MATMUL_F32 if len(oks) % 2 == 0 else S.NP_REDUCE_MIN
                oks.append(int(server.task(kind, 16)["ok"]))
                done += server.poll()
        done += server.drain()
        server.stop()
        out = np.zeros((len(asked), 3), np.int64)  # per request: digest of its distances, vertices reached, edges
        for r in done:
            out[r["id"] - first] = np.array([r["digest"], r["reached"], r["edges_scanned"]], np.uint64).astype(np.int64)
        return out, oks
    g, shape, case = st["graph"], st["shape"], st["case"]
    if app == "bfs":
        dist, stats = g.bfs(st["src"], **shape)
        return dist, stats["iterations"], stats["edges_scanned"]
    if app == "sssp":
        dist, stats = g.sssp(st["src"], **shape)
        return dist, stats["edges_scanned"]
    if app == "sssp_minplus":
        return g.sssp_minplus(st["src"], **shape)[0]
    if app == "color":
        out, stats = g.color(**shape)
        return out, stats["iterations"]
    if app == "mis":
        out, stats = g.mis(**shape)
        return out, stats["iterations"]
    if app == "pagerank":
        return g.pagerank(0.85, case["iterations"], **shape)[0]
    return g.bc(case["sources"], **shape)[0]


# ------------------------------------------------------------------- work
def _nm(case):
    if case["graph"] == "grid":
        r, c = case["rows"], case["cols"]
        return r * c, 2 * (r * (c - 1) + c * (r - 1))
    return case["n"], case["n"] * case["degree"] * (2 if case["graph"] == "rmat_sym" else 1)


def work(case):
    """Graph read once, result written once; PageRank and BC count their arithmetic too."""
    if case["app"] in ("batch", "serve"):
        tot = 0
        for it in G.batch_spec(case["count"], case["spec"], case["lo"], case["hi"]):
            n, m = (it.n, 4 * it.n) if it.kind == L.GRAPH_GRID else (it.n, 16 * it.n)
            tot += 8 * n + (8 if it.query == L.QUERY_SSSP else 4) * m
        if case["app"] == "serve":
            tot = tot * case["requests"] / case["count"]
        return dict(bytes=tot, flops=0)
    n, m = _nm(case)
    per_n = {"color": 12, "mis": 12, "bc": 12}.get(case["app"], 8)
    per_m = 8 if case["app"] in ("sssp", "sssp_minplus") else 4
    flops = {"pagerank": 2 * m * case.get("iterations", 0), "bc": 4 * m * case.get("sources", 0)}.get(case["app"], 0)
    return dict(bytes=per_n * n + per_m * m, flops=flops)


# ------------------------------------------------------------------ exact
def _minplus(n, src, dst, wt, s):
    """Distances from s by relaxing every arc until nothing falls."""
    d = torch.full((n,), INF, dtype=torch.int64, device="cuda")
    d[s] = 0
    while True:
        new = d.scatter_reduce(0, dst, d[src] + wt, "amin")
        if torch.equal(new, d):
            return d
        d = new


def _pagerank(n, src, dst, deg, iterations):
    # rank(v) = (1 - d) / n + d * sum over v's row of rank(u) / deg(u), with the damping the entry point gets (float32)
    d = float(np.float32(0.85))
    inv = torch.where(deg > 0, 1.0 / deg.clamp(min=1).double(), 0.0)
    r = torch.full((n,), 1.0 / n, dtype=torch.float64, device="cuda")
    for _ in range(iterations):
        s = torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, src, (r * inv)[dst])
        r = (1.0 - d) / n + d * s
    return r


def _bc(n, src, dst, sources):
    """Brandes' dependencies summed over the sources, all sources at once as the columns of dense matrices."""
    ones = torch.ones(len(src), dtype=torch.float64, device="cuda")
    out_adj = torch.sparse_coo_tensor(torch.stack([src, dst]), ones, (n, n)).coalesce()
    in_adj = torch.sparse_coo_tensor(torch.stack([dst, src]), ones, (n, n)).coalesce()
    total = torch.zeros(n, dtype=torch.float64, device="cuda")
    for a in range(0, sources, 1024):
        s = torch.arange(a, min(a + 1024, sources), device="cuda")
        k = torch.arange(len(s), device="cuda")
        level = torch.full((n, len(s)), -1, dtype=torch.int64, device="cuda")
        sigma = torch.zeros((n, len(s)), dtype=torch.float64, device="cuda")
        level[s, k], sigma[s, k] = 0, 1.0
        depth = 0
        while True:
            nxt = torch.sparse.mm(in_adj, torch.where(level == depth, sigma, 0.0))
            new = (level < 0) & (nxt > 0)
            if not bool(new.any()):
                break
            depth += 1
            level[new] = depth
            sigma = torch.where(new, nxt, sigma)
        delta = torch.zeros_like(sigma)
        for lv in range(depth - 1, -1, -1):
            coef = torch.where(level == lv + 1, (1.0 + delta) / sigma.clamp(min=1.0), 0.0)
            delta = torch.where(level == lv, sigma * torch.sparse.mm(out_adj, coef), delta)
        delta[s, k] = 0.0
        total += delta.sum(1)
    return total


def exact(case, seed):
    app = case["app"]
    if app in ("batch", "serve", "color", "mis"):  # whole numbers throughout
        return None
    g, s = _inputs(case, seed)
    deg = torch.from_numpy(np.diff(g.row_ptr)).cuda().long()
    src = torch.repeat_interleave(torch.arange(g.n, device="cuda"), deg)
    dst = torch.from_numpy(g.col).cuda().long()
    if app == "pagerank":
        return _pagerank(g.n, src, dst, deg, case["iterations"]).cpu().numpy()
    if app == "bc":
        return _bc(g.n, src, dst, case["sources"]).cpu().numpy()
    wt = torch.from_numpy(g.wt).cuda().long() if g.wt is not None else torch.ones_like(dst)
    d = _minplus(g.n, src, dst, wt, s)
    reached = int(deg[d < INF].sum())
    if app == "sssp_minplus":
        return torch.where(d == INF, L.BIG_NUM, d).cpu().numpy()
    if app == "sssp":
        return d.cpu().numpy(), reached
    out = d if app == "bfs_device" else d.cpu().numpy()
    return out, None, reached
