"""GPU parity of the apps on graphs whose rows span the kernels' row classes."""
import numpy as np
import pytest

import oracle
from gpu_workgroup_managment_amd import graphs as G

pytestmark = pytest.mark.gpu

# longest rows of each class of the standalone PageRank, one above, several segments, a partial last segment
ROWS = (0, 1, 4, 5, 8, 9, 63, 64, 65, 256, 2047, 2048, 2049, 4096, 9001)


def _rows_graph(n=20011, seed=3):
    """Directed: vertex i < len(ROWS) has ROWS[i] distinct out-edges, the others up to 12."""
    rng = np.random.default_rng(seed)
    src, dst = [], []
    for v, deg in enumerate(ROWS):
        src.append(np.full(deg, v))
        dst.append(len(ROWS) + rng.permutation(n - len(ROWS))[:deg])
    rest = np.repeat(np.arange(len(ROWS), n), rng.integers(0, 13, n - len(ROWS)))
    src.append(rest)
    dst.append((rest + rng.integers(1, n, len(rest))) % n)
    g = G.from_edges(n, np.concatenate(src), np.concatenate(dst))
    assert tuple(g.degrees()[: len(ROWS)]) == ROWS
    return g


def test_pagerank_row_classes(rt):
    """Ranks within the bound of the summation order, and the same bits for
    every launch shape. A row's sum of positive terms takes at most 32 + 6
    (lanes of a segment) + 1 + 6 (segments) roundings, then a product, an
    addition and the division of the contribution: 48 units of 2^-24 per
    iteration, damped by 0.85."""
    g = _rows_graph()
    ref = oracle.pagerank_f64(g.row_ptr, g.col, 0.85, 30)
    dg = rt.graph(g)
    base = None
    for wg, wgs in ((64, 3), (192, 40), (1024, 1), (1024, 0)):
        r, _ = dg.pagerank(0.85, 30, wg_size=wg, num_wgs=wgs)
        assert np.abs(r / ref - 1).max() <= 48 * 2.0 ** -24 / (1 - 0.85)
        base = r if base is None else base
        assert np.array_equal(r.view(np.uint32), base.view(np.uint32)), (wg, wgs)
    dg.close()


def _hub_graph(n, hubs):
    """Rows of degree `hubs`, spread evenly, and of up to 12 edges elsewhere."""
    rng = np.random.default_rng(n)
    src = [np.full(d, v * (n // len(hubs))) for v, d in enumerate(hubs)]
    dst = [rng.permutation(n)[:d] for d in hubs]
    rest = np.repeat(np.arange(n), rng.integers(0, 13, n))
    to = rng.integers(0, n, len(rest))
    return G.from_edges(n, np.concatenate(src + [rest]), np.concatenate(dst + [to]))


@pytest.mark.parametrize("n,hubs", [
    (7, (6,)), (1025, (64, 65, 5)), (16383, (2048, 2049, 4096, 4097)), (50001, (50000, 1023, 4)), (300001, (20000, 5)),
])
def test_pagerank_held_rows(rt, n, hubs):
    """Ranges whose rows lie in LDS (many workgroups), in memory (few), and both in one launch (a row longer than the
    LDS of a workgroup): the same bits, within the bound of the row classes above."""
    g = _hub_graph(n, hubs)
    ref = oracle.pagerank_f64(g.row_ptr, g.col, 0.85, 30)
    dg = rt.graph(g)
    base = None
    for wg, wgs in ((64, 3), (64, 0), (192, 40), (1024, 1), (1024, 0), (1024, 300)):
        r, _ = dg.pagerank(0.85, 30, wg_size=wg, num_wgs=wgs)
        assert np.abs(r / ref - 1).max() <= 48 * 2.0 ** -24 / (1 - 0.85)
        base = r if base is None else base
        assert np.array_equal(r.view(np.uint32), base.view(np.uint32)), (wg, wgs)
    dg.close()


def _symmetric(g):
    return G.from_edges(g.n, np.repeat(np.arange(g.n), g.degrees()), g.col, symmetric=True)


# rows at the edges of the scan's stages: 4 edges by the thread, 64 by eight lanes, the rest by a wave (256 a round)
STAGES = (1, 2, 4, 5, 12, 67, 68, 69, 132, 324, 325, 3000)


def _stage_graph():
    n, src, dst = 6007, [], []
    rng = np.random.default_rng(8)
    for v, deg in enumerate(STAGES):
        src.append(np.full(deg, v))
        dst.append(len(STAGES) + rng.permutation(n - len(STAGES))[:deg])
    return _symmetric(G.from_edges(n, np.concatenate(src), np.concatenate(dst)))


def _complete(n):
    i, j = np.divmod(np.arange(n * n), n)
    return G.from_edges(n, i[i != j], j[i != j])


OPEN_GRAPHS = {
    "stages": _stage_graph,
    "rmat": lambda: _symmetric(G.rmat(13, 16, seed=2)),
    "complete": lambda: _complete(131),  # as many colours as vertices: one long chain
    "mesh": lambda: G.grid(61, 83),
    "path": lambda: G.grid(1, 4099),
    "no edges": lambda: G.CSR(np.zeros(71, np.int32), np.zeros(0, np.int32)),
}


@pytest.mark.parametrize("name", list(OPEN_GRAPHS))
@pytest.mark.parametrize("wg,wgs", [(64, 1), (192, 19), (1024, 0)])
def test_color_mis_worklists(rt, name, wg, wgs):
    """Colours, sets and round counts of both forms of the worklist kernels."""
    g = OPEN_GRAPHS[name]()
    if name == "no edges":
        g.prio = np.arange(g.n, dtype=np.uint32)
    else:
        G.add_priorities(g)
    dg = rt.graph(g)
    ref, rounds = oracle.color(g.row_ptr, g.col, g.prio)
    out, st = dg.color(wg_size=wg, num_wgs=wgs)
    assert np.array_equal(out, ref) and st["iterations"] == rounds
    ref, rounds = oracle.mis(g.row_ptr, g.col, g.prio)
    out, st = dg.mis(wg_size=wg, num_wgs=wgs)
    assert np.array_equal(out, ref) and st["iterations"] == rounds
    dg.close()


@pytest.mark.parametrize("degree", [3, 9])
def test_color_directed_round_count(rt, degree):
    """Edges without a reverse: two neighbours may take the last colour in the
    same round, and the round count is one more."""
    n = 4001
    rng = np.random.default_rng(degree)
    g = G.add_priorities(G.from_edges(n, np.repeat(np.arange(n), degree), rng.integers(0, n, degree * n)))
    ref, rounds = oracle.color(g.row_ptr, g.col, g.prio)
    out, st = rt.graph(g).color(wg_size=256, num_wgs=24)
    assert np.array_equal(out, ref) and st["iterations"] == rounds


def _lds_limit():
    """Largest vertex count whose BC state is kept in LDS (18 bytes a vertex and four bitmaps in 160 KB - 1536)."""
    n = 8000
    while 16 * (n + 1) + (2 * (n + 1) + 3) // 4 * 4 + 16 * ((n + 32) // 32) + 1536 <= 160 << 10:
        n += 1
    return n


def _random_arcs(n, m, seed):
    rng = np.random.default_rng(seed)
    return G.from_edges(n, rng.integers(0, n, m), rng.integers(0, n, m))


BC_GRAPHS = {
    "lds limit": (lambda: _random_arcs(_lds_limit(), 30000, 1), 70),
    "above lds": (lambda: _random_arcs(_lds_limit() + 1, 30000, 1), 70),
    "row stages": (_stage_graph, 40),  # rows of 8, 9, 16, 17, 64, 65 edges and more, in both directions
    "stages, global": (lambda: _symmetric(G.from_edges(9001, np.r_[np.zeros(700, int), np.ones(64, int), np.full(17, 2)],
                                                       np.r_[np.arange(10, 710), np.arange(300, 364), np.arange(5, 22)])), 30),
    "many levels": (lambda: G.grid(1, 301), 301),
    "large counts": (lambda: G.grid(40, 41), 50),  # path counts far above 2^53
    "one vertex": (lambda: G.CSR(np.zeros(2, np.int32), np.zeros(0, np.int32)), 1),
    "no edges": (lambda: G.CSR(np.zeros(34, np.int32), np.zeros(0, np.int32)), 33),
    "two batches": (lambda: G.from_edges(12001, np.zeros(12000, int), np.arange(1, 12001), symmetric=True), 12001),
}


@pytest.mark.parametrize("name", list(BC_GRAPHS))
def test_bc_state_and_row_classes(rt, name):
    """Bit-exact sums wherever the state of a source is kept and whoever walks
    its rows, level count included."""
    make, sources = BC_GRAPHS[name]
    g = make()
    ref, levels = oracle.bc(g.row_ptr, g.col, sources)
    dg = rt.graph(g)
    for wg, wgs in ((64, 9), (256, 1024)) if g.n < 12000 else ((256, 1024),):
        out, st = dg.bc(sources, wg_size=wg, num_wgs=wgs)
        assert np.array_equal(out, ref) and st["iterations"] == levels, (wg, wgs)
    dg.close()


def _spans(n, span, seed):
    """Four out-edges a vertex (some fewer), none longer than `span` on the ring of n vertices."""
    rng = np.random.default_rng(seed)
    src = np.repeat(np.arange(n), rng.integers(0, 5, n))
    g = G.from_edges(n, src, (src + rng.integers(-span, span + 1, len(src))) % n)
    g.wt = rng.integers(0, 256, g.m).astype(np.int32)
    return g


LOW = {
    "one": lambda: G.CSR(np.zeros(2, np.int32), np.zeros(0, np.int32), np.zeros(0, np.int32)),
    "path": lambda: G.grid(1, 300),
    "spill": lambda: _spans(16384, 8192, 1),  # levels past the queues in LDS, any span
    "above": lambda: _spans(16385, 769, 2),  # past both lines
    "ring": lambda: _spans(40000, 768, 3),
    "bits": lambda: G.grid(512, 512),         # the last bit of the LDS bitmaps
    "past": lambda: G.grid(437, 600),         # 2^18 + 56 vertices
}


@pytest.mark.parametrize("name", LOW)
def test_low_degree_graphs(rt, name):
    """BFS and push SSSP where a low-degree graph moves to one workgroup, on
    both sides of each line; weights of 0 and 255, then one above the packed
    rows' 8 bits."""
    g = LOW[name]()
    if g.m and g.wt is None:
        g.wt = np.random.default_rng(5).integers(0, 256, g.m).astype(np.int32)
    src = g.n // 2 if name != "bits" else 0
    for top in (255, 256):
        if g.m:
            g.wt[g.m // 2] = top
        levels, n_levels = oracle.bfs(g.row_ptr, g.col, src)
        ref = oracle.sssp(g.row_ptr, g.col, g.wt, src)
        dg = rt.graph(g)
        for wg, wgs in ((64, 1), (320, 3), (512, 64), (1024, 0)):
            d, st = dg.bfs(src, wg_size=wg, num_wgs=wgs)
            assert np.array_equal(d, levels) and st["iterations"] == n_levels, (wg, wgs)
            d, _ = dg.sssp(src, wg_size=wg, num_wgs=wgs, mode=1)
            assert np.array_equal(d, ref), (wg, wgs)
        dg.close()


def _reverse(g):
    return G.from_edges(g.n, g.col, np.repeat(np.arange(g.n), g.degrees()))


BFS = {
    "hubs_out": lambda: _rows_graph(seed=6),             # few entries hold a level's edges
    "hubs_in": lambda: _reverse(_rows_graph(seed=7)),    # long rows scanned bottom-up
    "stages_in": lambda: _reverse(_stage_graph()),
    "rmat": lambda: G.rmat(12, 16, seed=11),
    "er": lambda: G.erdos_renyi(5003, 40000, seed=12),   # even degrees: no estimate
    "star": lambda: G.from_edges(3001, np.zeros(3000, int), np.arange(1, 3001), symmetric=True),
}


@pytest.mark.parametrize("name", BFS)
def test_bfs_bottom_up(rt, name):
    """Levels and their count where a level runs bottom-up, from one wave (many
    chunks of its range) to the whole grid."""
    g = BFS[name]()
    dg = rt.graph(g)
    for src in (0, g.n // 2, g.n - 1):
        levels, n_levels = oracle.bfs(g.row_ptr, g.col, src)
        for wg, wgs in ((64, 1), (192, 3), (512, 64), (1024, 0)):
            d, st = dg.bfs(src, wg_size=wg, num_wgs=wgs)
            assert np.array_equal(d, levels) and st["iterations"] == n_levels, (src, wg, wgs)
    dg.close()


def _in_rows(degrees, seed, lo=1, n=9001):
    """Vertex i has degrees[i % len] in-edges from random vertices; one vertex in 64 has none."""
    rng = np.random.default_rng(seed)
    deg = np.resize(np.asarray(degrees), n)
    deg[::64] = 0
    g = G.from_edges(n, rng.integers(0, n, deg.sum()), np.repeat(np.arange(n), deg))
    g.wt = rng.integers(lo, 256, g.m).astype(np.int32)
    return g


def _dag(n=3000, m=12000):
    rng = np.random.default_rng(31)
    a, b = rng.integers(0, n, (2, m))
    g = G.from_edges(n, np.minimum(a, b)[a != b], np.maximum(a, b)[a != b])
    g.wt = rng.integers(-5, 256, g.m).astype(np.int32)  # also lowers vertices that the source does not reach
    return g


def _fan(n):
    """Vertex 0 to all others, every 64th of those to its successor."""
    tail = np.arange(64, n - 1, 64)
    deg = np.zeros(n, np.int64)
    deg[0], deg[tail] = n - 1, 1
    col = np.concatenate([np.arange(1, n), tail + 1]).astype(np.int32)
    wt = np.concatenate([np.arange(1, n) % 251 + 1, tail % 7]).astype(np.int32)
    return G.CSR(np.concatenate([[0], np.cumsum(deg)]).astype(np.int32), col, wt)


MINPLUS = {
    "ones": lambda: _in_rows([1], 21),                     # 256 rows a block
    "blocks": lambda: _in_rows([255, 256, 257, 1, 2], 22, n=701),  # rows that end, begin and go on at a block's edge
    "steps": lambda: _in_rows([1025, 3, 64, 5000], 23, n=301),     # rows of several steps and waves
    "mixed": lambda: _in_rows([0, 3, 0, 0, 70, 17], 24),
    "edge": lambda: G.CSR(np.array([0, 1, 1], np.int32), np.array([1], np.int32), np.array([7], np.int32)),
    "none": lambda: G.CSR(np.zeros(4, np.int32), np.zeros(0, np.int32), np.zeros(0, np.int32)),
    "negative": _dag,
    "two_rows_a_bit": lambda: _in_rows([1, 3, 2], 25, n=1200007),
    "words_a_bit": lambda: _fan(33600000),
}


@pytest.mark.parametrize("name", MINPLUS)
def test_minplus_rows(rt, name):
    """Min-plus sweeps at the edges of blocks, steps and the LDS map; the
    number of sweeps stays within the Jacobi one's."""
    g = MINPLUS[name]()
    src = int(np.argmax(g.degrees()))
    ref, sweeps = oracle.sssp_minplus(g.row_ptr, g.col, g.wt, src)
    dg = rt.graph(g)
    for wg, wgs in ((1024, 0),) if g.n > 10 ** 6 else ((64, 1), (192, 7), (512, 64), (1024, 0)):
        d, st = dg.sssp_minplus(src, wg_size=wg, num_wgs=wgs)
        assert np.array_equal(d, ref), (wg, wgs)
        assert 1 <= st["iterations"] <= sweeps
    dg.close()


@pytest.mark.parametrize("n", [1, 16384, 16385, (1 << 19) - 1, (1 << 19) + 1, (1 << 22) + (1 << 19) + 3])
def test_results_arrive_whole(rt, n):
    """Results below and above a staging size, a chunk and the whole staging
    (4 bytes a vertex)."""
    g = _fan(n)
    ref, _ = oracle.sssp_minplus(g.row_ptr, g.col, g.wt, 0)
    dg = rt.graph(g)
    a, _ = dg.sssp_minplus(0)
    b, st = dg.sssp(0, mode=2)
    assert np.array_equal(a, ref) and np.array_equal(b, ref)
    assert st["edges_scanned"] == g.m
    dg.close()


def _steps(n, span, seed):
    """Up to four out-edges a vertex, one of them as long as `span` allows."""
    rng = np.random.default_rng(seed)
    src = np.repeat(np.arange(n), rng.integers(0, 5, n))
    dst = np.clip(src + rng.integers(-min(span, n - 1), min(span, n - 1) + 1, len(src)), 0, n - 1)
    src, dst = np.append(src, n // 2), np.append(dst, max(n // 2 - span, 0))
    g = G.from_edges(n, src, dst)
    keep = np.arange(g.m) - np.repeat(g.row_ptr[:-1], g.degrees()) < 4
    return G.from_edges(n, np.repeat(np.arange(n), g.degrees())[keep], g.col[keep])


@pytest.mark.parametrize("n,span", [(1, 0), (63, 9), (90001, 32767), (90001, 32768), (700001, 5000)])
def test_pagerank_low_degree(rt, n, span):
    """Ranks of graphs on both sides of the 16-bit rows' reach, with all of a
    range's rows in LDS and a part of them, the same bits for every launch
    shape. A term takes at most four additions, the product with the addition
    and the division of the contribution: 6 units of 2^-24 an iteration, damped
    by 0.85."""
    g = _steps(n, span, 4)
    ref = oracle.pagerank_f64(g.row_ptr, g.col, 0.85, 30)
    dg = rt.graph(g)
    base = None
    for wg, wgs in ((64, 3), (192, 40), (1024, 1), (1024, 0)):
        r, _ = dg.pagerank(0.85, 30, wg_size=wg, num_wgs=wgs)
        assert np.abs(r / ref - 1).max() <= 6 * 2.0 ** -24 / (1 - 0.85)
        base = r if base is None else base
        assert np.array_equal(r.view(np.uint32), base.view(np.uint32)), (wg, wgs)
    dg.close()


@pytest.mark.parametrize("n,m", [(1, 40000), (250, 32768), (257, 32767), (65537, 90000), (70001, 300007)])
def test_in_edges(rt, n, m):
    """The in-edge CSR of one, two and three sort passes, partial tiles and
    groups of tiles: betweenness needs its order bit for bit, the min-plus sweeps
    the weights beside it."""
    rng = np.random.default_rng(n)
    row = np.concatenate([[0], np.cumsum(np.bincount(rng.integers(0, n, m), minlength=n))]).astype(np.int32)
    g = G.CSR(row, (rng.integers(0, n, m) ** 2 % n).astype(np.int32), rng.integers(0, 256, m).astype(np.int32))
    dg = rt.graph(g)
    d, _ = dg.sssp_minplus(n // 2)
    assert np.array_equal(d, oracle.sssp_minplus(g.row_ptr, g.col, g.wt, n // 2)[0])
    b, _ = dg.bc(min(n, 9))
    assert np.array_equal(b, oracle.bc(g.row_ptr, g.col, min(n, 9))[0])
    dg.close()
