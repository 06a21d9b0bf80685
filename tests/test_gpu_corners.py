"""GPU parity at corners: weights that wrap, ids that share a word, shapes kept off before."""
import numpy as np
import pytest

import oracle
from gpu_workgroup_managment_amd import _lib as L
from gpu_workgroup_managment_amd import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1200002, 1200003, 2500004])
def test_minplus_source_without_in_edges(rt, n):
    """More than 2^20 vertices with in-edges, so that a bit of the sweeps' map
    stands for two or four of them. The source has no in-edge, one edge of a
    weight that wraps when added to an unreached distance, and one to the last
    vertex, the highest-numbered row: the first must never be followed."""
    heavy = 2 ** 31 - 6
    row = np.concatenate([[0], 2 + np.arange(n)]).astype(np.int32)  # the others have a loop each
    col = np.concatenate([[1, n - 1], np.arange(1, n)]).astype(np.int32)
    wt = np.concatenate([[heavy, 3], np.ones(n - 1)]).astype(np.int32)
    g = G.CSR(row, col, wt)
    ref, _ = oracle.sssp_minplus(g.row_ptr, g.col, g.wt, 0)
    pull = np.where(ref == L.BIG_NUM, oracle.INF, ref)
    dg = rt.graph(g)
    for wg, wgs in ((512, 64), (1024, 0)):
        d, _ = dg.sssp_minplus(0, wg_size=wg, num_wgs=wgs)
        assert np.array_equal(d, ref), (wg, wgs)
        d, _ = dg.sssp(0, wg_size=wg, num_wgs=wgs, mode=2)
        assert np.array_equal(d, pull), (wg, wgs)
    dg.close()


@pytest.mark.parametrize("wg", [64, 256, 512, 1024])
def test_two_level_barrier_at_full_occupancy(rt, wg):
    """The two-level barrier with every workgroup that fits, each epoch checked
    (every wait has a budget of spins: a wait that lasts too long ends the launch
    with an error)."""
    r = rt.barrier_bench(wg_size=wg, num_wgs=0, iterations=20, variant=L.BARRIER_XCD)
    assert r["epoch_errors"] == 0
    assert r["participating"] >= 256 and r["barriers"] == 200


@pytest.mark.parametrize("lowest", [1, -1])
def test_minplus_edges_scanned(rt, lowest):
    """The first sweep follows the source's edges (every edge where a weight is
    negative), each later one passes every edge."""
    n, src = 3001, 7
    rng = np.random.default_rng(lowest + 2)
    a, b = np.sort(rng.integers(0, n, (2, 9000)), axis=0)  # no cycles
    g = G.from_edges(n, a[a != b], b[a != b])
    g.wt = rng.integers(1, 256, g.m).astype(np.int32)
    g.wt[g.m // 2] = lowest
    dg = rt.graph(g)
    d, st = dg.sssp_minplus(src, wg_size=256, num_wgs=8)
    assert np.array_equal(d, oracle.sssp_minplus(g.row_ptr, g.col, g.wt, src)[0])
    first = g.degrees()[src] if lowest > 0 else g.m
    assert st["iterations"] > 1 and st["edges_scanned"] == first + (st["iterations"] - 1) * g.m
    dg.close()


def test_graph_bytes_count_what_the_apps_keep(rt):
    """The lists of the worklist apps (rows above 4 edges: two of 16 bytes a
    vertex), the ranks, BC's rows and in-edges."""
    n = 6007
    rng = np.random.default_rng(3)
    g = G.add_priorities(G.from_edges(n, rng.integers(0, n, 30000), rng.integers(0, n, 30000), symmetric=True))
    assert g.degrees().max() > 4
    dg = rt.graph(g)
    want = 4 * (n + 1) + 4 * g.m + 4 * n + 16
    assert dg.nbytes() == want
    dg.color(wg_size=64, num_wgs=3)
    want += 4 * n + 32 * n
    assert dg.nbytes() == want
    dg.mis(wg_size=64, num_wgs=3)
    want += 4 * n
    dg.pagerank(0.85, 2, wg_size=64, num_wgs=3)
    want += 12 * n
    assert dg.nbytes() == want
    dg.bc(9, wg_size=64, num_wgs=3)
    want += 4 * (n + 1) + 4 * g.m + 8 * 9 * n + 4 * 3 * (n + 2) + 8 * (n + 1) + 4 * (n + 1)
    assert dg.nbytes() == want
    dg.close()
