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
