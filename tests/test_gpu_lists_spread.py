"""Shortest paths over evenly spread columns, on both sides of the number of
rows from which they go by the tiles: distances are the one fixed point of
d[i] = min over i's entries of d[j] + w, d[source] = 0."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs,n,deg", [(8, 3 << 19, 24), (8, (3 << 19) + 1, 24), (16, 3 << 19, 8), (16, 1_600_007, 8)])
def test_spread(gbo, bs, n, deg):
    g = gbo.gen_er_m(n, n * deg // 2, 7)
    A = gbo.BsrMatrix.from_csr(g, bs)
    assert A.nblocks * (bs * bs // 8 + 4) > (192 << 20 if bs == 8 else 96 << 20)
    w = gbo.edge_weights(g, 1, 64, seed=3)
    source = 11
    d, _ = gbo.sssp(A, source, gbo.TileValues(A, g, w))
    inf = 0xFFFFFFFF
    dj = d[g.colind].astype(np.int64)
    cand = np.where(dj == inf, inf, dj + w)
    rows = np.flatnonzero(np.diff(g.rowptr))
    want = np.full(n, inf, np.int64)
    want[rows] = np.minimum.reduceat(cand, g.rowptr[rows])
    want[source] = 0
    assert np.array_equal(d.astype(np.int64), want)
    assert (d != inf).sum() > n // 2
    A.free()
