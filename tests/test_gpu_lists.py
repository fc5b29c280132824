"""Drivers on matrices large enough to be swept as edge lists: components,
shortest paths and PageRank on a graph with empty windows of 64 rows, rows and
tiles far denser than the rest, and a last window that is not whole."""
import numpy as np
import pytest
from scipy.sparse import csr_matrix
from scipy.sparse.csgraph import connected_components

pytestmark = pytest.mark.gpu
# bs: vertices, random neighbours of each, bytes of matrix from which many (few) sweeps use lists
SIZES = {8: (1_100_011, 17, 192 << 20, None), 16: (200_011, 16, 96 << 20, None),
         32: (150_011, 16, 48 << 20, 256 << 20), 64: (110_011, 16, 48 << 20, 512 << 20)}


@pytest.fixture(scope="module", params=sorted(SIZES))
def graph(request, gbo):
    bs = request.param
    n, deg, many, few = SIZES[bs]
    rng = np.random.default_rng(bs)
    live = n - 5000  # the rest: isolated, but for a path of ten
    m = live * deg // 2
    u, v = rng.integers(0, live, m), rng.integers(0, live, m)
    cu, cv = np.triu_indices(1000, 1)  # full tiles
    hub = rng.choice(live, live // 3, replace=False)
    path = np.arange(n - 2000, n - 1990)
    u = np.concatenate([u, cu + 3000, np.full(len(hub), 7), path[:-1]])
    v = np.concatenate([v, cv + 3000, hub, path[1:]])
    ok = u != v
    u, v = u[ok].astype(np.int64), v[ok].astype(np.int64)
    key = np.unique(np.concatenate([u * n + v, v * n + u]))
    rp = np.zeros(n + 1, np.int64)
    rp[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    g = gbo.Csr(n, n, rp.astype(np.int32), (key % n).astype(np.int32))
    A = gbo.BsrMatrix.from_csr(g, bs)
    size = A.nblocks * (bs * bs // 8 + 4)
    assert size >= many and (few is None or size >= few)
    return g, A, few is not None


def test_components(gbo, graph):
    g, A, listed = graph
    if not listed:
        pytest.skip("few sweeps: over the tiles at this block size")
    _, lab = connected_components(csr_matrix((np.ones(g.nnz, np.int8), g.colind, g.rowptr), (g.nrows, g.nrows)), False)
    first = np.full(lab.max() + 1, g.nrows)
    np.minimum.at(first, lab, np.arange(g.nrows))
    got, _ = gbo.cc(A)
    assert np.array_equal(got, first[lab])


@pytest.mark.parametrize("weighted", (False, True))
def test_shortest_paths(gbo, graph, weighted):
    """With positive weights the distances are the one fixed point of
    d[i] = min over i's entries of d[j] + w, d[source] = 0."""
    g, A, _ = graph
    w = gbo.edge_weights(g, 1, 64, seed=3) if weighted else np.ones(g.nnz, np.uint32)
    source = 11
    d, _ = gbo.sssp(A, source, gbo.TileValues(A, g, w) if weighted else None)
    inf = 0xFFFFFFFF
    dj = d[g.colind].astype(np.int64)
    cand = np.where(dj == inf, inf, dj + w)
    rows = np.flatnonzero(np.diff(g.rowptr))
    want = np.full(g.nrows, inf, np.int64)
    want[rows] = np.minimum.reduceat(cand, g.rowptr[rows])
    want[source] = 0
    assert np.array_equal(d.astype(np.int64), want)
    assert (d != inf).sum() > g.nrows // 2


def test_pagerank(gbo, graph):
    """As many iterations in float64.  Each of the engine's rounds three times a
    value (2^-24 relative, all terms positive) and the errors of earlier ones
    come in times alpha: 3 * 2^-24 / (1 - alpha) = 1.2e-6."""
    g, A, _ = graph
    n, alpha = g.nrows, np.float32(0.85)
    deg = np.diff(g.rowptr).astype(np.int32)
    p, iters, _ = gbo.pagerank(A, deg, float(alpha), 1e-7, 1000)
    M = csr_matrix((np.ones(g.nnz), g.colind, g.rowptr), (n, n))
    x = np.full(n, 1.0 / n)
    for _ in range(iters):
        x = M @ np.where(deg > 0, float(alpha) * x / np.maximum(deg, 1), 0.0) + (1.0 - float(alpha)) / n
    assert np.max(np.abs(p - x) / x) < 1.6e-6
