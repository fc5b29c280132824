"""Multi-source BFS over edge lists: matrices large enough for them, with empty
windows, rows and tiles far denser than the rest, isolated and repeated sources,
and every number of frontier words."""
import numpy as np
import pytest
from scipy.sparse import csr_matrix

pytestmark = pytest.mark.gpu
SIZES = {8: (100_011, 17), 16: (50_011, 14), 32: (24_011, 12), 64: (16_011, 8)}


def _levels(g, sources):
    M = csr_matrix((np.ones(g.nnz, np.int32), g.colind, g.rowptr), (g.nrows, g.nrows))
    level = np.full((g.nrows, len(sources)), -1, np.int32)
    F = np.zeros((g.nrows, len(sources)), np.int32)
    F[sources, np.arange(len(sources))] = 1
    depth = 0
    while F.any():
        level[F > 0] = depth
        F = ((M @ F > 0) & (level < 0)).astype(np.int32)
        depth += 1
    return level.T, depth


@pytest.mark.parametrize("bs, nsrc", [(8, 65), (16, 130), (32, 200), (64, 1), (64, 256)])
def test_levels(gbo, bs, nsrc):
    n, deg = SIZES[bs]
    rng = np.random.default_rng(bs)
    live = n - 1000
    m = live * deg // 2
    u, v = rng.integers(0, live, m), rng.integers(0, live, m)
    cu, cv = np.triu_indices(300, 1)
    hub = rng.choice(live, live // 3, replace=False)
    path = np.arange(n - 400, n - 390)
    u = np.concatenate([u, cu + 3000, np.full(len(hub), 7), path[:-1]])
    v = np.concatenate([v, cv + 3000, hub, path[1:]])
    ok = u != v
    u, v = u[ok].astype(np.int64), v[ok].astype(np.int64)
    key = np.unique(np.concatenate([u * n + v, v * n + u]))
    rp = np.zeros(n + 1, np.int64)
    rp[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    g = gbo.Csr(n, n, rp.astype(np.int32), (key % n).astype(np.int32))
    A = gbo.BsrMatrix.from_csr(g, bs)
    assert A.nblocks * (bs * bs // 8 + 4) >= 16 << 20
    sources = rng.integers(0, n, nsrc).astype(np.int32)
    sources[nsrc // 2] = path[0]
    sources[-1] = n - 1 if nsrc > 1 else path[3]
    want, depth = _levels(g, sources)
    got, nlev = gbo.bfs_multisource(A, sources)
    assert nlev == depth
    assert np.array_equal(np.asarray(got).reshape(nsrc, n), want)
