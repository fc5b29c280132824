"""Masked products sum(A * (A B)) over more ids than one bitmap holds: rows of
more keys than an item, lists that lie in one window, end at its edge or run over
all of them, for two to four windows; against scipy's integer products."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
WINDOW = 1 << 20


def csr(gbo, m):
    m.sort_indices()
    return gbo.Csr(m.shape[0], m.shape[1], m.indptr.astype(np.int32), m.indices.astype(np.int32))


@pytest.mark.parametrize("bs,n", [(8, WINDOW + 1), (64, 2 * WINDOW), (8, 3 * WINDOW + 77_777), (32, 3 * WINDOW + 77_777)])
def test_windows(gbo, bs, n):
    sp = pytest.importorskip("scipy.sparse")
    rng = np.random.default_rng(n % 1000 + bs)
    edges = np.array([x for w in range(0, n, WINDOW) for x in (w - 1, w, w + 1) if 0 <= x < n] + [n - 1])
    hubs = np.concatenate([edges, rng.choice(n, 4, replace=False)])
    r, c = [rng.integers(0, n, 20_000)], [rng.integers(0, n, 20_000)]
    for i, h in enumerate(np.unique(hubs)):
        d = (40, 600, 1500, 4000)[i % 4]
        # near one window's start, near its end, or anywhere
        at = (rng.integers(0, n, d), np.arange(d) + max(0, n - d - 5), np.arange(d) + (WINDOW - d // 2))[i % 3] % n
        r += [np.full(d, h), np.full(len(hubs), h)]
        c += [at, hubs]
    r, c = np.concatenate(r), np.concatenate(c)
    A = sp.coo_matrix((np.ones(2 * len(r), np.int64), (np.r_[r, c], np.r_[c, r])), (n, n)).tocsr()
    A.data[:] = 1
    B = sp.coo_matrix((np.ones(20_000, np.int64), (rng.integers(0, n, 20_000), rng.choice(hubs, 20_000))), (n, n)).tocsr()
    B.data[:] = 1
    for M, N in ((A, A), (A, B), (sp.tril(A, -1).tocsr(), sp.triu(A, 1).tocsr())):
        Ar, Bc = gbo.BsrMatrix.from_csr(csr(gbo, M), bs, 0), gbo.BsrMatrix.from_csr(csr(gbo, N), bs, 1)
        assert gbo.bsrbmm_tc(Ar, Bc) == int(M.multiply(M @ N).sum())
        Ar.free()
        Bc.free()
