"""Masked products sum(A * (A B)) with rows of A at the edges of the row
classes (eight rows to a wave, a wave each, a workgroup each, several items of
keys), sparse and dense tiles, and a B that is not A's transpose, against
scipy's integer products."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BS = (8, 16, 32, 64)


def csr(gbo, m):
    m.sort_indices()
    return gbo.Csr(m.shape[0], m.shape[1], m.indptr.astype(np.int32), m.indices.astype(np.int32))


def masked(gbo, A, B, bs):
    Ar, Bc = gbo.BsrMatrix.from_csr(csr(gbo, A), bs, 0), gbo.BsrMatrix.from_csr(csr(gbo, B), bs, 1)
    got = gbo.bsrbmm_tc(Ar, Bc)
    Ar.free()
    Bc.free()
    return got


def rand(sp, rng, n, nnz):
    m = sp.coo_matrix((np.ones(nnz, np.int64), (rng.integers(0, n, nnz), rng.integers(0, n, nnz))), (n, n)).tocsr()
    m.data[:] = 1
    return m


@pytest.mark.parametrize("bs", BS)
def test_row_classes(gbo, bs):
    sp = pytest.importorskip("scipy.sparse")
    n = 5000
    rng = np.random.default_rng(bs)
    rows, cols = [rng.integers(0, n, 15_000)], [rng.integers(0, n, 15_000)]
    for i, d in enumerate((1, 7, 8, 9, 31, 32, 33, 63, 64, 65, 511, 512, 513, 1025, n)):
        rows.append(np.full(d, 100 + 37 * i))
        cols.append(rng.permutation(n)[:d])
    A = sp.coo_matrix((np.ones(sum(map(len, rows)), np.int64), (np.concatenate(rows), np.concatenate(cols))), (n, n)).tocsr()
    A.data[:] = 1
    for B in (A.T.tocsr(), rand(sp, rng, n, 40_000), A):
        assert masked(gbo, A, B, bs) == int(A.multiply(A @ B).sum())


@pytest.mark.parametrize("bs", BS)
@pytest.mark.parametrize("n,p", [(63, 1.0), (520, 0.5), (1000, 0.93)])
def test_dense_tiles(gbo, bs, n, p):
    sp = pytest.importorskip("scipy.sparse")
    rng = np.random.default_rng(n)
    A = sp.csr_matrix((rng.random((n, n)) < p).astype(np.int64))
    B = sp.csr_matrix((rng.random((n, n)) < 0.4).astype(np.int64))
    assert masked(gbo, A, B, bs) == int(A.multiply(A @ B).sum())
    L = sp.tril(A, -1).tocsr()
    assert masked(gbo, L, L.T.tocsr(), bs) == int(L.multiply(L @ L.T).sum())


@pytest.mark.parametrize("bs", (8, 64))
def test_windows(gbo, bs):
    """More columns than a bitmap (or, at bs 8, a vector of tiles) holds: a
    dense block at each end of 1.3M vertices and heavy rows across them."""
    sp = pytest.importorskip("scipy.sparse")
    n = 1_300_003
    rng = np.random.default_rng(5)
    d = 80
    hub = np.concatenate([np.arange(d), n - 1 - np.arange(d), rng.integers(0, n, 3000)])
    block = np.concatenate([np.arange(d), n - 1 - np.arange(d)])
    r = np.concatenate([np.repeat(block, len(block)), np.full(len(hub), 7), np.full(len(hub), n - 3)])
    c = np.concatenate([np.tile(block, len(block)), hub, hub])
    A = sp.coo_matrix((np.ones(len(r), np.int64), (r, c)), (n, n)).tocsr()
    A.data[:] = 1
    assert masked(gbo, A, A.T.tocsr(), bs) == int(A.multiply(A @ A.T).sum())
    keep = sp.coo_matrix((np.ones(len(block) ** 2, np.int64), (np.repeat(block, len(block)), np.tile(block, len(block)))),
                         (n, n)).tocsr()  # dense tiles alone
    assert masked(gbo, keep, keep, bs) == int(keep.multiply(keep @ keep).sum())
