"""The library's own plan on matrices of dense tiles: at bs 8/16 its chunks stay
about as long as on sparse tiles, at bs 32/64 they are marked, and products over
them match the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def graph(gbo, n, part, density):
    """Rows below n * part hold `density` of the columns, the others three at random."""
    rng = np.random.default_rng(n)
    cut = int(n * part)
    m = rng.random((n, n), dtype=np.float32) < density
    m[cut:] = False
    m[np.repeat(np.arange(cut, n), 3), rng.integers(0, n, 3 * (n - cut))] = True
    r, c = np.nonzero(m)
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))])
    return gbo.Csr(n, n, rowptr.astype(np.int32), c.astype(np.int32))


@pytest.mark.parametrize("part, density", [(1.0, 1.0), (1.0, 0.3), (0.05, 0.9)])
@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_dense_tiles(gbo, po, bs, part, density):
    n = 2309  # full block rows of 289 tiles at bs 8 and 37 at bs 64: none is a chunk by itself
    g = graph(gbo, n, part, density)
    A = gbo.BsrMatrix.from_csr(g, bs)
    uniform = part == 1.0
    if bs <= 16:
        # about the same work everywhere: even chunks
        assert A.s.plan_even == (1 if uniform else 0)
        assert A.s.plan_nchunks * A.s.plan_chunk <= A.nblocks + 16 * A.s.plan_chunk
    else:
        assert A.s.plan_even == (3 if uniform else 0)
    rp, ci, tw = A.host_arrays()
    rng = np.random.default_rng(bs)
    xb = gbo.pack_vec(bs, (rng.random(n) < 0.4).astype(np.float32))
    vis = gbo.pack_vec(bs, (rng.random(n) < 0.3).astype(np.float32))
    w = gbo.edge_weights(g, 1, 64, seed=9)
    tv = gbo.TileValues(A, g, w)
    otv, owo = po.pack_values(bs, n, g.rowptr, g.colind, w, rp, ci, tw)
    d = rng.integers(0, 1000, n).astype(np.uint32)
    for _ in range(2):
        assert np.array_equal(gbo.bsrbmv_count(A, xb), po.count(bs, n, rp, ci, tw, xb))
        nx, cnt = gbo.bsrbmv_bfs_step(A, xb, vis)
        want, wcnt = po.bfs_step(bs, n, rp, ci, tw, xb, vis)
        assert np.array_equal(nx, want) and cnt == wcnt
        assert np.array_equal(gbo.bsrbmv_minplus(A, d), po.minplus(bs, n, rp, ci, tw, d))
        assert np.array_equal(gbo.bsrbmv_minplus(A, d, tv), po.minplus(bs, n, rp, ci, tw, d, otv, owo))
    A.free()


def test_count_over_even_chunks(gbo):
    """bs 8 from 6M tiles on: the count and the dense BFS step take chunks of their own."""
    scale, bs = 18, 8
    g = gbo.gen_rmat(scale, 24, seed=3)
    n = g.nrows
    A = gbo.BsrMatrix.from_csr(g, bs)
    assert A.nblocks >= 6 << 20 and A.s.plan_even == 0
    rng = np.random.default_rng(4)
    x = rng.random(n) < 0.4
    v = rng.random(n) < 0.3
    xb, vb = (gbo.pack_vec(bs, t.astype(np.float32)) for t in (x, v))
    want = np.diff(np.concatenate([[0], np.cumsum(x[g.colind], dtype=np.int64)])[g.rowptr]).astype(np.int32)
    dist = rng.integers(0, 1000, n).astype(np.uint32)
    first = gbo.bsrbmv_minplus(A, dist)
    for _ in range(2):
        assert np.array_equal(gbo.bsrbmv_count(A, xb), want)
        nx, cnt = gbo.bsrbmv_bfs_step(A, xb, vb)
        new = (want > 0) & ~v
        assert cnt == new.sum() and np.array_equal(nx, gbo.pack_vec(bs, new.astype(np.float32)))
    A.plan(100)
    assert np.array_equal(gbo.bsrbmv_count(A, xb), want)
    assert np.array_equal(gbo.bsrbmv_minplus(A, dist), first)
    A.free()
