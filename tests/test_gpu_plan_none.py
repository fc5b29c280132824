"""Products without a plan (one of even chunks made for the call) and on even
plans of a few tiles, against the oracle: block rows that end at, before and
after a chunk's end, run over many chunks, or are empty."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rows_of(bs, counts, seed):
    """One nonzero in each of counts[I] block columns of block row I."""
    rng = np.random.default_rng(seed)
    nbc = max(max(counts), 4) + 3
    n = max(len(counts), nbc) * bs - 3
    rows, cols = [], []
    for i, c in enumerate(counts):
        rows.append(i * bs + rng.integers(0, bs - 3, c))
        cols.append(np.sort(rng.choice(nbc - 1, c, replace=False)) * bs + rng.integers(0, bs, c))
    r, c = np.concatenate(rows), np.concatenate(cols)
    o = np.lexsort((c, r))
    rp = np.concatenate([[0], np.cumsum(np.bincount(r, minlength=n))])
    return n, rp.astype(np.int32), c[o].astype(np.int32)


@pytest.mark.parametrize("chunk", (None, 1, 7, 16))
@pytest.mark.parametrize("counts", [[16, 16, 16], [15, 17, 0, 0, 16, 1], [1] * 40, [300, 0, 5, 1000, 0], [0, 0, 3]])
@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_even_chunks(gbo, po, bs, counts, chunk):
    n, rowptr, colind = rows_of(bs, counts, bs + len(counts))
    g = gbo.Csr(n, n, rowptr, colind)
    A = gbo.BsrMatrix.from_csr(g, bs, plan=False)
    assert A.nblocks == sum(counts)
    if chunk:
        A.plan(chunk)
    rp, ci, tw = A.host_arrays()
    rng = np.random.default_rng(n)
    for _ in range(2):  # the count slots are clear for the second call
        xb = gbo.pack_vec(bs, (rng.random(n) < 0.4).astype(np.float32))
        vis = gbo.pack_vec(bs, (rng.random(n) < 0.3).astype(np.float32))
        assert np.array_equal(gbo.bsrbmv_count(A, xb), po.count(bs, n, rp, ci, tw, xb))
        nx, cnt = gbo.bsrbmv_bfs_step(A, xb, vis)
        want, wcnt = po.bfs_step(bs, n, rp, ci, tw, xb, vis)
        assert np.array_equal(nx, want) and cnt == wcnt
        xi = rng.integers(-2**31, 2**31 - 1, n).astype(np.int32)
        assert np.array_equal(gbo.bsrbmv_min_i32(A, xi), po.min_i32(bs, n, rp, ci, tw, xi))
        d = rng.integers(0, 1000, n).astype(np.uint32)
        assert np.array_equal(gbo.bsrbmv_minplus(A, d), po.minplus(bs, n, rp, ci, tw, d))
        x = rng.random(n).astype(np.float32)
        # the sum of FP32 terms in FP64, rounded once
        np.testing.assert_allclose(gbo.bsrbmv_sum_f32(A, x), po.sum_f64(bs, n, rp, ci, tw, x.astype(np.float64)),
                                   rtol=6.1e-8, atol=0)
    A.free()
