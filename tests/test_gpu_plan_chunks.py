"""Tiles per chunk of the library's own plans on both sides of the rule's lines:
the chunk that is chosen and the products over it against the oracle."""
import numpy as np
import pytest

from graphs import sym_csr

pytestmark = pytest.mark.gpu


def sparse_graph(gbo, n, m, core, seed):
    rng = np.random.default_rng(seed)
    u, v = [rng.integers(0, n, m)], [rng.integers(0, n, m)]
    if core:
        keep = np.triu(rng.random((core, core)) < 0.5, 1)
        a, b = np.nonzero(keep)
        u.append(a)
        v.append(b)
    rp, ci = sym_csr(n, np.concatenate(u), np.concatenate(v))
    return gbo.Csr(n, n, rp, ci)


@pytest.mark.parametrize("bs,n,m,core,chunk", [
    (8, 130_003, 500_000, 0, 128), (8, 130_003, 560_000, 0, 256), (8, 130_003, 560_000, 200, 128),
    (16, 100_003, 560_000, 0, 128), (32, 130_003, 210_000, 0, 96), (32, 130_003, 270_000, 0, 80),
    (32, 160_001, 800_000, 0, 256), (32, 130_003, 270_000, 300, 96),
    (64, 160_001, 250_001, 0, 96),
])
def test_chunks(gbo, po, bs, n, m, core, chunk):
    g = sparse_graph(gbo, n, m, core, bs + m)
    A = gbo.BsrMatrix.from_csr(g, bs)
    assert A.s.plan_chunk == chunk
    rp, ci, tw = A.host_arrays()
    rng = np.random.default_rng(n)
    xb = gbo.pack_vec(bs, (rng.random(n) < 0.3).astype(np.float32))
    assert np.array_equal(gbo.bsrbmv_count(A, xb), po.count(bs, n, rp, ci, tw, xb))
    xi = rng.integers(-2**31, 2**31 - 1, n).astype(np.int32)
    assert np.array_equal(gbo.bsrbmv_min_i32(A, xi), po.min_i32(bs, n, rp, ci, tw, xi))
    dist = rng.integers(0, 1000, n).astype(np.uint32)
    dist[rng.random(n) < 0.3] = gbo.INF_U32
    assert np.array_equal(gbo.bsrbmv_minplus(A, dist), po.minplus(bs, n, rp, ci, tw, dist))
    # the sum of FP32 terms in FP64, rounded once: half a unit in the last place of the FP64 sum's rounding
    x = rng.random(n).astype(np.float32)
    np.testing.assert_allclose(gbo.bsrbmv_sum_f32(A, x), po.sum_f64(bs, n, rp, ci, tw, x.astype(np.float64)),
                               rtol=6.1e-8, atol=0)
    A.free()
