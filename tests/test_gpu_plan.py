"""Products on the library's own plan (chunks of about equal work, shorter
where the tiles are dense) against the oracle, on matrices whose block rows
run over one to hundreds of chunks and whose tile count is at the edges of
the units the plan is cut in."""
import numpy as np
import pytest

from graphs import sym_csr

pytestmark = pytest.mark.gpu


def dense_core(gbo, n, core, hub, m, seed):
    """`core` vertices joined with probability 0.75 (dense tiles), a hub joined
    to all, m random edges."""
    rng = np.random.default_rng(seed)
    cu, cv = np.nonzero(rng.random((core, core)) < 0.5)
    u, v = [cu, rng.integers(0, n, m)], [cv, rng.integers(0, n, m)]
    if hub:
        u.append(np.full(n, n // 2))
        v.append(np.arange(n))
    rp, ci = sym_csr(n, np.concatenate(u), np.concatenate(v))
    return gbo.Csr(n, n, rp, ci)


@pytest.mark.parametrize("bs", (8, 16, 32, 64))
@pytest.mark.parametrize("n,core,hub,m", [(20_000, 700, True, 40_000), (4_099, 300, True, 3_000), (640, 640, False, 0),
                                          (65, 9, False, 20), (300_007, 400, True, 700_000)])
def test_own_plan(gbo, po, bs, n, core, hub, m):
    g = dense_core(gbo, n, core, hub, m, bs + n)
    A = gbo.BsrMatrix.from_csr(g, bs)
    rp, ci, tw = A.host_arrays()
    assert A.s.plan_nchunks >= 1 and 16 <= A.s.plan_chunk <= 256
    rng = np.random.default_rng(n)
    xb = gbo.pack_vec(bs, (rng.random(n) < 0.3).astype(np.float32))
    assert np.array_equal(gbo.bsrbmv_count(A, xb), po.count(bs, n, rp, ci, tw, xb))
    vis = gbo.pack_vec(bs, (rng.random(n) < 0.5).astype(np.float32))
    nx, cnt = gbo.bsrbmv_bfs_step(A, xb, vis)
    onx, ocnt = po.bfs_step(bs, n, rp, ci, tw, xb, vis)
    assert np.array_equal(nx, onx) and cnt == ocnt
    xi = rng.integers(-2**31, 2**31 - 1, n).astype(np.int32)
    assert np.array_equal(gbo.bsrbmv_min_i32(A, xi), po.min_i32(bs, n, rp, ci, tw, xi))
    dist = rng.integers(0, 1000, n).astype(np.uint32)
    dist[rng.random(n) < 0.3] = gbo.INF_U32
    assert np.array_equal(gbo.bsrbmv_minplus(A, dist), po.minplus(bs, n, rp, ci, tw, dist))
    w = gbo.edge_weights(g, 1, 64, seed=9)
    tv = gbo.TileValues(A, g, w)
    otv, owoff = po.pack_values(bs, n, g.rowptr, g.colind, w, rp, ci, tw)
    assert np.array_equal(gbo.bsrbmv_minplus(A, dist, tv), po.minplus(bs, n, rp, ci, tw, dist, otv, owoff))
    # the sum of FP32 terms in FP64, rounded once: half a unit in the last place of the FP64 sum's rounding
    x = rng.random(n).astype(np.float32)
    y = gbo.bsrbmv_sum_f32(A, x)
    np.testing.assert_allclose(y, po.sum_f64(bs, n, rp, ci, tw, x.astype(np.float64)), rtol=6.1e-8, atol=0)
    assert np.array_equal(y.view(np.uint32), gbo.bsrbmv_sum_f32(A, x).view(np.uint32))
    A.free()
