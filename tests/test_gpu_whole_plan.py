"""Plans whose chunks end at block rows: every product and step at the longest
block row that they are made for and one tile past it, with empty block rows
first, between and last, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
LONGEST = {8: 256, 16: 128, 32: 32, 64: 16}


def _matrix(gbo, bs, longest):
    rng = np.random.default_rng(bs)
    nbr = 700
    n = nbr * bs - 3
    rows, cols = [], []
    for R in range(nbr):
        k = 0 if R in (0, 1, 50, 51, 52, nbr - 1) else longest if R == 60 else rng.integers(1, min(longest, 12) + 1)
        J = rng.choice(nbr - 1, k, replace=False)
        for _ in range(2):
            rows.append(R * bs + rng.integers(0, bs, k))
            cols.append(J * bs + rng.integers(0, bs, k))
    e = np.unique(np.stack([np.concatenate(rows), np.concatenate(cols)], 1), axis=0)
    rp = np.r_[0, np.cumsum(np.bincount(e[:, 0], minlength=n))].astype(np.int32)
    return gbo.Csr(n, n, rp, e[:, 1].astype(np.int32))


@pytest.mark.parametrize("past", (0, 1))
@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_products(gbo, po, bs, past):
    g = _matrix(gbo, bs, LONGEST[bs] + past)
    n = g.nrows
    A = gbo.BsrMatrix.from_csr(g, bs)
    assert (A.s.plan_even == 2) == (past == 0)
    edge = np.repeat(np.arange(n), np.diff(g.rowptr))
    rng = np.random.default_rng(1)
    x = (rng.random(n) < 0.4).astype(np.float32)
    bits = gbo.pack_vec(bs, x)
    assert np.array_equal(gbo.bsrbmv_count(A, bits), np.bincount(edge, x[g.colind], n).astype(np.int32))
    v = rng.integers(-1000, 1000, n).astype(np.int32)
    want = np.full(n, np.iinfo(np.int32).max, np.int32)
    np.minimum.at(want, edge, v[g.colind])
    assert np.array_equal(gbo.bsrbmv_min_i32(A, v), want)
    f = rng.random(n).astype(np.float32)
    want = np.bincount(edge, f[g.colind].astype(np.float64), n).astype(np.float32)
    got = gbo.bsrbmv_sum_f32(A, f)
    assert np.all(np.abs(got - want) <= 2.0 ** -23 * want)  # FP64 sums, one rounding each
    d = np.where(rng.random(n) < 0.5, rng.integers(0, 1000, n), 0xFFFFFFFF).astype(np.uint32)
    w = gbo.edge_weights(g, 1, 64, seed=2)
    cand = np.minimum(d[g.colind].astype(np.int64) + w, 0xFFFFFFFF)
    want = d.astype(np.int64)
    np.minimum.at(want, edge, cand)
    assert np.array_equal(gbo.bsrbmv_minplus(A, d, gbo.TileValues(A, g, w)).astype(np.int64), want)
    vis = gbo.pack_vec(bs, (rng.random(n) < 0.3).astype(np.float32))
    nx, cnt = gbo.bsrbmv_bfs_step(A, bits, vis)
    onx, ocnt = po.bfs_step(bs, n, *A.host_arrays(), bits, vis)
    assert np.array_equal(nx, onx) and cnt == ocnt
