"""Personalized PageRank over every column layout (1 to 64 columns, padded
rows, 1 to 16 nonzeros at a time) on a directed graph with rows at the edges
of the segment lengths, against the FP64 fixed points of the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ALPHA = 0.85


@pytest.fixture(scope="module")
def hub_graph(gbo):
    """Rows of A^T of 0, 1, 63, 64, 65, 128, 4096, 4097 and 66000 nonzeros
    (one segment, several of 64, of 256 and of 1024) among random ones."""
    n = 66_037
    rng = np.random.default_rng(3)
    u, v = [rng.integers(0, n, 90_000)], [rng.integers(100, n - 7, 90_000)]  # the last vertices have no in-edges
    for row, deg in enumerate((1, 63, 64, 65, 128, 4096, 4097, 66_000)):
        u.append(rng.permutation(n)[:deg])
        v.append(np.full(deg, row))
    key = np.unique(np.concatenate(u).astype(np.int64) * n + np.concatenate(v))
    u, v = key // n, key % n
    keep = u != v
    u, v = u[keep], v[keep]
    rp = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))])
    return gbo.Csr(n, n, rp, v)


@pytest.mark.parametrize("bs,K", [(8, 1), (16, 3), (8, 4), (32, 5), (16, 8), (8, 9), (8, 16), (16, 17), (32, 31),
                                  (8, 33), (16, 37), (8, 64), (32, 64)])
def test_ppr_columns(gbo, po, hub_graph, bs, K):
    g = hub_graph
    n, deg, t = g.nrows, g.outdeg(), g.transpose()
    rng = np.random.default_rng(K)
    S = np.zeros((n, K))
    for k in range(K):
        S[rng.choice(n, 50, replace=False), k] = rng.dirichlet(np.full(50, 0.5))
    W = rng.standard_normal((n, K))
    S32, W32 = S.astype(np.float32), W.astype(np.float32)
    A, AT = gbo.BsrMatrix.from_csr(g, bs), gbo.BsrMatrix.from_csr(t, bs)
    # tolerance 1e-8: within 1e-6 L1 of the fixed point (a change of d leaves at
    # most d * alpha / (1 - alpha) to go; FP32 rounding of P adds 6e-8)
    P, it, _ = gbo.ppr_forward(AT, deg, S32, ALPHA, 1e-8, 400)
    want, _ = po.ppr_solve(n, t.rowptr, t.colind, deg, ALPHA, 0, S32)
    assert np.abs(P - want).sum(0).max() <= 1e-6
    gS, ga, _ = gbo.ppr_adjoint(A, AT, deg, S32, P, W32, ALPHA, 1e-8, 400)
    lam, _ = po.ppr_solve(n, g.rowptr, g.colind, deg, ALPHA, 1, W32)
    assert np.abs(gS - (1 - ALPHA) * lam).max() <= 1e-5 * np.abs((1 - ALPHA) * lam).max()
    PT = np.zeros_like(want)
    np.add.at(PT, np.repeat(np.arange(n), np.diff(t.rowptr)),
              (want / np.maximum(deg, 1)[:, None])[t.colind])
    wa = (lam * (PT - S32)).sum()
    assert abs(ga - wa) <= 1e-5 * np.abs(lam * (PT - S32)).sum()
    # an odd number of iterations, cut off: the iterate of that iteration, the same bits each time
    P3 = [gbo.ppr_forward(AT, deg, S32, ALPHA, 0.0, 3) for _ in range(2)]
    assert P3[0][1] == 3 and np.array_equal(P3[0][0].view(np.uint32), P3[1][0].view(np.uint32))
    p = S32.astype(np.float64)
    for _ in range(3):
        q = np.zeros_like(p)
        np.add.at(q, np.repeat(np.arange(n), np.diff(t.rowptr)), (p / np.maximum(deg, 1)[:, None])[t.colind])
        p = ALPHA * q + (1 - ALPHA) * S32
    assert np.abs(P3[0][0] - p).sum(0).max() <= 1e-6
    A.free()
    AT.free()
