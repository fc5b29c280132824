"""Products around the number of candidate pairs up to which a block row of C is
formed by one wave: every size of its sort, rows of more than a wave's tiles,
empty and long rows of B, unproductive pairs; and one block row past it."""
import numpy as np
import pytest

from test_gpu_spgemm import _check_product

pytestmark = pytest.mark.gpu
# tiles of a block row of A, tiles of the block rows of B that they meet
ROWS = [(1, 1), (2, 1), (1, 63), (64, 1), (65, 1), (1, 128), (129, 1), (3, 40), (0, 1), (16, 16), (85, 3), (255, 1),
        (256, 1), (1, 256), (300, 0)]


def _operands(gbo, bs, rows):
    rng = np.random.default_rng(bs)
    inner = sum(m for m, _ in rows)  # a block row of B for every tile of A
    A, B = [], []
    k0 = 0
    for i, (m, l) in enumerate(rows):
        for K in range(k0, k0 + m):
            A.append((i * bs + rng.integers(0, bs), K * bs + rng.integers(0, 2)))
            A.append((i * bs + rng.integers(0, bs), K * bs + rng.integers(0, 2)))
            J = rng.choice(300, l, replace=False)
            r = K * bs + rng.integers(0, 2 if bs > 8 else 3, l)  # some of A's columns meet empty rows
            B.extend(zip(r, J * bs + rng.integers(0, bs, l)))
        k0 += m

    def csr(entries, n, m):
        e = np.unique(np.array(entries, np.int64).reshape(-1, 2), axis=0)
        rp = np.r_[0, np.cumsum(np.bincount(e[:, 0], minlength=n))].astype(np.int32)
        return gbo.Csr(n, m, rp, e[:, 1].astype(np.int32))

    return csr(A, len(rows) * bs - 3, inner * bs) if A[-1][0] < len(rows) * bs - 3 else csr(
        A, len(rows) * bs, inner * bs), csr(B, inner * bs, 300 * bs)


@pytest.mark.parametrize("past", (False, True))
@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_rows_around_the_bound(gbo, po, bs, past):
    A, B = _operands(gbo, bs, ROWS + ([(257, 1)] if past else []))
    _check_product(gbo, po, A, B, bs)
