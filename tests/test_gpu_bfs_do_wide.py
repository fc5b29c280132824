"""Direction-optimizing BFS with hundreds of levels that are pushed by many
workgroups, one after another: frontiers of at most n/64 vertices with more
blocks or tiles than one workgroup takes.  A king grid from its middle has
them: level l is a ring of 8 l vertices."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def rings(m, x, y):
    """Levels of an m x m king grid: the Chebyshev distance from (x, y)."""
    i = np.arange(m)
    return np.maximum(np.abs(i[None, :] - x), np.abs(i[:, None] - y)).ravel().astype(np.int32)


@pytest.mark.parametrize("m,bs", [(768, 8), (1024, 8), (1024, 16), (1024, 32), (1024, 64), (2048, 8), (2048, 64)])
def test_king_from_the_middle(gbo, m, bs):
    A = gbo.BsrMatrix.from_csr(gbo.gen_king(m), bs)
    for x, y in ((m // 2, m // 2), (0, 0), (m // 3, m - 1)):
        want = rings(m, x, y)
        lv, sizes = gbo.bfs(A, y * m + x, A=A)
        assert np.array_equal(lv, want), (x, y)
        assert np.array_equal(sizes, np.bincount(want)), (x, y)
    A.free()
