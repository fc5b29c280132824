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


@pytest.mark.parametrize("bs", (8, 32))
def test_wide_and_narrow_in_turn(gbo, po, bs):
    """Four grids joined by paths: frontiers grow past what one workgroup takes
    and shrink to one vertex again."""
    m, path = 800, 40
    step = m * m + path
    k = gbo.gen_king(m)
    row = np.repeat(np.arange(k.nrows), np.diff(k.rowptr))
    u, v = [], []
    for q in range(4):
        o = q * step
        u.append(row + o)
        v.append(k.colind + o)
        # from the last row's middle, over the path, to the middle of the next grid's first row
        chain = np.concatenate([[o + m * (m - 1) + m // 2], o + m * m + np.arange(path), [o + step + m // 2]])
        chain = chain[chain < 4 * step]
        u += [chain[:-1], chain[1:]]
        v += [chain[1:], chain[:-1]]
    n = 4 * step
    key = np.unique(np.concatenate(u).astype(np.int64) * n + np.concatenate(v))
    rp = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))])
    g = gbo.Csr(n, n, rp, key % n)
    A = gbo.BsrMatrix.from_csr(g, bs)
    for s in (m // 2 * m + m // 2, 0, n - 1):
        want = po.bfs(n, g.rowptr, g.colind, s)
        lv, sizes = gbo.bfs(A, s, max_levels=8192, A=A)
        assert np.array_equal(lv, want), s
        assert np.array_equal(sizes, np.bincount(want)), s
    A.free()
