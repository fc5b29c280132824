"""Direction-optimizing BFS over graphs whose small frontiers run for many
levels in one launch: levels and level sizes against the oracle's queue BFS.
The graphs reach each way a run ends: the frontier empties, a launch's most
levels, a frontier of too many blocks, tiles or vertices, rows taken by the
whole workgroup."""
import numpy as np
import pytest

from graphs import sym_csr

pytestmark = pytest.mark.gpu
BS = (8, 16, 32, 64)


def check(gbo, po, g, bs, sources):
    A = gbo.BsrMatrix.from_csr(g, bs)
    for s in sources:
        want = po.bfs(g.nrows, g.rowptr, g.colind, s)
        lv, sizes = gbo.bfs(A, s, A=A)
        assert np.array_equal(lv, want), s
        assert np.array_equal(sizes, np.bincount(want[want >= 0])), s
    A.free()


def tree(gbo, fan, depth, seed):
    """Complete tree of the given fan-out, vertices numbered at random."""
    n = (fan ** (depth + 1) - 1) // (fan - 1)
    child = np.arange(1, n)
    p = np.random.default_rng(seed).permutation(n)
    rp, ci = sym_csr(n, p[child], p[(child - 1) // fan])
    return gbo.Csr(n, n, rp, ci), int(p[0])


@pytest.mark.parametrize("bs", BS)
def test_path(gbo, po, bs):
    n = 2600  # 2600 levels from one end: three launches
    rp, ci = sym_csr(n, np.arange(n - 1), np.arange(1, n))
    check(gbo, po, gbo.Csr(n, n, rp, ci), bs, (0, n - 1, n // 2))


@pytest.mark.parametrize("bs", BS)
def test_grid(gbo, po, bs):
    check(gbo, po, gbo.gen_king(150), bs, (0, 11_111))


@pytest.mark.parametrize("bs", BS)
def test_wide_tree(gbo, po, bs):
    g, root = tree(gbo, 3, 12, 5)  # 2187 -> 6561 vertices: more than 4096 blocks at bs 8
    check(gbo, po, g, bs, (root, 0))


@pytest.mark.parametrize("bs", BS)
def test_hubs(gbo, po, bs):
    """A path into a vertex of 6000 neighbours (rows of more than 256 tiles),
    on to one of 200,000 (more than 16384 tiles at bs 8), and out again."""
    n = 400_000
    rng = np.random.default_rng(9)
    mid, big = rng.choice(n, 6000, replace=False), rng.choice(n, 200_000, replace=False)
    u = [np.arange(20), np.full(6000, 20), np.full(200_000, mid[0]), np.array([big[0]])]
    v = [np.arange(1, 21), mid, big, np.array([n - 1])]
    rp, ci = sym_csr(n, np.concatenate(u), np.concatenate(v))
    check(gbo, po, gbo.Csr(n, n, rp, ci), bs, (0, 20, n - 1))


@pytest.mark.parametrize("bs", (8, 64))
def test_directed(gbo, po, bs):
    """A is the out-edge matrix, AT its transpose."""
    g = gbo.gen_rmat(12, 4, seed=3)
    row = np.repeat(np.arange(g.nrows), np.diff(g.rowptr))
    keep = (row < g.colind) | (row % 3 == 0)
    rp = np.concatenate([[0], np.cumsum(np.bincount(row[keep], minlength=g.nrows))])
    d = gbo.Csr(g.nrows, g.nrows, rp, g.colind[keep])
    A, AT = gbo.BsrMatrix.from_csr(d, bs), gbo.BsrMatrix.from_csr(d.transpose(), bs)
    for s in (0, 77, 1234):
        lv, _ = gbo.bfs(AT, s, A=A)
        assert np.array_equal(lv, po.bfs(d.nrows, d.rowptr, d.colind, s))
