"""Drivers that queue several iterations between two looks at their flags: runs
that end at, before and after each look, and more iterations than flags."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _path(gbo, n):
    i = np.arange(n)
    deg = np.where((i == 0) | (i == n - 1), 1, 2) if n > 1 else np.zeros(1, int)
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum(deg)
    ci = np.stack([i - 1, i + 1], 1).reshape(-1)
    return gbo.Csr(n, n, rp, ci[(ci >= 0) & (ci < n)].astype(np.int32))


@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_shortest_paths_on_paths(gbo, bs):
    for n in list(range(1, 26)) + [513, 3001]:
        d, it = gbo.sssp(gbo.BsrMatrix.from_csr(_path(gbo, n), bs), 0)
        assert np.array_equal(d, np.arange(n)) and it == n, n


@pytest.mark.parametrize("variant", (0, 1, 3))
@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_bfs_on_paths(gbo, bs, variant):
    for n in list(range(1, 26)) + [513, 3001]:
        A = gbo.BsrMatrix.from_csr(_path(gbo, n), bs).plan(0, variant)
        for source in {0, n // 2}:
            d = np.abs(np.arange(n) - source)
            want = np.bincount(d)
            level, sizes = gbo.bfs(A, source)
            assert np.array_equal(level, d) and np.array_equal(sizes, want), (n, source)
            out, got, nl = gbo.DeviceBuffer(4 * n), np.zeros(4096, np.int64), ctypes.c_int32()
            gbo._check(gbo.lib().gbo_bfs_noalloc(A.ref, source, out.ptr, got.ctypes.data, 4096, ctypes.byref(nl), None))
            assert np.array_equal(out.to_numpy(np.int32, n), d) and np.array_equal(got[:nl.value], want), (n, source)


@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_components_of_paths(gbo, bs):
    for n in (1, 2, 3, 5, 9, 70, 1000, 4097):
        lab, it = gbo.cc(gbo.BsrMatrix.from_csr(_path(gbo, n), bs))
        assert not lab.any() and it >= 1, n


@pytest.mark.parametrize("n", (300, 20000))  # one block sums the change, many do
@pytest.mark.parametrize("bs", (8, 64))
def test_pagerank_stops_at_max_iter(gbo, bs, n):
    """The iterate after exactly m iterations, in float64; three roundings of
    2^-24 each iteration (all terms positive): m * 3 * 2^-24 relative."""
    g = gbo.gen_er(n, 8 / n, 5)
    A = gbo.BsrMatrix.from_csr(g, bs)
    deg = np.diff(g.rowptr).astype(np.int32)
    rows = np.repeat(np.arange(n), deg)
    alpha = float(np.float32(0.85))
    x = np.full(n, 1.0 / n)
    for m in range(1, 13):
        s = np.where(deg > 0, alpha * x / np.maximum(deg, 1), 0.0)
        prev, x = x, np.bincount(rows, s[g.colind], n) + (1.0 - alpha) / n
        p, it, delta = gbo.pagerank(A, deg, alpha, 0.0, m)
        assert it == m
        assert np.max(np.abs(p - x) / x) < (m + 1) * 3 * 2.0 ** -24
        # each difference of the two iterates is off by their errors at most
        assert abs(delta - np.abs(x - prev).sum()) < (2 * m + 1) * 3 * 2.0 ** -24 * 2
