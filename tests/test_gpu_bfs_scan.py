"""BFS steps at bs 16 to 64 on block rows around the number of tiles a wave looks
at together, with frontiers of one vertex, of few and of all, partly visited."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _graph(gbo, bs):
    rng = np.random.default_rng(bs)
    n = 1030 * bs + 5
    counts = np.zeros(n, np.int64)
    for R, tiles in enumerate((0, 1, 63, 64, 65, 255, 256, 257, 1030)):
        counts[R * bs + rng.integers(0, bs)] = tiles  # one entry a tile
    counts[20 * bs:24 * bs] = 40
    counts[-1] = 300
    rp = np.r_[0, np.cumsum(counts)].astype(np.int32)
    rows = []
    for r in np.flatnonzero(counts):
        k = counts[r]
        blocks = rng.choice(1030, k, replace=False) if k <= 1030 else np.arange(k)
        rows.append(np.sort(blocks * bs + rng.integers(0, bs, k)))
    ci = np.concatenate(rows).astype(np.int32)
    return gbo.Csr(n, n, rp, ci)


@pytest.mark.parametrize("chunk", (0, 7, 300))  # rows whole and cut
@pytest.mark.parametrize("bs", (16, 32, 64))
def test_searches(gbo, bs, chunk):
    g = _graph(gbo, bs)
    n, ci = g.nrows, g.colind
    A = gbo.BsrMatrix.from_csr(g, bs)
    if chunk:
        A.plan(chunk)
    edge = np.repeat(np.arange(n), np.diff(g.rowptr))
    rng = np.random.default_rng(1)
    into = np.bincount(ci, minlength=n)
    for source in [int(np.argmax(into)), int(ci[0])] + list(rng.integers(0, n, 4)):
        level = np.full(n, -1, np.int32)
        front, depth = np.array([source]), 0
        while len(front):
            level[front] = depth
            depth += 1
            hit = np.unique(edge[np.isin(ci, front)])
            front = hit[level[hit] < 0]
        got, sizes = gbo.bfs(A, int(source))
        assert np.array_equal(got, level) and len(sizes) == depth


@pytest.mark.parametrize("chunk", (0, 7, 300))
@pytest.mark.parametrize("bs", (16, 32, 64))
def test_steps(gbo, po, bs, chunk):
    g = _graph(gbo, bs)
    n, rp, ci = g.nrows, g.rowptr, g.colind
    counts = np.diff(rp)
    rng = np.random.default_rng(2)
    A = gbo.BsrMatrix.from_csr(g, bs)
    A.plan(0, 0)  # at bs 16 the variant without the count kernel's form
    if chunk:
        A.plan(chunk, 0)
    edge = np.repeat(np.arange(n), counts)
    cnt = gbo.DeviceBuffer(8)
    for share in (0.0, 0.002, 0.3, 1.0):
        front = rng.random(n) < share
        front[rng.integers(0, n)] = True
        for seen in (0.0, 0.5, 1.0):
            vis = rng.random(n) < seen
            f, v = (po.pack_vec(bs, x.astype(np.float32)) for x in (front, vis))
            d_f, d_v = gbo.DeviceBuffer.from_numpy(f), gbo.DeviceBuffer.from_numpy(v)
            d_n = gbo.DeviceBuffer.from_numpy(np.full_like(f, 0x5A))
            gbo._check(gbo.lib().gbo_bsrbmv_bfs_step(A.ref, d_f.ptr, d_v.ptr, d_n.ptr, cnt.ptr, None))
            gbo.synchronize()
            want = np.bincount(edge[front[ci]], minlength=n).astype(bool) & ~vis
            assert np.array_equal(d_n.to_numpy(f.dtype, len(f)), po.pack_vec(bs, want.astype(np.float32)))
            assert cnt.to_numpy(np.int64, 1)[0] == want.sum()
