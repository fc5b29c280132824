"""Tiles whose padding (rows and columns past the matrix) holds bits, as a
caller's own packer may leave them: the listings of personalized PageRank and
of the triangle count take no row of the padding and no list past the last."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def with_tiles(gbo, A, tiles):
    """A's structure over other tile words."""
    d = gbo.DeviceBuffer.from_numpy(tiles)
    s = gbo.BsrStruct.from_buffer_copy(A.s)
    s.tiles, s.plan, s.plan_chunk, s.plan_nchunks = d.ptr, None, 0, 0
    return s, d


def last_rows(bs, n, rp):
    """Words of padding rows in the last block row: (tiles, rows)."""
    return slice(rp[-2], rp[-1]), slice(n % bs, bs)


@pytest.mark.parametrize("bs", (8, 16, 32))
@pytest.mark.parametrize("n,deg", [(1003, 6), (20_001, 16)])
def test_ppr_rows(gbo, bs, n, deg):
    g = gbo.gen_er_m(n, n * deg // 2, 3)
    A = gbo.BsrMatrix.from_csr(g, bs)
    rp, ci, tiles = A.host_arrays()
    dirty = tiles.reshape(-1, bs).copy()
    t, r = last_rows(bs, n, rp)
    assert t.stop > t.start and r.stop > r.start
    dirty[t, r] = np.iinfo(dirty.dtype).max
    ok = ci[t] < n // bs  # whole block columns: no column of the padding
    dirty[t][~ok] = tiles.reshape(-1, bs)[t][~ok]
    s, d = with_tiles(gbo, A, dirty.ravel())
    rng = np.random.default_rng(bs)
    S = rng.random((n, 5)).astype(np.float32)
    want, it, _ = gbo.ppr_forward(A, g.outdeg(), S, 0.85, 1e-6, 100)
    od, dS, dP = gbo.DeviceBuffer.from_numpy(g.outdeg()), gbo.DeviceBuffer.from_numpy(S), gbo.DeviceBuffer(S.nbytes)
    n_it, delta = ctypes.c_int32(), ctypes.c_double()
    gbo._check(gbo.lib().gbo_ppr_forward(ctypes.byref(s), od.ptr, 5, 0.85, dS.ptr, dP.ptr, 1e-6, 100,
                                         ctypes.byref(n_it), ctypes.byref(delta), None))
    assert n_it.value == it
    assert np.array_equal(dP.to_numpy(np.float32).reshape(n, 5), want)
    A.free()


@pytest.mark.parametrize("bs", (8, 16, 32, 64))
@pytest.mark.parametrize("n,deg", [(1003, 6), (5001, 120)])
def test_tc_columns(gbo, bs, n, deg):
    """Every row of L's last block column names the padding columns too (their
    lists are empty), and so may rows of all lengths."""
    g = gbo.gen_er_m(n, n * deg // 2, 4)
    L = g.tril()
    rows = np.repeat(np.arange(n), np.diff(L.rowptr))
    key = np.unique(np.concatenate([rows * n + L.colind, np.arange(n - 1) * n + n - 1]))  # a last column in most rows
    rp = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))])
    M = gbo.Csr(n, n, rp, key % n)
    A, B = gbo.BsrMatrix.from_csr(M, bs), gbo.BsrMatrix.from_csr(M.transpose(), bs, 1)
    want = gbo.bsrbmm_tc(A, B)
    brp, ci, tiles = A.host_arrays()
    dirty = tiles.reshape(-1, bs).copy()
    pad = bs - n % bs  # low bits of a word
    last = ci == n // bs
    assert last.sum() > n // bs // 2
    has = dirty[last] != 0
    dirty[last] |= np.where(has, dirty.dtype.type((1 << pad) - 1), dirty.dtype.type(0))
    s, d = with_tiles(gbo, A, dirty.ravel())
    cnt = gbo.DeviceBuffer(8)
    gbo._check(gbo.lib().gbo_bsrbmm_tc(ctypes.byref(s), B.ref, cnt.ptr, None))
    assert int(cnt.to_numpy(np.uint64)[0]) == want
    A.free()
    B.free()
