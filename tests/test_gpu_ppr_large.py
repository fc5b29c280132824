"""Personalized PageRank over more vertices, or vertices times columns, than a
launch has threads for (2^32): nearly empty graphs, the values at both ends."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
ALPHA = 0.85


def device_memory(gbo, need):
    gbo.lib()
    hip = ctypes.CDLL(gbo.hip_runtimes()[0])
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    if free.value < need << 30:
        pytest.skip(f"needs {need} GB of device memory")


def test_many_elements(gbo):
    """68.2M vertices of 63 columns, one edge u -> v between the last two;
    column 62 starts at u, column 0 at vertex 0, the others nowhere."""
    device_memory(gbo, 110)
    n, K, bs = 68_200_000, 63, 16
    assert n * K > 1 << 32
    u, v = n - 2, n - 1
    nbr = (n + bs - 1) // bs
    # A^T: row v has column u
    rp = gbo.DeviceBuffer.zeros(4 * (nbr + 1))
    rp.view(4 * nbr, 4).copy_from(np.ones(1, np.int32))
    ci = gbo.DeviceBuffer.from_numpy(np.array([u // bs], np.int32))
    assert u // bs == v // bs == nbr - 1
    tile = np.zeros(bs, np.uint16)
    tile[v % bs] = 1 << (bs - 1 - u % bs)
    tiles = gbo.DeviceBuffer.from_numpy(tile)
    s = gbo.BsrStruct(bs=bs, dir=0, nrows=n, ncols=n, nblockrows=nbr, nblockcols=nbr, nblocks=1, rowptr=rp.ptr,
                      colind=ci.ptr, tiles=tiles.ptr)
    deg = gbo.DeviceBuffer.zeros(4 * n)
    deg.view(4 * u, 4).copy_from(np.ones(1, np.int32))
    S, P = gbo.DeviceBuffer.zeros(4 * n * K), gbo.DeviceBuffer(4 * n * K)
    one = np.ones(1, np.float32)
    S.view(0, 4).copy_from(one)
    S.view(4 * (u * K + K - 1), 4).copy_from(one)
    gbo._check(gbo.lib().gbo_memset(P.ptr, 0xFF, P.nbytes))
    it, delta = ctypes.c_int32(), ctypes.c_double()
    gbo._check(gbo.lib().gbo_ppr_forward(ctypes.byref(s), deg.ptr, K, ALPHA, S.ptr, P.ptr, 1e-6, 50, ctypes.byref(it),
                                         ctypes.byref(delta), None))
    first, last = P.view(0, 4 * K).to_numpy(np.float32), P.view(4 * u * K, 8 * K).to_numpy(np.float32).reshape(2, K)
    a = np.float32(ALPHA)
    want0, want = np.zeros(K, np.float32), np.zeros((2, K), np.float32)
    want0[0] = 1 - a
    want[0, K - 1] = 1 - a
    want[1, K - 1] = a * (1 - a)
    np.testing.assert_allclose(first, want0, rtol=2e-7, atol=0)
    np.testing.assert_allclose(last, want, rtol=3e-7, atol=0)
    for x in (rp, ci, tiles, deg, S, P):
        x.free()


def test_many_block_rows(gbo):
    """2^29 vertices at bs 8, 2^26 block rows of one tile, each vertex with an
    edge to itself: p = s from the start."""
    device_memory(gbo, 130)
    n, bs = 1 << 29, 8
    nbr = n // bs
    rp = gbo.DeviceBuffer.from_numpy(np.arange(nbr + 1, dtype=np.int32))
    ci = gbo.DeviceBuffer.from_numpy(np.arange(nbr, dtype=np.int32))
    tiles = gbo.DeviceBuffer.from_numpy(np.tile(1 << np.arange(7, -1, -1), nbr).astype(np.uint8))
    s = gbo.BsrStruct(bs=bs, dir=0, nrows=n, ncols=n, nblockrows=nbr, nblockcols=nbr, nblocks=nbr, rowptr=rp.ptr,
                      colind=ci.ptr, tiles=tiles.ptr)
    deg = gbo.DeviceBuffer.from_numpy(np.ones(n, np.int32))
    val = np.zeros(n, np.float32)
    at = np.r_[0:4000, n // 2:n // 2 + 4000, n - 4000:n]
    val[at] = np.random.default_rng(1).random(len(at)).astype(np.float32) + 1
    S, P = gbo.DeviceBuffer.from_numpy(val), gbo.DeviceBuffer.zeros(4 * n)
    it, delta = ctypes.c_int32(), ctypes.c_double()
    gbo._check(gbo.lib().gbo_ppr_forward(ctypes.byref(s), deg.ptr, 1, ALPHA, S.ptr, P.ptr, 1e-5, 4, ctypes.byref(it),
                                         ctypes.byref(delta), None))
    # alpha s + (1 - alpha) s, each iteration rounded once
    np.testing.assert_allclose(P.to_numpy(np.float32), val, rtol=4 * 2.0 ** -24, atol=0)
    for x in (rp, ci, tiles, deg, S, P):
        x.free()
