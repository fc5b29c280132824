"""Calls that do not wait for their stream: they return while work that was
queued before them still runs, and their results are there once it has."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
NOT_READY = 600  # hipErrorNotReady


@pytest.mark.parametrize("scale,bs", [(8, 8), (16, 8), (14, 64)])
def test_bit_offsets_without_a_total(gbo, scale, bs):
    L = gbo.lib()
    gbo.lib()
    hip = ctypes.CDLL(gbo.hip_runtimes()[0])
    g = gbo.gen_rmat(scale, 8, seed=3)
    A = gbo.BsrMatrix.from_csr(g, bs)
    _, _, tiles = A.host_arrays()
    bits = np.unpackbits(tiles.view(np.uint8)).reshape(A.nblocks, -1).sum(1)
    want = np.concatenate([[0], np.cumsum(bits, dtype=np.int64)])
    st = ctypes.c_void_p()
    gbo._check(L.gbo_stream_create(ctypes.byref(st)))
    size = 1 << 30
    a, b = gbo.DeviceBuffer.zeros(size), gbo.DeviceBuffer(size)
    out = gbo.DeviceBuffer(8 * (A.nblocks + 1))
    gbo._check(L.gbo_bsr_bit_offsets(A.ref, out.ptr, None, st))  # whatever a first call sets up
    gbo.synchronize()
    gbo._check(L.gbo_memset(out.ptr, 0xFF, out.nbytes))
    for _ in range(300):  # some 100 ms of copies
        gbo._check(L.gbo_stream_copy(b.ptr, a.ptr, size, st))
    gbo._check(L.gbo_bsr_bit_offsets(A.ref, out.ptr, None, st))
    assert hip.hipStreamQuery(st) == NOT_READY
    gbo._check(L.gbo_stream_synchronize(st))
    assert np.array_equal(out.to_numpy(np.int64, A.nblocks + 1), want)
    nnz = ctypes.c_int64()
    gbo._check(L.gbo_bsr_bit_offsets(A.ref, out.ptr, ctypes.byref(nnz), st))
    assert nnz.value == want[-1]
    gbo._check(L.gbo_stream_destroy(st))
    for x in (a, b, out):
        x.free()
    A.free()
