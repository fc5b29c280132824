"""Blocks kept between calls: one too large to be kept sends no other off, and
those of a call of some GB are there for the next."""
import ctypes
import gc
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_large_blocks(gbo):
    gc.collect()  # no matrix of another test
    gbo.lib()
    hip = ctypes.CDLL(gbo.hip_runtimes()[0])

    def free():
        gbo.synchronize()
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    n, K, bs = (1 << 24) + 4096, 64, 8
    if free() < 40 << 30:
        pytest.skip("needs 40 GB of device memory")
    g = gbo.gen_er_m(1 << 20, 1 << 21, 1)
    A = gbo.BsrMatrix.from_csr(g, bs)
    rp = np.zeros(n + 1, np.int32)
    rp[n] = 1
    B = gbo.BsrMatrix.from_csr(gbo.Csr(n, n, rp, np.array([n - 1], np.int32)), bs)
    S, P, deg = gbo.DeviceBuffer.zeros(4 * n * K), gbo.DeviceBuffer(4 * n * K), gbo.DeviceBuffer.zeros(4 * n)
    it, delta = ctypes.c_int32(), ctypes.c_double()

    def ppr(M, rows):
        rc = gbo.lib().gbo_ppr_forward(M.ref, deg.ptr, K, 0.85, S.ptr, P.ptr, 1e-1, 3, ctypes.byref(it),
                                       ctypes.byref(delta), None)
        gbo._check(rc)
        return free()

    before = free()
    small = ppr(A, g.nrows)   # two iterates of 256 MB
    assert before - small > 500 << 20
    assert ppr(A, g.nrows) == small
    # two of 4 GB and more: nothing of the small call's goes (what is freed may
    # be counted as taken for a while longer, but not the other way round)
    assert ppr(B, n) <= small
    assert ppr(A, g.nrows) <= small
    A.free()
    B.free()
    for _ in range(50):
        if free() >= before:  # all of it goes with the last matrix
            break
        time.sleep(0.1)
    assert free() >= before
