"""Scratch of a general product that is sorted globally: what it holds at once is
its pairs' keys, as given and sorted, and the sort's own, not what the phases
before and after the sort used as well."""
import ctypes
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", (8, 32))
def test_symbolic(gbo, bs):
    gc.collect()
    gbo.lib()
    hip = ctypes.CDLL(gbo.hip_runtimes()[0])

    def free():
        gbo.synchronize()
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    n = 1 << 17
    g = gbo.gen_er_m(n, n * 6, 1)
    gbo.BsrMatrix.from_csr(g, bs).free()  # the last matrix: nothing is kept now
    A = gbo.BsrMatrix.from_csr(g, bs, plan=False)
    deg = np.diff(g.rowptr).astype(np.int64)
    pairs = int((deg * deg).sum())  # scalar products: at least the pairs of tiles with one
    d_rp, nb = gbo.DeviceBuffer(4 * (A.nblockrows + 1)), ctypes.c_int64()
    before = free()
    gbo._check(gbo.lib().gbo_bsrbmm_symbolic(A.ref, A.ref, d_rp.ptr, ctypes.byref(nb), None))
    held = before - free()
    # 8-byte keys three times and C's block rows, rounded up by an eighth at most; a few words per tile of A
    assert held <= (3 * 8 * pairs + 4 * nb.value) * 9 // 8 + 64 * A.nblocks
    assert held > 8 * nb.value
    A.free()
