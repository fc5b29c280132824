"""A matrix without columns has no nonzeros: whatever column its rows name is
out of range, in block rows of few nonzeros and of many."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_row", (0, 1, 40, 700))
@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_no_columns(gbo, bs, per_row):
    n = 2 * bs + 3
    rp = (np.arange(n + 1) * per_row).astype(np.int32)
    L, nb = gbo.lib(), ctypes.c_int64(-1)
    d_rp, d_brp = gbo.DeviceBuffer.from_numpy(rp), gbo.DeviceBuffer(4 * 4)
    for ci in (np.zeros(n * per_row, np.int32), np.tile(np.arange(per_row, dtype=np.int32), n)):
        d_ci = gbo.DeviceBuffer.from_numpy(ci)
        rc = L.gbo_csr2bsr_nnzb_dev(bs, d_rp.ptr, d_ci.ptr, n, 0, d_brp.ptr, ctypes.byref(nb), None)
        if per_row == 0:
            assert rc == 0 and nb.value == 0
        else:
            assert rc == -1 and b"range" in L.gbo_last_error()
