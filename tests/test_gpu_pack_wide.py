"""Packing of matrices of many block columns: block rows around the numbers of
nonzeros from which they are not merged, which grow with the width, and widths
at which they are merged in pieces.  Byte for byte the oracle's, and refused
where the narrow ones are."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
WINDOW = 1 << 18  # block columns of one bitmap
# windows, nonzeros of block rows at the bound there
WIDTHS = [(1, 256), (2, 384), (3, 576), (4, 768), (5, 768)]


def wide(bs, windows, above):
    """Block rows of about `above` nonzeros, none, one of a hub row, and a last
    one that is not whole; the last window holds one block column and a bit."""
    rng = np.random.default_rng(bs * 8 + windows)
    ncols = ((windows - 1) * WINDOW + 1) * bs + 3 if windows > 1 else WINDOW * bs
    counts = []
    for total in (above - 1, above, above + 1, 8 * bs, 8 * bs + 1, 2048, 2049):
        counts.append(np.bincount(rng.integers(0, bs, total), minlength=bs))
    counts.append(np.zeros(bs, np.int64))
    counts.append(np.r_[30000, rng.integers(0, 30, bs - 1)])
    counts.append(np.full(bs - 3, above // 4))
    counts = np.concatenate(counts)
    rows = [np.unique(rng.integers(0, ncols, k)) if k else np.zeros(0, np.int64) for k in counts]
    rows[8 * bs][-1] = ncols - 1
    rp = np.r_[0, np.cumsum([len(r) for r in rows])].astype(np.int32)
    return len(rows), ncols, rp, np.concatenate(rows).astype(np.int32)


@pytest.mark.parametrize("direction", (0, 1))
@pytest.mark.parametrize("windows,above", WIDTHS)
@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_wide(gbo, po, bs, windows, above, direction):
    n, ncols, rp, ci = wide(bs, windows, above)
    d_rp, d_ci = gbo.DeviceBuffer.from_numpy(rp), gbo.DeviceBuffer.from_numpy(ci)
    A = gbo.BsrMatrix.from_device_csr(d_rp, d_ci, n, ncols, bs, direction)
    for got, exp in zip(A.host_arrays(), po.pack(bs, n, rp, ci, direction)):
        assert np.array_equal(got, exp)
    A.free()
    L, nb, d_brp = gbo.lib(), ctypes.c_int64(), gbo.DeviceBuffer(4 * (n // bs + 2))
    hub = rp[8 * bs]
    for at, value, what in ((hub + 1, ncols, b"range"), (0, -1, b"range"), (rp[-1] - 1, ncols, b"range"),
                            (hub + 20000, 0, b"sorted"), (hub, ncols - 1, b"sorted")):
        bad = ci.copy()
        bad[at] = value
        d_bad = gbo.DeviceBuffer.from_numpy(bad)
        rc = L.gbo_csr2bsr_nnzb_dev(bs, d_rp.ptr, d_bad.ptr, n, ncols, d_brp.ptr, ctypes.byref(nb), None)
        assert rc == -1 and what in L.gbo_last_error(), (at, value)
    # a row pointer that ends elsewhere is refused before anything is written
    good = A_rowptr(gbo, L, bs, d_rp, d_ci, n, ncols, d_brp)
    brp = good.copy()
    brp[-1] += 1
    d_wrong, out = gbo.DeviceBuffer.from_numpy(brp), gbo.DeviceBuffer.from_numpy(np.full(64, 7, np.uint8))
    rc = L.gbo_csr2bsr_fill_dev(bs, direction, d_rp.ptr, d_ci.ptr, n, ncols, d_wrong.ptr, out.ptr, out.ptr, None)
    assert rc == -1 and b"rowptr" in L.gbo_last_error()
    assert (out.to_numpy(np.uint8, 64) == 7).all()


def A_rowptr(gbo, L, bs, d_rp, d_ci, n, ncols, d_brp):
    nb = ctypes.c_int64()
    gbo._check(L.gbo_csr2bsr_nnzb_dev(bs, d_rp.ptr, d_ci.ptr, n, ncols, d_brp.ptr, ctypes.byref(nb), None))
    return d_brp.to_numpy(np.int32, (n + bs - 1) // bs + 1)
