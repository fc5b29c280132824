"""Packing of block rows around and above the number of nonzeros from which
they are not merged: byte for byte the oracle's, on aligned and unaligned tile
buffers, and the refusals of the device path."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
BS = (8, 16, 32, 64)


def _csr(bs, above):
    """Block rows of above - 1, above and above + 1 nonzeros, none, one long row
    beside short ones, a dense band, and a last block row that is not whole;
    more block columns than one bitmap has, the last one not whole."""
    rng = np.random.default_rng(bs)
    ncols = (1 << 18) * bs + 3 * bs + 5
    counts = []
    for total in (above - 1, above, above + 1):
        counts.append(np.bincount(rng.integers(0, bs, total), minlength=bs))
    counts.append(np.zeros(bs, np.int64))
    counts.append(np.r_[40000, rng.integers(0, 30, bs - 1)])
    counts.append(np.full(bs, 2100))
    counts.append(np.full(bs - 3, above // 2))
    counts = np.concatenate(counts)
    rows = []
    for r, k in enumerate(counts):
        if k == 2100:  # neighbours, from another start in each row
            rows.append(np.arange(k) + ncols // 2 + 7 * (r % bs))
        else:
            rows.append(np.sort(rng.integers(0, ncols - k, k)) + np.arange(k))
    rows[0][-1] = ncols - 1
    rp = np.r_[0, np.cumsum(counts)].astype(np.int32)
    return len(counts), ncols, rp, np.concatenate(rows).astype(np.int32)


@pytest.mark.parametrize("direction", (0, 1))
@pytest.mark.parametrize("bs", BS)
def test_pack_around_the_bound(gbo, po, bs, direction):
    n, ncols, rp, ci = _csr(bs, max(128, 8 * bs))
    want = po.pack(bs, n, rp, ci, direction)
    d_rp, d_ci = gbo.DeviceBuffer.from_numpy(rp), gbo.DeviceBuffer.from_numpy(ci)
    A = gbo.BsrMatrix.from_device_csr(d_rp, d_ci, n, ncols, bs, direction)
    for got, exp in zip(A.host_arrays(), want):
        assert np.array_equal(got, exp)
    # tiles one word off any wider alignment
    nb, word = len(want[1]), bs // 8
    buf = gbo.DeviceBuffer.from_numpy(np.full((nb * bs + 2) * word, 0xA5, np.uint8))
    d_brp, d_bci = gbo.DeviceBuffer.from_numpy(want[0]), gbo.DeviceBuffer(4 * nb)
    gbo._check(gbo.lib().gbo_csr2bsr_fill_dev(bs, direction, d_rp.ptr, d_ci.ptr, n, ncols, d_brp.ptr, d_bci.ptr,
                                              buf.ptr + word, None))
    raw = buf.to_numpy(np.uint8, (nb * bs + 2) * word)
    assert np.array_equal(raw[word:-word].view(gbo.WORD_DTYPE[bs]), want[2])
    assert (raw[:word] == 0xA5).all() and (raw[-word:] == 0xA5).all()
    assert np.array_equal(d_bci.to_numpy(np.int32, nb), want[1])


@pytest.mark.parametrize("bs", BS)
def test_refusals_in_heavy_block_rows(gbo, bs):
    """A column out of range on either side, and a descent inside a row (also
    the row after empty ones); a descent from one row to the next is none."""
    n, ncols, rp, ci = _csr(bs, max(128, 8 * bs))
    hub = rp[4 * bs]
    d_rp = gbo.DeviceBuffer.from_numpy(rp)
    L, nb, d_brp = gbo.lib(), ctypes.c_int64(), gbo.DeviceBuffer(4 * (n // bs + 2))

    def refused(at, value, what):
        bad = ci.copy()
        bad[at] = value
        d_ci = gbo.DeviceBuffer.from_numpy(bad)
        rc = L.gbo_csr2bsr_nnzb_dev(bs, d_rp.ptr, d_ci.ptr, n, ncols, d_brp.ptr, ctypes.byref(nb), None)
        assert rc == -1 and what in L.gbo_last_error(), (at, value)

    for at in (hub, hub + 39999, rp[2 * bs]):
        refused(at, ncols, b"range")
        refused(at, -1, b"range")
    refused(hub, ncols - 1, b"sorted")            # the first of a row, after an empty block row
    refused(hub + 39999, 0, b"sorted")            # the last of a row
    refused(hub + 20000, 0, b"sorted")
    refused(rp[5 * bs + 1] + 2000, 0, b"sorted")  # the dense band
