"""Masked products sum(A * (A B)) counted by pairs of tiles: mask tiles of few
bits, of about as many as are listed, and full; block rows of one tile up to
some hundreds; a B that is not A's transpose; tiles at any address; against
scipy's integer products."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def csr(gbo, m):
    m = m.tocsr()
    m.sort_indices()
    return gbo.Csr(m.shape[0], m.shape[1], m.indptr.astype(np.int32), m.indices.astype(np.int32))


def by_tiles(sp, rng, bs, rows, nblocks, bits):
    """nblocks x nblocks tiles; block row I has rows[I] of them, each of a number
    of bits drawn from `bits`; the last block row and column are not whole."""
    n = nblocks * bs - 3
    r, c = [], []
    for i, k in enumerate(rows):
        for j in rng.choice(nblocks, k, replace=False):
            at = rng.choice(bs * bs, rng.choice(bits), replace=False)
            r.append(i * bs + at // bs)
            c.append(j * bs + at % bs)
    r, c = np.concatenate(r), np.concatenate(c)
    ok = (r < n) & (c < n)
    m = sp.coo_matrix((np.ones(ok.sum(), np.int64), (r[ok], c[ok])), (n, n)).tocsr()
    m.data[:] = 1
    return m


BITS = {8: (6, 20, 64), 16: (8, 60, 256), 32: (20, 319, 320, 321, 1024), 64: (5, 767, 768, 769, 4096)}


@pytest.mark.parametrize("bs,nblocks", [(8, 140), (16, 135), (32, 132), (64, 67)])
def test_tiles(gbo, bs, nblocks):
    sp = pytest.importorskip("scipy.sparse")
    rng = np.random.default_rng(bs)
    rows = [0, 1, 2, 63, 64, 65, min(129, nblocks), nblocks] + [int(rng.integers(0, 8)) for _ in range(nblocks - 8)]
    A = by_tiles(sp, rng, bs, rows, nblocks, BITS[bs])
    dense = by_tiles(sp, rng, bs, [20] * nblocks, nblocks, (bs * bs // 4,))
    for B in (A.T.tocsr(), A, dense):
        for M, N in ((A, B), (dense, B)):
            Ar, Bc = gbo.BsrMatrix.from_csr(csr(gbo, M), bs, 0), gbo.BsrMatrix.from_csr(csr(gbo, N), bs, 1)
            want = int(M.multiply(M @ N).sum())
            assert gbo.bsrbmm_tc(Ar, Bc) == want
            # the same tiles one word off any wider alignment
            word = bs // 8
            refs, keep = [], []
            for X in (Ar, Bc):
                _, _, tiles = X.host_arrays()
                buf = gbo.DeviceBuffer.from_numpy(np.concatenate([np.zeros(word, np.uint8), tiles.view(np.uint8)]))
                s = gbo.BsrStruct.from_buffer_copy(X.s)
                s.tiles, s.plan, s.plan_chunk, s.plan_nchunks = buf.ptr + word, None, 0, 0
                keep.append(buf)
                refs.append(s)
            cnt = gbo.DeviceBuffer(8)
            gbo._check(gbo.lib().gbo_bsrbmm_tc(ctypes.byref(refs[0]), ctypes.byref(refs[1]), cnt.ptr, None))
            assert int(cnt.to_numpy(np.uint64)[0]) == want
            Ar.free()
            Bc.free()


@pytest.mark.parametrize("bs", (8, 16, 32, 64))
def test_communities(gbo, bs):
    """Dense blocks along the diagonal of 2^18 vertices: by hand, k choose 3 each."""
    n, k = 1 << 18, 96
    m = n // k
    i, j = np.triu_indices(k, 1)
    off = np.arange(m)[:, None] * k
    u, v = (off + i).ravel(), (off + j).ravel()
    key = np.sort(np.concatenate([u * n + v, v * n + u]))
    rp = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))])
    assert gbo.tc(gbo.Csr(n, n, rp, key % n), bs) == m * k * (k - 1) * (k - 2) // 6
