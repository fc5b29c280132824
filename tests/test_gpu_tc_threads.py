"""Triangle counts of small and large graphs at once, each thread on a stream of
its own: what a call asks of a kernel (its LDS) is not another's to lower."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def operands(gbo, g, bs):
    L = g.tril()
    return gbo.BsrMatrix.from_csr(L, bs, plan=False), gbo.BsrMatrix.from_csr(L.transpose(), bs, 1, plan=False)


@pytest.mark.parametrize("bs,dense", [(8, False), (32, False), (8, True), (64, True)])
def test_small_and_large(gbo, bs, dense):
    if dense:  # word form: 0.8 of a small graph's entries; blocks of a larger one's diagonal
        small = gbo.gen_er(300, 0.8, 1)
        m, k = 512, 64
        i, j = np.triu_indices(k, 1)
        u = (np.arange(m)[:, None] * k + i).ravel()
        v = (np.arange(m)[:, None] * k + j).ravel()
        n = 64 * bs * m * 4 if bs == 8 else m * k * 8
        key = np.unique(np.concatenate([u * n + v, v * n + u]))
        rp = np.concatenate([[0], np.cumsum(np.bincount(key // n, minlength=n))])
        large = gbo.Csr(n, n, rp, key % n)
    else:
        small, large = gbo.gen_er_m(900, 60_000, 2), gbo.gen_rmat(20, 4, seed=2)
    mats = [operands(gbo, g, bs) for g in (small, large)]
    want = [gbo.bsrbmm_tc(*m) for m in mats]
    assert min(want) > 0
    bad = []

    def work(k):
        L, st = gbo.lib(), ctypes.c_void_p()
        gbo._check(L.gbo_stream_create(ctypes.byref(st)))
        cnt = gbo.DeviceBuffer(8)
        A, B = mats[k]
        for _ in range(60):
            rc = L.gbo_bsrbmm_tc(A.ref, B.ref, cnt.ptr, st)
            if rc or int(cnt.to_numpy(np.uint64)[0]) != want[k]:
                bad.append((k, rc, L.gbo_last_error()))
                break
        gbo._check(L.gbo_stream_destroy(st))

    th = [threading.Thread(target=work, args=(k % 2,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for m in mats:
        for A in m:
            A.free()
