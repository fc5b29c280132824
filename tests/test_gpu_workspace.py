"""Scratch kept between calls: calls from several threads and streams at once
get the results they get alone, and the memory goes back with the last
matrix."""
import ctypes
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_threads_and_streams(gbo, po):
    L = gbo.lib()
    graphs = [gbo.gen_rmat(12, 8, seed=s) for s in range(4)]
    mats = [gbo.BsrMatrix.from_csr(g, bs) for g, bs in zip(graphs, (8, 16, 32, 64))]
    gbo.synchronize()
    bad = []

    def work(k):
        g, A = graphs[k], mats[k]
        want = po.bfs(g.nrows, g.rowptr, g.colind, 1), po.cc(g.nrows, g.rowptr, g.colind)
        st = ctypes.c_void_p()
        gbo._check(L.gbo_stream_create(ctypes.byref(st)))
        out = gbo.DeviceBuffer(4 * g.nrows)
        n = ctypes.c_int32()
        for _ in range(20):
            gbo._check(L.gbo_bfs_do(A.ref, A.ref, 1, out.ptr, None, 0, ctypes.byref(n), st))
            if not np.array_equal(out.to_numpy(np.int32, g.nrows), want[0]):
                bad.append((k, "bfs"))
            gbo._check(L.gbo_cc(A.ref, out.ptr, ctypes.byref(n), st))
            if not np.array_equal(out.to_numpy(np.int32, g.nrows), want[1]):
                bad.append((k, "cc"))
        gbo._check(L.gbo_stream_destroy(st))

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad
    for A in mats:
        A.free()


def test_memory_goes_back(gbo):
    import gc

    gc.collect()
    hip = ctypes.CDLL(gbo.hip_runtimes()[0])
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        gbo.synchronize()
        assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    def step():
        g = gbo.gen_rmat(16, 16, seed=2)
        A = gbo.BsrMatrix.from_csr(g, 16)
        S = np.zeros((g.nrows, 64), np.float32)
        S[:, :] = 1.0 / g.nrows
        gbo.ppr_forward(A, g.outdeg(), S, 0.85, 1e-3, 10)
        held = free_bytes()
        A.free()
        return held

    step()  # the runtime's own first allocations
    gc.collect()
    before = free_bytes()
    held = step()
    gc.collect()
    # 16 MB of iterates and more are kept while a matrix lives, nothing once the last is freed
    assert before - held > (16 << 20)
    assert abs(free_bytes() - before) <= (4 << 20)
