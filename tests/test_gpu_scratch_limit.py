"""The blocks that the library keeps between calls are there for its own
allocations when the device has no other memory left."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
N = 160_000_000  # rows: scratch, arrays or vectors of 640 MB


def fill_pool(gbo, A, g):
    S = np.full((g.nrows, 64), 1.0 / g.nrows, np.float32)
    gbo.ppr_forward(A, g.outdeg(), S, 0.85, 1e-1, 2)


@pytest.fixture(scope="module")
def hog(gbo):
    """(take, give): take all of the device's memory but some 400 MB, with blocks of
    more than 500 MB kept by the library."""
    gbo.lib()
    hip = ctypes.CDLL(gbo.hip_runtimes()[0])
    g = gbo.gen_er_m(1 << 20, 1 << 21, 1)
    A = gbo.BsrMatrix.from_csr(g, 8)
    held = []

    def free():
        gbo.synchronize()
        f, t = ctypes.c_size_t(), ctypes.c_size_t()
        assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
        return f.value

    def grab(size):
        p = ctypes.c_void_p()
        rc = hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size))
        if rc:
            assert rc == 2  # hipErrorOutOfMemory
            hip.hipGetLastError()
            return False
        held.append(p)
        return True

    def take():
        fill_pool(gbo, A, g)
        assert grab(free() - (1 << 30))
        for _ in range(512):  # there is more than the runtime calls free
            if not grab(128 << 20):
                break
        else:
            pytest.skip("no end of device memory")
        for _ in range(3):
            assert hip.hipFree(held.pop()) == 0

    def give():
        while held:
            assert hip.hipFree(held.pop()) == 0

    yield take, give
    give()
    A.free()


def empty(gbo, n, bs, plan=False):
    """n x n with one nonzero, in the last row and column."""
    rp = np.zeros(n + 1, np.int32)
    rp[n] = 1
    return gbo.Csr(n, n, rp, np.array([n - 1], np.int32))


def test_products_without_a_plan(gbo, hog):
    take, give = hog
    A = gbo.BsrMatrix.from_csr(empty(gbo, N, 8), 8, plan=False)
    x, y = gbo.DeviceBuffer.zeros(N // 8 + 8), gbo.DeviceBuffer(4 * N)
    gbo._check(gbo.lib().gbo_memset(x.ptr, 0xFF, N // 8))
    take()
    rc = gbo.lib().gbo_bsrbmv_count(A.ref, x.ptr, y.ptr, 0, None)
    gbo.synchronize()
    give()
    gbo._check(rc)
    assert y.view(4 * (N - 2), 8).to_numpy(np.int32).tolist() == [0, 1]
    A.free()


def test_product_sum(gbo, hog):
    take, give = hog
    n = 40_000_000  # 16 bytes a column
    g = empty(gbo, n, 8)
    A, B = gbo.BsrMatrix.from_csr(g, 8, plan=False), gbo.BsrMatrix.from_csr(g, 8, 1, plan=False)
    d = gbo.DeviceBuffer(8)
    take()
    rc = gbo.lib().gbo_bsrbmm_sum(A.ref, B.ref, d.ptr, None)
    gbo.synchronize()
    give()
    gbo._check(rc)
    assert int(d.to_numpy(np.uint64)[0]) == 1
    A.free()
    B.free()


def test_host_csr(gbo, hog):
    take, give = hog
    g = empty(gbo, N, 64)
    nb = ctypes.c_int64()
    take()
    rc = gbo.lib().gbo_csr2bsr_nnzb(64, g.rowptr.ctypes.data, g.colind.ctypes.data, N, N, ctypes.byref(nb))
    give()
    gbo._check(rc)
    assert nb.value == 1


def test_own_plan_without_room(gbo):
    """The library's own plan where its allocation fits and the prefix sums it is
    cut by do not."""
    gbo.lib()
    hip = ctypes.CDLL(gbo.hip_runtimes()[0])
    n, deg, bs = 1 << 21, 12, 8
    g = gbo.gen_er_m(n, n * deg // 2, 1)
    A = gbo.BsrMatrix.from_csr(g, bs, plan=False)
    assert 20 << 20 < A.nblocks < 32 << 20
    # in MB: row counts 4 n, per chunk of 256 plan, start, tail, partials; prefix sums 20 bytes per 16 tiles
    plan = (4 * n + A.nblocks // 256 * (16 + 128)) >> 20
    cut = A.nblocks // 16 * 20 >> 20
    assert cut > 20
    held, leave = [], plan + cut // 2

    def grab(size):
        p = ctypes.c_void_p()
        if hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(size)):
            hip.hipGetLastError()
            return False
        held.append((p, size))
        return True

    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    gbo._check(gbo.lib().gbo_bsr_plan(A.ref, 256, None))  # whatever a first plan sets up
    gbo.lib().gbo_bsr_plan_free(A.ref)
    gbo.synchronize()
    assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    assert grab(f.value - (1 << 30))
    for size in (128 << 20, 2 << 20):
        for _ in range(600):
            if not grab(size):
                break
        else:
            pytest.skip("no end of device memory")
    # the kept blocks go with a failed allocation, and that is what there is then
    given = 0
    while held and given < leave << 20:
        p, size = held.pop()
        assert hip.hipFree(p) == 0
        given += size
    rc = gbo.lib().gbo_bsr_plan(A.ref, 0, None)
    gbo.synchronize()
    while held:
        assert hip.hipFree(held.pop()[0]) == 0
    gbo._check(rc)
    x = gbo.pack_vec(bs, (np.arange(n) % 3 == 0).astype(np.float32))
    y = gbo.bsrbmv_count(A, x)
    want = np.bincount(np.repeat(np.arange(n), np.diff(g.rowptr))[g.colind % 3 == 0], minlength=n)
    assert np.array_equal(y, want)
    A.free()
