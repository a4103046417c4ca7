"""Standalone products at the ends of the documented extents, whose operands
are made on the device; results in closed form."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _Device:
    """Device memory through the HIP runtime that the library is linked to."""

    def __init__(self, lib):
        self.lib, self.held = lib, []

    def call(self, name, *args):
        rc = getattr(self.lib, name)(*args)
        assert rc == 0, (name, rc)

    def free_bytes(self):
        free, total = C.c_size_t(), C.c_size_t()
        self.call("hipMemGetInfo", C.byref(free), C.byref(total))
        return free.value

    def zeros(self, entries):
        p = C.c_void_p()
        self.call("hipMalloc", C.byref(p), C.c_size_t(4 * entries))
        self.held.append(p)
        self.call("hipMemset", p, 0, C.c_size_t(4 * entries))
        return p.value

    def put(self, at, value):
        self.call("hipMemcpy", C.c_void_p(at), C.byref(C.c_float(value)), C.c_size_t(4), 1)

    def get(self, at, n):
        out = np.empty(n, np.float32)
        self.call("hipMemcpy", C.c_void_p(out.ctypes.data), C.c_void_p(at), C.c_size_t(4 * n), 2)
        return out

    def close(self):
        self.call("hipDeviceSynchronize")
        for p in self.held:
            self.call("hipFree", p)


def test_k_up_to_2_31(backend):
    """K = 2^31 - 1: the last K range reaches past 2^31 when rounded up.  The
    maximum sits at the first, a middle and the last entries of that range."""
    from tensorbranching_jl_amd import _lib
    M, K = 4, (1 << 31) - 1
    dev = _Device(_lib.tbh())
    if dev.free_bytes() < 4 * K * (M + 1) + (1 << 30):
        pytest.skip("needs 43 GB of device memory")
    try:
        A, B, out = dev.zeros(K * M), dev.zeros(K), dev.zeros(M)
        dev.put(A + 4 * (M * (K - 1) + 2), 3)
        for k, extra in ((K - (1 << 22) + 1, 0), (K - 12345, 0), (K - 1, 3)):
            dev.put(B + 4 * k, 5)
            dev.call("hipDeviceSynchronize")
            _lib.check(_lib.tbh().tbh_maxplus_gemm(backend.handle, 0, M, 1, K, 1, A, M, 0, B, K,
                                                   0, out, M, 0, _lib.TBH_DEVICE))
            want = np.full(M, 5, np.float32)
            want[2] += extra
            assert np.array_equal(dev.get(out, M), want), k
            dev.put(B + 4 * k, 0)
    finally:
        dev.close()


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
def test_2_24_products(backend, dtype):
    """A batch of 2^24 products of 4 x 1 x 5 (one A, overlapping windows as
    B): more workgroups of a tile each than one launch holds."""
    from tensorbranching_jl_amd import _lib
    M, K, batch = 4, 5, 1 << 24
    rng = np.random.default_rng(24)
    A = np.asfortranarray(rng.integers(-99, 100, (M, K)).astype(dtype))
    B = rng.integers(-999, 1000, batch + K - 1).astype(dtype)
    out = np.empty((batch, M), dtype)
    _lib.check(_lib.tbh().tbh_maxplus_gemm(
        backend.handle, 0 if dtype == np.float32 else 1, M, 1, K, batch, A.ctypes.data, M, 0,
        B.ctypes.data, K, 1, out.ctypes.data, M, M, _lib.TBH_HOST))
    for m in range(M):
        want = np.max([A[m, k] + B[k:k + batch] for k in range(K)], axis=0)
        assert np.array_equal(out[:, m], want), m
