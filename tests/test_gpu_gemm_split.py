"""The standalone GEMM's 64 x 64 tile kernel (csrc/tbh_gemm.hip) against the
oracle, bit for bit: extents at and around a tile, a K slab and a quad, K
ranges of their own workgroups, odd leading dimensions and strides on
operands whose columns are only 4-byte aligned, and the line to the 128 x 128 tiles."""
import numpy as np
import pytest

from conftest import rand_tropical

pytestmark = pytest.mark.gpu

SHAPES = [(4, 1, 4, 1), (5, 3, 7, 2), (7, 65, 31, 1), (63, 64, 32, 1), (64, 63, 33, 1),
          (65, 67, 36, 3), (66, 1, 127, 1), (67, 64, 128, 2), (64, 64, 256, 1),
          (130, 70, 257, 1), (61, 129, 1030, 2), (64, 64, 4099, 1), (9, 5, 2050, 5),
          (1021, 515, 77, 2), (512, 512, 300, 1), (2050, 1030, 40, 1),
          # K1 and its neighbours: 512 tiles of 128 x 128, K 256 and 260
          (128, 128, 16, 512), (4096, 2048, 256, 1), (4096, 2048, 260, 1),
          # below a quad
          (3, 200, 50, 2), (200, 90, 3, 1), (300, 20, 2, 1)]


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("shape", SHAPES)
def test_matches_oracle(backend, orc, dtype, shape):
    M, N, K, nb = shape
    rng = np.random.default_rng(M + 7 * N + 31 * K)
    A = rand_tropical(rng, (M, K, nb), dtype, lo=-1000)
    B = rand_tropical(rng, (K, N, nb), dtype, lo=-1000, neg_frac=0.3)
    A[:, :, 0][M // 2] = -np.inf if dtype == np.float32 else -(1 << 30)  # a zero row
    assert np.array_equal(backend.maxplus_gemm(A, B), orc.maxplus_gemm(A, B))


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("shape", [(1500, 1000, 384, 1), (1500, 1000, 383, 1),
                                   (1021, 515, 777, 3), (1600, 1500, 390, 1)])
def test_uneven_tile_counts(backend, orc, dtype, shape):
    """More tiles than CUs, split over K where they would not spread evenly
    over the CUs: at the shortest range, just below it, four ranges, 600
    tiles."""
    M, N, K, nb = shape
    rng = np.random.default_rng(M + K)
    A = rand_tropical(rng, (M, K, nb), dtype, lo=-1000)
    B = rand_tropical(rng, (K, N, nb), dtype, lo=-1000, neg_frac=0.3)
    assert np.array_equal(backend.maxplus_gemm(A, B), orc.maxplus_gemm(A, B))


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("shape", [(66, 70, 45, 3), (37, 20, 1029, 2), (64, 64, 64, 1)])
def test_odd_strides(backend, orc, dtype, shape):
    """Leading dimensions and batch strides past the matrices, so that most
    columns are only 4-byte aligned; every entry of C outside the M x N blocks
    stays."""
    from tensorbranching_jl_amd import _lib
    M, N, K, nb = shape
    lda, ldb, ldc = M + 1, K + 3, M + 2
    sA, sB, sC = lda * K + 1, ldb * N + 2, ldc * N + 3
    rng = np.random.default_rng(M + N + K)
    A = rand_tropical(rng, (M, K, nb), dtype)
    B = rand_tropical(rng, (K, N, nb), dtype)

    def flat(X, ld, stride):
        buf = np.full(stride * nb, 77, dtype)
        for t in range(nb):
            for c in range(X.shape[1]):
                o = t * stride + c * ld
                buf[o:o + X.shape[0]] = X[:, c, t]
        return buf

    a, b = flat(A, lda, sA), flat(B, ldb, sB)
    c = flat(np.full((M, N, nb), 5, dtype), ldc, sC)
    code = 0 if dtype == np.float32 else 1
    _lib.check(_lib.tbh().tbh_maxplus_gemm(backend.handle, code, M, N, K, nb, a.ctypes.data, lda,
                                           sA, b.ctypes.data, ldb, sB, c.ctypes.data, ldc, sC,
                                           _lib.TBH_HOST))
    assert np.array_equal(c, flat(orc.maxplus_gemm(A, B), ldc, sC))
