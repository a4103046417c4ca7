"""Standalone products in 32 x 32 tiles whose operands stay whole in LDS
(csrc/tbh_gemm.hip) against the oracle, bit for bit: extents at and around a
tile and a quad, K at and around each size of the kernel and the split among
its waves, aligned and odd columns, and the lines to the 64 x 64 tiles (K 513,
more tiles than the chip holds at once)."""
import numpy as np
import pytest

from conftest import rand_tropical

pytestmark = pytest.mark.gpu

SHAPES = [(4, 1, 4, 1), (5, 2, 7, 3), (31, 33, 15, 1), (32, 32, 16, 2), (33, 31, 17, 1),
          (36, 40, 63, 1), (64, 32, 64, 3), (61, 35, 65, 1), (96, 64, 128, 2), (97, 63, 127, 1),
          (40, 36, 129, 1), (128, 96, 256, 1), (127, 65, 255, 2), (64, 64, 260, 1),
          (33, 100, 257, 1), (512, 512, 512, 1), (511, 509, 511, 1), (516, 512, 512, 1),
          (32, 64, 513, 1), (68, 4, 500, 9), (1024, 512, 256, 1), (1028, 512, 256, 1),
          (896, 928, 64, 1), (32, 32, 8, 819), (32, 32, 8, 820)]


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("shape", SHAPES)
def test_matches_oracle(backend, orc, dtype, shape):
    M, N, K, nb = shape
    rng = np.random.default_rng(M + 7 * N + 31 * K + nb)
    A = rand_tropical(rng, (M, K, nb), dtype, lo=-1000)
    B = rand_tropical(rng, (K, N, nb), dtype, lo=-1000, neg_frac=0.3)
    A[:, :, 0][M // 2] = -np.inf if dtype == np.float32 else -(1 << 30)  # a zero row
    assert np.array_equal(backend.maxplus_gemm(A, B), orc.maxplus_gemm(A, B))


@pytest.mark.parametrize("shape", [(40, 36, 64, 2), (36, 33, 300, 2)])
def test_infinite_entries(backend, orc, shape):
    """+inf and -inf entries: a sum of both is dropped, as everywhere."""
    M, N, K, nb = shape
    rng = np.random.default_rng(K)
    A = rng.integers(-9, 10, (M, K, nb)).astype(np.float32)
    B = rng.integers(-9, 10, (K, N, nb)).astype(np.float32)
    A[3, 5, 0] = np.inf
    A[:, 7, 1] = -np.inf
    assert np.array_equal(backend.maxplus_gemm(A, B), orc.maxplus_gemm(A, B))
