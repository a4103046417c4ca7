"""Standalone products at the lines between the 128 x 128 (256 x 32) kernel and
the 64 x 64 one, on either side of each, against the oracle bit for bit."""
import numpy as np
import pytest

from conftest import rand_tropical

pytestmark = pytest.mark.gpu

SHAPES = [(256 * 224, 8, 64, 1), (256 * 223, 5, 64, 1), (256 * 192, 32, 16, 1),
          (256 * 191 - 4, 3, 16, 1), (256 * 160, 7, 20, 1), (256 * 159, 9, 20, 1),
          (300, 5, 64, 256), (2048, 4096, 260, 1), (256 * 487, 40, 260, 1),
          (71, 68, 15, 601), (71, 68, 16, 1500), (72, 68, 17, 601), (129, 65, 5, 400)]


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("shape", SHAPES)
def test_matches_oracle(backend, orc, dtype, shape):
    M, N, K, nb = shape
    rng = np.random.default_rng(M + 7 * N + 31 * K)
    A = rand_tropical(rng, (M, K, nb), dtype, lo=-1000)
    B = rand_tropical(rng, (K, N, nb), dtype, lo=-1000, neg_frac=0.3)
    A[:, :, 0][M // 2] = -np.inf if dtype == np.float32 else -(1 << 30)  # a zero row
    assert np.array_equal(backend.maxplus_gemm(A, B), orc.maxplus_gemm(A, B))
