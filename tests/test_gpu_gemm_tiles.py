"""Products that stay in K1's tiles (csrc/tbh_kernels.hip: aligned, at least
512 tiles, K up to 256) against the oracle, bit for bit: tiles whole (no
bounds to check) and cut in M, N or K, tile counts that are powers of two and
not, each of the three tile shapes, batches."""
import numpy as np
import pytest

from conftest import rand_tropical

pytestmark = pytest.mark.gpu

SHAPES = [(4096, 2048, 32, 1), (2944, 2948, 16, 1), (2944, 2944, 20, 1), (768, 764, 48, 15),
          (131072, 64, 32, 1), (131076, 64, 16, 1), (16384, 60, 20, 9), (131072, 32, 16, 1),
          (65540, 28, 36, 2)]


@pytest.mark.parametrize("dtype", [np.float32, np.int32])
@pytest.mark.parametrize("shape", SHAPES)
def test_matches_oracle(backend, orc, dtype, shape):
    M, N, K, nb = shape
    rng = np.random.default_rng(M + 7 * N + 31 * K)
    A = rand_tropical(rng, (M, K, nb), dtype, lo=-1000)
    B = rand_tropical(rng, (K, N, nb), dtype, lo=-1000, neg_frac=0.3)
    assert np.array_equal(backend.maxplus_gemm(A, B), orc.maxplus_gemm(A, B))
