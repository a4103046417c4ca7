// Host-side check of the standalone GEMM's dispatch (csrc/tbh_gemm_rule.hpp),
// built by tests/test_gemm_rule.py with UndefinedBehaviorSanitizer (g++, host
// code only): over extents up to 2^31 - 1 the K ranges of a split product
// follow one another from 0 to K, all but the last a multiple of a slab, and
// so does the one range of a product without a workspace; no launch passes
// 2^32 - 1 work-items.
#include <cstdio>

#include "tbh_gemm_rule.hpp"

using namespace tbh;

static int bad(const char* what, int64_t M, int64_t N, int64_t K, int64_t batch) {
  std::fprintf(stderr, "%s: M %ld N %ld K %ld batch %ld\n", what, (long)M, (long)N, (long)K,
               (long)batch);
  return 1;
}

static bool covers(const GemmSplit& g) {
  int64_t at = 0;
  for (int p = 0; p < g.ksplit; p++) {
    const int64_t kb = (int64_t)p * g.kpart;
    if (kb != at || kb >= g.K || kb % 32) return false;
    at = gemm_range_end(g, (int32_t)kb);
    if (at <= kb) return false;
  }
  return at == g.K;
}

int main() {
  const int64_t max = INT32_MAX;
  const int64_t ext[] = {4,    5,    63,   64,   65,    100,           513,           1021,
                         4096, 1500, 9999, 1024, 65536, (1ll << 20) + 1};
  const int64_t ks[] = {4,
                        31,
                        32,
                        33,
                        127,
                        128,
                        129,
                        255,
                        257,
                        383,
                        384,
                        777,
                        1030,
                        4099,
                        65537,
                        (1 << 24) + 1,
                        (1ll << 30) - 1,
                        1ll << 30,
                        (1ll << 30) + 64,
                        3ll << 29,
                        max - (1 << 22) - 1,
                        max - 63,
                        max - 32,
                        max - 31,
                        max - 30,
                        max - 1,
                        max};
  const int64_t batches[] = {1,   2,    3,         7,             129,
                             257, 512,  1000,      (1 << 24) - 1, 1 << 24,
                             1 << 25, 1 << 28, (1 << 28) + 1, max};
  long n = 0;
  for (int64_t M : ext)
    for (int64_t N : {(int64_t)1, (int64_t)3, (int64_t)64, (int64_t)515, (int64_t)4096})
      for (int64_t K : ks)
        for (int64_t batch : batches) {
          GemmSplit g{};
          if (!split_gemm(M, N, K, batch, false, ((M + 127) / 128) * ((N + 127) / 128) * batch,
                          256, &g))
            continue;
          n++;
          if (g.M != M || g.N != N || g.K != K || g.batch != batch)
            return bad("extents", M, N, K, batch);
          if (!covers(g)) return bad("K ranges", M, N, K, batch);
          const int64_t blocks = (int64_t)g.tiles_m * g.tiles_n * g.ksplit * g.batch;
          const int64_t quads = (M + 3) / 4 * N * batch;
          if (blocks * 256 >= 1ll << 32 ||
              (g.ksplit > 1 && (quads + 255) / 256 * 256 >= 1ll << 32))
            return bad("launch", M, N, K, batch);
          whole_k(&g);
          if (g.ksplit != 1 || !covers(g)) return bad("one range", M, N, K, batch);
        }
  std::printf("checked %ld products\n", n);
  return 0;
}
