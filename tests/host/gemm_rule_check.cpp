// Host-side check of the standalone GEMM's dispatch (csrc/tbh_gemm_rule.hpp),
// built by tests/test_gemm_rule.py with UndefinedBehaviorSanitizer (g++, host
// code only): over extents up to 2^31 - 1 the K ranges of a split product
// follow one another from 0 to K, all but the last a multiple of a slab, and
// so does the one range of a product without a workspace; no launch passes
// 2^32 - 1 work-items.  And at the lines between the two kernels, each product
// runs on the one that measured faster.
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

struct Line {
  int dtype;  // 0 Float32, 1 Int32
  int64_t M, N, K, batch;
  bool k1;
};
// (extents in multiples of 4 are aligned products)
static const Line kLines[] = {
    // narrow outputs in 256 x 32 tiles: 224 of them Float32, 192 at K <= 16,
    // 160 Int32
    {0, 256 * 224, 8, 64, 1, true}, {0, 256 * 223, 8, 64, 1, false},
    {0, 256 * 192, 8, 16, 1, true}, {0, 256 * 191, 8, 16, 1, false},
    {1, 256 * 160, 8, 64, 1, true}, {1, 256 * 159, 8, 64, 1, false},
    {0, 102400, 20, 1024, 1, true}, {1, 102400, 20, 1024, 1, true},
    {0, 768, 5, 452, 160, true},    {1, 600, 5, 64, 100, false},
    {1, 324, 3, 260, 1256, true},
    // K > 256: K1's tiles spread evenly, or not
    {0, 4096, 4096, 260, 1, true},  {1, 4096, 4096, 260, 1, true},
    {0, 2048, 4096, 512, 1, true},  {1, 2048, 4096, 512, 1, false},
    {0, 8192, 8192, 1024, 1, true}, {0, 3072, 3072, 1024, 1, false},
    {0, 6144, 6144, 4096, 1, true}, {0, 4096, 4096, 4096, 1, false},
    {0, 8, 12, 712, 1024, false},
    // unaligned, short K
    {0, 71, 68, 15, 1493, true},    {1, 200001, 65, 5, 1, true},
    {0, 85, 477, 6, 3097, true},    {0, 191, 4039, 5, 16, false},
    {0, 200001, 65, 17, 1, false},  {0, 50, 3133, 7, 586, false},
};

int main() {
  for (const Line& l : kLines) {
    const bool vec = l.M % 4 == 0 && l.K % 4 == 0;
    const int shape = vec ? gemm_shape(l.M, l.N) : 0;
    const int64_t tm = (l.M + gemm_bm(shape) - 1) / gemm_bm(shape),
                  tn = (l.N + gemm_bn(shape) - 1) / gemm_bn(shape);
    GemmSplit g{};
    if (split_gemm(l.dtype, l.M, l.N, l.K, l.batch, vec, tm * tn * l.batch, 256, &g) == l.k1)
      return bad("line", l.M, l.N, l.K, l.batch);
  }
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
          if (!split_gemm(0, M, N, K, batch, false, ((M + 127) / 128) * ((N + 127) / 128) * batch,
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
