// tbh_gemm_rule.hpp -- which kernel a standalone max-plus GEMM runs on (host
// code without HIP calls, so that the lines are tested without a GPU).
#pragma once
#include <algorithm>
#include <cstdint>

#include "tbh_internal.hpp"

namespace tbh {

// Workgroups of 256 in one launch: it holds at most 2^32 - 1 work-items (more
// wrap without an error).
constexpr int64_t kGemmMaxBlocks = ((int64_t)1 << 24) - 1;

// Whether K1 (128 x 128, 256 x 64 or 256 x 32 tiles; slabs of 16) takes a
// product that K1b could run: `tiles` 64 x 64 tiles, `k1_tiles` of K1's.  us per
// call, K1 / K1b, Float32 and Int32:
// - Aligned, at least 512 of K1's tiles, K <= 256: K1b's pass over the waves'
//   maxima, once per 64 x 64 outputs, costs more than its finer tiles give
//   (4096^2 x 16, kernels alone: 22 / 46; 64: 46 / 62; 256: 136 / 151).
// - Aligned, N <= 32: half of K1b's columns are padding.  K1's line lies at
//   7/8 of a tile (256 x 32) per CU for Float32, 5/8 for Int32, 6/8 at K <= 16.
//   400 tiles, K = 16 21 / 28, 23 / 30; 256, K = 64 28 / 27, 28 / 30; 240, 60
//   of 1000 x 5 x 452 86 / 93, 86 / 116; 200, K = 256 55 / 52, 55 / 68; 180 55 /
//   44, 56 / 57.  Int32 with rows of padding (600 in 768): 300 tiles, K = 64 33
//   / 30, 600 tiles equal.
// - Aligned, K > 256: where K1's tiles spread evenly over the CUs and are
//   whole, from two tiles per CU (Float32) or four (Int32): 4096^2 x 260 169 /
//   181, 234 / 249; 8192^2 x 1024 1833 / 1996, 2766 / 2908; 3840 x 2176 x 512
//   153 / 161, 227 / 223.  576 tiles (a last round of a quarter of the CUs):
//   3072^2 x 1024 402 / 322, 577 / 467.  The lead shrinks with K (4096^2 x 1024
//   3%, x 4096 -1%), but not on five tiles per CU and more (6144^2 x 4096 3%).
// - Unaligned, K <= 16: K1b fills half its slab or less, which its smaller
//   tiles make up for only on few tiles, or where K1's would hold much padding:
//   71 x 68 x 15, batch 1493 47 / 66, 52 / 72; 200001 x 65 x 5 58 / 65, 60 / 70;
//   85 x 477 x 6, batch 3097 311 / 431, 338 / 457; but 191 x 4039 x 5, batch 16
//   (1024 tiles) 53 / 42, 52 / 45; 15 x 3413 x 15, batch 424 210 / 202, 248 /
//   226; and K = 17, two of K1's slabs: 200001 x 65 75 / 65, 82 / 71.
inline bool k1_better(int dtype, int64_t M, int64_t N, int64_t K, int64_t batch, bool vec,
                      int64_t tiles, int64_t k1_tiles, int num_cus) {
  if (!vec)
    return K <= 16 && k1_tiles >= 600 && tiles * 5 >= k1_tiles * 13 &&
           (k1_tiles >= 1500 || M * N * batch * 10 < tiles * 4096 * 9);
  if (k1_tiles >= 512 && K <= 256) return true;
  const bool whole = tiles * 10 >= k1_tiles * 36;  // (of at most 4 per tile of K1's)
  if (gemm_shape(M, N) == 2) {
    const int eighths = dtype == 1 ? (whole ? 5 : 16) : K <= 16 ? 6 : 7;
    return k1_tiles * 8 >= (int64_t)num_cus * eighths;
  }
  const int64_t per_cu = (k1_tiles + num_cus - 1) / num_cus;
  return (K <= 1536 || per_cu >= 5) && k1_tiles > num_cus * (dtype == 1 ? 3 : 1) &&
         k1_tiles * 20 >= per_cu * num_cus * 19 && whole;
}

// Whether a standalone product runs on K1b (64 x 64 tiles), and in how many K
// ranges.  With few of its own tiles K1 leaves CUs idle (3072 x 2048 x 128 38 /
// 36; 2048^2 x 64 22 / 18; 1024^3 224 / 47; 512^3 114 / 19), and unaligned
// extents take K1's scalar loads (three 1021 x 515 x 777 Int32 238 / 92).  K1
// takes what k1_better says, and alone takes M or K below one quad and more
// tiles than K1b has workgroups in a launch (K1 walks its tiles).  Products of
// fewer than 256 tiles are split over K until 512 workgroups run, in ranges of
// at least 128 (64^2 outputs of K = 3428: 800 / 25; 256 or 768 workgroups, or
// ranges of 64, measured within 10% of this).  More tiles than CUs that would
// leave a tenth of the CUs' time idle (384 tiles are 2 on half of the 256 CUs)
// are split into the fewest ranges, up to four, that do not, while K / p >= 192
// (ranges are rounded up to slabs; what is left of K for the last, which starts
// last, may be shorter: K = 777 in four is 224, 224, 224 and 105). Whole /
// split, Float32 and Int32 us per call: 1500 x 1000 x 1000 89 / 75, 122 / 95;
// 1100^2 x 2000 158 / 111, 229 / 149; 1200^2 x 777 74 / 64, 101 / 79; three
// 1021 x 515 x 777 77 / 76, 100 / 94; 1600 x 1500 x 400 (600 tiles) 58 / 58, 76
// / 73. The second launch is made up for from K / p of (Float32 / Int32) 130 /
// 100 at 1100^2 in three ranges, 160 / 150 at 1200^2 and 190 / 150 at 1500 x
// 1000 in two, 150 / 120 at five 1000 x 300 in three, 210 / 165 at 1600 x 1500
// in two, 190 / 145 at three 1021 x 515 in four (97 there loses 12% / 5%): from
// 192 on all gain or are equal. Ranges that differ by at most a slab are equal
// or up to 8% slower: the short last one fills the end of the launch.
inline bool split_gemm(int dtype, int64_t M, int64_t N, int64_t K, int64_t batch, bool vec,
                       int64_t k1_tiles, int num_cus, GemmSplit* g) {
  if (M < 4 || K < 4) return false;
  const int64_t tm = (M + 63) / 64, tn = (N + 63) / 64;
  if (tm * tn > kGemmMaxBlocks || tm * tn * batch > kGemmMaxBlocks) return false;
  const int64_t tiles = tm * tn * batch;
  if (k1_better(dtype, M, N, K, batch, vec, tiles, k1_tiles, num_cus)) return false;
  int64_t parts = std::max<int64_t>(1, std::min<int64_t>(K / 128, 512 / tiles));
  auto even = [&](int64_t p) {
    const int64_t per_cu = (tiles * p + num_cus - 1) / num_cus;
    return tiles * p * 10 >= per_cu * num_cus * 9;
  };
  if (tiles > num_cus && !even(1))
    for (int64_t p = 2; p <= 4 && K / p >= 192; p++)
      if (even(p)) {
        parts = p;
        break;
      }
  g->M = (int32_t)M;
  g->N = (int32_t)N;
  g->K = (int32_t)K;
  g->batch = (int32_t)batch;
  g->tiles_m = (int32_t)tm;
  g->tiles_n = (int32_t)tn;
  const int64_t kpart = ((K + parts - 1) / parts + 31) / 32 * 32;
  g->kpart = (int32_t)std::min(kpart, K);
  g->ksplit = (int32_t)((K + kpart - 1) / kpart);
  return true;
}

// Whether a standalone product runs in 32 x 32 tiles with their operands whole
// in LDS: K up to 512 (132 KB), on at most 3.2 workgroups per CU, fewer as K
// grows past 160 (2 at 256, 1 at 512). A CU holds one workgroup at K > 256, two
// at K > 128 and at least four below, so between those sizes up to two rounds
// run; they are faster than 64 x 64 tiles all the same. Float32 and Int32 us
// per call, 64 x 64 tiles / 32 x 32: 512^2 x 512 (1 per CU) 27.3 / 20.6, past
// the line 640^2 x 512 29.5 / 37.8; 640^2 x 260 (1.6 per CU, one resident) 28.8
// / 24.3, 28.7 / 25.2; batches of 32^2, K = 260, 504 of them 41.6 / 25.1, 50.6
// / 26.2; 300 of K = 384 46.6 / 26.1, 59.1 / 27.4; 800 x 1000 x 160 (3.1 per
// CU, two resident) 26.2 / 23.9, 26.3 / 25.7; 1024 x 512 x 256 27.2 / 20.4,
// past it 768^2 28.0 / 23.3 but Int32 with odd extents no faster; K = 128: 768
// x 1024 23.2 / 19.9, 1024^2 23.3 / 21.3 (Int32 equal); K = 64: 512^2 18.9 /
// 16.2, 1024^2 equal, 1500 x 1000 20.8 / 21.4.
inline bool resident_gemm(int64_t tiles32, int64_t K, int num_cus) {
  return K <= 512 && tiles32 * std::max<int64_t>(K, 160) <= (int64_t)num_cus * 512;
}

// One K range per tile: no workspace.
inline void whole_k(GemmSplit* g) {
  g->ksplit = 1;
  g->kpart = g->K;
}

}  // namespace tbh
