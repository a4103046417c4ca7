// tbh_internal.hpp -- descriptors shared by the host planner and the gfx950
// kernels of libtbh.so.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace tbh {

constexpr int32_t kI32NegInf = -(1 << 30);
constexpr int32_t kI32NegThresh = -(1 << 29);
constexpr int kMaxRank = 30;     // largest tensor rank (2^30 entries)
constexpr int kMaxReduce = 12;   // reduced labels of one EW step
constexpr int kEwBlock = 256;    // threads per EW workgroup
constexpr int kTileBits = 12;    // a tile has at most 2^12 outputs
constexpr int kGemmScatter = 40; // GEMM output bit -> position table (rank + tile bits)
constexpr int kEpiElems = 8192;  // outputs per pass of a GEMM's LDS-staged epilogue
constexpr int kSubBits = 12;     // an LDS sub-tensor has at most 2^12 entries
// staged sub-tensors hold one pad entry per 2^TBH_LDS_PAD_SHIFT entries (0:
// none), which moves entries a multiple of that apart into different banks
#ifndef TBH_LDS_PAD_SHIFT
#define TBH_LDS_PAD_SHIFT 0
#endif
constexpr int kLdsElems =
    (1 << kSubBits) + (TBH_LDS_PAD_SHIFT ? ((1 << kSubBits) >> TBH_LDS_PAD_SHIFT) : 0);

// GEMM tile shape for an M x N output under a tile rule: 1 (default):
// tall-skinny outputs (N <= 64, M >= 256) take a 256-row tile so that a
// narrow N still fills it; 0: 128 x 128 tiles only; 2: 256 x 64 tiles up to
// N = 128 as well.
__host__ __device__ inline int gemm_shape(int64_t M, int64_t N, int rule = 1) {
  if (rule <= 0 || M < 256) return 0;
  if (N <= 32) return 2;
  if (N <= (rule >= 2 ? 128 : 64)) return 1;
  return 0;
}
// (shape 3: 64 x 64, each K slab split over the workgroup's waves)
constexpr int kGemm64 = 3, kGemmShapes = 4;
__host__ __device__ inline int gemm_bm(int shape) {
  return shape == kGemm64 ? 64 : shape ? 256 : 128;
}
__host__ __device__ inline int gemm_bn(int shape) {
  return shape == 2 ? 32 : shape == 0 ? 128 : 64;
}

// One EW step C = max over the reduced labels of A + B, tiled through LDS.
// The output labels split into tile labels (nT bits, ordered by C position)
// and outer labels (nO bits, one tile per configuration).  A tile first loads
// the sub-tensors of A and B it needs -- their tile and reduced labels, nSA /
// nSB bits in ascending operand position, so consecutive threads read
// consecutive addresses along the operand's lowest positions -- into LDS,
// then each of its outputs maxes A + B over the 2^nR reduced configurations
// and is written back contiguously along C's lowest positions.  Reduced
// labels beyond the sub-tensor budget are outer reduced labels (nRo): the
// tile repeats the load + max for each of their 2^nRo configurations,
// keeping its maxima in registers, before it writes.
// All positions are label positions (stride 2^p); -1 marks an absent label.
struct EwDesc {
  uint64_t a, b, c;        // device addresses; b == 0: unary step (B = tropical 1)
  int32_t nT, nO, nR;      // tile, outer and (sub-tensor) reduced bits
  int32_t nSA, nSB;        // sub-tensor bits of A and B
  int32_t tiles;           // 2^nO
  int32_t nRo;             // outer reduced bits (tiled steps only)
  int32_t mlay;            // MA in 1..3: tile bits 8..8+MA-1 are A-only labels and
                           // the rest of 8..11 B-only (a thread's 16 outputs are a
                           // 2^MA x 2^(4-MA) outer product); 0: no such layout
  int8_t qA[kMaxReduce];   // outer reduced bit -> A / B position
  int8_t qB[kMaxReduce];
  int8_t tC[kTileBits];    // tile bit -> C position
  int8_t tA[kTileBits];    // tile bit -> bit of A's sub-tensor
  int8_t tB[kTileBits];
  int8_t rA[kMaxReduce];   // reduced bit -> bit of A's / B's sub-tensor
  int8_t rB[kMaxReduce];
  int8_t sA[kSubBits];     // sub-tensor bit -> A position
  int8_t sB[kSubBits];
  int8_t oC[32], oA[32], oB[32];  // outer bit -> C / A / B position
};

__host__ __device__ inline uint32_t pos_stride(int8_t p) { return p >= 0 ? (1u << p) : 0u; }
__host__ __device__ inline uint32_t lds_pad(uint32_t i) {
  return TBH_LDS_PAD_SHIFT ? i + (i >> TBH_LDS_PAD_SHIFT) : i;
}

// One batched max-plus GEMM step (column-major, element strides).
struct GemmDesc {
  uint64_t a, b, c;         // device addresses
  int32_t M, N, K, batch;
  int64_t lda, ldb, ldc;
  int64_t sA, sB, sC;
  int32_t tiles_m, tiles_n; // tiles per batch entry
  int32_t shape;            // tile 0: 128 x 128, 1: 256 x 64, 2: 256 x 32, 3: 64 x 64
  // scatter: 0 C column-major with ldc; otherwise C has its own label order
  // (M, N, batch powers of two): bit q of (m, n, batch) -- m bits first,
  // then n, then batch -- sits at C position pc[q].  1: rows 0..4 sit at
  // positions 0..4, the tile stores its rows directly; 2: the tile is staged
  // in LDS and read back in ascending C position (ep), one pass of 2^ep_n
  // outputs (two passes split on the top column bit of the tile if ep_split)
  int32_t scatter;
  int8_t pc[kGemmScatter];  // -1 past the rank
  int8_t inv[32];           // C position -> output bit, -1 past the rank
  int8_t ep[16];            // tile bit b < 32: row bit b; 32 + b: column bit b
  int8_t epp[16];           // ... and its C position
  int32_t ep_n, ep_split;
};
static_assert(sizeof(GemmDesc) % 4 == 0 && sizeof(GemmDesc) <= 256, "a word per lane");

// One max-plus GEMM in 64 x 64 tiles (K1b, passed by value): ksplit K ranges
// of kpart (a multiple of 32 when ksplit > 1) per tile, their maxima to ws when
// ksplit > 1 (batch x ksplit x N x M).  M >= 4, K >= 4.
struct GemmSplit {
  uint64_t a, b, c, ws;
  int32_t M, N, K, batch;
  int64_t lda, ldb, ldc;
  int64_t sA, sB, sC;
  int32_t tiles_m, tiles_n, ksplit, kpart;
};
// The end of the K range that starts at kb (a sum of kb and kpart may pass 2^31).
__host__ __device__ inline int32_t gemm_range_end(const GemmSplit& g, int32_t kb) {
  return g.K - kb < g.kpart ? g.K : kb + g.kpart;
}

// Leaf tensor writes (vertex [0,w] or edge [0,0,0,-inf]).
struct LeafDesc {
  uint64_t p;      // device address
  int32_t kind;    // 1 = vertex, 2 = edge
  int32_t wbits;   // weight bit pattern of the dtype
};

// Per-slice epilogue: result = root + r (or r for an empty slice).
struct EpiDesc {
  uint64_t root;   // device address of the root scalar, 0: empty slice
  int32_t rbits;   // r as the dtype's bit pattern
  int32_t res;     // index of the result
};

// A fused part of the tree ("unit"): every step of a maximal connected part
// whose tensors all fit in LDS, contracted by one workgroup.  Tensors from
// outside it (ext) are copied to LDS first, only its root goes to memory.
// Inside a unit every tensor holds its labels in one global order (elimination
// time, latest first), so a step's union index is the output's bits, then the
// reduced labels'.
constexpr int kUnitWavesLog2 = 3;
constexpr int kUnitWaves = 1 << kUnitWavesLog2;  // waves of a unit's workgroup
constexpr int kUnitLds = 8192;     // LDS elements of a unit
constexpr int kUnitBits = 15;      // union labels of a unit's step
constexpr int kUnitRank = 14;      // output labels of a unit's step
constexpr int kUnitOperand = 12;   // labels of a tensor read from memory
constexpr int kUnitReduce = 6;     // reduced labels of a unit's step
// One wave's share of one step: chunks c0 .. c0+nc-1 of 64 outputs (nc a power
// of two, c0 a multiple), after `levels` more barriers than the wave has passed.
struct UnitItem {
  uint16_t mA, mB;  // the union bits of A and B; an operand holds its own in order
  uint16_t oA, oB;  // LDS element offsets of the operands at chunk c0
  uint16_t oC, c0;  // ... of the output (chunk 0)
  uint16_t f;       // output bits | reduced bits << 4 | kItemRoot | log2(nc) << 12
  uint16_t levels;
};
constexpr int kItemRoot = 1 << 8;  // the unit's output: to memory
struct UnitDesc {
  uint64_t c;        // device address of the output, 0: the slice's root scalar
  uint64_t pos;      // nibble k: the C position of output bit k
  uint32_t item0;    // first item; wave w's are item0 + start[w] .. start[w + 1] - 1
  uint32_t w0;       // first vertex weight
  uint32_t ext0;     // first tensor read from memory
  int32_t next;      // ... and their number
  int32_t nvert;     // vertex leaves, [0, w] at LDS 4 + 2 i (the edge tensor is at 0)
  int32_t res;       // c == 0: index of the slice's result
  int32_t rbits;     // ... and its r
  // no items at all: a leaf tensor (nvert 1: vertex, 0: edge)
  uint16_t start[kUnitWaves + 2];
};
struct UnitExt {
  uint64_t p;        // device address, labels in the units' order
  uint32_t off;      // LDS element offset
  uint32_t rank;
};

}  // namespace tbh
