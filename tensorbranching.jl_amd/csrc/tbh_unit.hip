// tbh_unit.hip -- K4 tbh_unit_kernel: a connected part of a slice's contraction
// tree in one workgroup, every tensor but its output in LDS.
//
// What bounds it: the chain of a unit's levels (10-30 of them), each a few
// LDS reads and a barrier; its arithmetic (at most 2^17 MACs) and bytes (16
// per step share, 4 per vertex weight, the output) are small.  One launch
// replaces the level-by-level launches of these steps (11-25 us each, about
// 93% of a slice's steps) and their 300-byte descriptors: the 22 slices of
// 3-regular n=100 at sc 10 are 22 units, 22 us against 862 us in 53 launches.
//
// A wave issues an instruction every 4 cycles at best and has its SIMD to
// itself, so a step's length is its instruction count.  An operand holds its
// labels in the union's order: its place of a union index is a bit extraction,
// read from a table of 6-bit extractions in LDS (4 KB, one load per thread); a
// step share's fields are taken from its 16 bytes for 64 shares at once, a
// share per lane, and read by lane.  Extraction by a loop over the bits and
// four waves in lockstep over rounds: 47 us where this takes 22, 40 / 24 for a
// slice of sc 15 (two launches), 17 / 10.7 per launch of two King's subgraphs.
//
// Eight waves and 36 KB of LDS per unit: the widest levels have 5-30 steps and
// four units stay resident per CU.  The steps of a level run side by side, one
// barrier per level; each wave has a list of its own.
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "tbh_device.hpp"

namespace tbh {

namespace {

// v[m << 6 | x]: the bits of x at the set bits of m, packed (6 bits).
struct BitTable {
  uint8_t v[4096];
  constexpr BitTable() : v{} {
    for (int m = 0; m < 64; m++)
      for (int x = 0; x < 64; x++) {
        int y = 0, n = 0;
        for (int k = 0; k < 6; k++)
          if (m >> k & 1) y |= (x >> k & 1) << n++;
        v[m << 6 | x] = (uint8_t)y;
      }
  }
};
__device__ constexpr BitTable kBits{};

// x's bit k at place p[k] (nibbles; 15: dropped), k < N.
template <int N>
__device__ __forceinline__ uint32_t place_bits(uint32_t x, uint64_t p) {
  uint32_t v = 0;
#pragma unroll
  for (int k = 0; k < N; k++) v |= ((x >> k) & 1u) << ((uint32_t)(p >> (4 * k)) & 15u);
  return v & 0x7fff;
}

__device__ __forceinline__ uint32_t lane_read(uint32_t v, uint32_t lane) {
  return __builtin_amdgcn_readlane(v, lane);
}
__device__ __forceinline__ uint64_t lane_read64(uint32_t lo, uint32_t hi, uint32_t lane) {
  return (uint64_t)lane_read(hi, lane) << 32 | lane_read(lo, lane);
}

}  // namespace

template <typename T>
__global__ __launch_bounds__(64 * kUnitWaves) void tbh_unit_kernel(
    const UnitDesc* __restrict__ units, const uint4* __restrict__ items,
    const uint32_t* __restrict__ weights, const UnitExt* __restrict__ ext,
    T* __restrict__ results) {
  __shared__ __align__(16) T lds[kUnitLds];
  __shared__ __align__(16) uint8_t bits[sizeof(BitTable)];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  static_assert(sizeof(BitTable) == 8 * 64 * kUnitWaves, "");
  const uint2 bt = reinterpret_cast<const uint2*>(kBits.v)[tid];
  // the descriptor by one load, a word per lane
  const uint32_t dw = reinterpret_cast<const uint32_t*>(units + blockIdx.x)[lane & 15];
#define TBH_FIELD(f) lane_read(dw, offsetof(UnitDesc, f) / 4)
  TBH_GLOBAL T* C = reinterpret_cast<TBH_GLOBAL T*>(
      (uint64_t)lane_read(dw, 1) << 32 | TBH_FIELD(c));
  const uint64_t pos = (uint64_t)lane_read(dw, 3) << 32 | TBH_FIELD(pos);
  const uint32_t* w = weights + TBH_FIELD(w0);
  const int nvert = TBH_FIELD(nvert), next = TBH_FIELD(next);
  const uint32_t ext0 = TBH_FIELD(ext0);
  constexpr uint32_t kStart = offsetof(UnitDesc, start) / 4;
  static_assert(sizeof(UnitDesc) == 64 && offsetof(UnitDesc, c) == 0 &&
                offsetof(UnitDesc, pos) == 8 && kStart * 4 == offsetof(UnitDesc, start), "");
  auto start_of = [&](uint32_t k) {
    return lane_read(dw, kStart + k / 2) >> (16 * (k & 1)) & 0xffff;
  };
  if (start_of(kUnitWaves) == 0) {  // a leaf tensor
    if (nvert) {
      if (tid < 2) C[tid] = tid ? __builtin_bit_cast(T, w[0]) : Trop<T>::one();
    } else if (tid < 4) {
      C[tid] = tid == 3 ? pad_zero<T>() : Trop<T>::one();
    }
    return;
  }
  // the wave's items, one per lane, 64 at a time, and the tensors from memory,
  // one per lane: they reach scalar registers by lane reads, with no further
  // memory access
  const uint32_t first = start_of(wave), count = start_of(wave + 1) - first;
  const uint4* my = items + (size_t)(TBH_FIELD(item0) + first);
  uint4 h{0, 0, 0, 0};
  if (lane < count) h = my[lane];
  uint32_t w0 = 0;
  if ((int)tid < nvert) w0 = w[tid];
  for (int q0 = 0; q0 < next; q0 += 64) {
    uint4 x{0, 0, 0, 0};
    if (q0 + (int)lane < next) x = reinterpret_cast<const uint4*>(ext)[ext0 + q0 + lane];
    const int nq = next - q0 < 64 ? next - q0 : 64;
    // straight to LDS, all in flight at once
    for (int q = 0; q < nq; q++) {
      const TBH_GLOBAL T* X = reinterpret_cast<const TBH_GLOBAL T*>(lane_read64(x.x, x.y, q));
      const uint32_t off = lane_read(x.z, q), n = 1u << lane_read(x.w, q);
      for (uint32_t i = (wave + q) % kUnitWaves * 64; i < n; i += 64 * kUnitWaves)
        if (i + lane < n)
          __builtin_amdgcn_global_load_lds(X + i + lane, (TBH_LDS T*)lds + off + i, 4, 0, 0);
    }
  }
  reinterpret_cast<uint2*>(bits)[tid] = bt;
  if (tid < 4) lds[tid] = tid == 3 ? pad_zero<T>() : Trop<T>::one();
  for (int i = tid; i < nvert; i += 64 * kUnitWaves) {
    lds[4 + 2 * i] = Trop<T>::one();
    lds[5 + 2 * i] = __builtin_bit_cast(T, i == (int)tid ? w0 : w[i]);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the copies to LDS (a barrier does not wait for them)
  __syncthreads();
  // Fields of the lane's item: rows of the table and offsets of its operands,
  // the strides of its first reduced bit, the output's place
  uint32_t rA = 0, rB = 0, oA = 0, oB = 0, dA = 0, dB = 0, oC = 0;
  for (uint32_t r = 0; r < count; r++) {
    const uint32_t at = r & 63;
    if (at == 0) {
      if (r && r + lane < count) h = my[r + lane];
      const uint32_t mA = h.x & 0xffff, mB = h.x >> 16, nP = h.w & 15, nR = (h.w >> 4) & 15;
      const uint32_t out = (1u << nP) - 1;
      rA = (mA & out & 63) << 6;
      rB = (mB & out & 63) << 6;
      oA = h.y & 0xffff;
      oB = h.y >> 16;
      dA = nR ? ((mA >> nP) & 1) << __builtin_popcount(mA & out) : 0;
      dB = nR ? ((mB >> nP) & 1) << __builtin_popcount(mB & out) : 0;
      oC = (h.z & 0xffff) + (h.z >> 16) * 64;
    }
    uint32_t a = lane_read(oA, at) + bits[lane_read(rA, at) + lane];
    uint32_t b = lane_read(oB, at) + bits[lane_read(rB, at) + lane];
    const uint32_t f = lane_read(h.w, at), nP = f & 15, nR = (f >> 4) & 15;
    const uint32_t c = lane_read(oC, at);
    const bool active = lane < (1u << nP);
    if ((f & (kItemRoot | 0xf000)) == 0 && nR < 2) {
      // most items: 64 outputs or fewer, to LDS, one reduced bit at most (none:
      // strides of 0, the same product twice)
      const uint32_t a1 = a + lane_read(dA, at), b1 = b + lane_read(dB, at);
      // the levels between (after the addresses: they need no data): every
      // wave passes each level's barrier once, as long as it has items left (a
      // wave that has ended is not waited for)
      for (uint32_t q = f >> 16; q > 0; q--) __syncthreads();
      // (maxed with the tropical zero: a NaN of an infinite weight is dropped)
      const T acc = Trop<T>::canon(max3(Trop<T>::zero(), Trop<T>::mul(lds[a], lds[b]),
                                        Trop<T>::mul(lds[a1], lds[b1])));
      if (active) lds[c + lane] = acc;
      continue;
    }
    // The chunk and reduced parts of the operands' places, one per lane, read
    // back by the loops.
    const uint32_t m = lane_read(h.x, at), mA = m & 0xffff, mB = m >> 16;
    const uint32_t out = (1u << nP) - 1, nc = 1u << ((f >> 12) & 15);
    uint32_t aC = 0, bC = 0, aR = 0, bR = 0;
    if (nc > 1) {
      aC = bits[(((mA >> 6) & (nc - 1)) << 6) + lane] << __builtin_popcount(mA & 63);
      bC = bits[(((mB >> 6) & (nc - 1)) << 6) + lane] << __builtin_popcount(mB & 63);
    }
    if (nR) {
      aR = bits[((mA >> nP) << 6) + lane] << __builtin_popcount(mA & out);
      bR = bits[((mB >> nP) << 6) + lane] << __builtin_popcount(mB & out);
    }
    // where an output goes: LDS (its own order), or the unit's C
    const bool root = f & kItemRoot;
    uint32_t pL = 0, pC = 0;
    if (root && C) {
      pL = place_bits<6>(lane & out, pos);
      if (nP > 6) pC = place_bits<8>((lane_read(h.z, at) >> 16) + lane, pos >> 24);
    }
    for (uint32_t q = f >> 16; q > 0; q--) __syncthreads();
    for (uint32_t k = 0; k < nc; k++) {
      const uint32_t ak = a + lane_read(aC, k), bk = b + lane_read(bC, k);
      T acc = Trop<T>::zero();
      if (nR < 2) {
        const uint32_t a1 = lane_read(aR, nR), b1 = lane_read(bR, nR);
        acc = max3(acc, Trop<T>::mul(lds[ak], lds[bk]),
                   Trop<T>::mul(lds[ak + a1], lds[bk + b1]));
      } else {
        for (uint32_t q = 0; q < (1u << nR); q += 4) {
          T v[4];
#pragma unroll
          for (int i = 0; i < 4; i++)
            v[i] = Trop<T>::mul(lds[ak + lane_read(aR, q + i)], lds[bk + lane_read(bR, q + i)]);
          acc = max3(max3(acc, v[0], v[1]), v[2], v[3]);
        }
      }
      acc = Trop<T>::canon(acc);
      if (!root) {
        if (active) lds[c + k * 64 + lane] = acc;
      } else if (C) {
        if (active) C[pL + lane_read(pC, k)] = acc;
      } else if (lane == 0) {
        // the slice's result: root + r
        results[TBH_FIELD(res)] =
            Trop<T>::canon(Trop<T>::mul(acc, __builtin_bit_cast(T, TBH_FIELD(rbits))));
      }
    }
  }
}

#undef TBH_FIELD

hipError_t launch_units(int dtype, const UnitDesc* units, const UnitItem* items,
                        const uint32_t* weights, const UnitExt* ext, int64_t n, void* results,
                        hipStream_t s) {
  const uint4* it = reinterpret_cast<const uint4*>(items);
  // a launch holds at most 2^32 - 1 work-items (more wrap without an error)
  constexpr int64_t kMost = ((int64_t)1 << 32) / (64 * kUnitWaves) - 1;
  for (int64_t i = 0; i < n; i += kMost) {
    const int blocks = (int)(n - i < kMost ? n - i : kMost);
    if (dtype == 0)
      tbh_unit_kernel<float><<<blocks, 64 * kUnitWaves, 0, s>>>(units + i, it, weights, ext,
                                                                static_cast<float*>(results));
    else
      tbh_unit_kernel<int32_t><<<blocks, 64 * kUnitWaves, 0, s>>>(
          units + i, it, weights, ext, static_cast<int32_t*>(results));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace tbh
