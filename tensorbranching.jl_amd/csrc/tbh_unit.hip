// tbh_unit.hip -- K4 tbh_unit_kernel: a connected part of a slice's contraction
// tree in one workgroup, every tensor but its output in LDS.
//
// What bounds it: the chain of a unit's levels (10-30 of them), each a few
// LDS reads and a barrier; its arithmetic (at most 2^17 MACs) and bytes (16
// per step share, 4 per vertex weight, the output) are small.  One launch
// replaces the level-by-level launches of these steps (11-25 us each, about
// 93% of a slice's steps) and their 300-byte descriptors: the 22 slices of
// 3-regular n=100 at sc 10 are 22 units, 45 us against 862 us in 53 launches;
// one n=100 slice of sc 15 takes 0.41 ms per call against 0.96 ms, the 301
// slices of n=200 at sc 20 16.6 against 23.9 ms (planning included).
//
// Four waves and 32 KB of LDS per unit: a level of a unit seldom has work for
// more waves, and five units stay resident per CU.  The steps of a level run
// side by side, one barrier per level.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tbh_device.hpp"

namespace tbh {

namespace {

// The bits of x at the set positions of m, packed to the low end (m the same
// in every lane): one field move per run of set bits.
__device__ __forceinline__ uint32_t gather_bits(uint32_t x, uint32_t m) {
  uint32_t v = 0, d = 0, at = 0;
  while (m) {
    const uint32_t z = __builtin_ctz(m);
    m >>= z;
    at += z;
    const uint32_t len = __builtin_ctz(~m);  // m has at most 16 bits
    v |= ((x >> at) & ((1u << len) - 1)) << d;
    d += len;
    at += len;
    m >>= len;
  }
  return v;
}

__device__ __forceinline__ uint32_t lane_read(uint32_t v, uint32_t lane) {
  return __builtin_amdgcn_readlane(v, lane);
}

}  // namespace

template <typename T>
__global__ __launch_bounds__(64 * kUnitWaves) void tbh_unit_kernel(
    const UnitDesc* __restrict__ units, const uint4* __restrict__ items,
    const uint32_t* __restrict__ weights, const UnitExt* __restrict__ ext,
    T* __restrict__ results) {
  __shared__ __align__(16) T lds[kUnitLds];
  const UnitDesc& u = units[blockIdx.x];
  const uint32_t tid = threadIdx.x, lane = tid & 63;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int rounds = u.rounds;
  const uint64_t pos = u.pos;
  const uint32_t* w = weights + u.w0;
  TBH_GLOBAL T* C = reinterpret_cast<TBH_GLOBAL T*>(u.c);
  if (rounds == 0) {  // a leaf tensor
    if (u.nvert) {
      if (tid < 2) C[tid] = tid ? __builtin_bit_cast(T, w[0]) : Trop<T>::one();
    } else if (tid < 4) {
      C[tid] = tid == 3 ? pad_zero<T>() : Trop<T>::one();
    }
    return;
  }
  // the wave's items, one per lane, 64 rounds at a time: a round's item
  // reaches scalar registers by a lane read, with no memory access
  const uint4* my = items + u.item0 + wave * rounds;
  uint4 held = (int)lane < rounds ? my[lane] : uint4{0, 0, 0, 0};
  // tensors from memory straight to LDS, all in flight at once
  for (int q = 0; q < u.next; q++) {
    const UnitExt x = ext[u.ext0 + q];
    const TBH_GLOBAL T* X = reinterpret_cast<const TBH_GLOBAL T*>(x.p);
    const uint32_t n = 1u << x.rank;
    for (uint32_t i = wave * 64; i < n; i += 64 * kUnitWaves)
      if (i + lane < n)
        __builtin_amdgcn_global_load_lds(X + i + lane, (TBH_LDS T*)lds + x.off + i, 4, 0, 0);
  }
  if (tid < 4) lds[tid] = tid == 3 ? pad_zero<T>() : Trop<T>::one();
  for (int i = tid; i < u.nvert; i += 64 * kUnitWaves) {
    lds[4 + 2 * i] = Trop<T>::one();
    lds[5 + 2 * i] = __builtin_bit_cast(T, w[i]);
  }
  __builtin_amdgcn_s_waitcnt(0);  // the copies to LDS (a barrier does not wait for them)
  __syncthreads();
  for (int r = 0; r < rounds; r++) {
    if (r && (r & 63) == 0) held = r + (int)lane < rounds ? my[r + lane] : uint4{0, 0, 0, 0};
    const uint32_t x = lane_read(held.x, r & 63), y = lane_read(held.y, r & 63);
    const uint32_t z = lane_read(held.z, r & 63), f = lane_read(held.w, r & 63) >> 16;
    const uint32_t nc = lane_read(held.w, r & 63) & 0xffff;
    if (nc) {
      const uint32_t mA = x & 0xffff, mB = x >> 16, oA = y & 0xffff, oB = y >> 16;
      const uint32_t oC = z & 0xffff, c0 = z >> 16;
      const uint32_t nP = f & 15, nR = (f >> 4) & 15;
      // union index = lane bits | chunk bits << 6 | reduced bits << nP; each
      // part keeps the operand's bits.  The chunk and reduced parts are held
      // one per lane and read back by the loops below.
      const uint32_t nl = nP < 6 ? nP : 6;
      const uint32_t lm = (1u << nl) - 1, cm = (1u << (nP - nl)) - 1;
      const uint32_t ml = lane & lm;
      const uint32_t aL = oA + gather_bits(ml, mA & lm), bL = oB + gather_bits(ml, mB & lm);
      const uint32_t sA = __builtin_popcount(mA & lm), sB = __builtin_popcount(mB & lm);
      uint32_t aC = 0, bC = 0, aR = 0, bR = 0;
      if (nP > 6) {
        aC = gather_bits(c0 + lane, (mA >> 6) & cm) << sA;
        bC = gather_bits(c0 + lane, (mB >> 6) & cm) << sB;
      }
      if (nR) {
        aR = gather_bits(lane, mA >> nP) << __builtin_popcount(mA & ((1u << nP) - 1));
        bR = gather_bits(lane, mB >> nP) << __builtin_popcount(mB & ((1u << nP) - 1));
      }
      // where an output goes: LDS (its own order), or the unit's C
      const bool root = f & (kItemRoot & 0xffff);
      uint32_t pL = 0, pC = 0;
      if (root && C) {
        for (uint32_t k = 0; k < nl; k++) pL |= ((lane >> k) & 1) << ((pos >> (4 * k)) & 15);
        for (uint32_t k = nl; k < nP; k++) pC |= (((c0 + lane) >> (k - nl)) & 1) << ((pos >> (4 * k)) & 15);
      }
      const bool active = lane <= lm;
      for (uint32_t c = 0; c < nc; c++) {
        const uint32_t a = aL + lane_read(aC, c), b = bL + lane_read(bC, c);
        T acc;
        if (nR == 0) {
          // (maxed with the tropical zero: a NaN of an infinite weight is dropped)
          acc = Trop<T>::add(Trop<T>::zero(), Trop<T>::mul(lds[a], lds[b]));
        } else if (nR == 1) {
          const uint32_t a1 = lane_read(aR, 1), b1 = lane_read(bR, 1);
          acc = max3(Trop<T>::zero(), Trop<T>::mul(lds[a], lds[b]),
                     Trop<T>::mul(lds[a + a1], lds[b + b1]));
        } else {
          acc = Trop<T>::zero();
          for (uint32_t q = 0; q < (1u << nR); q += 4) {
            T v[4];
#pragma unroll
            for (int i = 0; i < 4; i++)
              v[i] = Trop<T>::mul(lds[a + lane_read(aR, q + i)], lds[b + lane_read(bR, q + i)]);
            acc = max3(max3(acc, v[0], v[1]), v[2], v[3]);
          }
        }
        acc = Trop<T>::canon(acc);
        if (!root) {
          if (active) lds[oC + (c0 + c) * 64 + lane] = acc;
        } else if (C) {
          if (active) C[pL + lane_read(pC, c)] = acc;
        } else if (lane == 0) {
          // the slice's result: root + r
          results[u.res] = Trop<T>::canon(Trop<T>::mul(acc, __builtin_bit_cast(T, u.rbits)));
        }
      }
    }
    if (f & kItemBarrier) __syncthreads();
  }
}

hipError_t launch_units(int dtype, const UnitDesc* units, const UnitItem* items,
                        const uint32_t* weights, const UnitExt* ext, int64_t n, void* results,
                        hipStream_t s) {
  if (n <= 0) return hipSuccess;
  const uint4* it = reinterpret_cast<const uint4*>(items);
  if (dtype == 0)
    tbh_unit_kernel<float><<<(int)n, 64 * kUnitWaves, 0, s>>>(units, it, weights, ext,
                                                              static_cast<float*>(results));
  else
    tbh_unit_kernel<int32_t><<<(int)n, 64 * kUnitWaves, 0, s>>>(units, it, weights, ext,
                                                                static_cast<int32_t*>(results));
  return hipGetLastError();
}

}  // namespace tbh
