// tbh_gemm_epi.hpp -- output addressing shared by the GEMM kernels: a C in its
// consumer's label order (GemmDesc::scatter).
#pragma once
#include <stddef.h>

#include "tbh_device.hpp"

namespace tbh {

// A launch's descriptors and prefixes through the constant address space: scalar
// loads, which do not queue behind the tiles' vector loads.
#define TBH_CONST __attribute__((address_space(4)))
using KGemm = const TBH_CONST GemmDesc*;

// The step of tile `tile`: the last i with prefix[i] <= tile.
__device__ __forceinline__ int gemm_step(const TBH_CONST int64_t* prefix, int nops,
                                         int64_t tile) {
  int lo = 0, hi = nops;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= tile)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// The thread's index, opaque to the compiler: what a tile derives from it is
// not held in registers across tiles.
__device__ __forceinline__ int opaque_tid() {
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));
  return tid;
}

// The label positions of a tile's outputs are read from a GemmDesc held a word
// per lane, by lane reads: read from memory they are a byte each, one after
// another.
__device__ __forceinline__ uint32_t gemm_lanes(KGemm d) {
  const uint32_t lane = opaque_tid() & 63;
  return ((const uint32_t*)d)[lane < sizeof(GemmDesc) / 4 ? lane : 0];
}

// C position of output bit q (-1: none; only rows / columns past M / N, which
// are not written, have none).
__device__ __forceinline__ int gemm_pos(uint32_t w, uint32_t q) {
  const uint32_t o = (uint32_t)offsetof(GemmDesc, pc) + q;
  return (int)(int8_t)((uint32_t)__builtin_amdgcn_readlane((int)w, (int)(o >> 2)) >> (8 * (o & 3)));
}

// Offset in C of the wave-uniform output index x (m, then n, then batch bits):
// lane p decides C position p.
__device__ __forceinline__ int64_t gemm_offset(uint32_t w, uint32_t x) {
  const uint32_t p = opaque_tid() & 31;
  const uint32_t word =
      (uint32_t)__builtin_amdgcn_ds_bpermute((int)(offsetof(GemmDesc, inv) + (p & 28)), (int)w);
  const uint32_t q = (word >> (8 * (p & 3))) & 0xff;
  return (int64_t)(uint32_t)__ballot(q < 32 && ((x >> (q & 31)) & 1));
}

// A pass of 2^nbits staged outputs to C: the threads read LDS in ascending C
// position (enumeration bit k of output e = tid + 256 r is tile bit ep[k]), so
// that consecutive lanes store consecutive addresses.  In LDS, output (m, n)
// sits at (m ^ 4 (n & smask)) + 2^vm n.
template <typename T>
__device__ __forceinline__ void emit_staged(TBH_GLOBAL T* __restrict__ Ct,
                                            const T* __restrict__ st, int nbits, int vm,
                                            uint32_t smask, uint32_t w) {
  typedef T V __attribute__((ext_vector_type(4)));
  const int tid = opaque_tid();
  // enumeration bit k as its share of the LDS index (xk: XORed part, ak:
  // added part; row bit b: xk = 2^b; column bit b: xk = 4 (2^b & s), ak =
  // 2^(vm+b)) and of the C offset (gk), decoded once (uniform)
  uint32_t e[4], g[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    e[i] = (uint32_t)__builtin_amdgcn_readlane((int)w, (int)(offsetof(GemmDesc, ep) / 4) + i);
    g[i] = (uint32_t)__builtin_amdgcn_readlane((int)w, (int)(offsetof(GemmDesc, epp) / 4) + i);
  }
  uint32_t xk[13], ak[13], gk[13];
#pragma unroll
  for (int k = 0; k < 13; k++) {
    xk[k] = ak[k] = gk[k] = 0;
    if (k < nbits) {
      const uint32_t b = (e[k / 4] >> (8 * (k % 4))) & 0xff;
      const uint32_t bit = 1u << (b & 31);
      xk[k] = b < 32 ? bit : (bit & smask) << 2;
      ak[k] = b < 32 ? 0 : bit << vm;
      gk[k] = 1u << ((g[k / 4] >> (8 * (k % 4))) & 31);
    }
  }
  // enumeration bits 0 and 1 are C positions 0 and 1 (ep lists the pass's
  // bits by C position, and C's lowest positions are pass bits): a thread
  // owns 4 consecutive outputs, one aligned 16-byte store; bits 2..9 are
  // the thread, bits 10.. the iteration r
  uint32_t xt = 0, at = 0, gt = 0;
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const bool on = (tid >> k) & 1;
    xt ^= on ? xk[2 + k] : 0u;
    at += on ? ak[2 + k] : 0u;
    gt += on ? gk[2 + k] : 0u;
  }
  uint32_t li[4];
#pragma unroll
  for (int i = 0; i < 4; i++)
    li[i] = ((i & 1) ? xk[0] : 0u) ^ ((i & 2) ? xk[1] : 0u);
  const uint32_t a1 = ak[0], a2 = ak[1];
  const int R = 1 << (nbits - 10);  // 4 .. 8 per pass
#pragma unroll
  for (int r = 0; r < 8; r++) {
    if (r >= R) break;
    uint32_t xr = xt, ar = at, gr = gt;
#pragma unroll
    for (int k = 0; k < 3; k++)
      if ((r >> k) & 1) {
        xr ^= xk[10 + k];
        ar += ak[10 + k];
        gr += gk[10 + k];
      }
    V q;
    q.x = st[(xr ^ li[0]) + ar];
    q.y = st[(xr ^ li[1]) + ar + a1];
    q.z = st[(xr ^ li[2]) + ar + a2];
    q.w = st[(xr ^ li[3]) + ar + a1 + a2];
    *reinterpret_cast<TBH_GLOBAL V*>(Ct + gr) = q;
  }
}

}  // namespace tbh
