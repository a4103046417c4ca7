// tbh_gemm_epi.hpp -- output addressing shared by the GEMM kernels: a C in its
// consumer's label order (GemmDesc::scatter).
#pragma once
#include "tbh_device.hpp"

namespace tbh {

// Offset of the output bits x (bit b is GEMM output bit q0 + b) in a C whose
// bit q sits at position pc[q] (-1: no position; only rows / columns past M /
// N, which are not written, reach those).
__device__ __forceinline__ int64_t scatter_bits(const int8_t* __restrict__ pc, int q0, uint32_t x) {
  int64_t r = 0;
  for (int b = 0; x != 0 && q0 + b < kGemmScatter; b++, x >>= 1) {
    const int p = pc[q0 + b];
    if ((x & 1) && p >= 0) r += (int64_t)1 << p;
  }
  return r;
}

// A pass of 2^nbits staged outputs to C: the threads read LDS in ascending C
// position (enumeration bit k of output e = tid + 256 r is tile bit ep[k]), so
// that consecutive lanes store consecutive addresses.  In LDS, output (m, n)
// sits at (m ^ 4 (n & smask)) + 2^vm n.
template <typename T>
__device__ __forceinline__ void emit_staged(TBH_GLOBAL T* __restrict__ Ct,
                                            const T* __restrict__ st, int nbits, int vm,
                                            uint32_t smask, const int8_t* __restrict__ pc, int ma,
                                            const GemmDesc* __restrict__ d) {
  typedef T V __attribute__((ext_vector_type(4)));
  const int tid = threadIdx.x;
  // enumeration bit k as its share of the LDS index (xk: XORed part, ak:
  // added part; row bit b: xk = 2^b; column bit b: xk = 4 (2^b & s), ak =
  // 2^(vm+b)) and of the C offset (gk), decoded once (uniform)
  uint32_t xk[13], ak[13], gk[13];
#pragma unroll
  for (int k = 0; k < 13; k++) {
    xk[k] = ak[k] = gk[k] = 0;
    if (k < nbits) {
      const int b = d->ep[k];
      if (b < 32) {
        xk[k] = 1u << b;
        gk[k] = 1u << pc[b];
      } else {
        xk[k] = ((1u << (b - 32)) & smask) << 2;
        ak[k] = (1u << (b - 32)) << vm;
        gk[k] = 1u << pc[ma + b - 32];
      }
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
