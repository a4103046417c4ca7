// tbh_gemm.hip -- K1b: max-plus GEMMs in 64 x 64 tiles, for products whose
// 128 x 128 tiles would not fill the GPU, or whose extents or alignment are
// odd.  tbh_gemm_ksplit_kernel runs one product (the tbh_maxplus_gemm entry
// point), tbh_gemm64_kernel the GEMM steps of a wave (GemmDesc::shape 3).
//
// A workgroup of four waves owns one 64 x 64 output tile; every wave holds
// the whole tile (8 x 8 maxima per lane, the register blocking of K1) and
// takes a quarter of each K slab, so the tile is a quarter of K1's with K1's
// LDS traffic per MAC.  The waves' maxima meet in LDS at the end.  A K range
// per workgroup (ksplit > 1) spreads products of few tiles over the CUs:
// each range's raw maxima go to a workspace, and tbh_gemm_reduce_kernel maxes
// them into C.
//
// Operands are read 16 bytes at a time whatever their alignment (a global
// load needs only 4-byte alignment here); quads that cross an edge are read
// from the last four entries before it and shifted into place.
//
// Bound by the VALU for large products (4096^3 Float32 1742 us = 78.9 T op/s
// of the 82.1 measured for its instruction mix; 4093 x 4095 x 4091 71.9, 67.2
// with K1), by too little work in flight and the two launches for small ones
// (512^3 19 us, 114 with K1's 16 tiles; 64^3 10 us, 18.6 with K1, about 6 us
// of each the events around it): those whose 32 x 32 tiles fit the chip's LDS
// with all of K at once run in tbh_gemm32_kernel instead.  Short K: bound by handing the maxima over,
// which all four waves share (two waves alone: 4096^2 x 1024 491 us, 479 so;
// in one round of 48 KB instead of two of 24 KB: 486).  The grouped kernel
// runs the GEMM steps of 301 n=200 slices at 31 T op/s Int32 (K1: 19 of the
// 52 measured for the mix).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tbh_device.hpp"
#include "tbh_gemm_epi.hpp"

namespace tbh {

namespace {

constexpr int kTile = 64;   // output tile
constexpr int kSlab = 32;   // K per slab, 8 per wave
constexpr int kBRow = kTile + 4;

template <typename T>
struct Quad {
  typedef T V __attribute__((ext_vector_type(4)));                // LDS
  typedef T U __attribute__((ext_vector_type(4), aligned(4)));   // global memory
};

// x[d..3], then fill: the entries of a quad read d entries too early
template <typename T>
__device__ __forceinline__ typename Quad<T>::V shift_quad(typename Quad<T>::V x, int d, T fill) {
  if (d & 1) x = typename Quad<T>::V{x.y, x.z, x.w, fill};
  if (d & 2) x = typename Quad<T>::V{x.z, x.w, fill, fill};
  return x;
}

constexpr int kLdsA = kSlab * kTile, kLdsB = kSlab * kBRow;
constexpr int kGemmLds = 2 * (kLdsA + kLdsB);  // two slabs
static_assert(kGemmLds >= 6 * 1024 && kGemmLds >= kTile * kTile, "maxima handed over, the tile");

__device__ __forceinline__ int tile_col(int wave, int ty) {
  return 32 * (wave >> 1) + ty + 2 * (wave & 1);
}

// One tile over the K range [kb, ke): afterwards quad q of the thread (res[q])
// is rows 32 (q & 1) + tx .. + 3 of column tile_col(wave, ty) + (q >> 1).  EDGE:
// any extents >= 4 and alignment; else M and N are multiples of 64 and K is 16
// or a multiple of 32 (kb = 0, ke = K).
template <typename T, bool EDGE>
__device__ __forceinline__ void gemm64_tile(const TBH_GLOBAL T* __restrict__ A,
                                            const TBH_GLOBAL T* __restrict__ B, int M, int N,
                                            int K, int64_t lda, int64_t ldb, int kb, int ke,
                                            int m0, int n0, int tid, T* __restrict__ smem,
                                            T (&res)[4][4]) {
  T acc[8][8];
  using V = typename Quad<T>::V;
  using U = typename Quad<T>::U;
  constexpr int NA = kLdsA, NB = kLdsB;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const T pz = pad_zero<T>();
  // this thread's quads: A rows am..am+3 of slab columns ak and ak + 16, B
  // slab rows bk..bk+3 of columns bn and bn + 32
  const int aq = (tid & 15) * 4, ak = tid >> 4;
  const int bk = (tid & 7) * 4, bn = tid >> 3;
  V ra[2], rb[2];
  // rows past M read earlier ones, shifted so that valid rows stay in place
  const int am = !EDGE || m0 + aq < M - 4 ? m0 + aq : M - 4;
  const int as = m0 + aq - am < 4 ? m0 + aq - am : 0;
  const bool edge_m = m0 + kTile > M;
  const int bn0 = !EDGE || n0 + bn < N ? n0 + bn : N - 1;
  const int bn1 = !EDGE || n0 + bn + 32 < N ? n0 + bn + 32 : N - 1;
  // !EDGE: wave-uniform bases of the tile and one 32-bit byte offset per lane
  // and quad (M and K at most 2^24, the planner's rule), which leaves the
  // registers the maxima need
  const uint32_t oa = ((uint32_t)ak * (uint32_t)lda + aq) * 4;
  const uint32_t ob = ((uint32_t)bn * (uint32_t)ldb + bk) * 4;
  auto at = [](const TBH_GLOBAL T* base, uint32_t byte) {
    return *reinterpret_cast<const TBH_GLOBAL U*>(
        reinterpret_cast<const TBH_GLOBAL char*>(base) + byte);
  };
  auto load = [&](int k0) {
    if constexpr (!EDGE) {
      const TBH_GLOBAL T* Ak = A + m0 + (int64_t)k0 * lda;
      const TBH_GLOBAL T* Bk = B + (int64_t)n0 * ldb + k0;
      if ((uint32_t)k0 + kSlab <= (uint32_t)ke) {
        ra[0] = at(Ak, oa);
        ra[1] = at(Ak + 16 * lda, oa);
        rb[0] = at(Bk, ob);
        rb[1] = at(Bk + 32 * ldb, ob);
      } else {  // K = 16: half a slab
        ra[0] = at(Ak, oa);
        ra[1] = V{pz, pz, pz, pz};
        rb[0] = rb[1] = V{pz, pz, pz, pz};
        if (bk < 16) {
          rb[0] = at(Bk, ob);
          rb[1] = at(Bk + 32 * ldb, ob);
        }
      }
      return;
    }
    if ((uint32_t)k0 + kSlab <= (uint32_t)ke) {
#pragma unroll
      for (int e = 0; e < 2; e++)
        ra[e] = *reinterpret_cast<const TBH_GLOBAL U*>(A + (int64_t)(k0 + ak + 16 * e) * lda + am);
      rb[0] = *reinterpret_cast<const TBH_GLOBAL U*>(B + (int64_t)bn0 * ldb + k0 + bk);
      rb[1] = *reinterpret_cast<const TBH_GLOBAL U*>(B + (int64_t)bn1 * ldb + k0 + bk);
    } else {
      // the range's last slab: columns of A past it are the tropical zero,
      // and so are B's rows (a range ends at a multiple of 4, or at K)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int k = k0 + ak + 16 * e;
        if (k < ke)
          ra[e] = *reinterpret_cast<const TBH_GLOBAL U*>(A + (int64_t)k * lda + am);
        else
          ra[e] = V{pz, pz, pz, pz};
      }
      const int k = k0 + bk, kc = k < K - 4 ? k : K - 4;
      if (k < ke) {
        rb[0] = *reinterpret_cast<const TBH_GLOBAL U*>(B + (int64_t)bn0 * ldb + kc);
        rb[1] = *reinterpret_cast<const TBH_GLOBAL U*>(B + (int64_t)bn1 * ldb + kc);
        rb[0] = shift_quad<T>(rb[0], k - kc, pz);
        rb[1] = shift_quad<T>(rb[1], k - kc, pz);
      } else {
        rb[0] = rb[1] = V{pz, pz, pz, pz};
      }
    }
    if (edge_m) {
      ra[0] = shift_quad<T>(ra[0], as, pz);
      ra[1] = shift_quad<T>(ra[1], as, pz);
    }
  };
  auto store = [&](int buf) {
    T* As = smem + buf * (NA + NB);
    T* Bs = As + NA;
#pragma unroll
    for (int e = 0; e < 2; e++) *reinterpret_cast<V*>(As + (ak + 16 * e) * kTile + aq) = ra[e];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      Bs[(bk + q) * kBRow + bn] = rb[0][q];
      Bs[(bk + q) * kBRow + bn + 32] = rb[1][q];
    }
  };
  const int tx = (lane & 7) * 4, ty = (lane >> 3) * 4;
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int j = 0; j < 8; j++) acc[i][j] = Trop<T>::zero();
  if (kb < ke) load(kb);
  if (kb < ke) store(0);
  __syncthreads();
  int buf = 0;
  for (uint32_t k0 = kb; k0 < (uint32_t)ke; k0 += kSlab) {  // (ke + kSlab may pass 2^31)
    const bool more = k0 + kSlab < (uint32_t)ke;
    if (more) load(k0 + kSlab);
    const T* As = smem + buf * (NA + NB) + wave * 8 * kTile;
    const T* Bs = smem + buf * (NA + NB) + NA + wave * 8 * kBRow;
#pragma unroll
    for (int kk = 0; kk < 8; kk += 2) {
      T a0[8], a1[8], b0[8], b1[8];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        V v = *reinterpret_cast<const V*>(As + kk * kTile + 32 * h + tx);
        a0[4 * h] = v.x; a0[4 * h + 1] = v.y; a0[4 * h + 2] = v.z; a0[4 * h + 3] = v.w;
        v = *reinterpret_cast<const V*>(As + (kk + 1) * kTile + 32 * h + tx);
        a1[4 * h] = v.x; a1[4 * h + 1] = v.y; a1[4 * h + 2] = v.z; a1[4 * h + 3] = v.w;
        v = *reinterpret_cast<const V*>(Bs + kk * kBRow + 32 * h + ty);
        b0[4 * h] = v.x; b0[4 * h + 1] = v.y; b0[4 * h + 2] = v.z; b0[4 * h + 3] = v.w;
        v = *reinterpret_cast<const V*>(Bs + (kk + 1) * kBRow + 32 * h + ty);
        b1[4 * h] = v.x; b1[4 * h + 1] = v.y; b1[4 * h + 2] = v.z; b1[4 * h + 3] = v.w;
      }
#pragma unroll
      for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 8; j++)
          acc[i][j] = max3(acc[i][j], Trop<T>::mul(a0[i], b0[j]), Trop<T>::mul(a1[i], b1[j]));
      __builtin_amdgcn_sched_barrier(0);
    }
    if (more) store(buf ^ 1);
    __syncthreads();
    buf ^= 1;
  }
  // wave d ends with columns 2 d and 2 d + 1 of every lane's block: the others
  // hand it theirs, two waves' columns (24 KB) at a time
#pragma unroll
  for (int q = 0; q < 4; q++)
#pragma unroll
    for (int i = 0; i < 4; i++) res[q][i] = acc[4 * (q & 1) + i][q >> 1];  // wave 0's
#pragma unroll
  for (int half = 0; half < 2; half++) {
#pragma unroll
    for (int d = 2 * half; d < 2 * half + 2; d++) {
      if (wave != d) {
        T* p = smem + (((d & 1) * 3 + (wave < d ? wave : wave - 1)) * 256 + lane) * 4;
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const int j = 2 * d + (q >> 1), h = q & 1;
          T x0 = acc[4 * h][j], x1 = acc[4 * h + 1][j], x2 = acc[4 * h + 2][j],
            x3 = acc[4 * h + 3][j];
          asm volatile("" : "+v"(x0), "+v"(x1), "+v"(x2), "+v"(x3));  // keeps acc in registers
          *reinterpret_cast<V*>(p + q * 256) = V{x0, x1, x2, x3};
        }
      } else {
#pragma unroll
        for (int q = 0; q < 4; q++)
#pragma unroll
          for (int i = 0; i < 4; i++) res[q][i] = acc[4 * (q & 1) + i][2 * d + (q >> 1)];
      }
    }
    __syncthreads();
    if ((wave >> 1) == half) {
#pragma unroll
      for (int o = 0; o < 3; o++)
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const V v = *reinterpret_cast<const V*>(
              smem + ((((wave & 1) * 3 + o) * 4 + q) * 64 + lane) * 4);
#pragma unroll
          for (int i = 0; i < 4; i++) res[q][i] = Trop<T>::add(res[q][i], v[i]);
        }
    }
    if (half == 0) __syncthreads();
  }
}

}  // namespace

template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void
tbh_gemm_ksplit_kernel(const GemmSplit g) {
  using V = typename Quad<T>::V;
  using U = typename Quad<T>::U;
  __shared__ __align__(16) T smem[kGemmLds];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tx = (lane & 7) * 4, ty = (lane >> 3) * 4;
  uint32_t b = blockIdx.x;
  const int tm = b % g.tiles_m;
  b /= g.tiles_m;
  const int tn = b % g.tiles_n;
  b /= g.tiles_n;
  const int part = b % g.ksplit, t = b / g.ksplit;
  const int m0 = tm * kTile, n0 = tn * kTile;
  const int kb = part * g.kpart, ke = gemm_range_end(g, kb);
  const TBH_GLOBAL T* A = reinterpret_cast<const TBH_GLOBAL T*>(g.a) + t * g.sA;
  const TBH_GLOBAL T* B = reinterpret_cast<const TBH_GLOBAL T*>(g.b) + t * g.sB;
  T res[4][4];
  gemm64_tile<T, true>(A, B, g.M, g.N, g.K, g.lda, g.ldb, kb, ke, m0, n0, threadIdx.x, smem, res);
  // ksplit > 1: raw maxima to the workspace, dense M x N per (batch, part)
  const bool ws = g.ksplit > 1;
  const int64_t ld = ws ? g.M : g.ldc;
  TBH_GLOBAL T* C = ws ? reinterpret_cast<TBH_GLOBAL T*>(g.ws) +
                             ((int64_t)t * g.ksplit + part) * g.M * g.N
                       : reinterpret_cast<TBH_GLOBAL T*>(g.c) + t * g.sC;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const int n = n0 + tile_col(wave, ty) + (q >> 1), m = m0 + 32 * (q & 1) + tx;
    if (n >= g.N) continue;
    V v = V{res[q][0], res[q][1], res[q][2], res[q][3]};
    if (!ws)
      v = V{Trop<T>::canon(v.x), Trop<T>::canon(v.y), Trop<T>::canon(v.z), Trop<T>::canon(v.w)};
    TBH_GLOBAL T* p = C + n * ld + m;
    if (m + 4 <= g.M) {
      *reinterpret_cast<TBH_GLOBAL U*>(p) = v;
    } else {
      if (m < g.M) p[0] = v.x;
      if (m + 1 < g.M) p[1] = v.y;
      if (m + 2 < g.M) p[2] = v.z;
    }
  }
}

// Grouped: prefix[i] is the first tile of GEMM step i; a block walks tiles.
// Every extent is a power of two, M and N at least 64 (the planner's rule).
template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void tbh_gemm64_kernel(
    const GemmDesc* __restrict__ ops, const int64_t* __restrict__ prefix, int nops,
    int64_t total) {
  using V = typename Quad<T>::V;
  __shared__ __align__(16) T smem[kGemmLds];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int64_t tile = blockIdx.x; tile < total; tile += gridDim.x) {
    const int step = gemm_step((const TBH_CONST int64_t*)prefix, nops, tile);
    const KGemm d = (KGemm)(ops + step);
    const uint32_t w = gemm_lanes(d);
    // tiles along M, then N, then the batch, all powers of two
    uint32_t r = (uint32_t)(tile - ((const TBH_CONST int64_t*)prefix)[step]);
    const int M = d->M, N = d->N, K = d->K;
    const int tiles_m = d->tiles_m, tiles_n = d->tiles_n;
    const int tm = r & (tiles_m - 1);
    r >>= __builtin_ctz(tiles_m);
    const int tn = r & (tiles_n - 1);
    const int64_t t = r >> __builtin_ctz(tiles_n);
    const int m0 = tm * kTile, n0 = tn * kTile;
    const TBH_GLOBAL T* A =
        reinterpret_cast<const TBH_GLOBAL T*>(d->a) + t * d->sA;
    const TBH_GLOBAL T* B =
        reinterpret_cast<const TBH_GLOBAL T*>(d->b) + t * d->sB;
    TBH_GLOBAL T* C = reinterpret_cast<TBH_GLOBAL T*>(d->c);
    const int tid = opaque_tid();
    const int lane = tid & 63, tx = (lane & 7) * 4, ty = (lane >> 3) * 4;
    T res[4][4];
    gemm64_tile<T, false>(A, B, M, N, K, d->lda, d->ldb, 0, K, m0, n0, tid,
                          smem, res);
    auto quad = [&](int q) {
      return V{Trop<T>::canon(res[q][0]), Trop<T>::canon(res[q][1]), Trop<T>::canon(res[q][2]),
               Trop<T>::canon(res[q][3])};
    };
    const int nl = tile_col(wave, ty);
    const int scatter = d->scatter;
    if (scatter == 0) {
      C += t * d->sC;
      const int64_t ldc = d->ldc;
#pragma unroll
      for (int q = 0; q < 4; q++)
        *reinterpret_cast<TBH_GLOBAL V*>(C + (n0 + nl + (q >> 1)) * ldc + m0 + 32 * (q & 1) + tx) =
            quad(q);
    } else {
      const int ma = __builtin_ctz((uint32_t)M), nb = __builtin_ctz((uint32_t)N);
      C += gemm_offset(w, (uint32_t)m0 | (uint32_t)n0 << ma | (uint32_t)t << (ma + nb));
      if (scatter == 1) {
        // rows 0 and 1 at C positions 0 and 1: row quads are 16-byte runs
        uint32_t at = 0;
#pragma unroll
        for (int k = 2; k < 5; k++) at |= (((uint32_t)tx >> k) & 1) << gemm_pos(w, k);
#pragma unroll
        for (int k = 1; k < 6; k++) at |= (((uint32_t)nl >> k) & 1) << gemm_pos(w, ma + k);
        const uint32_t rh = 1u << gemm_pos(w, 5), c1 = 1u << gemm_pos(w, ma);
#pragma unroll
        for (int q = 0; q < 4; q++)
          *reinterpret_cast<TBH_GLOBAL V*>(C + (at | ((q & 1) ? rh : 0) | ((q >> 1) ? c1 : 0))) =
              quad(q);
      } else {
        // the tile through LDS, read back in ascending C position
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const uint32_t n = nl + (q >> 1), m = 32 * (q & 1) + tx;
          *reinterpret_cast<V*>(smem + ((m ^ ((n & 15) << 2)) + (n << 6))) = quad(q);
        }
        __syncthreads();
        emit_staged<T>(C, smem, d->ep_n, 6, 15, w);
      }
    }
    __syncthreads();
  }
}

// One product in 32 x 32 tiles with the tile's whole operands in LDS (K <=
// KMAX).  Bound by one pass through memory latency and the launch: every load
// of a workgroup is in flight at once, by DMA without registers, where a slab
// loop waits for each slab and a K range per workgroup needs a second launch.
// Twice the LDS reads per MAC of the 64 x 64 tile, so only for products of few
// tiles per CU (resident_gemm).  The waves split K (8 of them at K <= 256, 16
// above: 512^3 21.0 with 8, 20.6 us; 1024 x 512 x 256 20.4, 22.9 with 16; 4 at
// K <= 64).  Float32 us per call, 64 x 64 tiles / these: 64^3 18.5 / 15.8,
// 64^2 x 512 25.2 / 19.7, 256^3 25.0 / 17.2, 512^3 27.3 / 20.6, 511 x 512 x
// 509 30.5 / 22.1.
template <typename T, int KMAX, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void tbh_gemm32_kernel(const GemmSplit g, bool quads) {
  using V = typename Quad<T>::V;
  using U = typename Quad<T>::U;
  typedef T W __attribute__((ext_vector_type(2)));
  constexpr int S = KMAX + 4;  // column stride of B in LDS
  __shared__ __align__(16) T As[32 * KMAX];
  __shared__ __align__(16) T Bs[32 * S];
  static_assert(32 * KMAX >= 2 * WAVES * 256, "the waves' maxima meet in A's and B's LDS");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  uint32_t b = blockIdx.x;
  const int tm = b % g.tiles_m;
  b /= g.tiles_m;
  const int tn = b % g.tiles_n, t = b / g.tiles_n;
  const int m0 = tm * 32, n0 = tn * 32, M = g.M, N = g.N, K = g.K;
  const TBH_GLOBAL T* A = reinterpret_cast<const TBH_GLOBAL T*>(g.a) + t * g.sA;
  const TBH_GLOBAL T* B = reinterpret_cast<const TBH_GLOBAL T*>(g.b) + t * g.sB;
  // A as [k][32 rows], B as [32 columns][k]; rows and columns past M and N
  // repeat the last ones (their outputs are not stored)
#if defined(__HIP_DEVICE_COMPILE__)  // the host pass does not know gfx950's 16-byte form
  if (quads) {
    const int m = m0 + (lane & 7) * 4, mc = m < M ? m : M - 4;
    for (int e = wave; e * 8 < K; e += WAVES) {
      const int k = e * 8 + (lane >> 3);
      if (k < K)
        __builtin_amdgcn_global_load_lds(A + k * g.lda + mc, (TBH_LDS T*)As + e * 256, 16, 0, 0);
    }
  } else {
    const int m = m0 + (lane & 31), mc = m < M ? m : M - 1;
    for (int e = wave; e * 2 < K; e += WAVES) {
      const int k = e * 2 + (lane >> 5);
      if (k < K)
        __builtin_amdgcn_global_load_lds(A + k * g.lda + mc, (TBH_LDS T*)As + e * 64, 4, 0, 0);
    }
  }
  for (int n = wave; n < 32; n += WAVES) {
    const int nc = n0 + n < N ? n0 + n : N - 1;
    const TBH_GLOBAL T* Bn = B + nc * g.ldb;
    if (quads && KMAX >= 256) {
      for (int k0 = 0; k0 < K; k0 += 256)
        if (k0 + lane * 4 < K)
          __builtin_amdgcn_global_load_lds(Bn + k0 + lane * 4, (TBH_LDS T*)Bs + n * S + k0, 16, 0,
                                           0);
    } else {
      for (int k0 = 0; k0 < K; k0 += 64)
        if (k0 + lane < K)
          __builtin_amdgcn_global_load_lds(Bn + k0 + lane, (TBH_LDS T*)Bs + n * S + k0, 4, 0, 0);
    }
  }
#endif
  __builtin_amdgcn_s_waitcnt(0);  // the DMA's writes (a barrier does not wait for them)
  __syncthreads();
  // rows tx .. tx + 3, columns ty + 8 j; an equal part of K per wave
  const int tx = (lane & 7) * 4, ty = lane >> 3;
  T acc[4][4];
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int i = 0; i < 4; i++) acc[j][i] = Trop<T>::zero();
  const int per = (K + 2 * WAVES - 1) / (2 * WAVES) * 2;
  const int kb = wave * per, ke = K < kb + per ? K : kb + per;
  const T* Ap = As + tx;
  const T* Bp = Bs + ty * S;
  int k = kb;
#pragma unroll 4
  for (; k + 1 < ke; k += 2) {
    const V a0 = *reinterpret_cast<const V*>(Ap + k * 32);
    const V a1 = *reinterpret_cast<const V*>(Ap + k * 32 + 32);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const W w = *reinterpret_cast<const W*>(Bp + 8 * j * S + k);
#pragma unroll
      for (int i = 0; i < 4; i++)
        acc[j][i] = max3(acc[j][i], Trop<T>::mul(a0[i], w.x), Trop<T>::mul(a1[i], w.y));
    }
  }
  if (k < ke) {
    const V a0 = *reinterpret_cast<const V*>(Ap + k * 32);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const T w = Bp[8 * j * S + k];
#pragma unroll
      for (int i = 0; i < 4; i++) acc[j][i] = Trop<T>::add(acc[j][i], Trop<T>::mul(a0[i], w));
    }
  }
  __syncthreads();
  // the waves' maxima meet: wave w < 4 ends with column ty + 8 w.  Columns 0
  // and 1 go to A's LDS, 2 and 3 to B's
#pragma unroll
  for (int j = 0; j < 4; j++)
    *reinterpret_cast<V*>((j < 2 ? As : Bs) + (((j & 1) * WAVES + wave) * 64 + lane) * 4) =
        V{acc[j][0], acc[j][1], acc[j][2], acc[j][3]};
  __syncthreads();
  if (wave >= 4) return;
  const T* red = (wave < 2 ? As : Bs) + (wave & 1) * WAVES * 256;
  V v = *reinterpret_cast<const V*>(red + lane * 4);
#pragma unroll
  for (int o = 1; o < WAVES; o++) {
    const V x = *reinterpret_cast<const V*>(red + (o * 64 + lane) * 4);
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = Trop<T>::add(v[i], x[i]);
  }
#pragma unroll
  for (int i = 0; i < 4; i++) v[i] = Trop<T>::canon(v[i]);
  const int n = n0 + ty + 8 * wave, m = m0 + tx;
  if (n >= N) return;
  TBH_GLOBAL T* p = reinterpret_cast<TBH_GLOBAL T*>(g.c) + t * g.sC + n * g.ldc + m;
  if (m + 4 <= M) {
    *reinterpret_cast<TBH_GLOBAL U*>(p) = v;
  } else {
    if (m < M) p[0] = v.x;
    if (m + 1 < M) p[1] = v.y;
    if (m + 2 < M) p[2] = v.z;
  }
}

// C = the maximum over the K ranges' workspaces, one thread per four outputs
// of a column.
template <typename T>
__global__ __launch_bounds__(256) void tbh_gemm_reduce_kernel(const GemmSplit g) {
  using V = typename Quad<T>::V;
  using U = typename Quad<T>::U;
  const int64_t mq = (g.M + 3) / 4;
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= mq * g.N * g.batch) return;
  const int64_t m = i % mq * 4, n = i / mq % g.N, t = i / mq / g.N;
  const int64_t mn = (int64_t)g.M * g.N;
  // (M >= 4: a quad past M is the column's last four rows instead)
  const int64_t mc = m + 4 <= g.M ? m : g.M - 4;
  const TBH_GLOBAL T* w = reinterpret_cast<const TBH_GLOBAL T*>(g.ws) + t * g.ksplit * mn +
                          n * g.M + mc;
  V acc = *reinterpret_cast<const TBH_GLOBAL U*>(w);
  for (int p = 1; p < g.ksplit; p++) {
    const V v = *reinterpret_cast<const TBH_GLOBAL U*>(w + p * mn);
    acc = V{Trop<T>::add(acc.x, v.x), Trop<T>::add(acc.y, v.y), Trop<T>::add(acc.z, v.z),
            Trop<T>::add(acc.w, v.w)};
  }
  acc = V{Trop<T>::canon(acc.x), Trop<T>::canon(acc.y), Trop<T>::canon(acc.z),
          Trop<T>::canon(acc.w)};
  *reinterpret_cast<TBH_GLOBAL U*>(reinterpret_cast<TBH_GLOBAL T*>(g.c) + t * g.sC + n * g.ldc +
                                   mc) = acc;
}

template <typename T>
static void gemm32(const GemmSplit& g, bool quads, int blocks, hipStream_t s) {
  if (g.K <= 64)
    tbh_gemm32_kernel<T, 64, 4><<<blocks, 256, 0, s>>>(g, quads);
  else if (g.K <= 128)
    tbh_gemm32_kernel<T, 128, 8><<<blocks, 512, 0, s>>>(g, quads);
  else if (g.K <= 256)
    tbh_gemm32_kernel<T, 256, 8><<<blocks, 512, 0, s>>>(g, quads);
  else
    tbh_gemm32_kernel<T, 512, 16><<<blocks, 1024, 0, s>>>(g, quads);
}

// quads: every column of A and B starts at a multiple of 16 bytes and M and K
// are multiples of 4.
hipError_t launch_gemm32(int dtype, const GemmSplit& g, bool quads, hipStream_t s) {
  const int blocks = g.tiles_m * g.tiles_n * g.batch;
  if (dtype == 0)
    gemm32<float>(g, quads, blocks, s);
  else
    gemm32<int32_t>(g, quads, blocks, s);
  return hipGetLastError();
}

hipError_t launch_gemm_ksplit(int dtype, const GemmSplit& g, hipStream_t s) {
  const int64_t blocks = (int64_t)g.tiles_m * g.tiles_n * g.ksplit * g.batch;
  const int64_t quads = (int64_t)((g.M + 3) / 4) * g.N * g.batch;
  if (dtype == 0)
    tbh_gemm_ksplit_kernel<float><<<(int)blocks, 256, 0, s>>>(g);
  else
    tbh_gemm_ksplit_kernel<int32_t><<<(int)blocks, 256, 0, s>>>(g);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || g.ksplit == 1) return e;
  const int rb = (int)((quads + 255) / 256);
  if (dtype == 0)
    tbh_gemm_reduce_kernel<float><<<rb, 256, 0, s>>>(g);
  else
    tbh_gemm_reduce_kernel<int32_t><<<rb, 256, 0, s>>>(g);
  return hipGetLastError();
}

hipError_t launch_gemm64(int dtype, const GemmDesc* ops, const int64_t* prefix, int nops,
                         int64_t total, int grid, hipStream_t s) {
  if (total <= 0) return hipSuccess;
  if (dtype == 0)
    tbh_gemm64_kernel<float><<<grid, 256, 0, s>>>(ops, prefix, nops, total);
  else
    tbh_gemm64_kernel<int32_t><<<grid, 256, 0, s>>>(ops, prefix, nops, total);
  return hipGetLastError();
}

int gemm64_blocks_per_cu(int dtype) {
  int n = 0;
  const void* k = dtype == 0 ? (const void*)tbh_gemm64_kernel<float>
                             : (const void*)tbh_gemm64_kernel<int32_t>;
  const hipError_t err = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, 256, 0);
  return err == hipSuccess && n > 0 ? n : 2;
}

}  // namespace tbh
