// tbh_gemm.hip -- K1b tbh_gemm_ksplit_kernel: one max-plus GEMM (the
// tbh_maxplus_gemm entry point) whose 128 x 128 tiles would not fill the
// GPU, or whose extents or alignment are odd.
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
// (512^3 19 us, 114 with K1's 16 tiles; 64^3 10.5 us, 18.6 with K1, about 6 us
// of each the events around it).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tbh_device.hpp"

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

}  // namespace

template <typename T>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void
tbh_gemm_ksplit_kernel(const GemmSplit g) {
  using V = typename Quad<T>::V;
  using U = typename Quad<T>::U;
  constexpr int NA = kSlab * kTile, NB = kSlab * kBRow;
  constexpr int NRED = 2 * 64 * 64;  // two waves' maxima
  constexpr int NLDS = 2 * (NA + NB) > NRED ? 2 * (NA + NB) : NRED;
  __shared__ __align__(16) T smem[NLDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  uint32_t b = blockIdx.x;
  const int tm = b % g.tiles_m;
  b /= g.tiles_m;
  const int tn = b % g.tiles_n;
  b /= g.tiles_n;
  const int part = b % g.ksplit, t = b / g.ksplit;
  const int m0 = tm * kTile, n0 = tn * kTile;
  const int kb = part * g.kpart, ke = g.K < kb + g.kpart ? g.K : kb + g.kpart;
  const TBH_GLOBAL T* A = reinterpret_cast<const TBH_GLOBAL T*>(g.a) + t * g.sA;
  const TBH_GLOBAL T* B = reinterpret_cast<const TBH_GLOBAL T*>(g.b) + t * g.sB;
  const T pz = pad_zero<T>();
  // this thread's quads: A rows am..am+3 of slab columns ak and ak + 16, B
  // slab rows bk..bk+3 of columns bn and bn + 32
  const int aq = (tid & 15) * 4, ak = tid >> 4;
  const int bk = (tid & 7) * 4, bn = tid >> 3;
  // rows past M read earlier ones, shifted so that valid rows stay in place
  const int am = m0 + aq < g.M - 4 ? m0 + aq : g.M - 4;
  const int as = m0 + aq - am < 4 ? m0 + aq - am : 0;
  const bool edge_m = m0 + kTile > g.M;
  const int bn0 = n0 + bn < g.N ? n0 + bn : g.N - 1;
  const int bn1 = n0 + bn + 32 < g.N ? n0 + bn + 32 : g.N - 1;
  V ra[2], rb[2];
  auto load = [&](int k0) {
    if (k0 + kSlab <= ke) {
#pragma unroll
      for (int e = 0; e < 2; e++)
        ra[e] = *reinterpret_cast<const TBH_GLOBAL U*>(A + (int64_t)(k0 + ak + 16 * e) * g.lda + am);
      rb[0] = *reinterpret_cast<const TBH_GLOBAL U*>(B + (int64_t)bn0 * g.ldb + k0 + bk);
      rb[1] = *reinterpret_cast<const TBH_GLOBAL U*>(B + (int64_t)bn1 * g.ldb + k0 + bk);
    } else {
      // the range's last slab: columns of A past it are the tropical zero,
      // and so are B's rows (a range ends at a multiple of 4, or at K)
#pragma unroll
      for (int e = 0; e < 2; e++) {
        const int k = k0 + ak + 16 * e;
        if (k < ke)
          ra[e] = *reinterpret_cast<const TBH_GLOBAL U*>(A + (int64_t)k * g.lda + am);
        else
          ra[e] = V{pz, pz, pz, pz};
      }
      const int k = k0 + bk, kc = k < g.K - 4 ? k : g.K - 4;
      if (k < ke) {
        rb[0] = *reinterpret_cast<const TBH_GLOBAL U*>(B + (int64_t)bn0 * g.ldb + kc);
        rb[1] = *reinterpret_cast<const TBH_GLOBAL U*>(B + (int64_t)bn1 * g.ldb + kc);
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
  T acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; i++)
#pragma unroll
    for (int j = 0; j < 8; j++) acc[i][j] = Trop<T>::zero();
  if (kb < ke) load(kb);
  if (kb < ke) store(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = kb; k0 < ke; k0 += kSlab) {
    const bool more = k0 + kSlab < ke;
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
  // waves 2 and 3 hand their maxima to waves 0 and 1; then wave 0 takes
  // columns j < 4 of both and wave 1 the others
  T* red = smem;
  auto put = [&](int slot, int j0, int j1) {
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (j >= j0 && j < j1)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          T x0 = acc[4 * h][j], x1 = acc[4 * h + 1][j], x2 = acc[4 * h + 2][j],
            x3 = acc[4 * h + 3][j];
          asm volatile("" : "+v"(x0), "+v"(x1), "+v"(x2), "+v"(x3));  // keeps acc in registers
          *reinterpret_cast<V*>(red + ((slot * 16 + 2 * j + h) * 64 + lane) * 4) = V{x0, x1, x2, x3};
        }
  };
  auto take = [&](int slot, int j0, int j1) {
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (j >= j0 && j < j1)
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const V v = *reinterpret_cast<const V*>(red + ((slot * 16 + 2 * j + h) * 64 + lane) * 4);
          acc[4 * h][j] = Trop<T>::add(acc[4 * h][j], v.x);
          acc[4 * h + 1][j] = Trop<T>::add(acc[4 * h + 1][j], v.y);
          acc[4 * h + 2][j] = Trop<T>::add(acc[4 * h + 2][j], v.z);
          acc[4 * h + 3][j] = Trop<T>::add(acc[4 * h + 3][j], v.w);
        }
  };
  if (wave >= 2) put(wave - 2, 0, 8);
  __syncthreads();
  if (wave < 2) take(wave, 0, 8);
  __syncthreads();
  if (wave == 0) put(0, 4, 8);
  if (wave == 1) put(1, 0, 4);
  __syncthreads();
  if (wave >= 2) return;
  if (wave == 0) take(1, 0, 4);
  if (wave == 1) take(0, 4, 8);
  // ksplit > 1: raw maxima to the workspace, dense M x N per (batch, part)
  const bool ws = g.ksplit > 1;
  const int64_t ld = ws ? g.M : g.ldc;
  TBH_GLOBAL T* C = ws ? reinterpret_cast<TBH_GLOBAL T*>(g.ws) +
                             ((int64_t)t * g.ksplit + part) * g.M * g.N
                       : reinterpret_cast<TBH_GLOBAL T*>(g.c) + t * g.sC;
  auto write = [&](int j0) {
#pragma unroll
    for (int jj = 0; jj < 4; jj++) {
      const int j = j0 + jj, n = n0 + (j0 ? 32 : 0) + ty + jj;
      if (n >= g.N) continue;
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int m = m0 + 32 * h + tx;
        V v = V{acc[4 * h][j], acc[4 * h + 1][j], acc[4 * h + 2][j], acc[4 * h + 3][j]};
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
  };
  if (wave == 0)
    write(0);
  else
    write(4);
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

}  // namespace tbh
