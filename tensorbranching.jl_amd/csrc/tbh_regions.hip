// tbh_regions.hip -- branching tables of regions (tbh_region_tables), the
// table step of optimal_branches (src/branch.jl:79): for a region of a MIS
// problem and its boundary ("open") vertices, the reduced alpha tensor --
// per boundary configuration b the region's best weight with its boundary
// fixed to b, with the entries that a configuration using fewer boundary
// vertices matches or beats set to the tropical zero (GenericTensorNetworks'
// mis_compactify!) -- and, per surviving b, every region configuration that
// reaches it (the table rows of a BranchingTable).
//
// The alpha tensors are the SizeMax contraction of the region's network with
// its boundary fixed; they come in from the caller, or from tbh_region_alpha,
// which enumerates the region's 2^nv configurations (nv <= 24) as the table
// itself does.  A contraction per b (one scalar slice each: 2224 slices for 8
// regions of 14 vertices) took 45 ms, nearly all of it building and planning
// slices on the host; with the enumeration of the same regions, one launch,
// the tables take 1.6 ms:
//   tbh_alpha_kernel        a workgroup walks a run of a region's
//                           configurations, weighs the independent ones and
//                           keeps the best per boundary bits in LDS (up to
//                           2^12 of them, else straight in memory), merged by
//                           an integer atomic max on order-preserving keys;
//   tbh_compactify_kernel   one thread per (region, a): a survives unless a
//                           proper subset b of a has alpha[b] >= alpha[a];
//   tbh_configs_kernel      one thread per (region, x in {0,1}^nv): x is kept
//                           when it is independent in the region and its
//                           weight equals the pruned alpha of its boundary
//                           bits; pass 0 counts per (region, b), pass 1
//                           writes into each group's slots.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>

#include "tbh_runtime.hpp"

namespace tbh {

namespace {

constexpr int kRegionMaxNv = 24;    // 2^24 configurations per region at most
constexpr int kRegionMaxOpen = 16;  // 2^16 boundary configurations

struct RegionDesc {
  int32_t nv, nopen;
  uint32_t open;       // boundary vertices (bitmask over the region)
  int64_t x0;          // first configuration index of this region (prefix)
  int64_t a0;          // first alpha entry of this region (prefix)
  uint32_t adj[kRegionMaxNv];
  uint32_t wbits[kRegionMaxNv];  // dtype bit patterns (unit weights expanded)
};

// bits of x at the set positions of m, packed (x86 pext)
__device__ __forceinline__ uint32_t pext32(uint32_t x, uint32_t m) {
  uint32_t r = 0, k = 0;
  while (m) {
    const uint32_t low = m & (~m + 1u);
    if (x & low) r |= 1u << k;
    k++;
    m &= m - 1;
  }
  return r;
}

template <typename T>
__device__ __forceinline__ T tzero();
template <>
__device__ __forceinline__ float tzero<float>() { return -__builtin_inff(); }
template <>
__device__ __forceinline__ int32_t tzero<int32_t>() { return kI32NegInf; }

template <typename T>
__device__ __forceinline__ bool is_zero(T v) { return v <= tzero<T>(); }

// region of global index g: prefix[i] <= g < prefix[i + 1]
__device__ __forceinline__ int find_region(const int64_t* __restrict__ prefix, int n, int64_t g) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (prefix[mid] <= g)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// Order-preserving integer keys of the finite values of T (and the inverse);
// kNoKey: no configuration seen.
constexpr int32_t kNoKey = INT32_MIN;
__device__ __forceinline__ int32_t key_of(int32_t v) { return v; }
__device__ __forceinline__ int32_t key_of(float v) {
  const int32_t b = __builtin_bit_cast(int32_t, v);
  return b < 0 ? b ^ 0x7fffffff : b;
}
template <typename T>
__device__ __forceinline__ T of_key(int32_t k);
template <>
__device__ __forceinline__ int32_t of_key<int32_t>(int32_t k) { return k; }
template <>
__device__ __forceinline__ float of_key<float>(int32_t k) {
  return __builtin_bit_cast(float, k < 0 ? k ^ 0x7fffffff : k);
}

constexpr int kAlphaLdsBits = 12;    // boundary bits kept in LDS
constexpr int kAlphaRun = 1 << 12;   // configurations of one workgroup

__global__ __launch_bounds__(256) void tbh_alpha_fill_kernel(int64_t block0,
                                                              int32_t* __restrict__ keys,
                                                              int64_t total) {
  const int64_t g = (block0 + blockIdx.x) * blockDim.x + threadIdx.x;
  if (g < total) keys[g] = kNoKey;
}

// Workgroup w: configurations run0 .. of region r (bprefix: workgroups per
// region), in ascending vertex order of their weights' sum, as in
// tbh_configs_kernel.
template <typename T>
__global__ __launch_bounds__(256) void tbh_alpha_kernel(int64_t block0,
                                                        const RegionDesc* __restrict__ R,
                                                        const int64_t* __restrict__ bprefix,
                                                        int n, int32_t* __restrict__ keys) {
  __shared__ int32_t best[1 << kAlphaLdsBits];
  __shared__ uint32_t adj[kRegionMaxNv], wb[kRegionMaxNv];
  const int64_t block = block0 + blockIdx.x;
  const int r = find_region(bprefix, n, block);
  const RegionDesc& d = R[r];
  const int tid = threadIdx.x;
  const uint32_t open = d.open, entries = 1u << d.nopen;
  const bool lds = d.nopen <= kAlphaLdsBits;
  if (tid < kRegionMaxNv) {
    adj[tid] = d.adj[tid];
    wb[tid] = d.wbits[tid];
  }
  if (lds)
    for (uint32_t k = tid; k < entries; k += 256) best[k] = kNoKey;
  __syncthreads();
  const uint32_t total = 1u << d.nv;
  const uint32_t x0 = (uint32_t)(block - bprefix[r]) * kAlphaRun;
  const uint32_t x1 = x0 + kAlphaRun < total ? x0 + kAlphaRun : total;
  for (uint32_t x = x0 + tid; x < x1; x += 256) {
    T w = (T)0;
    bool ok = true;
    for (uint32_t m = x; m && ok; m &= m - 1) {
      const int v = __builtin_ctz(m);
      ok = (adj[v] & x) == 0;
      w += __builtin_bit_cast(T, wb[v]);
    }
    if (!ok) continue;
    const uint32_t e = pext32(x, open);
    if (lds)
      atomicMax(&best[e], key_of(w));
    else
      atomicMax(&keys[d.a0 + e], key_of(w));
  }
  if (!lds) return;
  __syncthreads();
  for (uint32_t k = tid; k < entries; k += 256)
    if (best[k] != kNoKey) atomicMax(&keys[d.a0 + k], best[k]);
}

// the keys as values, in place; no configuration: the tropical zero
template <typename T>
__global__ __launch_bounds__(256) void tbh_alpha_value_kernel(int64_t block0,
                                                              int32_t* __restrict__ keys,
                                                              int64_t total) {
  const int64_t g = (block0 + blockIdx.x) * blockDim.x + threadIdx.x;
  if (g >= total) return;
  const int32_t k = keys[g];
  reinterpret_cast<T*>(keys)[g] = k == kNoKey ? tzero<T>() : of_key<T>(k);
}

template <typename T>
__global__ __launch_bounds__(256) void tbh_compactify_kernel(int64_t block0,
                                                              const RegionDesc* __restrict__ R,
                                                              const int64_t* __restrict__ aprefix,
                                                              int n, int64_t total,
                                                              const T* __restrict__ in,
                                                              T* __restrict__ out) {
  const int64_t g = (block0 + blockIdx.x) * blockDim.x + threadIdx.x;
  if (g >= total) return;
  const int r = find_region(aprefix, n, g);
  const int64_t base = aprefix[r];
  const uint32_t a = (uint32_t)(g - base);
  const T va = in[g];
  bool dominated = false;
  // proper subsets b of a, from a - 1 down (b = (b - 1) & a)
  for (uint32_t b = (a - 1) & a; a != 0; b = (b - 1) & a) {
    if (in[base + b] >= va) {
      dominated = true;
      break;
    }
    if (b == 0) break;
  }
  out[g] = dominated ? tzero<T>() : va;
}

// PASS 0: counts[alpha entry] += 1 per matching configuration; PASS 1: writes
// x at slot[entry]++ within the entry's group (group offsets in `offs`).
template <typename T, int PASS>
__global__ __launch_bounds__(256) void tbh_configs_kernel(int64_t block0,
                                                           const RegionDesc* __restrict__ R,
                                                           const int64_t* __restrict__ xprefix,
                                                           int n, int64_t total,
                                                           const T* __restrict__ alpha,
                                                           uint32_t* __restrict__ counts,
                                                           const int64_t* __restrict__ offs,
                                                           uint32_t* __restrict__ configs) {
  const int64_t g = (block0 + blockIdx.x) * blockDim.x + threadIdx.x;
  if (g >= total) return;
  const int r = find_region(xprefix, n, g);
  const RegionDesc& d = R[r];
  const uint32_t x = (uint32_t)(g - xprefix[r]);
  T w = (T)0;
  for (uint32_t m = x; m; m &= m - 1) {
    const int v = __builtin_ctz(m);
    if (d.adj[v] & x) return;  // not independent
    T wv;
    __builtin_memcpy(&wv, &d.wbits[v], sizeof(T));
    w += wv;
  }
  const int64_t e = d.a0 + pext32(x, d.open);
  const T va = alpha[e];
  if (is_zero(va) || w != va) return;
  if (PASS == 0) {
    atomicAdd(&counts[e], 1u);
  } else {
    const uint32_t slot = atomicAdd(&counts[e], 1u);
    configs[offs[e] + slot] = x;
  }
}

// launch(block0, blocks) for runs of workgroups of 256 that a launch can hold:
// from 2^32 work-items on their number wraps, without an error.
template <class F>
hipError_t in_runs(int64_t blocks, F launch) {
  constexpr int64_t kMost = ((int64_t)1 << 24) - 1;
  for (int64_t b = 0; b < blocks; b += kMost) {
    launch(b, (int)std::min(blocks - b, kMost));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

template <typename T>
hipError_t launch_alpha(const RegionDesc* R, const int64_t* bprefix, int n, int64_t blocks,
                        int32_t* keys, int64_t total, hipStream_t s) {
  const int64_t ga = (total + 255) / 256;
  hipError_t e = in_runs(ga, [&](int64_t b, int grid) {
    tbh_alpha_fill_kernel<<<grid, 256, 0, s>>>(b, keys, total);
  });
  if (e == hipSuccess)
    e = in_runs(blocks, [&](int64_t b, int grid) {
      tbh_alpha_kernel<T><<<grid, 256, 0, s>>>(b, R, bprefix, n, keys);
    });
  if (e == hipSuccess)
    e = in_runs(ga, [&](int64_t b, int grid) {
      tbh_alpha_value_kernel<T><<<grid, 256, 0, s>>>(b, keys, total);
    });
  return e;
}

template <typename T>
hipError_t launch_compactify(const RegionDesc* R, const int64_t* aprefix, int n, int64_t total,
                             const void* in, void* out, hipStream_t s) {
  return in_runs((total + 255) / 256, [&](int64_t b, int grid) {
    tbh_compactify_kernel<T><<<grid, 256, 0, s>>>(b, R, aprefix, n, total, (const T*)in, (T*)out);
  });
}

template <typename T, int PASS>
hipError_t launch_configs(const RegionDesc* R, const int64_t* xprefix, int n, int64_t total,
                          const void* alpha, uint32_t* counts, const int64_t* offs,
                          uint32_t* configs, hipStream_t s) {
  return in_runs((total + 255) / 256, [&](int64_t b, int grid) {
    tbh_configs_kernel<T, PASS><<<grid, 256, 0, s>>>(b, R, xprefix, n, total, (const T*)alpha,
                                                     counts, offs, configs);
  });
}

}  // namespace
}  // namespace tbh

using namespace tbh;

// Checked descriptors of the regions and the prefixes of their
// configurations and alpha entries.
static int build_regions(tbh_dtype dtype, const tbh_region* regions, size_t n,
                         std::vector<RegionDesc>& desc, std::vector<int64_t>& xprefix,
                         std::vector<int64_t>& aprefix) {
  if (dtype != TBH_F32 && dtype != TBH_I32) {
    set_error("unknown dtype");
    return TBH_EINVAL;
  }
  desc.resize(n);
  xprefix.assign(n + 1, 0);
  aprefix.assign(n + 1, 0);
  for (size_t i = 0; i < n; i++) {
    const tbh_region& q = regions[i];
    if (q.nv < 0 || q.nv > kRegionMaxNv || (q.nv > 0 && !q.adj)) {
      set_error("region " + std::to_string(i) + ": needs 0 <= nv <= 24 and adjacency masks");
      return TBH_EINVAL;
    }
    const uint32_t all = q.nv == 32 ? ~0u : ((1u << q.nv) - 1u);
    if (q.open & ~all) {
      set_error("region " + std::to_string(i) + ": open vertex outside the region");
      return TBH_EINVAL;
    }
    RegionDesc& d = desc[i];
    std::memset(&d, 0, sizeof d);
    d.nv = q.nv;
    d.open = q.open;
    d.nopen = __builtin_popcount(q.open);
    if (d.nopen > kRegionMaxOpen) {
      set_error("region " + std::to_string(i) + ": more than 16 open vertices");
      return TBH_EINVAL;
    }
    for (int v = 0; v < q.nv; v++) {
      const uint32_t a = q.adj[v];
      if ((a & ~all) || ((a >> v) & 1u)) {
        set_error("region " + std::to_string(i) + ": adjacency of vertex " + std::to_string(v) +
                  " outside the region or a self loop");
        return TBH_EINVAL;
      }
      for (int u = 0; u < q.nv; u++)
        if (((a >> u) & 1u) != ((q.adj[u] >> v) & 1u)) {
          set_error("region " + std::to_string(i) + ": adjacency is not symmetric");
          return TBH_EINVAL;
        }
      d.adj[v] = a;
      if (!q.weights) {
        if (dtype == TBH_F32) {
          const float one = 1.0f;
          std::memcpy(&d.wbits[v], &one, 4);
        } else {
          d.wbits[v] = 1u;
        }
      } else {
        std::memcpy(&d.wbits[v], static_cast<const char*>(q.weights) + 4 * v, 4);
        if (dtype == TBH_F32) {
          float f;
          std::memcpy(&f, &d.wbits[v], 4);
          // configurations are matched by their weight: sums must be exact
          if (f != std::floor(f) || std::fabs(f) >= (float)(1 << 20)) {
            set_error("region " + std::to_string(i) +
                      ": Float32 table weights must be integers below 2^20");
            return TBH_EINVAL;
          }
        } else {
          const int32_t w = (int32_t)d.wbits[v];
          if (w <= -(1 << 24) || w >= (1 << 24)) {
            set_error("region " + std::to_string(i) + ": Int32 weights must satisfy |w| < 2^24");
            return TBH_EINVAL;
          }
        }
      }
    }
    d.x0 = xprefix[i];
    d.a0 = aprefix[i];
    xprefix[i + 1] = xprefix[i] + ((int64_t)1 << q.nv);
    aprefix[i + 1] = aprefix[i] + ((int64_t)1 << d.nopen);
  }
  return 0;
}

extern "C" int tbh_region_alpha(tbh_ctx* ctx, tbh_dtype dtype, const tbh_region* regions,
                                size_t n, void* alpha) {
  if (!ctx || (n && (!regions || !alpha))) {
    set_error("null argument");
    return TBH_EINVAL;
  }
  std::vector<RegionDesc> desc;
  std::vector<int64_t> xprefix, aprefix;
  int rc = build_regions(dtype, regions, n, desc, xprefix, aprefix);
  if (rc || n == 0) return rc;
  if (dtype == TBH_I32) {
    // the bound of an Int32 contraction, per boundary configuration: the
    // weights of its open vertices, summed, and the absolute weights of the
    // inner vertices it leaves stay below 2^28 together
    for (size_t i = 0; i < n; i++) {
      const RegionDesc& d = desc[i];
      double all = 0;
      for (int v = 0; v < d.nv; v++) all += std::fabs((double)(int32_t)d.wbits[v]);
      if (all < (double)(1 << 28)) continue;
      uint32_t b = 0;
      do {  // subsets of the open vertices
        double fixed = 0, inner = 0;
        uint32_t removed = 0;
        for (int v = 0; v < d.nv; v++)
          if ((b >> v) & 1u) {
            fixed += (double)(int32_t)d.wbits[v];
            removed |= d.adj[v];
          }
        for (int v = 0; v < d.nv; v++)
          if (!(((d.open | removed) >> v) & 1u)) inner += std::fabs((double)(int32_t)d.wbits[v]);
        if (!(removed & b) && std::fabs(fixed) + inner >= (double)(1 << 28)) {
          set_error("region " + std::to_string(i) +
                    ": Int32 regions need sum |w| < 2^28 for every boundary configuration");
          return TBH_EINVAL;
        }
        b = (b - d.open) & d.open;
      } while (b);
    }
  }
  std::vector<int64_t> bprefix(n + 1, 0);
  for (size_t i = 0; i < n; i++)
    bprefix[i + 1] = bprefix[i] + std::max<int64_t>(1, ((int64_t)1 << desc[i].nv) / kAlphaRun);
  if (bprefix[n] > INT32_MAX) {
    set_error("region tables: too many configurations in one call");
    return TBH_EINVAL;
  }
  const int64_t A = aprefix[n];
  std::lock_guard<std::mutex> g(ctx->mu);
  const size_t o_bp = (n * sizeof(RegionDesc) + 255) / 256 * 256;
  const size_t o_key = (o_bp + (n + 1) * 8 + 255) / 256 * 256;
  const int64_t doff = ctx->pool.alloc(o_key + 4 * A);
  if (doff < 0) {
    set_error("pool exhausted (region tables)");
    return TBH_ENOMEM;
  }
  char* dev = ctx->base + doff;
  int32_t* keys = (int32_t*)(dev + o_key);
  hipStream_t s = ctx->stream;
  const RegionDesc* dR = (const RegionDesc*)dev;
  const int64_t* dbp = (const int64_t*)(dev + o_bp);
  hipError_t e = hipSetDevice(ctx->device);
  if (e == hipSuccess)
    e = hipMemcpyAsync(dev, desc.data(), n * sizeof(RegionDesc), hipMemcpyHostToDevice, s);
  if (e == hipSuccess)
    e = hipMemcpyAsync(dev + o_bp, bprefix.data(), (n + 1) * 8, hipMemcpyHostToDevice, s);
  if (e == hipSuccess)
    e = dtype == TBH_F32 ? launch_alpha<float>(dR, dbp, (int)n, bprefix[n], keys, A, s)
                         : launch_alpha<int32_t>(dR, dbp, (int)n, bprefix[n], keys, A, s);
  if (e == hipSuccess) e = hipMemcpyAsync(alpha, keys, 4 * A, hipMemcpyDeviceToHost, s);
  const hipError_t es = hipStreamSynchronize(s);
  ctx->pool.free(doff);
  if (e != hipSuccess || es != hipSuccess) {
    set_error(std::string("region alpha: ") + hipGetErrorString(e != hipSuccess ? e : es));
    return TBH_EDEVICE;
  }
  return 0;
}

extern "C" int tbh_region_tables(tbh_ctx* ctx, tbh_dtype dtype, const tbh_region* regions,
                                 size_t n, void* alpha, size_t* group_ptr, uint32_t* configs,
                                 size_t cap, size_t* total) {
  if (!ctx || (n && (!regions || !alpha || !group_ptr || !total))) {
    set_error("null argument");
    return TBH_EINVAL;
  }
  if (total) *total = 0;
  std::vector<RegionDesc> desc;
  std::vector<int64_t> xprefix, aprefix;
  int rc0 = build_regions(dtype, regions, n, desc, xprefix, aprefix);
  if (rc0 || n == 0) return rc0;
  const int64_t X = xprefix[n], A = aprefix[n];
  std::lock_guard<std::mutex> g(ctx->mu);
  hipError_t e = hipSetDevice(ctx->device);
  if (e != hipSuccess) {
    set_error(std::string("hipSetDevice: ") + hipGetErrorString(e));
    return TBH_EDEVICE;
  }
  // device layout: descriptors, prefixes, alpha in / out, counts, offsets
  size_t off = 0;
  auto take = [&](size_t bytes) {
    const size_t o = (off + 255) / 256 * 256;
    off = o + bytes;
    return o;
  };
  const size_t o_desc = take(n * sizeof(RegionDesc));
  const size_t o_xp = take((n + 1) * sizeof(int64_t));
  const size_t o_ap = take((n + 1) * sizeof(int64_t));
  const size_t o_in = take(4 * A);
  const size_t o_out = take(4 * A);
  const size_t o_cnt = take(4 * A);
  const size_t o_offs = take(8 * (A + 1));
  const size_t head = off;
  const int64_t doff = ctx->pool.alloc(head);
  if (doff < 0) {
    set_error("pool exhausted (region tables)");
    return TBH_ENOMEM;
  }
  char* dev = ctx->base + doff;
  std::vector<int64_t> offs(A + 1, 0);
  std::vector<uint32_t> cnt(A, 0);
  int64_t cfg_off = -1;
  auto done = [&](int rc) {
    (void)hipStreamSynchronize(ctx->stream);
    ctx->pool.free(doff);
    if (cfg_off >= 0) ctx->pool.free(cfg_off);
    return rc;
  };
  auto fail = [&](hipError_t err, const char* what) {
    set_error(std::string("region tables (") + what + "): " + hipGetErrorString(err));
    return done(TBH_EDEVICE);
  };
  hipStream_t s = ctx->stream;
  const int G = 256;
  if ((e = hipMemcpyAsync(dev + o_desc, desc.data(), n * sizeof(RegionDesc),
                          hipMemcpyHostToDevice, s)) != hipSuccess ||
      (e = hipMemcpyAsync(dev + o_xp, xprefix.data(), (n + 1) * 8, hipMemcpyHostToDevice, s)) !=
          hipSuccess ||
      (e = hipMemcpyAsync(dev + o_ap, aprefix.data(), (n + 1) * 8, hipMemcpyHostToDevice, s)) !=
          hipSuccess ||
      (e = hipMemcpyAsync(dev + o_in, alpha, 4 * A, hipMemcpyHostToDevice, s)) != hipSuccess ||
      (e = hipMemsetAsync(dev + o_cnt, 0, 4 * A, s)) != hipSuccess)
    return fail(e, "upload");
  const RegionDesc* dR = (const RegionDesc*)(dev + o_desc);
  const int64_t* dxp = (const int64_t*)(dev + o_xp);
  const int64_t* dap = (const int64_t*)(dev + o_ap);
  uint32_t* dcnt = (uint32_t*)(dev + o_cnt);
  const int64_t* doffs = (const int64_t*)(dev + o_offs);
  if ((X + G - 1) / G > INT32_MAX) {
    set_error("region tables: too many configurations in one call");
    return done(TBH_EINVAL);
  }
  const char* dalpha = dev + o_out;
  e = dtype == TBH_F32 ? launch_compactify<float>(dR, dap, (int)n, A, dev + o_in, dev + o_out, s)
                       : launch_compactify<int32_t>(dR, dap, (int)n, A, dev + o_in, dev + o_out, s);
  if (e != hipSuccess) return fail(e, "compactify");
  e = dtype == TBH_F32
          ? launch_configs<float, 0>(dR, dxp, (int)n, X, dalpha, dcnt, doffs, nullptr, s)
          : launch_configs<int32_t, 0>(dR, dxp, (int)n, X, dalpha, dcnt, doffs, nullptr, s);
  if (e != hipSuccess) return fail(e, "count");
  if ((e = hipMemcpyAsync(alpha, dev + o_out, 4 * A, hipMemcpyDeviceToHost, s)) != hipSuccess ||
      (e = hipMemcpyAsync(cnt.data(), dcnt, 4 * A, hipMemcpyDeviceToHost, s)) != hipSuccess ||
      (e = hipStreamSynchronize(s)) != hipSuccess)
    return fail(e, "count readback");
  for (int64_t k = 0; k < A; k++) offs[k + 1] = offs[k] + cnt[k];
  const int64_t T = offs[A];
  *total = (size_t)T;
  for (size_t i = 0; i <= n; i++) group_ptr[i] = (size_t)offs[aprefix[i]];
  if (!configs || (size_t)T > cap) {
    if (configs) {
      set_error("region tables: " + std::to_string(T) + " configurations exceed the capacity " +
                std::to_string(cap));
      return done(TBH_ENOMEM);
    }
    return done(0);
  }
  if (T > 0) {
    cfg_off = ctx->pool.alloc((size_t)T * 4);
    if (cfg_off < 0) {
      set_error("pool exhausted (region table configurations)");
      return done(TBH_ENOMEM);
    }
    uint32_t* dcfg = (uint32_t*)(ctx->base + cfg_off);
    if ((e = hipMemcpyAsync(dev + o_offs, offs.data(), 8 * (A + 1), hipMemcpyHostToDevice, s)) !=
            hipSuccess ||
        (e = hipMemsetAsync(dcnt, 0, 4 * A, s)) != hipSuccess)
      return fail(e, "offsets");
    e = dtype == TBH_F32
            ? launch_configs<float, 1>(dR, dxp, (int)n, X, dalpha, dcnt, doffs, dcfg, s)
            : launch_configs<int32_t, 1>(dR, dxp, (int)n, X, dalpha, dcnt, doffs, dcfg, s);
    if (e != hipSuccess) return fail(e, "write");
    if ((e = hipMemcpyAsync(configs, dcfg, (size_t)T * 4, hipMemcpyDeviceToHost, s)) !=
            hipSuccess ||
        (e = hipStreamSynchronize(s)) != hipSuccess)
      return fail(e, "configurations readback");
    // each group's slots were taken in arrival order: ascending within groups
    for (int64_t k = 0; k < A; k++) std::sort(configs + offs[k], configs + offs[k + 1]);
  }
  return done(0);
}
