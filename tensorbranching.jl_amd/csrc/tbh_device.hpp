// tbh_device.hpp -- tropical arithmetic shared by the gfx950 kernels.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tbh_internal.hpp"

// Tensors are addressed in the global address space: their loads are
// global_load (counted by vmcnt only), not flat loads, which also count in
// lgkmcnt and so would make every wait for an LDS or scalar access wait for
// the data loads in flight too.
#define TBH_GLOBAL __attribute__((address_space(1)))
#define TBH_LDS __attribute__((address_space(3)))

namespace tbh {

template <typename T>
struct Trop;
template <>
struct Trop<float> {
  static __device__ __forceinline__ float zero() { return -__builtin_inff(); }
  static __device__ __forceinline__ float one() { return 0.0f; }
  static __device__ __forceinline__ float mul(float a, float b) { return a + b; }
  static __device__ __forceinline__ float add(float a, float b) { return __builtin_fmaxf(a, b); }
  static __device__ __forceinline__ float canon(float x) { return x; }
};
template <>
struct Trop<int32_t> {
  // accumulator start; sums of canonical values are >= -2^31
  static __device__ __forceinline__ int32_t zero() { return INT32_MIN; }
  static __device__ __forceinline__ int32_t one() { return 0; }
  static __device__ __forceinline__ int32_t mul(int32_t a, int32_t b) {
    return (int32_t)((uint32_t)a + (uint32_t)b);
  }
  static __device__ __forceinline__ int32_t add(int32_t a, int32_t b) { return a > b ? a : b; }
  static __device__ __forceinline__ int32_t canon(int32_t x) {
    return x < kI32NegThresh ? kI32NegInf : x;
  }
};
// max(a, b, c) as one v_max3 (the compiler forms it for only part of the
// GEMM's reductions).  Register operands only; inputs are never NaN.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
__device__ __forceinline__ int32_t max3(int32_t a, int32_t b, int32_t c) {
  int32_t r;
  asm("v_max3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

// zero used to pad GEMM operands (adds without overflow for Int32)
template <typename T>
__device__ __forceinline__ T pad_zero();
template <>
__device__ __forceinline__ float pad_zero<float>() { return -__builtin_inff(); }
template <>
__device__ __forceinline__ int32_t pad_zero<int32_t>() { return kI32NegInf; }

}  // namespace tbh
