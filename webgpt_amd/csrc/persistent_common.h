// Device helpers that the persistent kernels of any geometry share (prefill_persistent.hip, decode_generic.hip).
#ifndef WGPT_PERSISTENT_COMMON_H
#define WGPT_PERSISTENT_COMMON_H

#include <hip/hip_runtime.h>

#include "split_bf16.h"

namespace wgpt {
namespace {

constexpr int OUT = (int)0x80000000;  // a byte offset beyond every buffer: such a load returns zeros and moves nothing
constexpr int SC1 = 16;               // cache policy of device-scope loads

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (unsigned)bytes, 0x00020000);
}
template <int AUX>
__device__ __forceinline__ f32x4 load4(__amdgpu_buffer_rsrc_t b, int o, int so = 0) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b, o, so, AUX));
}
__device__ __forceinline__ unsigned ld_flag(const unsigned* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void st_agent(float* p, const f32x4& v) { asm volatile("global_store_dwordx4 %0, %1, off sc1" : : "v"(p), "v"(v) : "memory"); }
__device__ __forceinline__ void st_agent2(float* p, const u32x2& v) { asm volatile("global_store_dwordx2 %0, %1, off sc1" : : "v"(p), "v"(v) : "memory"); }

__device__ __forceinline__ void pair16(float v, float& a, float& b) {
  const unsigned u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
__device__ __forceinline__ void pair32(float v, float& a, float& b) {
  const unsigned u = __float_as_uint(v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  a = __uint_as_float(r[0]);
  b = __uint_as_float(r[1]);
}
// over the four lanes of equal lane & 15
__device__ __forceinline__ float quad_sum(float v) {
  float a, b;
  pair16(v, a, b);
  pair32(a + b, a, b);
  return a + b;
}
__device__ __forceinline__ float quad_max(float v) {
  float a, b;
  pair16(v, a, b);
  pair32(fmaxf(a, b), a, b);
  return fmaxf(a, b);
}
__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  return v;
}
__device__ __forceinline__ float gelu_ref(float x) {  // instructions.js:718-727
  const float x3 = x * x * x;
  const float cdf = 0.5f * (1.0f + tanhf(0.7978845608f * (x + 0.044715f * x3)));
  float r = x * cdf;
  r = x < -10.0f ? 0.0f : r;
  r = x > 10.0f ? x : r;
  return r;
}
// x / s with r = 1 / s at hand, rounded once (but for results under the smallest normal number), x finite. s infinite: 0, as the
// division gives it (the standard deviation of values from about 2^64 on; with r = 0 the finite number in its place changes nothing,
// where 0 * s would be no number).
__device__ __forceinline__ float quotient(float x, float s, float r) {
  const float q = x * r;
  return __builtin_fmaf(__builtin_fmaf(-q, fminf(s, 3.402823466e+38f), x), r, q);
}

// v, opaque to the optimiser: addresses built on the result are not kept in registers from one phase to the next.
__device__ __forceinline__ int opaque(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// n / m for 0 <= n < 2^20, r = 1 / m rounded
__device__ __forceinline__ int div_by(int n, int m, float r) {
  int q = (int)((float)n * r);
  q += (q + 1) * m <= n;
  q -= q * m > n;
  return q;
}

}  // namespace
}  // namespace wgpt

#endif
