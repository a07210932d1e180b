// The order in which GPT.generate selects tokens (selectTopK, globals.js:66-74), for the kernels that do it.
#ifndef WGPT_SELECT_KEY_H
#define WGPT_SELECT_KEY_H

#include <hip/hip_runtime.h>

#include <cmath>

namespace wgpt {
namespace {

// A logit and its index as one number whose order is the selection's: larger value first, lower index among equals
// (-0 and 0 are equal; NaN comes last).
typedef unsigned long long sel_key;
__device__ __forceinline__ unsigned order_bits(float v) {
  const unsigned b = __float_as_uint(v + 0.0f);
  return v != v ? 0u : (b & 0x80000000u ? ~b : b | 0x80000000u);
}
__device__ __forceinline__ sel_key make_key(float v, int i) { return (sel_key)order_bits(v) << 32 | (0xffffffffu - (unsigned)i); }
__device__ __forceinline__ float key_value(sel_key k) {
  const unsigned b = (unsigned)(k >> 32);
  return b == 0u ? NAN : __uint_as_float(b & 0x80000000u ? b & 0x7fffffffu : ~b);
}
__device__ __forceinline__ int key_index(sel_key k) { return (int)(0xffffffffu - (unsigned)k); }

// x[lane] of the wave, lane uniform
__device__ __forceinline__ double wave_read(double x, int lane) {
  const unsigned long long b = __double_as_longlong(x);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, lane), hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), lane);
  return __longlong_as_double((unsigned long long)hi << 32 | lo);
}

}  // namespace
}  // namespace wgpt

#endif
