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

template <int CTRL, int ROWS>
__device__ __forceinline__ sel_key dpp_first(sel_key v) {  // (lanes without a source get 0, which is no key)
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)v, CTRL, ROWS, 0xf, false);
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(v >> 32), CTRL, ROWS, 0xf, false);
  const sel_key o = (sel_key)hi << 32 | lo;
  return o > v ? o : v;
}
// The first key of the wave, wave-uniform; 0: none.
__device__ __forceinline__ sel_key wave_first(sel_key v) {
  v = dpp_first<0x111, 0xf>(v);
  v = dpp_first<0x112, 0xf>(v);
  v = dpp_first<0x114, 0xf>(v);
  v = dpp_first<0x118, 0xf>(v);
  v = dpp_first<0x142, 0xa>(v);
  v = dpp_first<0x143, 0xc>(v);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)v, 63), hi = __builtin_amdgcn_readlane((int)(unsigned)(v >> 32), 63);
  return (sel_key)hi << 32 | lo;
}
// The k first of the wave's keys, N a lane, in order: lane r has the r-th, the others 0.
template <int N>
__device__ __forceinline__ sel_key wave_firsts(const sel_key (&keys)[N], int k, int lane) {
  sel_key mine = 0, last = ~(sel_key)0;
  for (int r = 0; r < k; ++r) {
    sel_key best = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) best = keys[i] < last && keys[i] > best ? keys[i] : best;
    last = wave_first(best);
    if (lane == r) mine = last;
  }
  return mine;
}

// x[lane] of the wave, lane uniform
__device__ __forceinline__ double wave_read(double x, int lane) {
  const unsigned long long b = __double_as_longlong(x);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)b, lane), hi = __builtin_amdgcn_readlane((unsigned)(b >> 32), lane);
  return __longlong_as_double((unsigned long long)hi << 32 | lo);
}

}  // namespace
}  // namespace wgpt

#endif
