// Device code: an fp32 value as the sum of two fp16 values, and the order in which rows of such pairs travel from the kernel
// that finishes them to the product that reads them (gemm_pair.hip).
#ifndef WGPT_PAIR_F16_H
#define WGPT_PAIR_F16_H

#include <hip/hip_runtime.h>

#include "split_bf16.h"

namespace wgpt {
namespace {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// x = hi + lo, |lo| <= 2^-11 |hi|: eleven significand bits each and the sign of lo, so that what is left out is at most 2^-23 of x
// (in a quarter of all values; nothing in the others) where lo is a normal number, |x| >= 2^-2; below, at most 2^-25 whatever x is.
// Values are scaled by powers of two so that the largest one of a matrix is near 2^15.
__device__ __forceinline__ void pair_f16(float a, float b, unsigned& hi, unsigned& lo) {
  const f16x2 h = __builtin_convertvector((f32x2{a, b}), f16x2);
  hi = __builtin_bit_cast(unsigned, h);
  lo = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a - (float)h[0], b - (float)h[1]}), f16x2));
}

// int8 values 2 q and 2 q + 1 of the four of a word as fp16: a byte b + 128 under 0x64 is 1024 + b + 128
__device__ __forceinline__ unsigned f16_of_bytes(unsigned v, int q) {
  const unsigned x = __builtin_amdgcn_perm(0x64646464u, v ^ 0x80808080u, q ? 0x04030402u : 0x04010400u);
  return __builtin_bit_cast(unsigned, __builtin_bit_cast(f16x2, x) - f16x2{(_Float16)1152.f, (_Float16)1152.f});
}

// Rows in runs of 16 k: unit ((row / 32 * K16 + k / 16) * 2 + part) * 64 + (k / 8 % 2) * 32 + row % 32 of 16 bytes holds eight
// consecutive k of one part of a row, so that an operand of a 32x32x16 matrix instruction is one load of 1 KB of a wave.
__host__ __device__ __forceinline__ size_t pair_unit(int row, int k, int K16) {
  return ((size_t)(row >> 5) * K16 + (k >> 4)) * 128 + ((k >> 3) & 1) * 32 + (row & 31);
}

// One value, scaled already, at (row, k): for kernels whose threads end with single elements.
__device__ __forceinline__ void put_pair(void* rows, int K16, int row, int k, float v) {
  _Float16* p = static_cast<_Float16*>(rows) + pair_unit(row, k, K16) * 8 + (k & 7);
  const _Float16 h = (_Float16)v;
  p[0] = h;
  p[512] = (_Float16)(v - (float)h);
}

}  // namespace
}  // namespace wgpt

#endif
