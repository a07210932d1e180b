// Device code: an fp32 value as the sum of three bf16 values (exact from 2^-110 on), the operands of gemm_split.hip and attention_split.hip.
#ifndef WGPT_SPLIT_BF16_H
#define WGPT_SPLIT_BF16_H

#include <hip/hip_runtime.h>

namespace wgpt {
namespace {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));

// Two floats as bf16 pairs (round to nearest even): the first in bits 0-15.
__device__ __forceinline__ unsigned bf16_pair(float a, float b) {
  const f32x2 v = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

// x = hi + mid + lo exactly for |x| >= 2^-110 (8 + 8 + 8 significand bits, each remainder rounded to nearest and
// representable; below, lo falls under the smallest bf16 subnormal, 2^-133, and the sum is off by 2^-134 at most), the
// decomposition of Henry, Tang and Heinecke, "Leveraging the bfloat16 artificial intelligence datatype for
// higher-precision computations" (2019).
__device__ __forceinline__ void split_pair(float a, float b, unsigned& hi, unsigned& mid, unsigned& lo) {
  hi = bf16_pair(a, b);
  const float ra = a - __builtin_bit_cast(float, hi << 16), rb = b - __builtin_bit_cast(float, hi & 0xffff0000u);
  mid = bf16_pair(ra, rb);
  lo = bf16_pair(ra - __builtin_bit_cast(float, mid << 16), rb - __builtin_bit_cast(float, mid & 0xffff0000u));
}

struct Split8 {  // eight consecutive k of one row or column
  u32x4 hi, mid, lo;
};
__device__ __forceinline__ Split8 split8(const f32x4& a, const f32x4& b) {
  Split8 r;
  unsigned h[4], m[4], l[4];
  split_pair(a[0], a[1], h[0], m[0], l[0]);
  split_pair(a[2], a[3], h[1], m[1], l[1]);
  split_pair(b[0], b[1], h[2], m[2], l[2]);
  split_pair(b[2], b[3], h[3], m[3], l[3]);
  r.hi = u32x4{h[0], h[1], h[2], h[3]};
  r.mid = u32x4{m[0], m[1], m[2], m[3]};
  r.lo = u32x4{l[0], l[1], l[2], l[3]};
  return r;
}

}  // namespace
}  // namespace wgpt

#endif
