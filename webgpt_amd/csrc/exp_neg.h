// Device code: the exponential of the softmax in attention_split.hip and attention_pair.hip.
#ifndef WGPT_EXP_NEG_H
#define WGPT_EXP_NEG_H

#include <hip/hip_runtime.h>

namespace wgpt {
namespace {

// exp(x) for x <= 0 with the rounding of x * log2(e) made up for, times `up`: as exact as expf down to its smallest normal result
__device__ __forceinline__ float exp_neg(float x, float up = 1.f) {
  const float t = x * 1.44269504f;
  const float r = fmaf(x, 1.92596303e-8f, fmaf(x, 1.44269504f, -t));  // log2(e) = 1.44269502162933 + 1.92596303e-8
  const float e = __builtin_amdgcn_exp2f(t) * up;
  return fmaf(e, r * 0.693147181f, e);
}

}  // namespace
}  // namespace wgpt

#endif
