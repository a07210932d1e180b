// Matrix products of fp32 rows with fp32 or int8 weights on the bf16 matrix cores of gfx950 (gemm_split.hip).
#ifndef WGPT_GEMM_SPLIT_H
#define WGPT_GEMM_SPLIT_H

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace wgpt {

struct SplitGemmArgs {
  int M, N, K;
  const float* A;        // [M, lda]
  int lda;
  const void* W;         // [K, ldw]: floats, or words of four int8; or the order of launch_block_weights
  int ldw;
  bool blocked;
  const float* wscale;   // int8: per column
  const float* bias;     // may be null
  int epi;
  const float* resid;    // EPI_RESIDUAL: [M, ldc], may alias C
  float* C;              // [M, ldc]; with Kc only the columns below d are stored here
  int ldc;
  float *Kc, *Vc;        // null: no cache scatter (see KvAfter)
  int d, hs, ctx, pos0;
  float* part;           // not null: slice s of K leaves its sums, without bias and epilogue, at part + s * M * N
  int mt, nt, S;         // tiles along M and N, slices of K
};

// How a product is cut: which kernel, and into how many slices of K (1: the kernel finishes C itself).
struct SplitPlan {
  int kind, S;
};
// with_pass: a pass over the finished rows follows anyway (a LayerNorm), so that partial sums cost only their traffic.
SplitPlan plan_gemm_split(int M, int N, int K, bool i8, bool blocked, bool with_pass, bool may_slice);
// a.mt, a.nt and a.S are filled in from the plan. Bytes of A (M * lda floats) and W below 2^31.
hipError_t launch_gemm_split(const SplitPlan& p, SplitGemmArgs a, bool i8, hipStream_t s);

// Puts a matrix [K, N] of floats, or of int8 (four columns to a word), into the order that the products read with the fewest
// loads: [K / 4][N][4] floats or [K / 8][N][8] bytes, the same size. K a multiple of 8, N of 4; dst is not src.
hipError_t launch_block_weights(int K, int N, bool i8, const void* src, void* dst, hipStream_t s);

}  // namespace wgpt

#endif
