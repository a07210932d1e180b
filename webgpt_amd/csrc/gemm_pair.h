// Products of a prompt's rows with a model's weights on the fp16 matrix cores, both as pairs of fp16 values (gemm_pair.hip).
#ifndef WGPT_GEMM_PAIR_H
#define WGPT_GEMM_PAIR_H

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace wgpt {

inline int pair_k16(int K) { return (K + 15) / 16; }
// Bytes of `rows` rows of K values as pairs. What lies beyond the last row and beyond K has to be finite (zeros, once).
inline size_t pair_rows_bytes(int rows, int K) { return (size_t)((rows + 31) / 32) * pair_k16(K) * 2048; }
// Bytes of a weight matrix [K, N] as pairs: columns take the place of rows.
inline size_t pair_weights_bytes(int K, int N) { return pair_rows_bytes(N, K); }

// How a product ends.
enum PairEnd {
  PAIR_PART,      // slice s of K leaves its sums, scaled, at part + s * M * N
  PAIR_QKV,       // + bias; columns below d to C, the others to their rows of the cache
  PAIR_HEADS,     // + bias; as operands of the attention to heads[] (attention_pair.h), keys and values to their rows of the cache too
  PAIR_RESIDUAL,  // + bias + resid to C
  PAIR_GELU,      // GELU(+ bias), scaled by `pscale`, as pairs to P
};
struct PairGemmArgs {
  int M, N, K;
  const void* A;        // pairs
  const void* W;        // pairs; int8: the order of launch_block_weights
  const float* cscale;  // [N]: what a column's sums are multiplied with
  const float* bias;
  int end;
  float* C;
  int ldc;
  const float* resid;   // [M, ldc], may alias C
  float *Kc, *Vc;
  int d, hs, ctx;
  void* heads[3];       // q, keys, values
  int head_tiles;       // AttnPairArgs::tiles
  float hscale[3], rhs; // the scales of q, keys, values; 1 / hs
  void* P;
  float pscale;
  float* part;
  int mt, nt, S, row_blocks;  // filled in by launch_gemm_pair
};
struct PairPlan {
  int kind, S;
};
// may_slice: the caller sums the slices in a pass over the rows that it makes anyway.
PairPlan plan_gemm_pair(int M, int N, int K, bool i8, bool may_slice);
constexpr int PAIR_MAX_SLICES = 4;
hipError_t launch_gemm_pair(const PairPlan& p, PairGemmArgs a, bool i8, hipStream_t s);

// LayerNorm of rows that a pass finishes first: x = the sum of S slices at `part` + bias + x (S = 0: x as it is), out = the
// LayerNorm of x times `scale`, as pairs. out null: no LayerNorm.
struct PairLnArgs {
  int M, d, S;
  const float *part, *bias;
  float* x;
  const float *gamma, *beta;
  float scale;
  void* out;
};
hipError_t launch_ln_pair(const PairLnArgs& a, hipStream_t s);

// A weight matrix W [K, N] as pairs, columns scaled by powers of two; cscale[n] gets the inverse of column n's. out, cscale and few
// [N] hold zeros. What the products cannot take counts in stats[0] (see gemm_pair.hip).
hipError_t launch_pair_weights(int K, int N, const float* W, void* out, float* cscale, int* few, unsigned* stats, hipStream_t s);
// cscale[n] = scale[n] / 127 of an int8 matrix; stats[0] as above.
hipError_t launch_pair_scales(int N, const float* scale, float* cscale, unsigned* stats, hipStream_t s);
// Largest absolute value that (LayerNorm with gamma and beta) . W + bias can have in each of `runs` equal runs of the columns of W
// [K, N] (int8: words of four columns and scales), and that the LayerNorm itself can have: as floats at bound[run] and *ln_bound.
// Infinite where a column of the run, or a channel of the LayerNorm, has a bound, but zero, below spread.least, or .ln, of the largest: one
// scale does not fit both. sums: pair_bounds_floats(K, N) of memory.
struct PairSpread {
  float ln, least[3];
};
size_t pair_bounds_floats(int K, int N);
hipError_t launch_pair_bounds(int K, int N, int runs, PairSpread spread, const float* W, const int32_t* Wq, const float* wscale, const float* bias,
                              const float* gamma, const float* beta, float* sums, float* bound, float* ln_bound, hipStream_t s);
// cscale[n] *= factor (a power of two)
hipError_t launch_pair_rescale(int N, float factor, float* cscale, hipStream_t s);

}  // namespace wgpt

#endif
