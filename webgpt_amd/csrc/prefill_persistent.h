// Host interface of the persistent prefill kernel: the forward of a short prompt in one launch.
#ifndef WGPT_PREFILL_PERSISTENT_H
#define WGPT_PREFILL_PERSISTENT_H

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace wgpt {

constexpr int PP_GRID = 256;      // workgroups: one per compute unit of an MI355X
constexpr int PP_THREADS = 512;
constexpr int PP_ROWS = 16;       // rows of a row group: a matrix instruction's
constexpr int PP_MAX_GROUPS = 8;  // a wave of the attention takes the keys of one row group
constexpr int PP_MAX_T = PP_ROWS * PP_MAX_GROUPS;
constexpr int PP_FLAGS = PP_MAX_GROUPS * PP_GRID + 64;  // words of PrefillArgs::flags, the launch's error word among them

// What the products are made of: fp32 values, int8 weights and rows of three bf16 values each, or rows (and fp32 weights) that are
// pairs of fp16 values as those of gemm_pair.hip.
// Pairs are for rows above PP_PAIR_ABOVE: logits of 6 layers of 512, 90 tokens, 2.8e-7 from 64-bit arithmetic with them against 2.7e-7; 8
// layers of 576, 100 tokens, 2.8e-7 against 2.9e-7.
constexpr int PP_PAIR_ABOVE = 512;
enum PrefillMode { PP_PLAIN_F32 = 0, PP_SPLIT_I8 = 1, PP_PAIR_F32 = 2, PP_PAIR_I8 = 3 };

// One layer's weights in the order of launch_block_weights (PP_PAIR_F32: of launch_pair_weights), and its small parameters
// (device pointers).
struct PrefillLayer {
  const void *wA, *wC, *wD, *wE;                            // c_attn, attention c_proj, c_fc, mlp c_proj
  // int8 column scales, or what the columns of pairs are multiplied with (null for plain fp32); biases
  const float *sA, *sC, *sD, *sE, *bA, *bC, *bD, *bE;
  const float *ln1g, *ln1b, *ln2g, *ln2b;
};
// Scales of the rows that its four products read, as pairs. (Apart from the pointers, which are a power of two of bytes without them: as part of
// them they cost the kernel on plain values, which has no use for them, up to 1 %: 6 layers of 384 columns, 5, 40 and 120 tokens, 159.3, 183.8
// and 194.8 us against 158.1, 181.7 and 193.3.)
struct PrefillScales {
  float A, C, D, E;
};

struct PrefillArgs {
  int T, L, H, hs, d, ctx, V;
  float scale;
  const int32_t* tok;  // [T], memory that the device can read
  const float *wte, *wpe, *lnf_g, *lnf_b;
  const PrefillLayer* layers;  // [L], device memory; behind them the PrefillScales [L]
  float* x;                     // [T, d]: the residual stream after the last layer
  // exchanged between workgroups, for prefill_rows(T) rows: queries [T, d]; the residual stream, the same behind the attention and
  // the attention's output (d floats a row), the hidden rows (4 d), in the order that their readers load
  float *q, *xe, *x1, *att, *h;
  float* kv;                    // [L][2][H][ctx][hs]: rows 0..T-1 are written
  float *logits, *host_logits;  // [V]: of the last row, the second in pinned host memory
  unsigned* flags;              // [PP_FLAGS], cleared once; epochs only grow (see prefill_epochs)
  unsigned ebase;               // last epoch of earlier launches
  unsigned spin_limit;
  int* host_err;                // pinned: left alone by a launch that has run to its end with sums that could all be split
  // filled in by launch_prefill_persistent
  int groups, per_xcd, cols;    // row groups; column groups of each XCD; columns groups in all
  int cpA, cpC, cpD;            // columns of a workgroup: q/k/v, the two projections, hidden rows
  int rows_per_wg;              // vocabulary rows
  float rcpA, rcpC, rcpD, rhs;  // reciprocals of the columns and of the head size
};

enum { PP_ERR_WAIT = 1, PP_ERR_SPLIT = 2 };  // *host_err: a bounded wait expired; sums that the split operands may have spoilt

inline int prefill_rows(int T) { return (T + PP_ROWS - 1) / PP_ROWS * PP_ROWS; }
// Floats of the exchange buffers q, xe, x1, att, h of such prompts, one behind the other.
inline size_t prefill_exchange_floats(int T, int d) { return (size_t)8 * prefill_rows(T) * d; }
inline unsigned prefill_epochs(int L) { return 5u * (unsigned)L + 1u; }
// The longest prompt that the kernel takes of such a model, 0: none (compute_units of the device at hand).
int prefill_persistent_rows(int d, int H, int hs, int V, bool i8, int compute_units);
hipError_t launch_prefill_persistent(PrefillArgs a, PrefillMode mode, hipStream_t s);

}  // namespace wgpt

#endif
