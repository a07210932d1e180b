// Attention of a longer prompt on pairs of fp16 values (attention_pair.hip).
#ifndef WGPT_ATTENTION_PAIR_H
#define WGPT_ATTENTION_PAIR_H

#include <hip/hip_runtime.h>

#include <cstddef>

namespace wgpt {

constexpr int PAIR_ATTN_ROWS = 32;      // queries of a block, keys of a tile
inline bool pair_attn_takes(int hs) { return hs % 8 == 0 && hs <= 128; }

__host__ __device__ inline int pair_attn_steps(int hs) { return 2 * ((hs + 31) / 32); }
// Bytes of the operands of up to T rows of H heads of q, keys or values: [H][block or tile][steps][2 parts][64 lanes] units of 16
// bytes, the eight values that the lane supplies to the step. q and keys: row lane % 32, dimensions 16 step + 8 (lane / 32) ..;
// values: dimension 32 (step / 2) + lane % 32, and of the sixteen keys of step % 2 the eight 4 (lane / 32) .. + 3 and + 8 .. + 11.
// Dimensions beyond the head size are zeros (once); rows beyond the last of its block or tile hold anything, values of them zeros.
inline int pair_attn_tiles(int T) { return (T + PAIR_ATTN_ROWS - 1) / PAIR_ATTN_ROWS; }
inline size_t pair_attn_bytes(int T, int H, int hs) {
  return (size_t)H * pair_attn_tiles(T) * pair_attn_steps(hs) * 2048;
}

struct AttnPairArgs {
  int T, H, hs, tiles;      // tiles: of a head in the operands, at least those of T rows, and the same for every T
  const void *q, *k, *v;
  float scale;              // of a score, the operands' scales taken out
  void* out;                // pairs of rows (pair_f16.h), H * hs wide, with the values' scale
  int K16;
  int blocks;               // of queries; filled in by launch_attention_pair
};
hipError_t launch_attention_pair(AttnPairArgs a, hipStream_t s);

}  // namespace wgpt

#endif
