// Causal attention of a longer prompt (AttentionBlock: formatQ, fusedWeights, softmax and attentionValues of
// instructions.js:1129-1212) on the fp16 matrix cores, between two products of gemm_pair.hip, for head sizes of 8, 16, .. 128.
//
// q, keys and values are pairs of fp16 values (pair_f16.h) that the product in front has left in the order of the operands, so
// that one load of a wave is 1 KB and nothing is split, moved or transposed here; three of the four partial products are taken.
// Scales are those of bounds that the weights give (gemm_pair.hip), for q and keys one each: a score is a sum times a constant.
// A key that is no number has scores that are none, its value is stored as zero, and so it reaches the queries that see it and
// no others. Weights of a softmax, at most 1, are taken 2^15 times (their sum too), values as they come.
// Everything is computed transposed, S^T = K Q^T and O^T = V^T P^T: an accumulator holds 16 keys of ONE query per lane, so the
// softmax needs one exchange between lanes and the weights are where the second product wants them. A workgroup owns 32
// queries of a head, its waves share the keys in runs of 32-key tiles and are merged at the end, into pairs for c_proj.
//
// What bounds it is the chain of one workgroup and the vector instructions of the softmax: a tile is 24 matrix instructions (of
// 32 cycles) at head size 64, and 16 vector instructions per weight. Against attention_split.hip with its pass over the operands, or
// fp32 matrix instructions below 700 rows, us at head size 64: 943 rows of 12 heads 30.6 -> 13.4, 512 of 16 17.3 -> 7.5, 300 of 25
// 14.7 -> 7.4; the product in front takes 2 us more for the operands. Logits are closer to 64-bit arithmetic: 117M 943 tokens
// 4.3e-7 (4.4e-7 with the other attention), 345M 512 5.4e-7, and so at all other shapes measured.
#include "attention_pair.h"

#include <cmath>

#include "exp_neg.h"
#include "pair_f16.h"

namespace wgpt {
namespace {

constexpr int APQ = PAIR_ATTN_ROWS;  // queries per workgroup, keys per tile
constexpr int AP_MERGE = APQ + 1;    // row stride of a wave's O^T[dim][query] in the merge
constexpr float AP_UP = 0x1p15f;

__device__ __forceinline__ f32x16 mfma(const u32x4& p, const u32x4& q, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, p), __builtin_bit_cast(f16x8, q), c, 0, 0, 0);
}
// the products of a run of steps, smallest first
template <int N>
__device__ __forceinline__ f32x16 pair_mfma(const u32x4 (*w)[2], const u32x4 (*x)[2]) {
  f32x16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
  for (int s = 0; s < N; ++s) acc = mfma(w[s][1], x[s][0], acc);
#pragma unroll
  for (int s = 0; s < N; ++s) acc = mfma(w[s][0], x[s][1], acc);
#pragma unroll
  for (int s = 0; s < N; ++s) acc = mfma(w[s][0], x[s][0], acc);
  return acc;
}

// DB: blocks of 32 dimensions that hold a head. Registers: the operands of a block of queries and of a tile's keys and values (16
// DB each), O (16 DB), the tile's part of it and the scores; from three blocks on a wave needs more than half a SIMD's, so
// four waves fill the compute unit.
template <int DB, int NWV>
__global__ __launch_bounds__(NWV * 64, DB < 3 ? 2 : 1) void attention_pair_kernel(AttnPairArgs a) {
  constexpr int KS = 2 * DB, DIMS = 32 * DB, WAVE_FLOATS = DIMS * AP_MERGE + 2 * APQ;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  // the longest rows of keys first; the heads go round, so that an XCD sees as few of them as 8 and their number allow
  const int item = (int)blockIdx.x, h = item % a.H, qb = a.blocks - 1 - item / a.H;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l32 = lane & 31, hh = lane >> 5;
  const int nt = qb + 1, tb = nt * wave / NWV, te = nt * (wave + 1) / NWV;
  const size_t head = (size_t)h * a.tiles;
  const auto fetch = [&](u32x4 (&f)[KS][2], const void* base, int t) {
    const u32x4* src = static_cast<const u32x4*>(base) + (head + t) * (KS * 128) + lane;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int p = 0; p < 2; ++p) f[s][p] = src[(s * 2 + p) * 64];
  };
  f32x16 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
  float m = -INFINITY, lsum = 0.f;
  if (tb < te) {
    u32x4 qf[KS][2], kf[KS][2], vf[KS][2];
    fetch(kf, a.k, tb);
    fetch(qf, a.q, qb);
    for (int t = tb; t < te; ++t) {
      fetch(vf, a.v, t);
      f32x16 sc = pair_mfma<KS>(kf, qf);
      fetch(kf, a.k, t + 1 < te ? t + 1 : t);
      if (t == qb) {  // keys that not all queries see: key (r / 4) * 8 + hh * 4 + r % 4 of query l32
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[r] = (r >> 2) * 8 + hh * 4 + (r & 3) <= l32 ? sc[r] : -INFINITY;
      }
      float top = sc[0];
#pragma unroll
      for (int r = 1; r < 16; ++r) top = fmaxf(top, sc[r]);
      top = fmaxf(top, __shfl_xor(top, 32));
      const float mnew = fmaxf(m, top * a.scale);  // (finite: a query sees a key of every tile)
      const float corr = m > -INFINITY ? exp_neg(m - mnew) : 0.f;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float w = exp_neg(fmaf(sc[r], a.scale, -mnew), AP_UP);
        sc[r] = sc[r] == -INFINITY ? 0.f : w;
      }
      float psum = 0.f;
#pragma unroll
      for (int r = 0; r < 16; r += 4) psum += (sc[r] + sc[r + 1]) + (sc[r + 2] + sc[r + 3]);
      lsum = lsum * corr + psum;
      m = mnew;
      u32x4 pf[2][2];
#pragma unroll
      for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          unsigned hi, lo;
          pair_f16(sc[8 * s + 2 * i], sc[8 * s + 2 * i + 1], hi, lo);
          pf[s][0][i] = hi, pf[s][1][i] = lo;
        }
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        const f32x16 part = pair_mfma<2>(vf + 2 * b, pf);
#pragma unroll
        for (int r = 0; r < 16; ++r) o[b][r] = fmaf(o[b][r], corr, part[r]);
      }
    }
    lsum += __shfl_xor(lsum, 32);  // the two halves of a column saw disjoint keys, the same maximum
  }

  float* Om = lds + wave * WAVE_FLOATS;  // [DIMS][AP_MERGE], then maxima and sums of the 32 queries
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) Om[(b * 32 + (r >> 2) * 8 + hh * 4 + (r & 3)) * AP_MERGE + l32] = o[b][r];
  if (hh == 0) {
    Om[DIMS * AP_MERGE + l32] = m;
    Om[DIMS * AP_MERGE + APQ + l32] = lsum;
  }
  __syncthreads();
  const int qi = tid & 31, row = qb * APQ + qi;
  float f[NWV], M = -INFINITY, den = 0.f;
#pragma unroll
  for (int w = 0; w < NWV; ++w) {
    f[w] = lds[w * WAVE_FLOATS + DIMS * AP_MERGE + qi];
    M = fmaxf(M, f[w]);
  }
#pragma unroll
  for (int w = 0; w < NWV; ++w) {
    f[w] = f[w] > -INFINITY ? exp_neg(f[w] - M) : 0.f;
    den += lds[w * WAVE_FLOATS + DIMS * AP_MERGE + APQ + qi] * f[w];
  }
  if (row >= a.T) return;
  for (int dq = tid >> 5; 4 * dq < a.hs; dq += NWV * 2) {  // four dimensions of a query
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NWV; ++w)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] += lds[w * WAVE_FLOATS + (4 * dq + e) * AP_MERGE + qi] * f[w];
    unsigned hi[2], lo[2];
    pair_f16(v[0] / den, v[1] / den, hi[0], lo[0]);
    pair_f16(v[2] / den, v[3] / den, hi[1], lo[1]);
    const int k = h * a.hs + 4 * dq;
    u32x2* to = static_cast<u32x2*>(a.out) + 2 * pair_unit(row, k, a.K16) + ((k >> 2) & 1);
    to[0] = u32x2{hi[0], hi[1]};
    to[128] = u32x2{lo[0], lo[1]};
  }
}

template <int DB, int NWV>
hipError_t launch_waves(const AttnPairArgs& a, hipStream_t s) {
  constexpr size_t lds = sizeof(float) * NWV * (32 * DB * AP_MERGE + 2 * APQ);
  static bool enabled = false;  // dynamic LDS size already raised
  if (lds > 64 * 1024 && !enabled) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_pair_kernel<DB, NWV>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    enabled = true;
  }
  attention_pair_kernel<DB, NWV><<<(unsigned)(a.H * a.blocks), NWV * 64, lds, s>>>(a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_attention_pair(AttnPairArgs a, hipStream_t s) {
  a.blocks = pair_attn_tiles(a.T);
  if (a.T < 1 || a.tiles < a.blocks || !pair_attn_takes(a.hs) || (long)a.H * a.blocks > 0x7fffffffL) return hipErrorInvalidValue;
  // Eight waves to a workgroup halve the chain of the longest one, four (two workgroups to a compute unit) merge less. Head size 64,
  // us with eight and four: 300 rows of 25 heads 8.2 and 7.4, 512 of 16 7.6 and 7.5, 943 of 12 13.4 and 13.5.
  const bool many = a.blocks > 16;
  switch ((a.hs + 31) / 32) {
    case 1: return many ? launch_waves<1, 8>(a, s) : launch_waves<1, 4>(a, s);
    case 2: return many ? launch_waves<2, 8>(a, s) : launch_waves<2, 4>(a, s);
    case 3: return launch_waves<3, 4>(a, s);
    default: return launch_waves<4, 4>(a, s);
  }
}

}  // namespace wgpt
