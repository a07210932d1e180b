// Causal attention of a prompt (AttentionBlock: formatQ, fusedWeights, softmax and attentionValues of
// instructions.js:1129-1212) on the bf16 matrix cores, for head sizes up to 128.
//
// Operands are split into three bf16 values each and the six largest partial products taken, as in gemm_split.hip: an error
// no larger than that of fp32 products at 2.7 times their rate. q, K and V are split once, by a pass in front
// (attention_operands), which also lays them out so that every operand of a matrix instruction is one load of 1 KB of
// neighbouring bytes per wave: no LDS, no transposition and no conversion in the loop over the keys, where only the weights
// are split. Everything is computed transposed, S^T = K Q^T and O^T = V^T P^T: an accumulator then holds 16 keys of ONE query
// per lane, so that the softmax needs one exchange between lanes and the weights are where the second product wants them.
// A workgroup owns 32 queries of a head, its waves share the keys in runs of 32-key tiles and are merged at the end.
// Bound by what a compute unit takes from L2 (12 KB per 32 keys at head size 64, read by every block of 32 queries).
#include <cmath>

#include "exp_neg.h"
#include "kernels.h"
#include "pair_f16.h"

namespace wgpt {
namespace {

constexpr int ASQ = 32;         // queries per workgroup, keys per tile
constexpr int AS_MERGE = ASQ + 1;  // row stride of a wave's O^T[dim][query] in the merge

struct AttnSplitArgs {
  int Tq, pos0, H, hs, nq, nt;  // nq, nt: blocks of 32 queries, tiles of 32 keys
  float scale;
  const float* q;
  int ldq;
  const float *Kc, *Vc;
  size_t hstride;
  int ldkv;
  float* out;
  int ldo;
  PairRows pairs;
  u32x4 *Q3, *K3, *V3;  // [H][block or tile][KS steps][3 parts][64 lanes]
};

__device__ __forceinline__ void put(const AttnSplitArgs& a, int row, int h, int dim, float v) {
  if (a.pairs.rows) put_pair(a.pairs.rows, a.pairs.K16, row, h * a.hs + dim, v * a.pairs.scale);
  else a.out[(size_t)row * a.ldo + (size_t)h * a.hs + dim] = v;
}

// Operands of one block of queries or tile of keys: unit (step, part, lane) of 16 bytes holds the eight values that the lane
// supplies to the step. q and K: row lane % 32, dimensions 16 step + 8 (lane / 32) ..; V: dimension 32 (step / 2) + lane % 32,
// and of the sixteen keys of step % 2 the eight that the accumulator of S^T leaves in this half of the wave.
// Values beyond the head size, the last query or the last key are zeros.
__global__ void attention_operands(AttnSplitArgs a) {
  const int lane = threadIdx.x & 63, step = threadIdx.x >> 6, steps = blockDim.x >> 6;
  const int h = blockIdx.y, r = lane & 31, half = lane >> 5, nkeys = a.pos0 + a.Tq;
  int t = blockIdx.x;
  f32x4 v[2];
  u32x4* dst;
  if (t < a.nq + a.nt) {
    const bool isq = t < a.nq;
    if (!isq) t -= a.nq;
    const int row = t * ASQ + r;
    const bool live = row < (isq ? a.Tq : nkeys);
    const float* p = isq ? a.q + (size_t)row * a.ldq + (size_t)h * a.hs : a.Kc + h * a.hstride + (size_t)row * a.ldkv;
    const int d0 = 16 * step + 8 * half;
#pragma unroll
    for (int i = 0; i < 2; ++i)
      v[i] = live && d0 + 4 * i < a.hs ? *reinterpret_cast<const f32x4*>(p + d0 + 4 * i) : f32x4{0.f, 0.f, 0.f, 0.f};
    dst = isq ? a.Q3 + (size_t)(h * a.nq + t) * steps * 192 : a.K3 + (size_t)(h * a.nt + t) * steps * 192;
  } else {
    t -= a.nq + a.nt;
    const int dim = 32 * (step >> 1) + r, k0 = t * ASQ + 16 * (step & 1) + 4 * half;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int key = k0 + 8 * (j >> 2) + (j & 3);
      v[j >> 2][j & 3] = dim < a.hs && key < nkeys ? a.Vc[h * a.hstride + (size_t)key * a.ldkv + dim] : 0.f;
    }
    dst = a.V3 + (size_t)(h * a.nt + t) * steps * 192;
  }
  const Split8 s = split8(v[0], v[1]);
  dst += step * 192 + lane;
  dst[0] = s.hi;
  dst[64] = s.mid;
  dst[128] = s.lo;
}

__device__ __forceinline__ f32x16 mfma(const u32x4& p, const u32x4& q, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, p), __builtin_bit_cast(bf16x8, q), c, 0, 0, 0);
}
// The product of the leading parts goes to its own sum: what the other five, 2^-8 of it and less, add up to meets it once
// per tile, and the sum of a tile is rounded three times instead of twelve.
__device__ __forceinline__ void split_mfma(const u32x4 (&w)[3], const u32x4 (&x)[3], f32x16& lead, f32x16& rest) {
  rest = mfma(w[2], x[0], rest);
  lead = mfma(w[0], x[0], lead);
  rest = mfma(w[0], x[2], rest);
  rest = mfma(w[1], x[1], rest);
  rest = mfma(w[1], x[0], rest);
  rest = mfma(w[0], x[1], rest);
}

// Sums or maxima of four values over the workgroup; sh: four floats per wave.
template <int NT, bool MAX>
__device__ __forceinline__ f32x4 over_workgroup(f32x4 v, f32x4* sh) {
  const auto with = [](const f32x4& x, const f32x4& y) {
    f32x4 r;
#pragma unroll
    for (int u = 0; u < 4; ++u) r[u] = MAX ? fmaxf(x[u], y[u]) : x[u] + y[u];
    return r;
  };
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = with(v, f32x4{__shfl_xor(v[0], off), __shfl_xor(v[1], off), __shfl_xor(v[2], off), __shfl_xor(v[3], off)});
  __syncthreads();  // (everyone has read what sh held)
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  v = sh[0];
#pragma unroll
  for (int w = 1; w < NT / 64; ++w) v = with(v, sh[w]);
  return v;
}

// The outputs of the queries q0 + (bits of `left`) with plain fp32 products, four at a time by the whole workgroup, over runs of
// AS_RUN keys: for operands that have no split (infinite ones, see gemm_split.hip), for NaN, and for values so small that their
// third part is lost (under 2^-110: outputs under 2^-60 are taken again, as sums are in gemm_split.hip). Weights are as small
// for keys whose scores are AS_FAR below the largest one, and exp_neg has none under 2^-126: queries with such keys have their
// outputs under 2^-20 taken again, zeros among them, which leaves out such weights on values of about 2^80 and more. Scores
// that are not numbers end it, as nothing else can come out. An attention block of 12 heads x 48 at 943 rows takes 325 us where every output is taken again (128 us where none is; 21.6 ms with a loop
// over the keys per output).
constexpr int AS_RUN = 1024;
constexpr float AS_FAR = 76.f;  // exp(-76) is 2^-109.6
template <int NT>
__device__ __forceinline__ void plain_rows(const AttnSplitArgs& a, int h, int q0, unsigned left, float* lds) {
  float* const scores = lds;  // [4][AS_RUN]
  f32x4* const red = reinterpret_cast<f32x4*>(lds + 4 * AS_RUN);
  f32x4 *const sh = red + NT, *const qs = sh + NT / 64;  // qs: [4][32]
  const int tid = threadIdx.x, n4 = a.hs >> 2;
  int lpk = 1;  // lanes to a row of V
  while (lpk < n4) lpk <<= 1;
  const int sub = tid & (lpk - 1), grp = tid / lpk, ngrp = NT / lpk;
  const bool act = sub < n4;
  const float* V = a.Vc + h * a.hstride + 4 * sub;
#pragma unroll 1
  while (left) {
    int row[4];
    f32x4 acc[4], m, l;
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // (fewer than four: the last one again)
      row[u] = left ? q0 + __builtin_ctz(left) : row[u > 0 ? u - 1 : 0];
      left &= left - 1;
      if (tid < n4) qs[u * 32 + tid] = *reinterpret_cast<const f32x4*>(a.q + (size_t)row[u] * a.ldq + (size_t)h * a.hs + 4 * tid);
      acc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      m[u] = -3.402823e+38f;
      l[u] = 0.f;
    }
    __syncthreads();
    const int nkeys = a.pos0 + row[3] + 1;
#pragma unroll 1
    for (int j0 = 0; j0 < nkeys; j0 += AS_RUN) {
      const int n = min(AS_RUN, nkeys - j0);
      // four lanes to a key, four keys to a lane at a time
      for (int j1 = tid >> 2; j1 < n + (tid >> 2); j1 += NT) {
        float dot[4][4];
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int u = 0; u < 4; ++u) dot[t][u] = 0.f;
#pragma unroll 1
        for (int c = tid & 3; c < n4; c += 4) {
          f32x4 y[4];
#pragma unroll
          for (int t = 0; t < 4; ++t) {
            const int j = j1 + t * (NT / 4);
            y[t] = *reinterpret_cast<const f32x4*>(a.Kc + h * a.hstride + (size_t)(j0 + (j < n ? j : n - 1)) * a.ldkv + 4 * c);
          }
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const f32x4 x = qs[u * 32 + c];
#pragma unroll
            for (int t = 0; t < 4; ++t) dot[t][u] += (x[0] * y[t][0] + x[1] * y[t][1]) + (x[2] * y[t][2] + x[3] * y[t][3]);
          }
        }
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            float s = dot[t][u];
            s += __shfl_xor(s, 1);
            s += __shfl_xor(s, 2);
            const int j = j1 + t * (NT / 4);
            if ((tid & 3) == u && j < n) scores[u * AS_RUN + j] = j0 + j <= a.pos0 + row[u] ? s * a.scale : -INFINITY;
          }
      }
      __syncthreads();
      f32x4 top = m, sum = {0.f, 0.f, 0.f, 0.f};
      for (int j = tid; j < n; j += NT)
#pragma unroll
        for (int u = 0; u < 4; ++u) top[u] = fmaxf(top[u], scores[u * AS_RUN + j]);
      top = over_workgroup<NT, true>(top, sh);
      for (int j = tid; j < n; j += NT)
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float e = expf(scores[u * AS_RUN + j] - top[u]);
          scores[u * AS_RUN + j] = e;
          sum[u] += e;
        }
      sum = over_workgroup<NT, false>(sum, sh);
      bool live = false;
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const float corr = expf(m[u] - top[u]);
        l[u] = l[u] * corr + sum[u];
        acc[u] *= corr;
        live = live || l[u] < INFINITY;
      }
      m = top;
      if (!live) break;
      if (act) {
#pragma unroll 4
        for (int j = grp; j < n; j += ngrp) {
          const f32x4 y = *reinterpret_cast<const f32x4*>(V + (size_t)(j0 + j) * a.ldkv);
#pragma unroll
          for (int u = 0; u < 4; ++u)
            if (j0 + j <= a.pos0 + row[u]) acc[u] += scores[u * AS_RUN + j] * y;
        }
      }
      __syncthreads();
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      red[tid] = acc[u];
      __syncthreads();
      if (tid < a.hs) {
        float o = 0.f;
        for (int g = 0; g < ngrp; ++g) o += red[g * lpk + (tid >> 2)][tid & 3];
        put(a, row[u], h, tid, l[u] < INFINITY ? o / l[u] : NAN);
      }
      __syncthreads();
    }
  }
}

// DB: blocks of 32 dimensions that hold a head. Registers: the operands of a tile's K and V (24 DB each), O (16 DB) and the
// sums; q fits beside them for DB = 1 only and waits in LDS otherwise. From three blocks on a wave needs more than half a
// SIMD's registers, so four waves fill the compute unit.
template <int DB, int NWV>
__global__ __launch_bounds__(NWV * 64, NWV / 4) void attention_split_kernel(AttnSplitArgs a) {
  constexpr int KS = 2 * DB, DIMS = 32 * DB, WAVE_FLOATS = DIMS * AS_MERGE + 3 * ASQ;
  constexpr bool QREG = DB == 1;
  static_assert(4 * AS_RUN + 4 * NWV * 64 + 4 * NWV + 4 * 128 <= NWV * WAVE_FLOATS, "plain_rows' memory");
  extern __shared__ __attribute__((aligned(16))) float as_lds[];
  __shared__ unsigned again;  // queries with an output that the split may have spoilt
  // consecutive blocks go to one XCD, whose L2 then holds the K and V of few heads; the longest rows of keys first
  const int total = a.H * a.nq, per = (total + 7) >> 3, item = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || item >= total) return;
  const int h = item / a.nq, qb = a.nq - 1 - item % a.nq, q0 = qb * ASQ;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l32 = lane & 31, hh = lane >> 5;
  const int qpos = a.pos0 + q0 + l32;  // keys 0..qpos are visible to this lane's query (which may be beyond the last one)
  const int nt = (a.pos0 + min(q0 + ASQ, a.Tq) + ASQ - 1) / ASQ;
  const int tb = nt * wave / NWV, te = nt * (wave + 1) / NWV;

  const u32x4* qsrc = a.Q3 + (size_t)(h * a.nq + qb) * KS * 192;
  u32x4* qlds = reinterpret_cast<u32x4*>(as_lds);
  u32x4 qr[QREG ? KS : 1][3];
  if constexpr (QREG) {
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int p = 0; p < 3; ++p) qr[s][p] = qsrc[(s * 3 + p) * 64 + lane];
  } else {
    for (int i = threadIdx.x; i < KS * 192; i += NWV * 64) qlds[i] = qsrc[i];
    __syncthreads();
  }
  f32x16 o[DB];
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[b][r] = 0.f;
  float m = -INFINITY, lsum = 0.f, least = INFINITY;
  u32x4 kf[KS][3], vf[KS][3];
  const auto fetch = [&](u32x4 (&f)[KS][3], const u32x4* base, int t) {
    const u32x4* src = base + (size_t)(h * a.nt + t) * KS * 192 + lane;
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int p = 0; p < 3; ++p) f[s][p] = src[(s * 3 + p) * 64];
  };
  if (tb < te) fetch(kf, a.K3, tb);
  for (int t = tb; t < te; ++t) {
    fetch(vf, a.V3, t);
    f32x16 sacc, rest;
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[r] = rest[r] = 0.f;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if constexpr (QREG) {
        split_mfma(kf[s], qr[s], sacc, rest);
      } else {
        const u32x4 x[3] = {qlds[(s * 3 + 0) * 64 + lane], qlds[(s * 3 + 1) * 64 + lane], qlds[(s * 3 + 2) * 64 + lane]};
        split_mfma(kf[s], x, sacc, rest);
      }
    }
    fetch(kf, a.K3, t + 1 < te ? t + 1 : t);
    float tmax = -INFINITY;
    if (t * ASQ + ASQ - 1 > a.pos0 + q0) {  // keys that not all queries see
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int key = t * ASQ + (r >> 2) * 8 + hh * 4 + (r & 3);
        sacc[r] = key <= qpos ? (sacc[r] + rest[r]) * a.scale : -INFINITY;
        least = fminf(least, key <= qpos ? sacc[r] : INFINITY);
        tmax = fmaxf(tmax, sacc[r]);
      }
    } else {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        sacc[r] = (sacc[r] + rest[r]) * a.scale;
        least = fminf(least, sacc[r]);
        tmax = fmaxf(tmax, sacc[r]);
      }
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
    const float mnew = fmaxf(m, tmax);
    // a query with no visible key so far keeps m = -inf: guard the exponentials
    const float corr = m > -INFINITY ? exp_neg(m - mnew) : 0.f;
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      sacc[r] = sacc[r] == -INFINITY ? 0.f : exp_neg(sacc[r] - mnew);  // (not a number stays that: plain_rows)
    }
#pragma unroll
    for (int r = 0; r < 16; r += 4) psum += (sacc[r] + sacc[r + 1]) + (sacc[r + 2] + sacc[r + 3]);
    lsum = lsum * corr + psum;
    m = mnew;
#pragma unroll
    for (int b = 0; b < DB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[b][r] *= corr;
    u32x4 pf[2][3];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const Split8 w = split8(f32x4{sacc[8 * s], sacc[8 * s + 1], sacc[8 * s + 2], sacc[8 * s + 3]},
                              f32x4{sacc[8 * s + 4], sacc[8 * s + 5], sacc[8 * s + 6], sacc[8 * s + 7]});
      pf[s][0] = w.hi;
      pf[s][1] = w.mid;
      pf[s][2] = w.lo;
    }
#pragma unroll
    for (int b = 0; b < DB; ++b) {
#pragma unroll
      for (int r = 0; r < 16; ++r) rest[r] = 0.f;
      split_mfma(vf[2 * b], pf[0], o[b], rest);
      split_mfma(vf[2 * b + 1], pf[1], o[b], rest);
#pragma unroll
      for (int r = 0; r < 16; ++r) o[b][r] += rest[r];
    }
  }
  lsum += __shfl_xor(lsum, 32);  // the two halves of a column saw disjoint keys, the same maximum
  least = fminf(least, __shfl_xor(least, 32));

  if constexpr (!QREG) __syncthreads();
  float* Om = as_lds + wave * WAVE_FLOATS;  // [DIMS][AS_MERGE], then maxima, sums and least scores of the 32 queries
#pragma unroll
  for (int b = 0; b < DB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) Om[(b * 32 + (r >> 2) * 8 + hh * 4 + (r & 3)) * AS_MERGE + l32] = o[b][r];
  if (hh == 0) {
    Om[DIMS * AS_MERGE + l32] = m;
    Om[DIMS * AS_MERGE + ASQ + l32] = lsum;
    Om[DIMS * AS_MERGE + 2 * ASQ + l32] = least;
  }
  if (threadIdx.x == 0) again = 0u;
  __syncthreads();
  for (int e = threadIdx.x; e < ASQ * DIMS; e += NWV * 64) {
    const int qi = e / DIMS, dim = e % DIMS;
    if (q0 + qi >= a.Tq || dim >= a.hs) continue;
    float mw[NWV], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      mw[w] = as_lds[w * WAVE_FLOATS + DIMS * AS_MERGE + qi];
      M = fmaxf(M, mw[w]);
    }
    float num = 0.f, den = 0.f, lo = INFINITY;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const float f = mw[w] > -INFINITY ? exp_neg(mw[w] - M) : 0.f;
      num += as_lds[w * WAVE_FLOATS + dim * AS_MERGE + qi] * f;
      den += as_lds[w * WAVE_FLOATS + DIMS * AS_MERGE + ASQ + qi] * f;
      lo = fminf(lo, as_lds[w * WAVE_FLOATS + DIMS * AS_MERGE + 2 * ASQ + qi]);
    }
    const float v = num / den;
    put(a, q0 + qi, h, dim, v);
    // twice the bits, so without the sign: not finite, or under 2^-60 and no zero (far keys: under 2^-20, or zero)
    constexpr unsigned HI = 0xff000000u;
    const bool far = lo < M - AS_FAR;
    const unsigned v2 = __float_as_uint(v) << 1, limit = (far ? 127 - 20 : 127 - 60) << 24;
    if (v2 >= HI || (v2 < limit && (far || v2 != 0u))) atomicOr(&again, 1u << qi);
  }
  __syncthreads();
  const unsigned left = __builtin_amdgcn_readfirstlane(again);
  if (left) plain_rows<NWV * 64>(a, h, q0, left, as_lds);
}

template <int DB, int NWV>
hipError_t launch_waves(const AttnSplitArgs& a, hipStream_t s) {
  const size_t merge = sizeof(float) * NWV * (32 * DB * AS_MERGE + 3 * ASQ), ql = DB > 1 ? (size_t)2 * DB * 192 * 16 : 0;
  const size_t lds = merge > ql ? merge : ql;
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_split_kernel<DB, NWV>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const long grid = ((long)a.H * a.nq + 7) / 8 * 8;
  if (grid > 0x7fffffffL) return hipErrorInvalidValue;
  attention_split_kernel<DB, NWV><<<(unsigned)grid, NWV * 64, lds, s>>>(a);
  return hipGetLastError();
}

}  // namespace

size_t attention_split_bytes(int Tq, int pos0, int H, int hs) {
  const size_t per = (size_t)2 * ((hs + 31) / 32) * 192 * 16;
  return per * H * ((Tq + ASQ - 1) / ASQ + 2 * (size_t)((pos0 + Tq + ASQ - 1) / ASQ));
}

hipError_t launch_attention_split(int Tq, int pos0, int H, int hs, float scale, const float* q, int ldq, const float* Kc, const float* Vc,
                                  size_t hstride, int ldkv, float* out, int ldo, void* ws, hipStream_t s, const PairRows* pairs) {
  if (hs > 128 || (hs & 3) || H > 65535) return hipErrorInvalidValue;
  AttnSplitArgs a{Tq, pos0, H, hs, (Tq + ASQ - 1) / ASQ, (pos0 + Tq + ASQ - 1) / ASQ, scale, q, ldq, Kc, Vc, hstride, ldkv, out, ldo, pairs ? *pairs : PairRows{}, nullptr, nullptr, nullptr};
  const int DB = (hs + 31) / 32;
  const size_t unit = (size_t)2 * DB * 192;
  a.Q3 = static_cast<u32x4*>(ws);
  a.K3 = a.Q3 + unit * H * a.nq;
  a.V3 = a.K3 + unit * H * a.nt;
  attention_operands<<<dim3(a.nq + 2 * a.nt, H), 2 * DB * 64, 0, s>>>(a);
  switch (DB) {
    case 1: return launch_waves<1, 8>(a, s);
    case 2: return launch_waves<2, 8>(a, s);
    case 3: return launch_waves<3, 4>(a, s);
    default: return launch_waves<4, 4>(a, s);
  }
}

}  // namespace wgpt
