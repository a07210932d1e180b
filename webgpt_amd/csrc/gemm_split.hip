// FastMatMulBlock (instructions.js:157-319) for prompts, and its int8 weight-only form (other/int8-gemm.js:117-229).
//
// The operands are fp32 (the weights perhaps int8), the multiplications run on the bf16 matrix cores: an fp32 value of 2^-110
// and more is the exact sum of three bf16 values, x = hi + mid + lo with |mid| <= 2^-8 |x| and |lo| <= 2^-17 |x| (smaller
// values: spoilt), and of the nine partial products of x y the six largest are taken, all of them exact in the fp32
// accumulator's input. The three left out (mid lo, lo mid, lo lo) are together at most 2^-24 |x y|, an fp32 rounding of one
// product; with sums of sixteen products rounded once instead of two at a time the sum of four products and more is at least
// as close to the exact one as that of v_mfma_f32_32x32x2_f32 (emulated, norm of the errors: K = 4 2.6e-8 against 3.1e-8,
// K = 768 3.1e-7 against 3.7e-7), unless few of sixteen products are not zero (nine of ten columns of A zero: 1.5 times as far).
// An int8 weight is one bf16 value (8 significand bits), so three products do, and
// the column's scale[n] / 127 is applied to the finished sum; where that sum leaves the range of fp32, which the scaled
// one need not, it is taken again with weights that are scaled first (plain_sums). A value that is infinite, or rounds to an
// infinite bf16, has no such split (inf + nan + nan): every sum it takes part in comes out as NaN or infinite, and a wave that
// finds one among its sums takes them again with fp32 matrix instructions (plain_sums).
// bf16 runs at 16 times the rate of fp32 here, six products are therefore 2.7 times (int8: 5.3 times) faster.
#include "gemm_split.h"

#include <cmath>
#include <type_traits>

#include "kernels.h"
#include "split_bf16.h"

namespace wgpt {
namespace {

template <int R>
struct SplitBlock;
template <>
struct SplitBlock<32> {
  typedef f32x16 acc_t;
  static constexpr int NACC = 16;
  static __device__ __forceinline__ acc_t mfma(const u32x4& w, const u32x4& a, const acc_t& c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
  }
  // fp32 operands: one k for each half of the wave
  static __device__ __forceinline__ acc_t plain(float w, float a, const acc_t& c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(w, a, c, 0, 0, 0); }
  // column (of W) of the four consecutive ones in accumulator registers 4q..4q+3 of a lane
  static __device__ __forceinline__ int row4(int q, int lane) { return 8 * q + 4 * (lane >> 5); }
};
template <>
struct SplitBlock<16> {
  typedef f32x4 acc_t;
  static constexpr int NACC = 4;
  static __device__ __forceinline__ acc_t mfma(const u32x4& w, const u32x4& a, const acc_t& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), c, 0, 0, 0);
  }
  static __device__ __forceinline__ acc_t plain(float w, float a, const acc_t& c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(w, a, c, 0, 0, 0); }
  static __device__ __forceinline__ int row4(int, int lane) { return 4 * (lane >> 4); }
};


__device__ __forceinline__ float gelu_ref(float x) {
  const float x3 = x * x * x;
  const float cdf = 0.5f * (1.0f + tanhf(0.7978845608f * (x + 0.044715f * x3)));
  float r = x * cdf;
  r = x < -10.0f ? 0.0f : r;
  r = x > 10.0f ? x : r;
  return r;
}

// ---- operands of one wave: RUN consecutive k per lane and step of 32. Loads are raw buffer loads whose per-lane offset
// never changes: the step's place is in the scalar offset, so no vector instruction goes into addresses. ----
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void* p, unsigned bytes = 0x7fffffffu) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, bytes, 0x00020000);
}
__device__ __forceinline__ f32x4 buf_f4(__amdgpu_buffer_rsrc_t b, int v, int s) {
  return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b, v, s, 0));
}
// Lane (c, kg) of a block of R columns supplies k = RUN8 pieces: step s, chunk (STEPS > 1 ? 2 * s + kg : kg) of eight.
template <int R>
__device__ __forceinline__ int chunk_of(int s, int kg) { return R == 32 ? 2 * s + kg : kg; }

// W as the caller's matrices come, [K, N]: one row of 32 (or 16) columns per load. BLK: as a model keeps it (block_weights),
// [K / 4][N][4] floats or [K / 8][N][8] int8: a lane's eight consecutive k in two (one) loads of 16 (8) bytes, neighbours
// next to each other. A compute unit takes a load instruction every 10-15 ns whatever its width; a step of 32 k is four (two)
// of them instead of sixteen. Cold weights, best shape of each: int8 300x6400x1600 37.9 -> 25.8 us, 943x6400x1600 97.0 ->
// 64.8 us, 16x4800x1600 8.7 -> 7.4 us; fp32, where the splitting of W costs more than its loads, 128x3072x768 11.5 -> 10.2 us,
// 16x3072x1024 8.9 -> 7.0 us, 943x3072x768 37.2 -> 36.9 us.
template <int R, bool I8, bool BLK>
struct WRaw {
  static constexpr int STEPS = R == 32 ? 2 : 1;
  unsigned v[BLK && I8 ? 2 * STEPS : 8 * STEPS];
  static __device__ __forceinline__ int offset(const SplitGemmArgs& a, int n, int kg) {
    if constexpr (BLK) return I8 ? 8 * (n + kg * a.N) : 16 * (n + kg * 2 * a.N);
    else return 4 * ((I8 ? n >> 2 : n) + kg * 8 * a.ldw);
  }
  __device__ __forceinline__ void load(const SplitGemmArgs& a, __amdgpu_buffer_rsrc_t b, int off, int it) {
    if constexpr (BLK && I8) {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) put2(s, __builtin_amdgcn_raw_buffer_load_b64(b, off, 8 * (it * 4 + 2 * s) * a.N, 0));
    } else if constexpr (BLK) {
#pragma unroll
      for (int i = 0; i < 2 * STEPS; ++i) put4(i, __builtin_amdgcn_raw_buffer_load_b128(b, off, 16 * (it * 8 + (i >> 1) * 4 + (i & 1)) * a.N, 0));
    } else {
#pragma unroll
      for (int i = 0; i < 8 * STEPS; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b32(b, off, 4 * (it * 32 + (i >> 3) * 16 + (i & 7)) * a.ldw, 0);
    }
  }
  // the step that reaches beyond K: rows (runs of eight, K a multiple of eight) past the last one repeat it (their A is zero)
  __device__ __forceinline__ void load_tail(const SplitGemmArgs& a, __amdgpu_buffer_rsrc_t b, int n, int kg, int it) {
    if constexpr (BLK) {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        const int c = it * 4 + chunk_of<R>(s, kg), last = (a.K >> 3) - 1, u = c < last ? c : last;
        if constexpr (I8) {
          put2(s, __builtin_amdgcn_raw_buffer_load_b64(b, 8 * (u * a.N + n), 0, 0));
        } else {
          put4(2 * s, __builtin_amdgcn_raw_buffer_load_b128(b, 16 * (2 * u * a.N + n), 0, 0));
          put4(2 * s + 1, __builtin_amdgcn_raw_buffer_load_b128(b, 16 * ((2 * u + 1) * a.N + n), 0, 0));
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8 * STEPS; ++i) {
        const int k = it * 32 + chunk_of<R>(i >> 3, kg) * 8 + (i & 7);
        v[i] = __builtin_amdgcn_raw_buffer_load_b32(b, 4 * ((I8 ? n >> 2 : n) + (k < a.K ? k : a.K - 1) * a.ldw), 0, 0);
      }
    }
  }
  __device__ __forceinline__ void put2(int i, u32x2 x) { v[2 * i] = x[0], v[2 * i + 1] = x[1]; }
  __device__ __forceinline__ void put4(int i, u32x4 x) { v[4 * i] = x[0], v[4 * i + 1] = x[1], v[4 * i + 2] = x[2], v[4 * i + 3] = x[3]; }
  __device__ __forceinline__ Split8 get(int s, int n) const {
    if constexpr (I8) {
      Split8 r;
      unsigned h[4];
      if constexpr (BLK) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const unsigned x = v[2 * s + (i >> 1)], sh = 16 * (i & 1);
          h[i] = bf16_pair((float)((int)(x << (24 - sh)) >> 24), (float)((int)(x << (16 - sh)) >> 24));
        }
      } else {
        const int sh = 24 - 8 * (n & 3);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          h[i] = bf16_pair((float)((int)(v[8 * s + 2 * i] << sh) >> 24), (float)((int)(v[8 * s + 2 * i + 1] << sh) >> 24));
      }
      r.hi = u32x4{h[0], h[1], h[2], h[3]};
      return r;
    } else {
      const u32x4 a = {v[8 * s], v[8 * s + 1], v[8 * s + 2], v[8 * s + 3]}, b = {v[8 * s + 4], v[8 * s + 5], v[8 * s + 6], v[8 * s + 7]};
      return split8(__builtin_bit_cast(f32x4, a), __builtin_bit_cast(f32x4, b));
    }
  }
  // value e of the eight of step s
  __device__ __forceinline__ float plain(int s, int e, int n) const {
    if constexpr (!I8) return __builtin_bit_cast(float, v[8 * s + e]);
    else if constexpr (BLK) return (float)((int)(v[2 * s + (e >> 2)] << (24 - 8 * (e & 3))) >> 24);
    else return (float)((int)(v[8 * s + e] << (24 - 8 * (n & 3))) >> 24);
  }
};
// A of a lane, straight from memory (rows of A, fp32)
template <int R>
struct ARaw {
  static constexpr int STEPS = R == 32 ? 2 : 1;
  f32x4 v[2 * STEPS];
  static __device__ __forceinline__ int offset(const SplitGemmArgs& a, int m, int kg) { return 4 * ((m < a.M ? m : a.M - 1) * a.lda + kg * 8); }
  __device__ __forceinline__ void load(const SplitGemmArgs&, __amdgpu_buffer_rsrc_t b, int off, int it) {
#pragma unroll
    for (int i = 0; i < 2 * STEPS; ++i) v[i] = buf_f4(b, off, 128 * it + 64 * (i >> 1) + 16 * (i & 1));
  }
  __device__ __forceinline__ void load_tail(const SplitGemmArgs& a, __amdgpu_buffer_rsrc_t b, int m, int kg, int it) {
#pragma unroll
    for (int i = 0; i < 2 * STEPS; ++i) {
      const int k = it * 32 + chunk_of<R>(i >> 1, kg) * 8 + 4 * (i & 1);
      const f32x4 x = buf_f4(b, 4 * ((m < a.M ? m : a.M - 1) * a.lda + (k < a.K ? k : a.K - 4)), 0);
      v[i] = k < a.K ? x : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  }
  __device__ __forceinline__ Split8 get(int s) const { return split8(v[2 * s], v[2 * s + 1]); }
  __device__ __forceinline__ float plain(int s, int e) const { return v[2 * s + (e >> 2)][e & 3]; }
};

template <bool I8>
__device__ __forceinline__ f32x4 scaled(const SplitGemmArgs& a, int n, f32x4 v) {
  if constexpr (I8) {
    const f32x4 s = *reinterpret_cast<const f32x4*>(a.wscale + n);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] *= s[i] / 127.0f;
  }
  return v;
}

__device__ __forceinline__ void split_epilogue(const SplitGemmArgs& a, int m, int n, int slice, f32x4 v) {
  if (a.part) {
    *reinterpret_cast<f32x4*>(a.part + ((size_t)slice * a.M + m) * a.N + n) = v;
    return;
  }
  if (a.bias) v += *reinterpret_cast<const f32x4*>(a.bias + n);
  if (a.epi == EPI_GELU) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = gelu_ref(v[i]);
  } else if (a.epi == EPI_RESIDUAL) {
    v += *reinterpret_cast<const f32x4*>(a.resid + (size_t)m * a.ldc + n);
  }
  float* c = a.C + (size_t)m * a.ldc + n;
  if (a.Kc && n >= a.d) {
    const bool val = n >= 2 * a.d;
    const int e = n - (val ? 2 : 1) * a.d, h = e / a.hs;
    c = (val ? a.Vc : a.Kc) + ((size_t)h * a.ctx + a.pos0 + m) * a.hs + (e - h * a.hs);
  }
  *reinterpret_cast<f32x4*>(c) = v;
}

// position of a workgroup in the grid of tiles: consecutive tiles (m fastest: they share the columns of W) go to one XCD
__device__ __forceinline__ bool tile_of(const SplitGemmArgs& a, int& m, int& n, int& slice) {
  const int total = a.mt * a.nt * a.S, per = (total + 7) >> 3;
  int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || t >= total) return false;
  m = t % a.mt;
  t /= a.mt;
  n = t % a.nt;
  slice = t / a.nt;
  return true;
}

template <int R, int MB, int NB, bool I8>
__device__ __forceinline__ void split_products(const Split8 (&ws)[NB], const Split8 (&xs)[MB], typename SplitBlock<R>::acc_t (&acc)[MB][NB]) {
  typedef SplitBlock<R> B;
  // smallest products first; the three that are left out are at most 2^-24 of a product
#define SPLIT_STEP(wp, xp)                                                                        \
  _Pragma("unroll") for (int i = 0; i < MB; ++i) _Pragma("unroll") for (int j = 0; j < NB; ++j) \
      acc[i][j] = B::mfma(ws[j].wp, xs[i].xp, acc[i][j])
  if constexpr (!I8) SPLIT_STEP(lo, hi);
  SPLIT_STEP(hi, lo);
  if constexpr (!I8) SPLIT_STEP(mid, mid);
  if constexpr (!I8) SPLIT_STEP(mid, hi);
  SPLIT_STEP(hi, mid);
  SPLIT_STEP(hi, hi);
#undef SPLIT_STEP
}

// Are there sums in the wave's tile that the split may have spoilt? Those that are not finite; unscaled int8 ones of 2^124 and
// more, so that the eight of a workgroup have a finite sum; and tiny ones: a value under 2^-110 loses what its third part
// would hold under the smallest bf16 subnormal, 2^-134 at most, which shows in sums under SPLIT_TINY unless the other operand
// has values of about 2^50 and more. (One instruction per two registers for the largest and one for the smallest; the largest
// lets NaN through. Zeros are no tiny sums: a value up to 2^-134 has no bf16 part at all, and a sum of nothing but products with
// such values stays zero, as where subnormal numbers are flushed. To look for them where sums are zero, in no more than a wave's
// first step, makes every launch longer: 128x2304x768 10.9 -> 11.1 us, 943x3072x768 35.7 -> 36.8 us.)
constexpr float SPLIT_TINY = 0x1p-60f;
template <int R, int MB, int NB, bool I8>
__device__ __forceinline__ bool spoilt(const typename SplitBlock<R>::acc_t (&acc)[MB][NB]) {
  float most = 0.f, least = INFINITY;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < SplitBlock<R>::NACC; ++e) {
        most = __builtin_elementwise_maximum(most, fabsf(acc[i][j][e]));
        least = __builtin_elementwise_minimum(least, fabsf(acc[i][j][e]));
      }
  bool bad = !(most < (I8 ? 0x1p124f : INFINITY));
  if (least < SPLIT_TINY) {
    unsigned tiny = ~0u;  // (twice the bits, less one: the sign is gone and a zero is the largest)
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int e = 0; e < SplitBlock<R>::NACC; ++e) tiny = min(tiny, (__float_as_uint(acc[i][j][e]) << 1) - 1u);
    bad = bad || tiny < (__float_as_uint(SPLIT_TINY) << 1) - 1u;
  }
  return __builtin_amdgcn_ballot_w64(bad) != 0;
}

// The sums of a wave's tile from row m0 of A over its steps it0, it0 + by, .. below it1 (and the one that reaches beyond K) with
// fp32 matrix instructions (and int8 weights scaled), for operands that cannot be split: 2.7 times (int8: 5.3 times) the matrix time of the sums that they
// replace, and only the waves with such operands pay it: 943x3072x768 with nothing but NaN 37 -> about 92 us (1.7 ms with one
// product after the other).
// (Inlined: a call would cost every launch of these kernels 5 us, for the stack that it needs.)
template <int R, int MB, int NB, bool I8, bool BLK>
__device__ __forceinline__ void plain_sums(const SplitGemmArgs& a, __amdgpu_buffer_rsrc_t wb, __amdgpu_buffer_rsrc_t xb, int m0, const int (&nn)[NB],
                                           int it0, int it1, int by, bool tail, typename SplitBlock<R>::acc_t (&acc)[MB][NB]) {
  typedef SplitBlock<R> B;
  const int lane = threadIdx.x & 63, r = lane & (R - 1), kg = lane / R;
  WRaw<R, I8, BLK> w[NB];
  ARaw<R> x[MB];
  float scale[NB];
  if constexpr (I8) {
#pragma unroll
    for (int j = 0; j < NB; ++j) scale[j] = a.wscale[nn[j]] / 127.0f;
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < B::NACC; ++e) acc[i][j][e] = 0.f;
  const auto multiply = [&](int kend) {  // kend: how many of a chunk's eight k there are
#pragma unroll
    for (int s = 0; s < WRaw<R, I8, BLK>::STEPS; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          // (beyond K the loads repeat the last row of W, which may be infinite, and A is zero)
          float wv = chunk_of<R>(s, kg) * 8 + e < kend ? w[j].plain(s, e, nn[j]) : 0.f;
          if constexpr (I8) wv *= scale[j];
#pragma unroll
          for (int i = 0; i < MB; ++i) acc[i][j] = B::plain(wv, x[i].plain(s, e), acc[i][j]);
        }
  };
#pragma unroll 1
  for (int it = it0; it < it1; it += by) {
#pragma unroll
    for (int j = 0; j < NB; ++j) w[j].load(a, wb, WRaw<R, I8, BLK>::offset(a, nn[j], kg), it);
#pragma unroll
    for (int i = 0; i < MB; ++i) x[i].load(a, xb, ARaw<R>::offset(a, m0 + i * R + r, kg), it);
    multiply(32);
  }
  if (tail) {
    const int it = a.K >> 5;
#pragma unroll
    for (int j = 0; j < NB; ++j) w[j].load_tail(a, wb, nn[j], kg, it);
#pragma unroll
    for (int i = 0; i < MB; ++i) x[i].load_tail(a, xb, m0 + i * R + r, kg, it);
    multiply(a.K & 31);
  }
}

// Sum of NP partial tiles (LDS, 64 float4 per entry) and epilogue. A tile's columns belong to NWN waves; `plain`, int8 only: a
// flag for each wave, partial tile by partial tile, whose sums are scaled already.
template <int R, int MB, int NB, int NP, int NWN, int THREADS, bool I8>
__device__ __forceinline__ void finish_tile(const SplitGemmArgs& a, const f32x4* red, const int* plain, int m0, int n0, int slice) {
  typedef SplitBlock<R> B;
  constexpr int Q = B::NACC / 4, ENT = MB * NB * Q;
  int some = 0;
  if constexpr (I8) {
#pragma unroll
    for (int u = 0; u < NP * NWN; ++u) some |= plain[u];
  }
  for (int e = threadIdx.x; e < ENT * 64; e += THREADS) {
    const int ln = e & 63, b = e >> 6, q = b % Q, ij = b / Q;
    const int m = m0 + (ij / NB) * R + (ln & (R - 1)), n = n0 + (ij % NB) * R + B::row4(q, ln);
    if (m >= a.M || n >= a.N) continue;
    f32x4 v;
    if (I8 && some) {
      f32x4 done = {0.f, 0.f, 0.f, 0.f};
      v = done;
#pragma unroll 1
      for (int u = 0; u < NP; ++u) {
        if (plain[u * NWN + (ij % NB) / (NB / NWN)]) done += red[u * ENT * 64 + e];
        else v += red[u * ENT * 64 + e];
      }
      v = scaled<I8>(a, n, v) + done;
    } else {
      v = red[e];
#pragma unroll
      for (int u = 1; u < NP; ++u) v += red[u * ENT * 64 + e];
      v = scaled<I8>(a, n, v);
    }
    split_epilogue(a, m, n, slice, v);
  }
}

// The waves of a workgroup split K, each holds the whole tile and takes its operands straight from memory: no barrier and no
// LDS until the sums meet. Bound by the load instructions of a compute unit up to ~100 rows (10-15 ns each whatever their
// width), beyond that by matrix and vector instructions one after the other (six products per pair against eleven vector
// instructions per two values split). Dependent launches, cold weights: 13x2304x768 5.5 us, 13x768x3072 in four slices 5.1 us
// (219 and 193 us with the fp32 tile kernel that served 5 to 15 rows before); 64x64 tiles: 512x4096x1024 32.4 us = 132
// TFLOP/s (39.9 us with v_mfma_f32_32x32x2_f32), int8 300x6400x1600 38.8 us (73).
template <int R, int MB, int NB, int NW, bool I8, bool BLK>
__global__ __launch_bounds__(NW * 64, MB == 2 ? 2 : 4) void gemm_split_rows(SplitGemmArgs a) {
  typedef SplitBlock<R> B;
  constexpr int STEPS = WRaw<R, I8, BLK>::STEPS, Q = B::NACC / 4, ENT = MB * NB * Q;
  extern __shared__ __attribute__((aligned(16))) float gs_lds[];
  int m0, n0, slice;
  if (!tile_of(a, m0, n0, slice)) return;
  m0 *= MB * R;
  n0 *= NB * R;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & (R - 1), kg = lane / R;
  const int iters = a.K >> 5, part = slice * NW + wave, parts = a.S * NW;
  const int it0 = (int)((long)iters * part / parts), it1 = (int)((long)iters * (part + 1) / parts);
  const __amdgpu_buffer_rsrc_t wb = buffer_of(a.W), xb = buffer_of(a.A);
  int nn[NB], wo[NB], xo[MB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    nn[j] = n0 + j * R + r < a.N ? n0 + j * R + r : a.N - 1;
    wo[j] = WRaw<R, I8, BLK>::offset(a, nn[j], kg);
  }
#pragma unroll
  for (int i = 0; i < MB; ++i) xo[i] = ARaw<R>::offset(a, m0 + i * R + r, kg);
  typename B::acc_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < B::NACC; ++e) acc[i][j][e] = 0.f;
  WRaw<R, I8, BLK> w[NB];
  ARaw<R> x[MB];
  Split8 ws[STEPS][NB], xs[STEPS][MB];
  auto fetch = [&](int it) {
#pragma unroll
    for (int j = 0; j < NB; ++j) w[j].load(a, wb, wo[j], it);
#pragma unroll
    for (int i = 0; i < MB; ++i) x[i].load(a, xb, xo[i], it);
  };
  auto convert = [&] {
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
#pragma unroll
      for (int j = 0; j < NB; ++j) ws[s][j] = w[j].get(s, nn[j]);
#pragma unroll
      for (int i = 0; i < MB; ++i) xs[s][i] = x[i].get(s);
    }
  };
  if (it0 < it1) fetch(it0);
  for (int it = it0; it < it1; ++it) {
    convert();
    fetch(it + 1 < it1 ? it + 1 : it);
    __builtin_amdgcn_sched_barrier(0);  // the requests leave before the products, not where their values are first needed
#pragma unroll
    for (int s = 0; s < STEPS; ++s) split_products<R, MB, NB, I8>(ws[s], xs[s], acc);
  }
  if ((a.K & 31) && part == parts - 1) {
#pragma unroll
    for (int j = 0; j < NB; ++j) w[j].load_tail(a, wb, nn[j], kg, iters);
#pragma unroll
    for (int i = 0; i < MB; ++i) x[i].load_tail(a, xb, m0 + i * R + r, kg, iters);
    convert();
#pragma unroll
    for (int s = 0; s < STEPS; ++s) split_products<R, MB, NB, I8>(ws[s], xs[s], acc);
  }
  __shared__ int plain[NW];
  const bool again = spoilt<R, MB, NB, I8>(acc);
  if (again) plain_sums<R, MB, NB, I8, BLK>(a, wb, xb, m0, nn, it0, it1, 1, (a.K & 31) && part == parts - 1, acc);
  if constexpr (I8) plain[wave] = again;
  f32x4* red = reinterpret_cast<f32x4*>(gs_lds);
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < Q; ++q)
        red[(wave * ENT + (i * NB + j) * Q + q) * 64 + lane] = f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
  __syncthreads();
  finish_tile<R, MB, NB, NW, 1, NW * 64, I8>(a, red, plain, m0, n0, slice);
}

__device__ __forceinline__ void lds_barrier() {  // orders LDS accesses only: loads from memory stay in flight
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// KG groups of NWN waves; a group takes every KG-th step of 32 k. Its waves own 32 * NB columns each, for all rows of the
// tile: W goes straight from memory into registers, A through LDS, split once per workgroup on its way in. A step is two halves of
// 16 k; between the products of a half stand the reads of the next half's A from LDS and the splitting of its W, so that no product
// waits for either: with the reads of a step in front of its products, where all waves of a compute unit make them at once,
// the matrix cores stood still for a third of the time (cold weights, us before and now: 943x3072x768 in 96x128 tiles 32.5, 29.9,
// in 128x128 tiles 37.9, 32.9; 512x3072x1024 in 64x128 27.5, 23.9; 512x1024x1024 in 32x64 13.2, 11.2). A step of 128x128 takes 1.04 us
// with all units at work and 0.85 with 32 of them, its products 0.64 at the matrix cores' rate. 96x128 tiles are for row counts
// of which 128 leave units idle: 943x2304x768 180 workgroups, 26.6 us, where 144 of 128x128 take 31.0 and 64x64 tiles of the kernel above 37.4.
template <int MB, int NB, int NWN, int KG, bool I8, bool BLK, int OCC, int D>
__global__ __launch_bounds__(NWN * KG * 64, OCC) void gemm_split_tile(SplitGemmArgs a) {
  constexpr int R = 32;
  typedef SplitBlock<R> B;
  constexpr int MT = MB * R, GT = NWN * 64, Q = 4;
  constexpr int CH = MT + 2;               // units of 16 bytes between chunks of eight k: conflict-free writes and reads
  constexpr int BUF = 3 * 4 * CH;          // units of one buffer: planes x chunks
  constexpr int AV = (MT * 4 + GT - 1) / GT;          // runs of eight k that a thread stages per step
  extern __shared__ __attribute__((aligned(16))) float gs_lds[];
  int m0, n0, slice;
  if (!tile_of(a, m0, n0, slice)) return;
  m0 *= MT;
  n0 *= NB * NWN * R;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int grp = wave / NWN, wn = wave % NWN, gt = threadIdx.x % GT;
  const int r = lane & 31, kg = lane >> 5;
  // the v-th run of this thread among the tile's MT * 4; where the last ones do not reach all threads, the others repeat one
  const auto run_of = [&](int v) { return gt + v * GT < MT * 4 ? gt + v * GT : gt + (v - 1) * GT; };
  u32x4* abuf = reinterpret_cast<u32x4*>(gs_lds) + grp * 2 * BUF;
  const int full = a.K >> 5;
  const int s0 = (int)((long)full * slice / a.S), s1 = (int)((long)full * (slice + 1) / a.S);
  const int rounds = (s1 - s0 + KG - 1) / KG;
  const __amdgpu_buffer_rsrc_t wb = buffer_of(a.W), xb = buffer_of(a.A);
  int nn[NB], wo[NB], xo[AV], xl[AV];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = n0 + (wn * NB + j) * R + r;
    nn[j] = n < a.N ? n : a.N - 1;
    wo[j] = WRaw<R, I8, BLK>::offset(a, nn[j], kg);
  }
#pragma unroll
  for (int v = 0; v < AV; ++v) {
    const int u = run_of(v), row = u >> 2, c = u & 3;
    xo[v] = 4 * ((m0 + row < a.M ? m0 + row : a.M - 1) * a.lda + c * 8);
    xl[v] = c * CH + row;
  }
  typename B::acc_t acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < B::NACC; ++e) acc[i][j][e] = 0.f;
  static_assert(D % 2 == 0, "the buffer of a step is a constant of the unrolled loop");
  WRaw<R, I8, BLK> w[D][NB];
  f32x4 x[D][AV][2];
  Split8 ws[2][NB], xs[2][MB];  // of the two halves of a step
  const auto clamp_step = [&](int i) { const int t = s0 + i * KG + grp; return t < s1 ? t : s1 - 1; };
  const auto fetch_w = [&](int u, int i) {
    const int t = clamp_step(i);
#pragma unroll
    for (int j = 0; j < NB; ++j) w[u][j].load(a, wb, wo[j], t);
  };
  // steps beyond the slice's end are asked for out of the buffer's range and come back as zeros
  const auto fetch_x = [&](int u, int i) {
    const int t = s0 + i * KG + grp;
#pragma unroll
    for (int v = 0; v < AV; ++v) {
      const int o = t < s1 ? xo[v] : -32;
      x[u][v][0] = buf_f4(xb, o, t < s1 ? 128 * t : 0);
      x[u][v][1] = buf_f4(xb, o + 16, t < s1 ? 128 * t : 0);
    }
  };
  const auto stage = [&](int u, int buf) {
#pragma unroll
    for (int v = 0; v < AV; ++v) {
      const Split8 p = split8(x[u][v][0], x[u][v][1]);
      u32x4* d = abuf + buf * BUF + xl[v];
      d[0] = p.hi;
      d[4 * CH] = p.mid;
      d[8 * CH] = p.lo;
    }
  };
  const auto convert = [&](int u, int h) {
#pragma unroll
    for (int j = 0; j < NB; ++j) ws[h][j] = w[u][j].get(h, nn[j]);
  };
  const auto read = [&](int buf, int h) {
#pragma unroll
    for (int i = 0; i < MB; ++i) {
      const u32x4* p = abuf + buf * BUF + (2 * h + kg) * CH + i * R + r;
      xs[h][i].hi = p[0];
      xs[h][i].mid = p[4 * CH];
      xs[h][i].lo = p[8 * CH];
    }
  };
  constexpr int NMF = MB * NB * (I8 ? 3 : 6), VW = NB * (I8 ? 14 : 46), VA = AV * 48;  // matrix and vector instructions of half a step
  const auto interleave = [&](auto vector) {
    constexpr int NVAL = decltype(vector)::value / NMF + 1;
    __builtin_amdgcn_sched_group_barrier(0x100, 3 * MB, 0);
#pragma unroll
    for (int m = 0; m < NMF; ++m) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, NVAL, 0);
    }
  };
  if (rounds > 0) {
#pragma unroll
    for (int u = 0; u < D; ++u) {
      fetch_x(u, u);
      fetch_w(u, u);
    }
    stage(0, 0);
    fetch_x(0, D);
    convert(0, 0);
    lds_barrier();
    read(0, 0);
    for (int i = 0; i < rounds; i += D) {
#pragma unroll
      for (int u = 0; u < D; ++u) {
        if (u > 0 && i + u >= rounds) break;
        // Half a step's products, between them the second half's operands and the splitting of the next step's A ..
        read(u & 1, 1);
        split_products<R, MB, NB, I8>(ws[0], xs[0], acc);
        convert(u, 1);
        stage((u + 1) % D, (u + 1) & 1);
        fetch_w(u, i + u + D);
        fetch_x((u + 1) % D, i + u + 1 + D);
        interleave(std::integral_constant<int, VW + VA>());
        lds_barrier();
        // .. the other half's, and the next step's first operands
        read((u + 1) & 1, 0);
        split_products<R, MB, NB, I8>(ws[1], xs[1], acc);
        convert((u + 1) % D, 0);
        interleave(std::integral_constant<int, VW>());
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if ((a.K & 31) && slice == a.S - 1) {  // the last, partial step: group 0
    lds_barrier();
    if (grp == 0) {
#pragma unroll
      for (int v = 0; v < AV; ++v) {
        const int u = run_of(v), row = u >> 2, m = m0 + row < a.M ? m0 + row : a.M - 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int k = full * 32 + (gt & 3) * 8 + 4 * h;
          const f32x4 t = buf_f4(xb, 4 * (m * a.lda + (k < a.K ? k : a.K - 4)), 0);
          x[0][v][h] = k < a.K ? t : f32x4{0.f, 0.f, 0.f, 0.f};
        }
      }
      stage(0, 0);
#pragma unroll
      for (int j = 0; j < NB; ++j) w[0][j].load_tail(a, wb, nn[j], kg, full);
    }
    lds_barrier();
    if (grp == 0) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        convert(0, h);
        read(0, h);
        split_products<R, MB, NB, I8>(ws[h], xs[h], acc);
      }
    }
    lds_barrier();
  }
  __shared__ int plain[KG * NWN];
  const bool again = spoilt<R, MB, NB, I8>(acc);
  if (again)
    plain_sums<R, MB, NB, I8, BLK>(a, wb, xb, m0, nn, s0 + grp, s1, KG, grp == 0 && (a.K & 31) && slice == a.S - 1, acc);
  if constexpr (I8) plain[wave] = again;
  f32x4* red = reinterpret_cast<f32x4*>(gs_lds);
  constexpr int NBW = NWN * NB, ENT = MB * NBW * Q;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < Q; ++q)
        red[(grp * ENT + (i * NBW + wn * NB + j) * Q + q) * 64 + lane] = f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
  __syncthreads();
  finish_tile<R, MB, NBW, KG, NWN, NWN * KG * 64, I8>(a, red, plain, m0, n0, slice);
}

// [K, N] to the order that WRaw<.., BLK> reads; a thread makes one run of four (int8: eight) k of a column.
__global__ __launch_bounds__(256) void block_weights_f32(int K, int N, const float* __restrict__ W, f32x4* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)(K >> 2) * N) return;
  const size_t k = i / N * 4, n = i % N;
  out[i] = f32x4{W[k * N + n], W[(k + 1) * N + n], W[(k + 2) * N + n], W[(k + 3) * N + n]};
}
__global__ __launch_bounds__(256) void block_weights_i8(int K, int N, const signed char* __restrict__ W, u32x2* __restrict__ out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)(K >> 3) * N) return;
  const size_t k = i / N * 8, n = i % N;
  u32x2 v = {0, 0};
#pragma unroll
  for (int j = 0; j < 8; ++j) v[j >> 2] |= (unsigned)(unsigned char)W[(k + j) * N + n] << (8 * (j & 3));
  out[i] = v;
}

// ---- launches ----
// A launch takes about fixed + rounds * (one + more * (ceil(workgroups / 256) - 1)) us, where a workgroup needs
// ceil(steps of its slice / kpar) rounds: a compute unit that gets a second workgroup determines the launch. The numbers
// are least-squares fits to launches on MI355X (8 to 1024 rows, 384 to 6400 columns, K from 384 to 6400, 1 to 8 slices; 39800 of
// them, those within 1.5 or 2 times the best shape's time). The shape that they choose is within 1.0 to 1.7 % of the best one
// (geometric mean). Zeros: a form of W for which the shape is not needed (without it the choice is no worse, or 0.1 %) or not built.
struct Shape {
  int mtile, ntile, kpar;  // tile; steps of 32 k that a workgroup works on at a time
  struct Fit { float fixed, one, more; } f32, i8, f32_blk, i8_blk;
};
constexpr Shape SHAPES[] = {
    {16, 16, 8, {2.74f, 0.85f, 0.90f}, {3.61f, 0.50f, 0.53f}, {3.34f, 0.56f, 0.78f}, {3.62f, 0.39f, 0.57f}},  // gemm_split_rows<16, 1, 1, 8>
    {16, 32, 8, {3.36f, 0.94f, 1.11f}, {3.58f, 0.70f, 0.87f}, {3.84f, 0.68f, 0.95f}, {3.68f, 0.47f, 0.70f}},  // gemm_split_rows<16, 1, 2, 8>
    {32, 32, 8, {3.35f, 1.24f, 1.55f}, {3.68f, 1.14f, 1.26f}, {3.63f, 1.10f, 1.51f}, {3.83f, 0.73f, 1.27f}},  // gemm_split_rows<32, 1, 1, 8>
    {64, 64, 4, {5.17f, 1.38f, 1.78f}, {5.53f, 1.10f, 1.47f}, {4.85f, 1.33f, 1.89f}, {0, 0, 0}},              // gemm_split_rows<32, 2, 2, 4>
    {64, 64, 8, {4.72f, 2.68f, 3.90f}, {0, 0, 0}, {0, 0, 0}, {0, 0, 0}},                                      // gemm_split_rows<32, 2, 2, 8>
    {32, 64, 4, {5.10f, 0.93f, 1.14f}, {5.50f, 0.72f, 0.90f}, {4.76f, 0.74f, 1.12f}, {4.74f, 0.39f, 0.70f}},  // gemm_split_tile<1, 1, 2, 4>
    {128, 128, 2, {8.59f, 1.98f, 3.36f}, {10.50f, 1.40f, 2.32f}, {7.98f, 1.85f, 3.54f}, {0, 0, 0}},           // gemm_split_tile<4, 1, 4, 2>
    {64, 128, 2, {0, 0, 0}, {0, 0, 0}, {5.95f, 1.05f, 1.98f}, {6.67f, 0.57f, 0.99f}},                         // gemm_split_tile<2, 1, 4, 2>
    {96, 128, 2, {0, 0, 0}, {0, 0, 0}, {6.96f, 1.57f, 2.82f}, {0, 0, 0}},                                     // gemm_split_tile<3, 1, 4, 2>
};
constexpr int NSHAPES = sizeof(SHAPES) / sizeof(SHAPES[0]);
constexpr const Shape::Fit& fit_of(const Shape& sh, bool i8, bool blocked) { return blocked ? (i8 ? sh.i8_blk : sh.f32_blk) : i8 ? sh.i8 : sh.f32; }
constexpr bool built(int kind, bool i8, bool blocked) { return fit_of(SHAPES[kind], i8, blocked).fixed > 0; }

constexpr size_t rows_lds(int R, int MB, int NB, int NW) { return (size_t)NW * MB * NB * R * R * sizeof(float); }
constexpr size_t tile_lds(int MB, int NB, int NWN, int KG) {
  const size_t red = (size_t)KG * MB * NB * NWN * 32 * 32 * sizeof(float), stage = (size_t)KG * 2 * 3 * 4 * (MB * 32 + 2) * 16;
  return red > stage ? red : stage;
}

template <typename K>
hipError_t launch_kernel(K kernel, const SplitGemmArgs& a, int threads, size_t lds, hipStream_t s) {
  if (lds > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
  }
  const long grid = ((long)a.mt * a.nt * a.S + 7) / 8 * 8;
  if (grid > 0x7fffffffL) return hipErrorInvalidValue;
  kernel<<<(unsigned)grid, threads, lds, s>>>(a);
  return hipGetLastError();
}

template <bool I8, bool BLK>
hipError_t launch_shape(int kind, const SplitGemmArgs& a, hipStream_t s) {
  switch (kind) {
    case 0: return launch_kernel(gemm_split_rows<16, 1, 1, 8, I8, BLK>, a, 512, rows_lds(16, 1, 1, 8), s);
    case 1: return launch_kernel(gemm_split_rows<16, 1, 2, 8, I8, BLK>, a, 512, rows_lds(16, 1, 2, 8), s);
    case 2: return launch_kernel(gemm_split_rows<32, 1, 1, 8, I8, BLK>, a, 512, rows_lds(32, 1, 1, 8), s);
    case 3:
      if constexpr (built(3, I8, BLK)) return launch_kernel(gemm_split_rows<32, 2, 2, 4, I8, BLK>, a, 256, rows_lds(32, 2, 2, 4), s);
      break;
    case 4:
      if constexpr (built(4, I8, BLK)) return launch_kernel(gemm_split_rows<32, 2, 2, 8, I8, BLK>, a, 512, rows_lds(32, 2, 2, 8), s);
      break;
    case 5: return launch_kernel(gemm_split_tile<1, 1, 2, 4, I8, BLK, 2, 2>, a, 512, tile_lds(1, 1, 2, 4), s);
    case 6:
      if constexpr (built(6, I8, BLK)) return launch_kernel(gemm_split_tile<4, 1, 4, 2, I8, BLK, 2, 2>, a, 512, tile_lds(4, 1, 4, 2), s);
      break;
    case 7:
      if constexpr (built(7, I8, BLK)) return launch_kernel(gemm_split_tile<2, 1, 4, 2, I8, BLK, 2, 2>, a, 512, tile_lds(2, 1, 4, 2), s);
      break;
    case 8:
      if constexpr (built(8, I8, BLK)) return launch_kernel(gemm_split_tile<3, 1, 4, 2, I8, BLK, 2, 2>, a, 512, tile_lds(3, 1, 4, 2), s);
      break;
  }
  return hipErrorInvalidValue;
}

}  // namespace

SplitPlan plan_gemm_split(int M, int N, int K, bool i8, bool blocked, bool with_pass, bool may_slice) {
  SplitPlan best = {0, 1};
  double best_t = 1e30;
  const int steps = (K + 31) / 32;
  for (int c = 0; c < NSHAPES; ++c) {
    const Shape& sh = SHAPES[c];
    const Shape::Fit& f = fit_of(sh, i8, blocked);
    if (!built(c, i8, blocked)) continue;
    const double tiles = (double)((M + sh.mtile - 1) / sh.mtile) * ((N + sh.ntile - 1) / sh.ntile);
    for (int S = 1; S <= (may_slice ? 8 : 1); ++S) {
      if (S > 1 && steps < 4 * S) break;
      const double load = std::ceil(tiles * S / 256.0);
      const double rounds = ((steps + S - 1) / S + sh.kpar - 1) / sh.kpar;
      double t = f.fixed + rounds * (f.one + f.more * (load - 1));
      if (S > 1) t += (with_pass ? 0.0 : 4.0) + (double)S * M * N * 8.0 / 5.0e6;  // the pass over the partial sums, at 5 TB/s
      if (t < best_t) {
        best_t = t;
        best = {c, S};
      }
    }
  }
  return best;
}

hipError_t launch_block_weights(int K, int N, bool i8, const void* src, void* dst, hipStream_t s) {
  if ((K & 7) || (N & 3)) return hipErrorInvalidValue;
  const size_t n = (size_t)(i8 ? K >> 3 : K >> 2) * N;
  if (i8) block_weights_i8<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(K, N, static_cast<const signed char*>(src), static_cast<u32x2*>(dst));
  else block_weights_f32<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(K, N, static_cast<const float*>(src), static_cast<f32x4*>(dst));
  return hipGetLastError();
}

hipError_t launch_gemm_split(const SplitPlan& p, SplitGemmArgs a, bool i8, hipStream_t s) {
  a.mt = (a.M + SHAPES[p.kind].mtile - 1) / SHAPES[p.kind].mtile;
  a.nt = (a.N + SHAPES[p.kind].ntile - 1) / SHAPES[p.kind].ntile;
  a.S = p.S;
  if (a.blocked) return i8 ? launch_shape<true, true>(p.kind, a, s) : launch_shape<false, true>(p.kind, a, s);
  return i8 ? launch_shape<true, false>(p.kind, a, s) : launch_shape<false, false>(p.kind, a, s);
}

}  // namespace wgpt
