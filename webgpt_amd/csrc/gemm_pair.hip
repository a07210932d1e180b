// The products of a model's longer prompts (FastMatMulBlock, instructions.js:157-319; int8 weights: other/int8-gemm.js:117-229)
// on the fp16 matrix cores, with the LayerNorm passes that make their rows (instructions.js:451-550).
//
// Every operand is a pair of fp16 values (pair_f16.h), made once: the weights' when a model is loaded (4 bytes a value, as in fp32;
// int8 ones are fp16 values as they are), the rows' by the kernel that finishes them. Of the four partial products of x y three
// are taken (int8: both of two). A value's pair is at most one fp32 rounding away from it, the product left out is at most 2^-22
// of x y, and a sum is rounded once per sixteen products and part, half as often as with the six products of three bf16 values
// (gemm_split.hip): from 64-bit arithmetic the sums are, norm of the errors and K slices of a launch alike, K = 576 1.25e-7 away
// against 1.32e-7, 768 1.36e-7 against 1.52e-7, 3072 2.3e-7 against 3.0e-7; below K = 384 they are further (256 1.05e-7
// against 0.90e-7), and such models keep the six products.
//
// fp16's range: a matrix of rows has one scale, a power of two from a bound that its values cannot leave. Behind a LayerNorm a
// normalised value is at most sqrt(d), so a row times gamma plus beta, its product with a column (Cauchy), GELU of that and
// averages of it (attention) are bounded by the weights alone (launch_pair_bounds). A column of weights has a scale of its own.
// Values 17 bits below the bound lose relative precision, not absolute: 2^-40 of the bound. A value behind a LayerNorm is about the root of
// the width below its column's bound, an average of T such values the root of T further, and columns below the widest one by the difference:
// how far they may be, a LayerNorm's channels too (PairSpread, model.hip), is where the error of their pairs begins to grow. Models with wider rows,
// or whose weights span more than 2^17 (more than one in 64 of a column), or leave 2^-80 .. 2^80, or are not finite, are found when they are loaded and
// keep the six products. A LayerNorm's row is finite or nothing but NaN, so no sum has to be taken again.
//
// The four waves of a workgroup split K: each holds the whole tile, its operands come straight from memory in loads of 1 KB,
// requested two steps of 16 k ahead: no barrier, no LDS and no vector instruction in the loop (int8: ten for eight weights).
// Then the waves exchange quarters of their tiles through LDS, and each finishes a quarter. What bounds it (counters of prompts of 943 x 768,
// 512 x 1024 and, int8, 300 x 1600): operands. 64 to 286 MB a launch come out of L2, 22 to 47 bytes per ns and compute unit over the whole
// launch, of which 2.5 us are stream time, 1.5 first loads, and the exchange; the matrix units, at 32 cycles an instruction, are busy in 24 to
// 32 % of the compute units' cycles (14 and 16 % in the narrow products of the attention), and these run at 1.6 to 1.9 per ns, 2.2 where few units multiply.
#include "gemm_pair.h"

#include <cmath>
#include <type_traits>
#include <utility>

#include "attention_pair.h"
#include "pair_f16.h"
#include "persistent_common.h"

namespace wgpt {
namespace {

template <class F, int... I>
__device__ __forceinline__ void unrolled_(F&& f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, class F>  // f(0) .. f(N - 1), the index a constant
__device__ __forceinline__ void unrolled(F&& f) { unrolled_(f, std::make_integer_sequence<int, N>{}); }

__device__ __forceinline__ f32x16 mfma(const u32x4& w, const u32x4& a, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, a), c, 0, 0, 0);
}
// A lane's four values in a row become one value of each of its quad's four: element `lane % 4` of lanes 0 .. 3.
__device__ __forceinline__ f32x4 transpose_quad(f32x4 v) {
  const auto swap = [](float& a, float& b, bool odd, auto perm) {
    const float got = __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(odd ? a : b), decltype(perm)::value, 0xf, 0xf, false));
    (odd ? a : b) = got;
  };
  const bool o1 = threadIdx.x & 1, o2 = threadIdx.x & 2;
  float e[4] = {v[0], v[1], v[2], v[3]};
  const std::integral_constant<int, 0xB1> by1;
  const std::integral_constant<int, 0x4E> by2;
  swap(e[0], e[1], o1, by1);
  swap(e[2], e[3], o1, by1);
  swap(e[0], e[2], o2, by2);
  swap(e[1], e[3], o2, by2);
  return f32x4{e[0], e[1], e[2], e[3]};
}
__device__ __forceinline__ unsigned ror8(unsigned v) { return __builtin_amdgcn_mov_dpp(v, 0x128, 0xf, 0xf, false); }  // from lane ^ 8
// Values of a q/k/v product, of row r of a block of rows and columns n8 + 4 half .. + 3: to the operands of attention_pair.hip, and keys
// and values to the cache too. The eight columns at n8 are a wave's, of one head (d and hs are multiples of 8), so all but the lane's place
// in them is scalar: with head, dimension and unit found by every lane the product of 512 x 3072 x 1024 took 20.2 us instead of 18.7.
// The other half of a lane's unit is with the lane 32 on (q and keys: eight dimensions of a row) or 8 on (values: eight keys):
// one of the two keeps the hi, the other the lo, and each writes 16 bytes.
__device__ __forceinline__ void put_heads(const PairGemmArgs& a, int block, int r, int half, int n8, const f32x4& v) {
  const int which = n8 < a.d ? 0 : n8 < 2 * a.d ? 1 : 2, e = n8 - which * a.d;
  const int h = __builtin_amdgcn_readfirstlane(div_by(e, a.hs, a.rhs)), dim = e - h * a.hs;
  const bool row = block * 32 + r < a.M;
  if (which && row) {
    float* const rows = (which == 2 ? a.Vc : a.Kc) + ((size_t)h * a.ctx + block * 32) * a.hs + dim;
    *reinterpret_cast<f32x4*>(rows + (r * a.hs + 4 * half)) = v;
  }
  f32x4 x = v * (which == 0 ? a.hscale[0] : which == 1 ? a.hscale[1] : a.hscale[2]);
  u32x4* const units = static_cast<u32x4*>(which == 0 ? a.heads[0] : which == 1 ? a.heads[1] : a.heads[2]) +
                       (size_t)(h * a.head_tiles + block) * (pair_attn_steps(a.hs) * 128);
  unsigned hi[2], lo[2];
  if (which == 2) {
    // (finite in fp16: a row's values are no numbers or within the bound; the rows beyond the last come from what another layer of an
    // earlier, longer prompt has left in A, for which that bound does not hold)
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = row && fabsf(x[i]) < INFINITY ? x[i] : 0.f;
    x = transpose_quad(x);  // four keys of a dimension
    pair_f16(x[0], x[1], hi[0], lo[0]);
    pair_f16(x[2], x[3], hi[1], lo[1]);
    const bool low = r & 8;
    const unsigned g0 = ror8(low ? hi[0] : lo[0]), g1 = ror8(low ? hi[1] : lo[1]);
    units[(dim >> 5) * 256 + (dim & 31) + ((r >> 4) * 128 + (low ? 64 : 0) + ((r >> 2) & 1) * 32 + 4 * half + (r & 3))] =
        low ? u32x4{g0, g1, lo[0], lo[1]} : u32x4{hi[0], hi[1], g0, g1};
  } else {
    pair_f16(x[0], x[1], hi[0], lo[0]);
    pair_f16(x[2], x[3], hi[1], lo[1]);
    const auto s0 = __builtin_amdgcn_permlane32_swap(hi[0], lo[0], false, false), s1 = __builtin_amdgcn_permlane32_swap(hi[1], lo[1], false, false);
    units[(dim >> 4) * 128 + ((dim >> 3) & 1) * 32 + (64 * half + r)] = u32x4{s0[0], s1[0], s0[1], s1[1]};
  }
}

// MB x NB blocks of 32 rows and 32 columns. Two workgroups to a compute unit (three of the small tiles), which fill each other's waits.
template <int MB, int NB, bool I8>
__global__ __launch_bounds__(256, MB * NB <= 4 ? 3 : 2) void gemm_pair_kernel(PairGemmArgs a) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  // consecutive tiles (rows fastest: they share the columns of W) go to one XCD
  const int total = a.mt * a.nt * a.S, per = (total + 7) >> 3;
  int t = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || t >= total) return;
  const int mi = t % a.mt;
  t /= a.mt;
  const int ni = t % a.nt, slice = t / a.nt;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, half = lane >> 5;
  const int K16 = (a.K + 15) >> 4, part = slice * 4 + wave, parts = a.S * 4;
  const int it0 = (int)((long)K16 * part / parts), it1 = (int)((long)K16 * (part + 1) / parts);
  const int col_blocks = (a.N + 31) >> 5;
  const __amdgpu_buffer_rsrc_t xb = buffer_of(a.A, (size_t)a.row_blocks * K16 * 2048);
  const __amdgpu_buffer_rsrc_t wb = buffer_of(a.W, I8 ? (size_t)a.K * a.N : (size_t)col_blocks * K16 * 2048);
  const int l16 = 16 * lane;
  int xo[MB], wo[NB];  // byte offsets of the blocks (int8: of the lane's column); blocks beyond the last repeat it
#pragma unroll
  for (int i = 0; i < MB; ++i) {
    const int b = mi * MB + i;
    xo[i] = (b < a.row_blocks ? b : a.row_blocks - 1) * K16 * 2048;
  }
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    if constexpr (I8) {
      const int n = (ni * NB + j) * 32 + r;
      wo[j] = 8 * ((n < a.N ? n : a.N - 1) + half * a.N);
    } else {
      const int b = ni * NB + j;
      wo[j] = (b < col_blocks ? b : col_blocks - 1) * K16 * 2048;
    }
  }
  f32x16 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  // two steps' operands: parts 0 (hi) and 1 (lo); int8 weights as they come, and as fp16
  u32x4 x[2][MB][2], w[2][NB][I8 ? 1 : 2], wf[2][NB];
  const auto load_x = [&](int u, int it, int i, int p) {
    x[u][i][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(xb, l16, xo[i] + it * 2048 + p * 1024, 0));
  };
  const auto load_w = [&](int u, int it, int j, int p) {
    if constexpr (I8) {  // (a run of eight k beyond K comes back as zeros; the rows are zeros there too)
      const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(wb, wo[j], 16 * it * a.N, 0);
      w[u][j][0][0] = v[0], w[u][j][0][1] = v[1];
    } else {
      w[u][j][p] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(wb, l16, wo[j] + it * 2048 + p * 1024, 0));
    }
  };
  const auto convert = [&](int u, int o) {
    wf[u][o >> 2][o & 3] = f16_of_bytes(w[u][o >> 2][0][(o >> 1) & 1], o & 1);
  };
  // smallest products first
  constexpr int SEC = MB * NB, NMF = SEC * (I8 ? 2 : 3), NCV = I8 ? 4 * NB : 0, CV0 = NMF / 4;
  if (it0 < it1) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int it = it0 + u < it1 ? it0 + u : it1 - 1;
#pragma unroll
      for (int p = I8 ? 0 : 1; p >= 0; --p)
#pragma unroll
        for (int j = 0; j < NB; ++j) load_w(u, it, j, p);
#pragma unroll
      for (int p = 1; p >= 0; --p)
#pragma unroll
        for (int i = 0; i < MB; ++i) load_x(u, it, i, p);
    }
    unrolled<NCV>([&](auto o) { convert(0, decltype(o)::value); });
    for (int it = it0; it < it1; it += 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        if (u > 0 && it + u >= it1) break;
        const int nx = it + u + 2 < it1 ? it + u + 2 : it1 - 1;
        // One matrix instruction at a time, behind it the loads into registers that no later one of this step reads, and a
        // share of the next step's conversions.
        unrolled<NMF>([&](auto mc) {
          constexpr int m = decltype(mc)::value, sec = m / SEC, q = m % SEC, i = q / NB, j = q % NB;
          constexpr int xp = (I8 ? sec == 0 : sec == 1) ? 1 : 0;
          if constexpr (I8) {
            acc[i][j] = mfma(wf[u][j], x[u][i][xp], acc[i][j]);
            if constexpr (m < NB) load_w(u, nx, m, 0);
            if constexpr (sec == 1 && q < MB) load_x(u, nx, q, 1);
            if constexpr (m >= CV0) {
              constexpr int o0 = (m - CV0) * NCV / (NMF - CV0), o1 = (m - CV0 + 1) * NCV / (NMF - CV0);
              unrolled<o1 - o0>([&](auto o) { convert(u ^ 1, o0 + decltype(o)::value); });
            }
          } else {
            acc[i][j] = mfma(w[u][j][sec == 0 ? 1 : 0], x[u][i][xp], acc[i][j]);
            if constexpr (sec == 1 && q < NB) load_w(u, nx, q, 1);
            if constexpr (sec == 2 && q < MB) load_x(u, nx, q, 1);
          }
          if constexpr (m == NMF - 1) {
#pragma unroll
            for (int n = 0; n < NB; ++n)
              if constexpr (!I8) load_w(u, nx, n, 0);
#pragma unroll
            for (int n = 0; n < MB; ++n) load_x(u, nx, n, 0);
          }
          __builtin_amdgcn_sched_barrier(0);
        });
      }
    }
  }

  // Wave v finishes the columns 8 v .. 8 v + 7 of every block (accumulator registers 4 v .. 4 v + 3: row r, columns 8 v + 4 half ..).
  const int n_of = 8 * wave + 4 * half;
  f32x4 cs[NB], bias[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = (ni * NB + j) * 32 + n_of, nc = n < a.N ? n : 0;
    cs[j] = *reinterpret_cast<const f32x4*>(a.cscale + nc);
    if (a.end != PAIR_PART) bias[j] = *reinterpret_cast<const f32x4*>(a.bias + nc);
  }
  f32x4* red = reinterpret_cast<f32x4*>(lds);  // [finishing wave][the other three in ascending order][block][lane]
  f32x4 own[SEC];
  unrolled<4>([&](auto vc) {
    constexpr int v = decltype(vc)::value;
    if (v == wave) {
#pragma unroll
      for (int b = 0; b < SEC; ++b) own[b] = f32x4{acc[b / NB][b % NB][4 * v], acc[b / NB][b % NB][4 * v + 1], acc[b / NB][b % NB][4 * v + 2], acc[b / NB][b % NB][4 * v + 3]};
    } else {
      f32x4* to = red + ((v * 3 + (wave < v ? wave : wave - 1)) * SEC) * 64 + lane;
#pragma unroll
      for (int b = 0; b < SEC; ++b) to[b * 64] = f32x4{acc[b / NB][b % NB][4 * v], acc[b / NB][b % NB][4 * v + 1], acc[b / NB][b % NB][4 * v + 2], acc[b / NB][b % NB][4 * v + 3]};
    }
  });
  __syncthreads();
  const f32x4* from = red + wave * 3 * SEC * 64 + lane;
#pragma unroll
  for (int b = 0; b < SEC; ++b) {
    const int j = b % NB, m = (mi * MB + b / NB) * 32 + r, n = (ni * NB + j) * 32 + n_of;
    f32x4 v = (own[b] + from[b * 64]) + (from[(SEC + b) * 64] + from[(2 * SEC + b) * 64]);
    v *= cs[j];
    if (a.end == PAIR_PART) {
      if (m < a.M && n < a.N) *reinterpret_cast<f32x4*>(a.part + ((size_t)slice * a.M + m) * a.N + n) = v;
      continue;
    }
    v += bias[j];
    if (a.end == PAIR_GELU) {
      unsigned h[2], l[2];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gelu_ref(v[e]) * a.pscale;
      pair_f16(v[0], v[1], h[0], l[0]);
      pair_f16(v[2], v[3], h[1], l[1]);
      // the lane's row and the one 32 lanes on hold eight consecutive columns: one keeps their hi, the other their lo
      const auto s0 = __builtin_amdgcn_permlane32_swap(h[0], l[0], false, false), s1 = __builtin_amdgcn_permlane32_swap(h[1], l[1], false, false);
      if (m < a.M && n < a.N)
        static_cast<u32x4*>(a.P)[pair_unit(m, n & ~7, (a.N + 15) >> 4) + 64 * half] = u32x4{s0[0], s1[0], s0[1], s1[1]};
      continue;
    }
    if (a.end == PAIR_HEADS) {
      const int n8 = (ni * NB + j) * 32 + 8 * wave;
      if (mi * MB + b / NB < a.row_blocks && n8 < a.N) put_heads(a, mi * MB + b / NB, r, half, n8, v);  // (rows beyond the last have their place in its block)
      continue;
    }
    if (m >= a.M || n >= a.N) continue;
    float* c = a.C + (size_t)m * a.ldc + n;
    if (a.end == PAIR_RESIDUAL) {
      v += *reinterpret_cast<const f32x4*>(a.resid + (size_t)m * a.ldc + n);
    } else if (n >= a.d) {
      const bool val = n >= 2 * a.d;
      const int e = n - (val ? 2 : 1) * a.d, h = e / a.hs;
      c = (val ? a.Vc : a.Kc) + ((size_t)h * a.ctx + m) * a.hs + (e - h * a.hs);
    }
    *reinterpret_cast<f32x4*>(c) = v;
  }
}

// W = 1: a wave per row, four rows a workgroup. W = 4: a workgroup per row. Each lane holds eight values in G runs of 512 W.
// (layernorm_kernel's steps; memory and its latency bound it: a row is read once, with the sums of its slices in flight together.)
template <int G, int W>
__global__ __launch_bounds__(256) void ln_pair_kernel(PairLnArgs a) {
  __shared__ float sh[8];
  constexpr int RUN = 512 * W;
  const int row = W > 1 ? (int)blockIdx.x : (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6), lane = W > 1 ? threadIdx.x : threadIdx.x & 63;
  if (row >= a.M) return;
  const auto row_sum = [&](float v, float* to) {
    v = wave_sum(v);
    if constexpr (W == 1) return v;
    if ((lane & 63) == 0) to[lane >> 6] = v;
    __syncthreads();
    return (to[0] + to[1]) + (to[2] + to[3]);
  };
  // (loads of a lane beyond the row, or of a slice too many, ask for nothing and give zeros: under a branch each would be waited for)
  const size_t row_bytes = 4 * (size_t)a.d;
  float* const xr = a.x + (size_t)row * a.d;
  const __amdgpu_buffer_rsrc_t xb = buffer_of(xr, row_bytes), gb = buffer_of(a.gamma, row_bytes), bb = buffer_of(a.beta, row_bytes);
  f32x4 v[G][2], ga[G][2], be[G][2];
  float sum = 0.f;
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int h = 0; h < 2; ++h) v[g][h] = load4<0>(xb, 4 * RUN * g + 32 * lane + 16 * h);
  if (a.S > 0) {
    const __amdgpu_buffer_rsrc_t sb = buffer_of(a.bias, row_bytes);
    f32x4 p[G][2][PAIR_MAX_SLICES], bias[G][2];
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int o = 4 * RUN * g + 32 * lane + 16 * h;
#pragma unroll
        for (int s = 0; s < PAIR_MAX_SLICES; ++s) p[g][h][s] = load4<0>(buffer_of(a.part + ((size_t)s * a.M + row) * a.d, s < a.S ? row_bytes : 0), o);
        bias[g][h] = load4<0>(sb, o);
      }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        v[g][h] += ((p[g][h][0] + p[g][h][1]) + (p[g][h][2] + p[g][h][3])) + bias[g][h];
        const int k = RUN * g + 8 * lane + 4 * h;
        if (k < a.d) *reinterpret_cast<f32x4*>(xr + k) = v[g][h];
      }
  }
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      ga[g][h] = load4<0>(gb, 4 * RUN * g + 32 * lane + 16 * h);
      be[g][h] = load4<0>(bb, 4 * RUN * g + 32 * lane + 16 * h);
      sum += (v[g][h][0] + v[g][h][1]) + (v[g][h][2] + v[g][h][3]);
    }
  if (!a.out) return;
  const float mean = row_sum(sum, sh) / (float)a.d;
  float q = 0.f;
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      if (RUN * g + 8 * lane + 4 * h < a.d) {
        const f32x4 e = v[g][h] - mean;
        q += (e[0] * e[0] + e[1] * e[1]) + (e[2] * e[2] + e[3] * e[3]);
      }
  const float stdev = sqrtf(row_sum(q, sh + 4) / (float)a.d + 1e-5f), rstd = 1.0f / stdev;
  u32x4* out = static_cast<u32x4*>(a.out);
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int k = RUN * g + 8 * lane;
    if (k >= a.d) continue;
    u32x4 hi, lo;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f32x4 y;
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = (ga[g][h][i] * quotient(v[g][h][i] - mean, stdev, rstd) + be[g][h][i]) * a.scale;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        unsigned hh, ll;
        pair_f16(y[2 * i], y[2 * i + 1], hh, ll);
        hi[2 * h + i] = hh, lo[2 * h + i] = ll;
      }
    }
    const size_t u = pair_unit(row, k, (a.d + 15) >> 4);
    out[u] = hi;
    out[u + 64] = lo;
  }
}

// ---- at load ----
constexpr float PAIR_LEAST = 0x1p-80f, PAIR_MOST = 0x1p80f;
__device__ __forceinline__ bool in_range(float v) { return v == 0.f || (fabsf(v) >= PAIR_LEAST && fabsf(v) <= PAIR_MOST); }

// Workgroups of these take 32 columns times CHUNK of K, eight threads to a column. (A workgroup for all of K: 17 ms more for the
// 96 matrices of 345M to load, 10 % of it.)
constexpr int CHUNK = 128;
struct ColumnChunk {
  int c, p, n, k0, k1;
  __device__ __forceinline__ ColumnChunk(int K, int n0) {
    c = threadIdx.x & 31, p = threadIdx.x >> 5, n = n0 + (int)blockIdx.x * 32 + c;
    k0 = (int)blockIdx.y * CHUNK, k1 = k0 + CHUNK < K ? k0 + CHUNK : K;
  }
};
// Largest absolute values of the columns, as bits (zeros before); infinite where there is one or a NaN.
__global__ __launch_bounds__(256) void pair_column_max(int K, int N, const float* __restrict__ W, unsigned* top) {
  __shared__ float sh[8][32];
  const ColumnChunk t(K, 0);
  float most = 0.f;
  if (t.n < N) {
#pragma unroll
    for (int i = 0; i < CHUNK / 8; ++i) {
      const int k = t.k0 + 8 * i + t.p;
      const float v = k < t.k1 ? fabsf(W[(size_t)k * N + t.n]) : 0.f;
      most = fmaxf(most, v < INFINITY ? v : INFINITY);
    }
  }
  sh[t.p][t.c] = most;
  __syncthreads();
  if (t.p || t.n >= N) return;
#pragma unroll
  for (int i = 0; i < 8; ++i) most = fmaxf(most, sh[i][t.c]);
  atomicMax(&top[t.n], __float_as_uint(most));
}
// most = m 2^e with m in [0.5, 1): the column times 2^(15 - e)
__device__ __forceinline__ int column_exponent(float most) {
  int e = 15;
  if (most > 0.f && in_range(most)) (void)frexpf(most, &e);
  return e;
}
__global__ __launch_bounds__(256) void pair_weights_kernel(int K, int N, const float* __restrict__ W, u32x4* __restrict__ out, const float* top, int* few) {
  __shared__ int sh[8][32];
  const ColumnChunk t(K, 0);
  const float up = t.n < N ? ldexpf(1.f, 15 - column_exponent(top[t.n])) : 0.f;
  int tiny = 0;
#pragma unroll
  for (int i = 0; i < CHUNK / 64; ++i) {  // runs of eight k
    const int k8 = t.k0 / 8 + 8 * i + t.p;
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      v[u] = t.n < N && 8 * k8 + u < t.k1 ? W[(size_t)(8 * k8 + u) * N + t.n] * up : 0.f;
      tiny += v[u] != 0.f && fabsf(v[u]) < 0.25f;
    }
    u32x4 hi, lo;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      unsigned h, l;
      pair_f16(v[2 * u], v[2 * u + 1], h, l);
      hi[u] = h, lo[u] = l;
    }
    if (8 * k8 < t.k1) {
      u32x4* o = out + pair_unit((int)blockIdx.x * 32 + t.c, 8 * k8, (K + 15) >> 4);
      o[0] = hi;
      o[64] = lo;
    }
  }
  sh[t.p][t.c] = tiny;
  __syncthreads();
  if (t.p || t.n >= N) return;
#pragma unroll
  for (int i = 1; i < 8; ++i) tiny += sh[i][t.c];
  if (tiny) atomicAdd(&few[t.n], tiny);
}
// The columns' factors in the place of their largest values.
__global__ __launch_bounds__(256) void pair_weights_end(int K, int N, float* top, const int* few, unsigned* stats) {
  const int n = (int)blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  const float most = top[n];
  if (!in_range(most) || 64 * few[n] > K) atomicAdd(stats, 1u);
  top[n] = ldexpf(1.f, column_exponent(most) - 15);
}

__global__ __launch_bounds__(256) void pair_scales_kernel(int N, const float* __restrict__ scale, float* __restrict__ cscale, unsigned* stats) {
  const int n = (int)blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  cscale[n] = scale[n] / 127.0f;
  if (!in_range(scale[n])) atomicAdd(stats, 1u);
}

// |LN(x) . w + b| <= sqrt(K) |gamma w| + |beta . w + b|: the two sums of a chunk of a column at sums[chunk][column]
__global__ __launch_bounds__(256) void pair_bounds_kernel(int K, int N, const float* __restrict__ W, const int32_t* __restrict__ Wq,
                                                          const float* __restrict__ wscale, const float* __restrict__ gamma, const float* __restrict__ beta,
                                                          float2* sums) {
  __shared__ float2 sh[8][32];
  const ColumnChunk t(K, 0);
  float s = 0.f, d = 0.f;
  if (t.n < N) {
    const float ws = Wq ? wscale[t.n] / 127.0f : 1.f;
#pragma unroll
    for (int i = 0; i < CHUNK / 8; ++i) {
      const int k = t.k0 + 8 * i + t.p;
      if (k >= t.k1) break;
      const float w = Wq ? (float)((int)(Wq[(size_t)k * (N >> 2) + (t.n >> 2)] << (24 - 8 * (t.n & 3))) >> 24) * ws : W[(size_t)k * N + t.n];
      const float g = gamma[k] * w;
      s += g * g;
      d += beta[k] * w;
    }
  }
  sh[t.p][t.c] = make_float2(s, d);
  __syncthreads();
  if (t.p || t.n >= N) return;
#pragma unroll
  for (int i = 1; i < 8; ++i) s += sh[i][t.c].x, d += sh[i][t.c].y;
  sums[(size_t)blockIdx.y * N + t.n] = make_float2(s, d);
}
// A workgroup per run of n columns.
__global__ __launch_bounds__(1024) void pair_bounds_end(int K, int N, int n, PairSpread spread, const float* __restrict__ bias, float2* sums, float* bound) {
  __shared__ unsigned most;
  __shared__ int low;
  if (threadIdx.x == 0) most = 0u, low = 0;
  __syncthreads();
  const int n0 = (int)blockIdx.x * n;
  float top = 0.f;
  for (int c = n0 + threadIdx.x; c < n0 + n; c += 1024) {
    float s = 0.f, d = 0.f;
    for (int i = 0; i * CHUNK < K; ++i) {
      const float2 p = sums[(size_t)i * N + c];
      s += p.x, d += p.y;
    }
    float b = sqrtf((float)K * s) + fabsf(d + bias[c]);
    b = b < INFINITY ? b : INFINITY;
    sums[c].x = b;  // (this thread's own)
    top = fmaxf(top, b);
  }
  atomicMax(&most, __float_as_uint(top));
  __syncthreads();
  top = __uint_as_float(most);
  const float least = spread.least[blockIdx.x] * top;
  for (int c = n0 + threadIdx.x; c < n0 + n; c += 1024)
    if (sums[c].x != 0.f && sums[c].x < least) low = 1;
  __syncthreads();
  if (threadIdx.x == 0) bound[blockIdx.x] = low ? INFINITY : top;
}
// One workgroup: the largest |LayerNorm|, infinite where a channel can only be far below it, but zero: with one gain, or one bias, far
// above the others', one scale does not fit both.
__global__ __launch_bounds__(256) void pair_ln_bound_kernel(int d, float least, const float* __restrict__ gamma, const float* __restrict__ beta, float* bound) {
  __shared__ float sh[2][256];
  __shared__ int low;
  const float root = sqrtf((float)d);
  float g = 0.f, b = 0.f;
  bool odd = false;
  for (int k = threadIdx.x; k < d; k += 256) {
    odd = odd || !(fabsf(gamma[k]) < INFINITY) || !(fabsf(beta[k]) < INFINITY);
    g = fmaxf(g, fabsf(gamma[k]));
    b = fmaxf(b, fabsf(beta[k]));
  }
  sh[0][threadIdx.x] = odd ? INFINITY : g;
  sh[1][threadIdx.x] = b;
  if (threadIdx.x == 0) low = 0;
  __syncthreads();
  for (int i = 0; i < 256; ++i) g = fmaxf(g, sh[0][i]), b = fmaxf(b, sh[1][i]);
  const float v = root * g + b;
  for (int k = threadIdx.x; k < d; k += 256) {
    const float own = root * fabsf(gamma[k]) + fabsf(beta[k]);
    if (own != 0.f && own < least * v) low = 1;
  }
  __syncthreads();
  if (threadIdx.x == 0) *bound = v < INFINITY && !low ? v : INFINITY;
}
__global__ __launch_bounds__(256) void pair_rescale_kernel(int N, float factor, float* cscale) {
  const int n = (int)blockIdx.x * 256 + threadIdx.x;
  if (n < N) cscale[n] *= factor;
}

// ---- launches ----
// A launch takes about fixed + steps * one + (load - 1) * (again + steps * more) us: steps of 16 k that a wave takes, load =
// workgroups / 256, rounded up. Least-squares fits to 6000 launches on MI355X (136 to 1024 rows, 512 to 6400 columns, K from 512 to
// 6400, 1 to 4 slices; those within twice the best shape's time). The shape that they choose is 2.4 % (int8 3.6 %) from the best one in the
// geometric mean, the noise of small launches included. Tiles of 64x128, 96x96 and 128x96, of which a compute unit holds one, were the best
// for one launch in fifteen (943x3072x768: 22.9 us in 128x96, 19.4 in 64x96, two to a unit) and are not built; 32x128 neither.
struct Shape {
  int mb, nb;
  struct Fit { float fixed, one, more, again; } f32, i8;
};
constexpr Shape SHAPES[] = {
    {2, 2, {3.64f, 0.462f, 0.395f, 0.68f}, {3.95f, 0.313f, 0.198f, 0.87f}},
    {2, 3, {3.92f, 0.620f, 0.513f, 0.99f}, {4.36f, 0.382f, 0.272f, 1.30f}},
    {3, 2, {4.13f, 0.602f, 0.499f, 0.96f}, {4.46f, 0.398f, 0.304f, 1.22f}},
    {1, 2, {3.45f, 0.313f, 0.283f, 0.32f}, {3.39f, 0.240f, 0.123f, 0.55f}},
};
constexpr int NSHAPES = sizeof(SHAPES) / sizeof(SHAPES[0]);

template <int MB, int NB, bool I8>
hipError_t launch_shape(const PairGemmArgs& a, hipStream_t s) {
  constexpr size_t lds = (size_t)12 * MB * NB * 1024;
  static bool enabled = false;  // dynamic LDS size already raised
  if (lds > 64 * 1024 && !enabled) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_pair_kernel<MB, NB, I8>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    enabled = true;
  }
  const long grid = ((long)a.mt * a.nt * a.S + 7) / 8 * 8;
  if (grid > 0x7fffffffL) return hipErrorInvalidValue;
  gemm_pair_kernel<MB, NB, I8><<<(unsigned)grid, 256, lds, s>>>(a);
  return hipGetLastError();
}
template <bool I8>
hipError_t launch_kind(int kind, const PairGemmArgs& a, hipStream_t s) {
  switch (kind) {
    case 0: return launch_shape<2, 2, I8>(a, s);
    case 1: return launch_shape<2, 3, I8>(a, s);
    case 2: return launch_shape<3, 2, I8>(a, s);
    case 3: return launch_shape<1, 2, I8>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace

PairPlan plan_gemm_pair(int M, int N, int K, bool i8, bool may_slice) {
  PairPlan best = {0, 1};
  double best_t = 1e30;
  for (int c = 0; c < NSHAPES; ++c) {
    const Shape& sh = SHAPES[c];
    const Shape::Fit& f = i8 ? sh.i8 : sh.f32;
    const double tiles = (double)((M + 32 * sh.mb - 1) / (32 * sh.mb)) * ((N + 32 * sh.nb - 1) / (32 * sh.nb));
    for (int S = 1; S <= (may_slice ? PAIR_MAX_SLICES : 1); ++S) {
      const double steps = std::ceil((K + 15) / 16 / (4.0 * S)), load = std::ceil(tiles * S / 256.0);
      const double t = f.fixed + steps * f.one + (load - 1) * (f.again + steps * f.more) + (S > 1 ? (double)S * M * N * 4.0 / 5.0e6 : 0.0);  // slices read at 5 TB/s
      if (t < best_t) best_t = t, best = {c, S};
    }
  }
  return best;
}

hipError_t launch_gemm_pair(const PairPlan& p, PairGemmArgs a, bool i8, hipStream_t s) {
  a.mt = (a.M + 32 * SHAPES[p.kind].mb - 1) / (32 * SHAPES[p.kind].mb);
  a.nt = (a.N + 32 * SHAPES[p.kind].nb - 1) / (32 * SHAPES[p.kind].nb);
  a.S = p.S;
  a.row_blocks = (a.M + 31) / 32;
  // 32-bit offsets of the loads
  if (pair_rows_bytes(a.M, a.K) >= 0x80000000u || pair_weights_bytes(a.K, a.N) >= 0x80000000u || p.S < 1 || p.S > PAIR_MAX_SLICES) return hipErrorInvalidValue;
  return i8 ? launch_kind<true>(p.kind, a, s) : launch_kind<false>(p.kind, a, s);
}

hipError_t launch_ln_pair(const PairLnArgs& a, hipStream_t s) {
  // Few rows leave compute units without one of four waves' rows: a workgroup per row. Passes of a prompt (some of them with slices), us with
  // a wave and with a workgroup per row, at 150, 300, 400, 500 and 1000 rows: 768 columns 5.1 4.1, 5.4 4.8, 5.4 5.2, 5.9 5.7, 6.0 6.6; 1024 5.1 4.4, 5.2 5.4, 5.8 5.7,
  // 5.8 6.0, 5.3 6.2; 1280 6.1 4.9, 6.2 5.6, 6.3 5.9, 6.6 6.3, 6.6 7.4; 1600 6.9 5.1, 6.9 5.9, 7.3 6.5, 6.3 6.4, 8.1 8.7; 2048 7.7 5.7, 7.5 6.5, 6.5 6.5, 6.8 7.0,
  // 8.4 10.2: the sides meet between 300 and 600 rows. (Rows above 2048 would be two runs of a workgroup, which are not built.)
  if (a.M <= 400 && a.d <= 2048) {
    ln_pair_kernel<1, 4><<<(unsigned)a.M, 256, 0, s>>>(a);
    return hipGetLastError();
  }
  const unsigned grid = (unsigned)(a.M + 3) / 4;
  switch ((a.d + 511) / 512) {
    case 1: ln_pair_kernel<1, 1><<<grid, 256, 0, s>>>(a); break;
    case 2: ln_pair_kernel<2, 1><<<grid, 256, 0, s>>>(a); break;
    case 3: ln_pair_kernel<3, 1><<<grid, 256, 0, s>>>(a); break;
    case 4: ln_pair_kernel<4, 1><<<grid, 256, 0, s>>>(a); break;
    case 5:
    case 6: ln_pair_kernel<6, 1><<<grid, 256, 0, s>>>(a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_pair_weights(int K, int N, const float* W, void* out, float* cscale, int* few, unsigned* stats, hipStream_t s) {
  const dim3 grid((N + 31) / 32, (K + CHUNK - 1) / CHUNK);
  pair_column_max<<<grid, 256, 0, s>>>(K, N, W, reinterpret_cast<unsigned*>(cscale));
  pair_weights_kernel<<<grid, 256, 0, s>>>(K, N, W, static_cast<u32x4*>(out), cscale, few);
  pair_weights_end<<<(N + 255) / 256, 256, 0, s>>>(K, N, cscale, few, stats);
  return hipGetLastError();
}
hipError_t launch_pair_scales(int N, const float* scale, float* cscale, unsigned* stats, hipStream_t s) {
  pair_scales_kernel<<<(N + 255) / 256, 256, 0, s>>>(N, scale, cscale, stats);
  return hipGetLastError();
}
size_t pair_bounds_floats(int K, int N) { return (size_t)2 * ((K + CHUNK - 1) / CHUNK) * N; }
hipError_t launch_pair_bounds(int K, int N, int runs, PairSpread spread, const float* W, const int32_t* Wq, const float* wscale, const float* bias,
                              const float* gamma, const float* beta, float* sums, float* bound, float* ln_bound, hipStream_t s) {
  float2* const p = reinterpret_cast<float2*>(sums);
  pair_bounds_kernel<<<dim3((N + 31) / 32, (K + CHUNK - 1) / CHUNK), 256, 0, s>>>(K, N, W, Wq, wscale, gamma, beta, p);
  pair_bounds_end<<<runs, 1024, 0, s>>>(K, N, N / runs, spread, bias, p, bound);
  pair_ln_bound_kernel<<<1, 256, 0, s>>>(K, spread.ln, gamma, beta, ln_bound);
  return hipGetLastError();
}
hipError_t launch_pair_rescale(int N, float factor, float* cscale, hipStream_t s) {
  pair_rescale_kernel<<<(N + 255) / 256, 256, 0, s>>>(N, factor, cscale);
  return hipGetLastError();
}

}  // namespace wgpt
