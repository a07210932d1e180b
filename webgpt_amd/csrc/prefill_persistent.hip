// The forward of a short prompt (GPT.run, model.js:104-268, on a window of up to PP_MAX_T tokens) as one persistent launch.
//
// A launch per block costs a short prompt 3 to 5 us of fixed time for each of its 7 or 8 dependent launches a layer, more than
// its operations and bytes (117M, 13 tokens: 86 launches in 0.50 ms for 340 MB of weights, 52 us at the rate of reads).
// Calls of wgpt_prefill with launches, with this kernel on plain values (three bf16 values each beside int8 weights), and on pairs of
// fp16 values, ms: 117M 1 token 0.50, 0.37, 0.35, 13 0.55, 0.39, 0.37, 45 0.45 (plain), 0.41, 128 0.79, 0.56, 0.48; toy 64 0.28, 0.17 (plain).
// Twelve layers, plain and pairs: 345M 100 tokens 0.71, 0.59, 774M 64 0.71, 0.62, 128 1.01, 0.85; 24 of 1.5B int8, 16 tokens 1.10, 0.99, 128
// 1.90, 1.71. Clock stamps of a layer of 117M on plain values, which is 30 us with them at 13 rows and 43 at 128: from the last flag to the end of a wait 0.3 to 1.4 us (0.4 to 1.4 at 128 rows), sums,
// epilogue, stores and the flag 0.8 to 1.1 a phase (0.6 to 1.2), loads with LayerNorm and products c_attn 2.5 (7.3), attention 2.7 (4.0), c_proj
// 2.1 (2.4), c_fc 3.1 (8.6), the second MLP product 5.7 (9.1; at 13 rows a compute unit reads all hidden rows for four columns), the last workgroup 0.6
// to 2.4 behind the median. The matrix units were busy for 11 % of the launch at 13 rows and 31 % at 128, 14 us a layer of the 27 in its
// products; on pairs for 10 % at 128, 4 us a layer.
// The compiler spills 218 to 329 scalar registers into vector lanes.
// Here one workgroup per compute unit stays for the whole forward and the blocks are phases of it:
//
//   - workgroups form a grid of row groups (16 rows of the prompt, the rows of a matrix instruction) times column groups;
//     a linear layer's output columns are dealt to the column groups. The workgroups of one column group are on one XCD, so
//     the weights that they share come out of its L2;
//   - inside a workgroup the eight waves split the contraction; a wave multiplies its slice of the 16 rows with its slice of
//     all columns of the workgroup on the matrix cores, and the partial tiles meet in LDS. Weights and rows are the pairs of fp16
//     values and the scales of gemm_pair.hip where the model has them and its rows are wide enough (PP_PAIR_ABOVE); the attention's
//     output and the hidden rows travel as pairs. Else fp32 values are multiplied as they are, and beside int8 weights rows are
//     exact sums of three bf16 values (split_bf16.h, gemm_split.hip);
//   - LayerNorm is applied to the rows in registers on their way in (statistics of a row: each wave about its own mean,
//     merged through LDS), GELU, bias and residual are epilogues, and a workgroup keeps the residual stream of its columns;
//   - rows pass from phase to phase through memory with write-through stores at device scope; a workgroup that has finished a
//     phase waits for its stores and raises its flag to the phase's epoch, and a wave waits for the flags of those workgroups
//     whose columns it multiplies. The first weights of a phase are requested before that wait;
//   - a (head, row group) of the attention is one workgroup, a wave of it the 16 keys of one row group, with fp32 matrix
//     instructions; the waves' outputs are merged in LDS;
//   - at the end all workgroups normalise the last row and take their run of the vocabulary.
//
// No buffer is overwritten while somebody may still read it: every wave range of a phase waits for all workgroups that write
// its columns, the eight waves of a workgroup together for all writers, and between a buffer's use in a layer and its next
// writing in the layer behind it lies the second MLP product, for which every writer of hidden rows must have finished. Keys and
// values, which later row groups read too, have rows of their own in the cache.
//
// Every wait is bounded. A wait that expires, and sums that the split may have spoilt (spoilt, gemm_split.hip), end the launch
// early with a word for the host, which then runs the prompt with a launch per block. A flag is looked at with relaxed atomic loads at device
// scope, and the rows behind it are read with device-scope loads (sc1) that the compiler cannot move above them; they were stored
// at that scope and had arrived (s_waitcnt) before the flag was raised.
#include "prefill_persistent.h"

#include "pair_f16.h"
#include "persistent_common.h"

namespace wgpt {
namespace {

constexpr int NT = PP_THREADS, NW = NT / 64;
struct Flags {
  unsigned* flags;
  unsigned ebase, spin_limit;
  int* host_err;
  int* bail;  // LDS
  __device__ __forceinline__ int bailed() const { return __hip_atomic_load(bail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
  __device__ __forceinline__ unsigned* word(int rg, int cg) const { return flags + 64 + rg * PP_GRID + cg; }
  // The launch cannot go on: other workgroups find its epoch in the error word, the host the reason.
  __device__ __forceinline__ void give_up(int why) const {
    *bail = 1;
    __hip_atomic_store(flags, ebase + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    *host_err = why;
  }
  // One wave: n flags, the i-th that of at(i), have reached epoch ep (or the launch has given up).
  template <class At>
  __device__ __forceinline__ void wait(int n, unsigned ep, int lane, At at, bool patient = false) const {
    for (int i0 = 0; i0 < n; i0 += 64) {
      const unsigned* p = i0 + lane < n ? at(i0 + lane) : nullptr;
      for (unsigned spins = 0;;) {
        const bool missing = p && (int)(ld_flag(p) - ep) < 0;
        if (!__builtin_amdgcn_ballot_w64(missing)) break;
        if (bailed()) return;
        ++spins;
        if (spins > spin_limit) {
          if (lane == 0) give_up(PP_ERR_WAIT);
          return;
        }
        if ((spins & 15u) == 0 && ld_flag(flags) == ebase + 1u) {
          *bail = 1;
          return;
        }
        if (patient) __builtin_amdgcn_s_sleep(64);
        else __builtin_amdgcn_s_sleep(1);
      }
    }
    asm volatile("" ::: "memory");
  }
};

constexpr bool is_i8(int mode) { return mode & 1; }
constexpr bool is_pair(int mode) { return mode & 2; }

// Eight consecutive k of one column: floats, the hi and lo halves of pairs, or bytes.
template <int MODE>
struct WSlice8 {
  unsigned v[is_i8(MODE) ? 2 : 8];
  __device__ __forceinline__ u32x4 bf16() const {
    u32x4 h;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const unsigned x = v[i >> 1], sh = 16 * (i & 1);
      h[i] = bf16_pair((float)((int)(x << (24 - sh)) >> 24), (float)((int)(x << (16 - sh)) >> 24));
    }
    return h;
  }
  __device__ __forceinline__ u32x4 f16() const { return u32x4{f16_of_bytes(v[0], 0), f16_of_bytes(v[0], 1), f16_of_bytes(v[1], 0), f16_of_bytes(v[1], 1)}; }
};
// The same for NS steps of 32 k, in the order of launch_block_weights, or of pair_unit.
template <int MODE, int NS>
struct WSlice {
  WSlice8<MODE> s[NS];
  // Column n of N (nok: there is one) from step `step` on, cnt steps of them; a lane's place in the step is its kg, the step's
  // a scalar offset.
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, int N, int K8, int n, bool nok, int step, int cnt, int kg) {
    constexpr bool I8 = is_i8(MODE), UNITS = MODE == PP_PAIR_F32;
    const int o = nok ? (UNITS ? ((n >> 5) * ((K8 + 1) >> 1) + (kg >> 1)) * 2048 + (kg & 1) * 512 + (n & 31) * 16 : (I8 ? 8 : 32) * kg * N + (I8 ? 8 : 16) * n) : OUT;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
      const int left = i < cnt ? K8 - 4 * (step + i) : 0, so = UNITS ? 4096 * (i < cnt ? step + i : 0) : (I8 ? 32 : 128) * N * (i < cnt ? step + i : 0);
      const int oi = kg < left ? o : OUT;
      if constexpr (I8) {
        const u32x2 x = __builtin_amdgcn_raw_buffer_load_b64(b, oi, so, 0);
        s[i].v[0] = x[0], s[i].v[1] = x[1];
      } else {
        const u32x4 x = __builtin_amdgcn_raw_buffer_load_b128(b, oi, so, 0), y = __builtin_amdgcn_raw_buffer_load_b128(b, oi, so + (UNITS ? 1024 : 16 * N), 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[i].v[e] = x[e], s[i].v[4 + e] = y[e];
      }
    }
  }
};
// The memory of a weight matrix [K, N].
template <int MODE>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t weights_of(const void* W, size_t K, int N) {
  return buffer_of(W, MODE == PP_PAIR_F32 ? (size_t)((N + 31) >> 5) * ((K + 15) >> 4) * 2048 : K * N * (is_i8(MODE) ? 1 : 4));
}

// Eight k of one row as the products take them, from two runs of four floats, or from the hi and lo halves of pairs.
template <int MODE>
struct Operand {
  u32x4 hi, lo;
  __device__ __forceinline__ void set(const f32x4 (&x)[2]) { hi = __builtin_bit_cast(u32x4, x[0]), lo = __builtin_bit_cast(u32x4, x[1]); }
};
template <>
struct Operand<PP_SPLIT_I8> {
  Split8 v;
  __device__ __forceinline__ void set(const f32x4 (&x)[2]) { v = split8(x[0], x[1]); }
};
template <>
struct Operand<PP_PLAIN_F32> {
  f32x4 v[2];
  __device__ __forceinline__ void set(const f32x4 (&x)[2]) { v[0] = x[0], v[1] = x[1]; }
};
template <int MODE, int N>
struct Operands {
  Operand<MODE> v[N];
  __device__ __forceinline__ void set(const f32x4 (&x)[N][2]) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i].set(x[i]);
  }
};
__device__ __forceinline__ f32x4 mfma(const u32x4& w, const u32x4& x, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma_f16(const u32x4& w, const u32x4& x, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, x), c, 0, 0, 0);
}
// Products of N steps of 32 k. Pairs: all four products (with the three of gemm_pair.hip the logits of 12 layers of 117M at 128 tokens
// were 3.3e-7 from 64-bit arithmetic; 3.1e-7 with four, and 3.1e-7 with plain values; at 117M's other lengths and from 576 to
// 1600 columns four are as close as plain values or closer).
// Else, int8: a weight is one bf16 value, a row's the sum of three (the products of gemm_split.hip).
// fp32: fp32 matrix instructions, which round after every product; four sums and their tree keep the chains short: the logits
// of 8 layers of 117M are 3.3e-7 from 64-bit arithmetic (one chain in two 4.5e-7; the launches of gemm_split.hip 3.8e-7). (Six
// bf16 products for an fp32 one take a third of the matrix units' time of these eight instructions, but eleven vector
// instructions for every two weights and rows: c_fc of 13 rows of 768 2.1 us of its phase, 1.5 with these.)
template <int N>
__device__ __forceinline__ f32x4 products(const WSlice8<PP_PAIR_F32> (&w)[N], const Operands<PP_PAIR_F32, N>& x) {
  f32x4 acc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const u32x4 hi = {w[i].v[0], w[i].v[1], w[i].v[2], w[i].v[3]}, lo = {w[i].v[4], w[i].v[5], w[i].v[6], w[i].v[7]};
    acc[0] = mfma_f16(lo, x.v[i].lo, acc[0]);
    acc[1] = mfma_f16(hi, x.v[i].lo, acc[1]);
    acc[0] = mfma_f16(lo, x.v[i].hi, acc[0]);
    acc[2 + (i & 1)] = mfma_f16(hi, x.v[i].hi, acc[2 + (i & 1)]);
  }
  return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}
template <int N>
__device__ __forceinline__ f32x4 products(const WSlice8<PP_PAIR_I8> (&w)[N], const Operands<PP_PAIR_I8, N>& x) {
  f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const u32x4 wv = w[i].f16();
    acc[0] = mfma_f16(wv, x.v[i].lo, acc[0]);
    acc[1] = mfma_f16(wv, x.v[i].hi, acc[1]);
  }
  return acc[0] + acc[1];
}
template <int N>
__device__ __forceinline__ f32x4 products(const WSlice8<PP_SPLIT_I8> (&w)[N], const Operands<PP_SPLIT_I8, N>& x) {
  f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const u32x4 wv = w[i].bf16();
    acc[0] = mfma(wv, x.v[i].v.lo, acc[0]);
    acc[1] = mfma(wv, x.v[i].v.mid, acc[1]);
    acc[0] = mfma(wv, x.v[i].v.hi, acc[0]);
  }
  return acc[0] + acc[1];
}
template <int N>
__device__ __forceinline__ f32x4 products(const WSlice8<PP_PLAIN_F32> (&w)[N], const Operands<PP_PLAIN_F32, N>& x) {
  f32x4 acc[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) acc[e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < N; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e & 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[i].v[e]), x.v[i].v[e >> 2][e & 3], acc[e & 3], 0, 0, 0);
  return (acc[0] + acc[1]) + (acc[2] + acc[3]);
}
// int8 sums that the split may have spoilt, as in gemm_split.hip: not finite, from 2^124 on, under 2^-60 but zero. (Of the prompt's rows
// only: those of the last row group beyond it hold what earlier prompts or other owners of the memory have left.)
template <int MODE>
__device__ __forceinline__ bool spoilt(const f32x4& v) {
  bool bad = false;
  if constexpr (MODE == PP_SPLIT_I8) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float m = fabsf(v[i]);
      bad = bad || !(m < 0x1p124f) || (m < 0x1p-60f && m > 0.f);
    }
  }
  return bad;
}

// The launch's arguments where they lie: what a phase needs of them is read again (scalar loads) rather than kept in, and
// spilled from, registers for the whole kernel.
typedef const __attribute__((address_space(4))) PrefillArgs ConstArgs;
__device__ __forceinline__ ConstArgs* fresh_args() {
  ConstArgs* p = (ConstArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}
typedef const __attribute__((address_space(4))) PrefillLayer ConstLayer;
__device__ __forceinline__ ConstLayer* fresh_layer(int li) {
  ConstLayer* p = (ConstLayer*)(size_t)fresh_args()->layers + li;
  asm volatile("" : "+s"(p));
  return p;
}
typedef const __attribute__((address_space(4))) PrefillScales ConstScales;
template <int MODE>
__device__ __forceinline__ float row_scale(int li, float PrefillScales::*of) {
  if constexpr (!is_pair(MODE)) return 1.f;
  ConstArgs* a = fresh_args();
  return ((ConstScales*)((ConstLayer*)(size_t)a->layers + a->L) + li)->*of;
}

// Rows travel between the workgroups of a row group in the order in which their readers load them, [K / 8][2][16 rows][4]: a
// load of a wave is 256 contiguous bytes for each of its four k. (With rows of K floats the sixteen rows of a load lie in one
// or a few channels of the L2, the same ones for every workgroup: the second MLP product of 128 rows of 768 took 19.8 us, 12.4
// in this order and with requests two chunks ahead.)
__device__ __forceinline__ int row_offset(int r, int k) { return ((k >> 2) * PP_ROWS + r) * 4; }
// Four values of a row of the attention's output or the hidden rows to their readers: as pairs, where these take pairs (made by every
// reader, 96 values a lane at 13 rows of 3072 would be 0.9 us of the phase), with hi and lo in the place of the two runs of four.
template <int MODE>
__device__ __forceinline__ void put_row(float* rows, int r, int k, const f32x4& v, float scale) {
  if constexpr (is_pair(MODE)) {
    unsigned hi[2], lo[2];
    pair_f16(v[0] * scale, v[1] * scale, hi[0], lo[0]);
    pair_f16(v[2] * scale, v[3] * scale, hi[1], lo[1]);
    float* const p = rows + row_offset(r, k & ~7) + ((k >> 1) & 2);
    st_agent2(p, u32x2{hi[0], hi[1]});
    st_agent2(p + 4 * PP_ROWS, u32x2{lo[0], lo[1]});
  } else {
    st_agent(rows + row_offset(r, k), v);
  }
}

// HJ: head sizes up to 16 HJ.
template <int MODE, int NS, int HJ>
__global__ __launch_bounds__(NT, 2) void prefill_persistent_kernel(PrefillArgs) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  constexpr bool I8 = is_i8(MODE), PAIR = is_pair(MODE), SCALED = I8 || PAIR;  // (columns have factors)
  constexpr int LN = 256 * NS;  // the widest row of this instantiation
  constexpr int CH = NS < 3 ? NS : 3;  // steps of a chunk of the 4d-long contraction
  __shared__ int bail;
  __shared__ float2 stat[NW][PP_ROWS], cnt[NW];
  __shared__ f32x4 lnp[LN / 2];
  ConstArgs* const a0 = fresh_args();
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d = a0->d, T = a0->T, L = a0->L, groups = a0->groups, cpA = a0->cpA, cpC = a0->cpC, cpD = a0->cpD;
  const int slot = blockIdx.x >> 3, rg = slot % groups, cg = (blockIdx.x & 7) * a0->per_xcd + slot / groups;
  const bool rows_here = slot < groups * a0->per_xcd;
  const Flags fl = {a0->flags, a0->ebase, a0->spin_limit, a0->host_err, &bail};
  f32x4* red = reinterpret_cast<f32x4*>(lds);

  const auto cols_of = [&](int N, int cp) { const int n = N - cg * cp; return n > cp ? cp : n < 0 ? 0 : n; };
  const int ncA = cols_of(3 * d, cpA), ncC = cols_of(d, cpC), ncD = cols_of(4 * d, cpD);
  const int tilesA = (ncA + 15) >> 4, tilesC = (ncC + 15) >> 4, tilesD = (ncD + 15) >> 4;
  // slices of the contraction, in steps of 32
  const int st1 = (d + 31) >> 5, st4 = (4 * d + 31) >> 5, K81 = d >> 3, K84 = d >> 1;
  const int s1 = st1 * wave / NW, n1 = st1 * (wave + 1) / NW - s1, s4 = st4 * wave / NW, n4 = st4 * (wave + 1) / NW - s4;
  const auto last_col = [&](int step, int n, int K) { const int k = 32 * (step + n); return (k < K ? k : K) - 1; };
  if (tid < NW) {
    const int k0 = 32 * (st1 * tid / NW), k1 = 32 * (st1 * (tid + 1) / NW), n = (k1 < d ? k1 : d) - k0;  // elements of a row in wave tid
    cnt[tid] = make_float2((float)n, n > 0 ? 1.0f / (float)n : 0.f);
  }
  if (tid == 0) bail = 0;
  __syncthreads();

  // what a thread finishes of a [16, columns] result: four columns of a row in tiles et, et + 8
  const int er = tid & 15, ec = 4 * ((tid >> 4) & 3), et = wave;
  const int em = rg * PP_ROWS + er;
  f32x4 res = {0.f, 0.f, 0.f, 0.f};  // residual stream: row em, columns cg * cpC + 16 * et + ec ..
  // What the next phase needs first is requested when this one has raised its flag, in front of the wait for the others'. (A phase
  // earlier, behind the requests for the rows, the weights were in the way of the stores and flags of the phase: 117M, 13 tokens
  // 0.495 ms against 0.415.)
  WSlice<MODE, NS> w_next;                    // weights of its first tile
  f32x4 bias_next[2], scale_next[2];        // of this thread's columns
  constexpr int RING = I8 || NS < 6 ? 2 : 1;  // tiles whose weights are on their way
  const auto request_w = [&](WSlice<MODE, NS>& to, const void* W, int N, int cp, int nc, int t) {
    const int o = opaque(lane), n = 16 * t + (o & 15);
    to.load(weights_of<MODE>(W, d, N), N, K81, cg * cp + n, n < nc, s1, n1, o >> 4);
  };
  const auto request_cols = [&](const float* b, const float* s, int N, int cp, int nc) {
    const __amdgpu_buffer_rsrc_t bb = buffer_of(b, 4 * (size_t)N), sb = buffer_of(SCALED ? s : b, 4 * (size_t)N);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int n = 16 * (et + NW * i) + (4 * (opaque(tid) >> 4) & 12), o = n < nc ? 4 * (cg * cp + n) : OUT;
      bias_next[i] = load4<0>(bb, o);
      if constexpr (SCALED) scale_next[i] = load4<0>(sb, o);
    }
  };
  // Gamma and beta of the next LayerNorm: a float4 of each per thread, on their way while the workgroup waits for the rows.
  f32x4 gamma = {0.f, 0.f, 0.f, 0.f}, beta = gamma;
  const auto request_ln = [&](const float* g, const float* b) {
    const int o = 4 * opaque(tid) < d ? 16 * opaque(tid) : OUT;
    gamma = load4<0>(buffer_of(g, 4 * (size_t)d), o);
    beta = load4<0>(buffer_of(b, 4 * (size_t)d), o);
  };
  // N steps of the rows that the row group exchanges in `src` (K8 runs of eight a row), from step `step` on, cnt of them.
  const auto load_rows = [&](auto& x, const float* src, int K8, int step, int cnt) {
    constexpr int N = sizeof(x) / sizeof(x[0]);
    const __amdgpu_buffer_rsrc_t b = buffer_of(src + (size_t)rg * PP_ROWS * 8 * K8, (size_t)PP_ROWS * 32 * K8);
    const int ol = opaque(lane), kg = ol >> 4, base = 32 * PP_ROWS * kg + 16 * (ol & 15);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int left = i < cnt ? K8 - 4 * (step + i) : 0, so = 128 * PP_ROWS * (i < cnt ? step + i : 0), o = kg < left ? base : OUT;
      x[i][0] = load4<SC1>(b, o, so);
      x[i][1] = load4<SC1>(b, o, so + 16 * PP_ROWS);
    }
  };
  // LayerNorm of the wave's slice (instructions.js:451-550), as pairs where the products take them; all waves take part.
  const auto normalise = [&](f32x4 (&x)[NS][2], float scale) {
    const int ol = opaque(lane), row = ol & 15, kg = ol >> 4;
    float sum = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
      for (int h = 0; h < 2; ++h) sum += (x[s][h][0] + x[s][h][1]) + (x[s][h][2] + x[s][h][3]);
    sum = quad_sum(sum);
    const float mw = sum * cnt[wave].y;
    float q = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const bool in = s < n1 && (s1 + s) * 4 + kg < K81;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const float e0 = x[s][h][0] - mw, e1 = x[s][h][1] - mw, e2 = x[s][h][2] - mw, e3 = x[s][h][3] - mw;
        q += in ? (e0 * e0 + e1 * e1) + (e2 * e2 + e3 * e3) : 0.f;
      }
    }
    q = quad_sum(q);
    if (kg == 0) stat[wave][row] = make_float2(sum, q);
    if (tid < LN / 4) {
      lnp[tid] = gamma;
      lnp[LN / 4 + tid] = beta;
    }
    __syncthreads();
    float total = 0.f, m2 = 0.f;
    float2 p[NW];
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      p[v] = stat[v][row];
      total += p[v].x;
    }
    const float fd = (float)d, rd = 1.0f / fd, mean = quotient(total, fd, rd);
#pragma unroll
    for (int v = 0; v < NW; ++v) {
      const float2 c = cnt[v];
      const float e = p[v].x * c.y - mean;
      m2 += p[v].y + (c.x * e) * e;  // (0 for a wave without elements, also where e * e overflows)
    }
    const float stdev = sqrtf(m2 / fd + 1e-5f), rstd = 1.0f / stdev;  // (m2 may be infinite)
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int k8 = (s1 + s) * 4 + kg;
      // beyond the slice the weights are zero and x becomes zero too, whatever the mean: an entry behind the row, of zeros (a row that
      // fills all entries has nothing beyond a slice)
      const bool in = s < n1 && k8 < K81;
      const f32x4* lg = lnp + 2 * (in ? k8 : K81);
      const float r = in ? rstd : 0.f;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const f32x4 g = lg[h], be = lg[LN / 4 + h];
#pragma unroll
        for (int i = 0; i < 4; ++i) x[s][h][i] = g[i] * quotient(x[s][h][i] - mean, stdev, r) + be[i];
      }
      if constexpr (PAIR) {
        u32x4 hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          unsigned a, b;
          pair_f16(x[s][i >> 1][2 * (i & 1)] * scale, x[s][i >> 1][2 * (i & 1) + 1] * scale, a, b);
          hi[i] = a, lo[i] = b;
        }
        x[s][0] = __builtin_bit_cast(f32x4, hi), x[s][1] = __builtin_bit_cast(f32x4, lo);
      }
    }
  };
  // Products of the wave's slice of a d-long contraction with the workgroup's columns; partial tiles to `red`.
  const auto multiply = [&](const f32x4 (&x)[NS][2], WSlice<MODE, NS> (&w)[RING], const void* W, int N, int cp, int nc, int tiles) {
    Operands<MODE, NS> xs;
    xs.set(x);
    bool bad = false;
    const auto tile = [&](WSlice<MODE, NS>& wt, int t) {
      const f32x4 v = products(wt.s, xs);
      if (t + RING < tiles) request_w(wt, W, N, cp, nc, t + RING);
      bad = bad || (em < T && spoilt<MODE>(v));
      red[(wave * tiles + t) * 64 + opaque(lane)] = v;
    };
#pragma unroll 1
    for (int t = 0; t < tiles; t += RING) {
      tile(w[0], t);
      if (RING > 1 && t + 1 < tiles) tile(w[RING - 1], t + 1);
    }
    if (__builtin_amdgcn_ballot_w64(bad) && lane == 0) fl.give_up(PP_ERR_SPLIT);
  };
  // Sum of the eight partial tiles: tile et + 8 i, this thread's row and columns.
  const auto finished = [&](int tiles, int slot, const f32x4 (&bias)[2], const f32x4 (&scale)[2]) {
    const f32x4* p = red + (et + NW * slot) * 64 + opaque(lane);
    f32x4 u[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) u[i] = p[i * tiles * 64];
    f32x4 v = ((u[0] + u[1]) + (u[2] + u[3])) + ((u[4] + u[5]) + (u[6] + u[7]));
    if constexpr (PAIR) v *= scale[slot];
    else if constexpr (I8) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= scale[slot][e] / 127.0f;
    }
    return v + bias[slot];
  };
  // All stores of the workgroup have reached the level at which the compute units agree; its flag says so.
  const auto raise = [&](unsigned ep) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) __hip_atomic_store(fl.word(rg, cg), ep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  const auto wait_cols = [&](int cp, float rcp, int c0, int c1, unsigned ep) {  // columns c0..c1 of this row group
    const int g0 = div_by(c0, cp, rcp);
    fl.wait(div_by(c1, cp, rcp) - g0 + 1, ep, lane, [&](int i) { return fl.word(rg, g0 + i); });
  };
  // (A workgroup without columns of a phase requests nothing with the same instructions: registers that are written on one path
  // only would have to be kept through all phases.)
  const auto request_A = [&](int li) {
    ConstLayer* ly = fresh_layer(li);
    request_w(w_next, ly->wA, 3 * d, cpA, ncA, 0);
    request_ln(ly->ln1g, ly->ln1b);
    request_cols(ly->bA, ly->sA, 3 * d, cpA, ncA);
  };
  const auto request_D = [&](int li) {
    ConstLayer* ly = fresh_layer(li);
    request_w(w_next, ly->wD, 4 * d, cpD, ncD, 0);
    request_ln(ly->ln2g, ly->ln2b);
    request_cols(ly->bD, ly->sD, 4 * d, cpD, ncD);
  };
  // The phase takes over what was requested for it; the weights of its second tile.
  const auto take = [&](WSlice<MODE, NS> (&w)[RING], f32x4 (&bias)[2], f32x4 (&scale)[2], const void* W, int N, int cp, int nc) {
    w[0] = w_next;
    if (RING > 1) request_w(w[RING - 1], W, N, cp, nc, 1);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      bias[i] = bias_next[i];
      if constexpr (SCALED) scale[i] = scale_next[i];
    }
  };

  if (rows_here) {
    request_A(0);
    if (et < tilesC && 16 * et + ec < ncC) {
      const int n = cg * cpC + 16 * et + ec, m = em < T ? em : T - 1;
      res = *reinterpret_cast<const f32x4*>(a0->wte + (size_t)a0->tok[m] * d + n) + *reinterpret_cast<const f32x4*>(a0->wpe + (size_t)m * d + n);
    }
    unsigned ep = fl.ebase;
    for (int li = 0; li < L; ++li, ep += 5) {
      // ---- c_attn: LN1, q/k/v; keys and values to their rows of the cache ----
      if (tilesA) {
        f32x4 x[NS][2], bias[2], scale[2];
        WSlice<MODE, NS> w[RING];
        ConstArgs* a = fresh_args();
        if (li == 0) {  // the embedding (instructions.js:795-821)
          const int ol = opaque(lane), m = rg * PP_ROWS + (ol & 15), row = m < T ? m : T - 1;
          const float *te = a->wte + (size_t)a->tok[row] * d, *pe = a->wpe + (size_t)row * d;
#pragma unroll
          for (int s = 0; s < NS; ++s) {
            const int k8 = (s1 + s) * 4 + (ol >> 4);
            x[s][0] = x[s][1] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (s < n1 && k8 < K81) {
              x[s][0] = *reinterpret_cast<const f32x4*>(te + 8 * k8) + *reinterpret_cast<const f32x4*>(pe + 8 * k8);
              x[s][1] = *reinterpret_cast<const f32x4*>(te + 8 * k8 + 4) + *reinterpret_cast<const f32x4*>(pe + 8 * k8 + 4);
            }
          }
        } else {
          if (n1 > 0) wait_cols(cpC, a->rcpC, 32 * s1, last_col(s1, n1, d), ep);
          load_rows(x, a->xe, K81, s1, n1);
        }
        ConstLayer* ly = fresh_layer(li);
        take(w, bias, scale, ly->wA, 3 * d, cpA, ncA);
        normalise(x, row_scale<MODE>(li, &PrefillScales::A));
        multiply(x, w, ly->wA, 3 * d, cpA, ncA, tilesA);
        __syncthreads();
        if (bail) return;
        a = fresh_args();
        const int hs = a->hs, ctx = a->ctx;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int n = 16 * (et + NW * i) + ec, col = cg * cpA + n;
          if (n >= ncA || em >= T) continue;
          const f32x4 v = finished(tilesA, i, bias, scale);
          if (col < d) {
            st_agent(a->q + (size_t)em * d + col, v);
          } else {
            const int e = col < 2 * d ? col - d : col - 2 * d, h = div_by(e, hs, a->rhs);
            st_agent(a->kv + (((size_t)(2 * li + (col >= 2 * d)) * a->H + h) * ctx + em) * hs + (e - h * hs), v);
          }
        }
        raise(ep + 1);
      }
      {
        ConstLayer* ly = fresh_layer(li);
        request_w(w_next, ly->wC, d, cpC, ncC, 0);
        request_cols(ly->bC, ly->sC, d, cpC, ncC);
      }

      // ---- attention: heads cg, cg + cols, .. of this row group ----
      {
        ConstArgs* a = fresh_args();
        const int hs = a->hs, stride = hs + 4, H = a->H;
        for (int h = cg; h < H; h += a->cols) {
          if (wave <= rg) {  // the keys of row group `wave`
            const float rcp = a->rcpA, ascale = a->scale;
            const int q0 = div_by(h * hs, cpA, rcp), k0 = div_by(d + h * hs, cpA, rcp), v0 = div_by(2 * d + h * hs, cpA, rcp);
            const int nq = div_by(h * hs + hs - 1, cpA, rcp) - q0 + 1, nk = div_by(d + h * hs + hs - 1, cpA, rcp) - k0 + 1;
            const int nv = div_by(2 * d + h * hs + hs - 1, cpA, rcp) - v0 + 1;
            fl.wait(nq + nk + nv, ep + 1, lane, [&](int i) {
              return i < nq ? fl.word(rg, q0 + i) : i < nq + nk ? fl.word(wave, k0 + i - nq) : fl.word(wave, v0 + i - nq - nk);
            });
            const int keys = T - wave * PP_ROWS < PP_ROWS ? T - wave * PP_ROWS : PP_ROWS;
            const float* Kc = a->kv + (((size_t)2 * li * H + h) * a->ctx + wave * PP_ROWS) * hs;
            const __amdgpu_buffer_rsrc_t qb = buffer_of(a->q, (size_t)T * d * 4), kb = buffer_of(Kc, (size_t)keys * hs * 4);
            const __amdgpu_buffer_rsrc_t vb = buffer_of(Kc + (size_t)H * a->ctx * hs, (size_t)keys * hs * 4);
            const int ol = opaque(lane), r = ol & 15, kg = ol >> 4, row = rg * PP_ROWS + r < T ? rg * PP_ROWS + r : T - 1;
            f32x4 kf[HJ], qf[HJ];
            float vf[HJ][4];
#pragma unroll
            for (int j = 0; j < HJ; ++j) {
              const bool in = 16 * j + 4 * kg < hs;
              qf[j] = load4<SC1>(qb, in ? 4 * (row * d + h * hs + 16 * j + 4 * kg) : OUT);
              kf[j] = load4<SC1>(kb, in && r < keys ? 4 * (r * hs + 16 * j + 4 * kg) : OUT);
            }
#pragma unroll
            for (int j = 0; j < HJ; ++j)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                vf[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(vb, 16 * j + r < hs && 4 * kg + e < keys ? 4 * ((4 * kg + e) * hs + 16 * j + r) : OUT, 0, SC1));
            f32x4 sc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int j = 0; j < HJ; ++j)
              if (16 * j < hs) {
#pragma unroll
                for (int e = 0; e < 4; ++e) sc[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][e], qf[j][e], sc[e & 1], 0, 0, 0);
              }
            float p[4], m = -INFINITY, l = 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int key = wave * PP_ROWS + 4 * kg + e;
              p[e] = key <= row ? (sc[0][e] + sc[1][e]) * ascale : -INFINITY;
              m = fmaxf(m, p[e]);
            }
            m = quad_max(m);
            const float base = m == -INFINITY ? 0.f : m;  // (scores of -inf only: weights of 0, which other waves' keys outweigh)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              p[e] = wave * PP_ROWS + 4 * kg + e <= row ? expf(p[e] - base) : 0.f;
              l += p[e];
            }
            l = quad_sum(l);
            float* o = lds + (size_t)(wave * PP_ROWS + r) * stride;
            bool odd = false;  // a value that is not finite would reach queries that do not see its key
#pragma unroll
            for (int j = 0; j < HJ; ++j)
              if (16 * j < hs) {
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                  odd = odd || !(fabsf(vf[j][e]) < INFINITY);
                  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[j][e], p[e], acc, 0, 0, 0);
                }
                if (16 * j + 4 * kg < hs) *reinterpret_cast<f32x4*>(o + 16 * j + 4 * kg) = acc;
              }
            if (kg == 0) {
              o[hs] = m;
              o[hs + 1] = l;
            }
            if (__builtin_amdgcn_ballot_w64(odd) && lane == 0) fl.give_up(PP_ERR_SPLIT);
          }
          __syncthreads();
          if (bail) return;
          for (int e = tid; e < 4 * hs; e += NT) {  // sixteen rows, four elements of each
            const int qr = e & 15, c = 4 * (e >> 4);
            if (rg * PP_ROWS + qr >= T) continue;
            float M = -INFINITY;
            for (int u = 0; u <= rg; ++u) M = fmaxf(M, lds[(size_t)(u * PP_ROWS + qr) * stride + hs]);
            float l = 0.f;
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
            for (int u = 0; u <= rg; ++u) {
              const float* o = lds + (size_t)(u * PP_ROWS + qr) * stride;
              const float f = expf(o[hs] - M);
              l += f * o[hs + 1];
              const f32x4 ov = *reinterpret_cast<const f32x4*>(o + c);
#pragma unroll
              for (int i = 0; i < 4; ++i) v[i] += f * ov[i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] /= l;
            put_row<MODE>(a->att + (size_t)rg * PP_ROWS * d, qr, h * hs + c, v, row_scale<MODE>(li, &PrefillScales::C));
          }
          if (h + a->cols < H) __syncthreads();
        }
        if (cg < H) raise(ep + 2);
      }

      // ---- attention c_proj + residual ----
      if (tilesC) {
        ConstArgs* a = fresh_args();
        if (n1 > 0) {
          const int h0 = div_by(32 * s1, a->hs, a->rhs), h1 = div_by(last_col(s1, n1, d), a->hs, a->rhs), cols = a->cols;
          fl.wait(h1 - h0 + 1, ep + 2, lane, [&](int i) { return fl.word(rg, (h0 + i) % cols); });
        }
        f32x4 x[NS][2], bias[2], scale[2];
        WSlice<MODE, NS> w[RING];
        load_rows(x, a->att, K81, s1, n1);
        ConstLayer* ly = fresh_layer(li);
        take(w, bias, scale, ly->wC, d, cpC, ncC);
        multiply(x, w, ly->wC, d, cpC, ncC, tilesC);
        __syncthreads();
        if (bail) return;
        if (16 * et + ec < ncC && em < T) {
          res += finished(tilesC, 0, bias, scale);
          st_agent(fresh_args()->x1 + (size_t)rg * PP_ROWS * d + row_offset(er, cg * cpC + 16 * et + ec), res);
        }
        raise(ep + 3);
      }
      request_D(li);

      // ---- c_fc: LN2, GELU ----
      WSlice<MODE, CH> we;  // the second MLP product's first weights
      const auto request_E = [&] {
        ConstLayer* ly = fresh_layer(li);
        const int ol = opaque(lane), r = ol & 15;
        we.load(weights_of<MODE>(ly->wE, (size_t)4 * d, d), d, K84, cg * cpC + r, r < ncC, s4, n4, ol >> 4);
        request_cols(ly->bE, ly->sE, d, cpC, ncC);
      };
      if (tilesD) {
        f32x4 x[NS][2], bias[2], scale[2];
        WSlice<MODE, NS> w[RING];
        ConstArgs* a = fresh_args();
        if (n1 > 0) wait_cols(cpC, a->rcpC, 32 * s1, last_col(s1, n1, d), ep + 3);
        load_rows(x, a->x1, K81, s1, n1);
        ConstLayer* ly = fresh_layer(li);
        take(w, bias, scale, ly->wD, 4 * d, cpD, ncD);
        normalise(x, row_scale<MODE>(li, &PrefillScales::D));
        multiply(x, w, ly->wD, 4 * d, cpD, ncD, tilesD);
        __syncthreads();
        if (bail) return;
        float* h = fresh_args()->h + (size_t)rg * PP_ROWS * 4 * d;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int n = 16 * (et + NW * i) + ec;
          if (n >= ncD || em >= T) continue;
          f32x4 v = finished(tilesD, i, bias, scale);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = gelu_ref(v[e]);
          put_row<MODE>(h, er, cg * cpD + n, v, row_scale<MODE>(li, &PrefillScales::E));
        }
        raise(ep + 4);
      }
      request_E();

      // ---- mlp c_proj + residual ----
      if (tilesC) {
        ConstArgs* a = fresh_args();
        constexpr int TM = 2;  // tiles of a pass over the slice
        const __amdgpu_buffer_rsrc_t b = weights_of<MODE>(fresh_layer(li)->wE, (size_t)4 * d, d);
        const float* hidden = a->h;
        const int ol = opaque(lane), r = ol & 15, kg = ol >> 4;
        if (n4 > 0) wait_cols(cpD, a->rcpD, 32 * s4, last_col(s4, n4, 4 * d), ep + 4);
        f32x4 x[2][CH][2];
        load_rows(x[0], hidden, K84, s4, n4);
        load_rows(x[1], hidden, K84, s4 + CH, n4 - CH);
        f32x4 bias[2], scale[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          bias[i] = bias_next[i];
          if constexpr (SCALED) scale[i] = scale_next[i];
        }
        WSlice<MODE, CH> w[2] = {we, we};
        bool bad = false;
#pragma unroll 1
        for (int t0 = 0; t0 < tilesC; t0 += TM) {
          const bool two = t0 + 1 < tilesC;
          const auto request_we = [&](int t, int c) { const int n = 16 * (t0 + t) + r; w[t].load(b, d, K84, cg * cpC + n, n < ncC, s4 + c, n4 - c, kg); };
          if (t0) {
            request_we(0, 0);
            load_rows(x[0], hidden, K84, s4, n4);
            load_rows(x[1], hidden, K84, s4 + CH, n4 - CH);
          }
          request_we(1, 0);
          f32x4 sum[TM];
#pragma unroll
          for (int t = 0; t < TM; ++t) sum[t] = f32x4{0.f, 0.f, 0.f, 0.f};
          const auto chunk = [&](f32x4 (&xc)[CH][2], int c) {
            Operands<MODE, CH> xs;
            xs.set(xc);
            load_rows(xc, hidden, K84, s4 + c + 2 * CH, n4 - c - 2 * CH);
            sum[0] += products(w[0].s, xs);
            request_we(0, c + CH);
            if (two) {
              sum[1] += products(w[1].s, xs);
              request_we(1, c + CH);
            }
          };
#pragma unroll 1
          for (int c = 0; c < n4; c += 2 * CH) {
            chunk(x[0], c);
            if (c + CH < n4) chunk(x[1], c + CH);
          }
#pragma unroll
          for (int t = 0; t < TM; ++t)
            if (t0 + t < tilesC) {
              bad = bad || (em < T && spoilt<MODE>(sum[t]));
              red[(wave * tilesC + t0 + t) * 64 + lane] = sum[t];
            }
        }
        if (__builtin_amdgcn_ballot_w64(bad) && lane == 0) fl.give_up(PP_ERR_SPLIT);
        __syncthreads();
        if (bail) return;
        if (16 * et + ec < ncC && em < T) {
          res += finished(tilesC, 0, bias, scale);
          const int n = cg * cpC + 16 * et + ec;
          st_agent(a->xe + (size_t)rg * PP_ROWS * d + row_offset(er, n), res);
          if (li + 1 == L) *reinterpret_cast<f32x4*>(a->x + (size_t)em * d + n) = res;
        }
        raise(ep + 5);
      }
      request_A(li + 1 < L ? li + 1 : li);  // (behind the last layer nobody waits for them)
    }
  }

  // ---- final LayerNorm of the last row, vocabulary projection (instructions.js:849-856, 916-943) ----
  {
    constexpr int R = NS > 4 ? 2 : 4;  // table rows of a wave in flight
    ConstArgs* a = fresh_args();
    const int V = a->V, per = a->rows_per_wg, v0 = blockIdx.x * per, v1 = v0 + per < V ? v0 + per : V;
    const float* wte = a->wte;
    f32x4 t[R][NS];
    const auto table = [&](int v) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const float* e = wte + (size_t)(v + i) * d;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
          t[i][s] = f32x4{0.f, 0.f, 0.f, 0.f};
          if (v + i < v1 && 256 * s + 4 * lane < d) t[i][s] = *reinterpret_cast<const f32x4*>(e + 256 * s + 4 * lane);
        }
      }
    };
    table(v0 + R * wave);
    const int lg = (T - 1) / PP_ROWS, lr = (T - 1) % PP_ROWS;
    fl.wait((d + cpC - 1) / cpC, fl.ebase + 5u * L, lane, [&](int i) { return fl.word(lg, i); }, !rows_here);
    const __amdgpu_buffer_rsrc_t xb = buffer_of(a->xe + (size_t)lg * PP_ROWS * d, (size_t)PP_ROWS * d * 4);
    f32x4 x[NS];
    float sum = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) x[s] = load4<SC1>(xb, 256 * s + 4 * lane < d ? 4 * row_offset(lr, 256 * s + 4 * lane) : OUT);
#pragma unroll
    for (int s = 0; s < NS; ++s) sum += (x[s][0] + x[s][1]) + (x[s][2] + x[s][3]);
    const float mean = wave_sum(sum) / (float)d;
    float q = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const float e0 = x[s][0] - mean, e1 = x[s][1] - mean, e2 = x[s][2] - mean, e3 = x[s][3] - mean;
      q += 256 * s + 4 * lane < d ? (e0 * e0 + e1 * e1) + (e2 * e2 + e3 * e3) : 0.f;
    }
    const float stdev = sqrtf(wave_sum(q) / (float)d + 1e-5f), rstd = 1.0f / stdev;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      if (256 * s + 4 * lane < d) {
        const f32x4 g = *reinterpret_cast<const f32x4*>(a->lnf_g + 256 * s + 4 * lane), be = *reinterpret_cast<const f32x4*>(a->lnf_b + 256 * s + 4 * lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) x[s][i] = g[i] * quotient(x[s][i] - mean, stdev, rstd) + be[i];
      }
    __syncthreads();  // (every wave is past its wait: the row of logits may take the place of the tiles)
    if (bail) return;
#pragma unroll 1
    for (int v = v0 + R * wave; v < v1; v += R * NW) {
      float z[R];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        float acc = 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s) acc += (t[i][s][0] * x[s][0] + t[i][s][1] * x[s][1]) + (t[i][s][2] * x[s][2] + t[i][s][3] * x[s][3]);
        z[i] = acc;
      }
      table(v + R * NW);
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const float zz = wave_sum(z[i]);
        if (lane == 0 && v + i < v1) lds[v + i - v0] = zz;
      }
    }
    __syncthreads();
    for (int e = tid; e < v1 - v0; e += NT) {
      a->logits[v0 + e] = lds[e];
      a->host_logits[v0 + e] = lds[e];
    }
  }
}

constexpr int MAX_LDS = 144 * 1024;  // beside the static part

int columns_of(int N, int groups) { return ((N + groups - 1) / groups + 3) / 4 * 4; }

// The grid of a prompt of T rows.
void cut(PrefillArgs& a) {
  a.groups = (a.T + PP_ROWS - 1) / PP_ROWS;
  a.per_xcd = PP_GRID / 8 / a.groups;
  a.cols = 8 * a.per_xcd;
  a.cpA = columns_of(3 * a.d, a.cols);
  a.cpC = columns_of(a.d, a.cols);
  a.cpD = columns_of(4 * a.d, a.cols);
  a.rows_per_wg = (a.V + PP_GRID - 1) / PP_GRID;
  a.rcpA = 1.0f / (float)a.cpA, a.rcpC = 1.0f / (float)a.cpC, a.rcpD = 1.0f / (float)a.cpD, a.rhs = 1.0f / (float)a.hs;
}
size_t lds_bytes(const PrefillArgs& a) {
  const int widest = a.cpD > a.cpA ? a.cpD : a.cpA;
  size_t need = (size_t)NW * ((widest + 15) / 16) * 64 * 16;
  const size_t att = (size_t)NW * PP_ROWS * (a.hs + 4) * 4, run = 4 * (size_t)a.rows_per_wg;
  if (att > need) need = att;
  if (run > need) need = run;
  return need > 84 * 1024 ? need : 84 * 1024;  // more than half of a compute unit's, so that exactly one workgroup lives on each
}

template <int MODE, int NS, int HJ>
hipError_t launch_hj(const PrefillArgs& a, hipStream_t s) {
  const size_t lds = lds_bytes(a);
  static bool enabled = false;  // dynamic LDS size already raised
  if (!enabled) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(prefill_persistent_kernel<MODE, NS, HJ>), hipFuncAttributeMaxDynamicSharedMemorySize, MAX_LDS);
    if (e != hipSuccess) return e;
    enabled = true;
  }
  prefill_persistent_kernel<MODE, NS, HJ><<<PP_GRID, NT, lds, s>>>(a);
  return hipGetLastError();
}
template <int MODE, int NS>
hipError_t launch_ns(const PrefillArgs& a, hipStream_t s) {
  return a.hs <= 64 ? launch_hj<MODE, NS, 4>(a, s) : launch_hj<MODE, NS, 8>(a, s);
}
template <int MODE>
hipError_t launch_any(const PrefillArgs& a, hipStream_t s) {
  if (a.d <= PP_PAIR_ABOVE) {
    if constexpr (is_pair(MODE)) return hipErrorInvalidValue;
    else return launch_ns<MODE, 2>(a, s);
  }
  if (a.d <= 768) return launch_ns<MODE, 3>(a, s);
  if (a.d <= 1024) return launch_ns<MODE, 4>(a, s);
  if (a.d <= 1280) return launch_ns<MODE, 5>(a, s);
  return launch_ns<MODE, 7>(a, s);
}

}  // namespace

int prefill_persistent_rows(int d, int H, int hs, int V, bool i8, int compute_units) {
  if (compute_units < PP_GRID || d % 8 || hs % 4 || hs > 128 || d > 1792 || H * hs != d) return 0;
  PrefillArgs a{};
  a.d = d, a.hs = hs, a.V = V, a.T = PP_MAX_T;
  cut(a);  // (the widest shares are those of the longest prompt)
  // a thread finishes at most one float4 of a projection and two of the others, and the widest tiles fit beside the static part
  if (a.cpC > 16 * NW || a.cpA > 32 * NW || a.cpD > 32 * NW || lds_bytes(a) > (size_t)MAX_LDS) return 0;
  // With fp32 rows above 1280 a wave has the registers for one tile of weights ahead, too few for the two and more tiles of longer
  // prompts: twelve layers of d = 1600 1.07 ms against 1.18 with launches at 64 rows, 1.54 against 1.44 at 128 (d = 1280: 1.04
  // against 1.18).
  return !i8 && d > 1280 ? 64 : PP_MAX_T;
}

hipError_t launch_prefill_persistent(PrefillArgs a, PrefillMode mode, hipStream_t s) {
  if (a.T < 1 || a.T > PP_MAX_T || a.T > a.ctx) return hipErrorInvalidValue;
  cut(a);
  switch (mode) {
    case PP_PLAIN_F32: return launch_any<PP_PLAIN_F32>(a, s);
    case PP_SPLIT_I8: return launch_any<PP_SPLIT_I8>(a, s);
    case PP_PAIR_F32: return launch_any<PP_PAIR_F32>(a, s);
    case PP_PAIR_I8: return launch_any<PP_PAIR_I8>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace wgpt
