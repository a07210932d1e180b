// Greedy decode steps of GPT.run (model.js:104-268) in one persistent launch, for any width and head size.
//
// A token as one launch per block is 5 L + 3 dependent launches of 4 to 6 us, whatever they move (token_launches, model.hip).
// us per token with launches and with this kernel, 40 positions and on (layers x width, head size): 4 x 576, 48, 111 -> 59, int8
// 149 -> 59; 4 x 320, 16, 96 -> 52; 6 x 1280, 128, 251 -> 165 (480 MB of weights, 74 us at the rate of reads); 3 x 64, 16, 73 -> 40.
// At the widest and at long contexts (four layers, position 100 and 900): 1600, 32, 197 and 205 -> 141 and 148, int8 240 and 248 -> 95 and 102;
// 1792, 128, 205 and 239 -> 158 and 167, int8 242 and 275 -> 98 and 108; 1288, 92, 175 and 209 -> 124 and 132; 64, 16, 90 -> 57 (800).
// What is left, as clock stamps of 4 x 576 have it: a layer is 13.7 us, of which 6.4 pass between the last word of an exchange and its readers
// (0.8 the attention's, 1.0 to 1.7 each other one), 5.3 are the phases (1.9 the attention, 1.2 c_fc, 1.0 c_attn, 0.5 and 0.7 the projections), 2.0
// workgroups behind the median one; a step's end is 6.3. The compiler spills 144 to 191 scalar registers into vector lanes, and of fp32
// rows above 1280 7 vector registers (sampled 28) to scratch.
// Here one workgroup per compute unit stays for all steps and the blocks are phases of it, as in decode_persistent.hip, whose
// phases are compiled for one width and heads of 64 each. This kernel has its geometry in registers; only the number of 256-wide
// segments of a row (NS) and the key rows that a wave holds (R) are compile-time, so that weights and keys have registers:
//
//   - c_attn and c_fc: whole columns of the decode slabs per wave; the input row is gathered in LDS and normalised by every wave;
//   - both projections: a wave multiplies its segments of the row with all columns of the workgroup, partial sums meet in LDS.
//     A wave waits for its own segments only, so the row needs no gathering;
//   - attention: a workgroup per (head, slice of the context); the slices are merged by the waves of the projection;
//   - rows pass between workgroups as {value, epoch} words, written and polled at device scope; a word validates itself;
//   - weights of a phase, keys and values are requested before the wait in front of it;
//   - at the end of a step every workgroup finds the arg-max of all workgroups' candidates, so a step needs no broadcast. With
//     top_k up to PD_TOPK a workgroup's candidates are its top_k first logits and every wave samples from the first of all (us per
//     token at top_k 2 and 8, before with a launch and a selection for each: 4 x 576 of 5003 tokens 77 -> 61.5 and 67, 3 x 64
//     57 -> 44.5 and 52, 6 x 1280 of 50257 210 -> 191.5 and 196). Above eight the words would outgrow a poll of four a thread.
//
// No word is overwritten while somebody may still wait for its epoch: an exchange is written again only by a workgroup that has
// seen, through the exchanges between, the results of everyone who reads it. The candidates, which workgroups without
// columns read too, alternate between two buffers. A key or value is read by other workgroups one step later: its stores have
// completed before its workgroup's candidate of that step.
//
// Every wait is bounded; one that expires ends the launch with the error word, and the host repeats the call with launches.
#include "decode_generic.h"

#include <type_traits>

#include "persistent_common.h"
#include "select_key.h"

namespace wgpt {
namespace {

typedef unsigned long long u64;

constexpr int NT = PD_THREADS, NW = NT / 64, G = PD_GRID;
constexpr int SEG = 256;                          // contraction elements of a slab item
template <int N>
using Count = std::integral_constant<int, N>;
// Polls: volatile, which makes them system scope (sc0 sc1). A poll sees a word that another XCD's compute unit has stored at device scope
// because neither the L1 nor a stale line of its own L2 answers it, and it is made again in every round because the loops also hold relaxed
// atomic loads, across which the compiler moves no read (a loop of nothing but such loads is one load: volatile or not, it is a plain
// read of memory to the compiler).
constexpr int POLL = SC1 | (int)0x80000000;

template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp_add(float v) {
  return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xf, true));
}
// N sums over the 64 lanes side by side, wave-uniform.
template <int N>
__device__ __forceinline__ void wave_sums(float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = dpp_add<0x111, 0xf>(v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = dpp_add<0x112, 0xf>(v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = dpp_add<0x114, 0xf>(v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = dpp_add<0x118, 0xf>(v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = dpp_add<0x142, 0xa>(v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = dpp_add<0x143, 0xc>(v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v[i]), 63));
}
__device__ __forceinline__ float wave_total(float v) {
  float a[1] = {v};
  wave_sums(a);
  return a[0];
}
template <int CTRL>
__device__ __forceinline__ float dpp_get(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}
// Over the lpk lanes of a key (4, 8, 16 or 32 adjacent ones), every lane gets it.
__device__ __forceinline__ float key_sum(float v, int lpk) {
  v += dpp_get<0xB1>(v);
  v += dpp_get<0x4E>(v);
  if (lpk > 4) v += dpp_get<0x141>(v);
  if (lpk > 8) v += dpp_get<0x140>(v);
  if (lpk > 16) {
    float a, b;
    pair16(v, a, b);
    v = a + b;
  }
  return v;
}
// Over the lanes at one place of every key.
template <class Op>
__device__ __forceinline__ float across_keys(float v, int lpk, Op op) {
  if (lpk <= 4) v = op(v, dpp_get<0x124>(v));
  if (lpk <= 8) v = op(v, dpp_get<0x128>(v));
  float a, b;
  if (lpk <= 16) {
    pair16(v, a, b);
    v = op(a, b);
  }
  pair32(v, a, b);
  return op(a, b);
}
__device__ __forceinline__ float dot4(const f32x4& a, const f32x4& b) { return (a[0] * b[0] + a[1] * b[1]) + (a[2] * b[2] + a[3] * b[3]); }

// Four consecutive k of one column.
template <bool I8>
struct Weight {
  f32x4 v;
  static constexpr int BYTES = 16;
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, int o, int so) { v = load4<0>(b, o, so); }
  __device__ __forceinline__ f32x4 value() const { return v; }
};
template <>
struct Weight<true> {
  int v;
  static constexpr int BYTES = 4;
  __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t b, int o, int so) { v = __builtin_amdgcn_raw_buffer_load_b32(b, o, so, 0); }
  __device__ __forceinline__ f32x4 value() const { return f32x4{(float)(v << 24 >> 24), (float)(v << 16 >> 24), (float)(v << 8 >> 24), (float)(v >> 24)}; }
};

struct Waits {
  int* err;
  unsigned spin_limit;
  int* bail;  // LDS
  __device__ __forceinline__ int bailed() const { return __hip_atomic_load(bail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); }
  // One wave: the pairs of {value, epoch} words at byte offsets off of a buffer are all of epoch ep (or the launch has given up).
  // A lane that needs fewer waits for one of its words again: no masks to keep.
  template <int N>
  __device__ __forceinline__ void words(__amdgpu_buffer_rsrc_t b, const int (&off)[N], u32x4 (&v)[N], unsigned ep) const {
    for (unsigned spins = 0;;) {
#pragma unroll
      for (int i = 0; i < N; ++i) v[i] = __builtin_amdgcn_raw_buffer_load_b128(b, off[i], 0, POLL);
      bool missing = false;
#pragma unroll
      for (int i = 0; i < N; ++i) missing = missing || v[i][1] != ep || v[i][3] != ep;
      if (!__builtin_amdgcn_ballot_w64(missing)) return;
      if (bailed()) return;
      ++spins;
      if (spins > spin_limit) {
        *bail = 1;
        __hip_atomic_store(err, (int)ep, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
      }
      if ((spins & 15u) == 0 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        *bail = 1;
        return;
      }
    }
  }
};
__device__ __forceinline__ void publish(u64* p, float v, unsigned ep) {
  __hip_atomic_store(p, ((u64)ep << 32) | __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The launch's arguments where they lie, read again (scalar loads) by each phase rather than kept in registers for all of them.
typedef const __attribute__((address_space(4))) PersistentArgs ConstArgs;
__device__ __forceinline__ ConstArgs* fresh_args() {
  ConstArgs* p = (ConstArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return p;
}
__device__ __forceinline__ int opaque_s(int v) {
  asm volatile("" : "+s"(v));
  return v;
}
__device__ __forceinline__ void nap(int units) {  // about 64 clocks each
  for (int i = 0; i < units; ++i) __builtin_amdgcn_s_sleep(1);
}

// NS: segments of a row. R: key rows of a lane, 8 for heads of more than 64. SAMPLE: tokens are sampled from the top_k first logits.
template <bool I8, int NS, int R, bool SAMPLE>
__global__ __launch_bounds__(NT, 2) void decode_generic_kernel(PersistentArgs) {
  constexpr int CWA = (3 * NS + NW - 1) / NW, CWD = (4 * NS + NW - 1) / NW;  // columns of a wave, segments of a wave of the 4d-long row
  constexpr int FULL = NS == 7 ? 5 : NS - 1;                                 // segments that every width of this instantiation fills (launch_any)
  constexpr int PW = Weight<I8>::BYTES;
  constexpr int NP = (NS * SEG / 2 + NT - 1) / NT;                           // pairs of words of a row per thread
  extern __shared__ __attribute__((aligned(16))) float run[];                // this workgroup's logits
  __shared__ __attribute__((aligned(16))) float row[NS * SEG], part[NW][8], heads[NW][136];
  __shared__ float out[4 * NS], far_out[I8 ? 4 * NS : 1], far_part[I8 ? NW : 1][8];
  __shared__ float best_v[NW];
  __shared__ int best_i[NW], bail;
  __shared__ sel_key firsts[NW * PD_TOPK];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wg = blockIdx.x;
  ConstArgs* const a0 = fresh_args();
  const int d = a0->d, H = a0->H, hs = d / H, L = a0->L, V = a0->V;
  const int S = (d + SEG - 1) / SEG, SH = (4 * d + SEG - 1) / SEG;
  const auto share = [&](int N, int& c0) {  // columns of this workgroup
    const int per = (N + G - 1) / G;
    c0 = wg * per;
    const int n = N - c0;
    return n > per ? per : n < 0 ? 0 : n;
  };
  int cA, cC, cD;
  const int ncA = share(3 * d, cA), ncC = share(d, cC), ncD = share(4 * d, cD);
  const int lsh = hs <= 16 ? 2 : hs <= 32 ? 3 : hs <= 64 ? 4 : 5, lpk = 1 << lsh, kpw = 64 >> lsh;  // lanes of a key, keys of a wave's load
  const int most = H * DG_SPLIT <= G ? DG_SPLIT : G / H;
  const float rhs = 1.0f / (float)hs;
  const LayerParamOffsets po = layer_param_offsets(d);
  const Waits wt = {a0->err, a0->spin_limit, &bail};

  for (int i = tid; i < NS * SEG; i += NT) row[i] = 0.f;
  if (tid == 0) bail = 0;
  __syncthreads();

  Weight<I8> w[NS * CWD];
  f32x4 gam[NS], bet[NS];
  float bias = 0.f, scale = 1.f;
  const auto matrix = [&](int li, size_t off, int N, int segs) {
    const int per = (N + G - 1) / G;
    ConstArgs* a = fresh_args();
    return buffer_of(static_cast<const char*>(a->slabs) + ((size_t)li * a->slab_stride + off) * PW, (size_t)G * per * segs * 64 * PW);
  };
  const auto request_finish = [&](int li, int c0, int nc, int bo, int so) {  // of this thread's column
    const float* lp = fresh_args()->lparams + (size_t)li * po.stride;
    const __amdgpu_buffer_rsrc_t b = buffer_of(lp, (size_t)po.stride * 4);
    const int t = opaque(tid), c = t < nc ? 4 * (c0 + t) : OUT;
    bias = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, c, 4 * bo, 0));
    if constexpr (I8) scale = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, c, 4 * so, 0));
  };
  const auto request_ln = [&](const float* g, const float* b) {
    const __amdgpu_buffer_rsrc_t gb = buffer_of(g, 4 * (size_t)d), bb = buffer_of(b, 4 * (size_t)d);
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const int e = SEG * s + 4 * opaque(lane), o = e < d ? 4 * e : OUT;
      gam[s] = load4<0>(gb, o);
      bet[s] = load4<0>(bb, o);
    }
  };
  // Columns wave, wave + 8, .. of the workgroup's nc, all segments.
  const auto request_columns = [&](__amdgpu_buffer_rsrc_t b, int c0, int nc, auto cw) {
    const int o = opaque(lane) * PW, u = opaque_s(wave), segs = opaque_s(S);
#pragma unroll
    for (int j = 0; j < cw(); ++j)
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const int c = u + NW * j;
        const bool in = c < nc && s < segs;
        w[j * NS + s].load(b, in ? o : OUT, in ? ((c0 + c) * segs + s) * 64 * PW : 0);
      }
  };
  // Segments wave, wave + 8, .. of the workgroup's nc columns.
  const auto request_segments = [&](__amdgpu_buffer_rsrc_t b, int segs, auto cw) {
    const int o = opaque(lane) * PW, u = opaque_s(wave), c0 = opaque_s(cC);
#pragma unroll
    for (int c = 0; c < NS; ++c)
#pragma unroll
      for (int j = 0; j < cw(); ++j) {
        const int s = u + NW * j;
        const bool in = c < ncC && s < segs;
        w[c * cw() + j].load(b, in ? o : OUT, in ? ((c0 + c) * segs + s) * 64 * PW : 0);
      }
  };
  const auto request_A = [&](int li) {
    request_columns(matrix(li, 0, 3 * d, S), cA, ncA, Count<CWA>());
    request_finish(li, cA, ncA, po.bA, po.sA);
    if constexpr (I8) {
      const float* lp = fresh_args()->lparams + (size_t)li * po.stride;
      request_ln(lp + po.ln1g, lp + po.ln1b);
    }
  };
  const auto request_C = [&](int li) {
    request_segments(matrix(li, fresh_args()->slab_offC, d, S), S, Count<1>());
    request_finish(li, cC, ncC, po.bC, po.sC);
  };
  const auto request_D = [&](int li) {
    request_columns(matrix(li, fresh_args()->slab_offD, 4 * d, S), cD, ncD, Count<CWD>());
    request_finish(li, cD, ncD, po.bD, po.sD);
    if constexpr (I8) {
      const float* lp = fresh_args()->lparams + (size_t)li * po.stride;
      request_ln(lp + po.ln2g, lp + po.ln2b);
    }
  };
  const auto request_E = [&](int li) {
    request_segments(matrix(li, fresh_args()->slab_offE, d, SH), SH, Count<CWD>());
    request_finish(li, cC, ncC, po.bE, po.sE);
  };
  // The d words of an exchange into `row`, for all waves.
  const auto gather_row = [&](const u64* buf, unsigned ep) {
    const __amdgpu_buffer_rsrc_t b = buffer_of(buf, 8 * (size_t)d);
    int off[NP];
    u32x4 v[NP];
    const int t = opaque(tid);
#pragma unroll
    for (int i = 0; i < NP; ++i) off[i] = 16 * (2 * (t + NT * i) < d ? t + NT * i : 0);
    wt.words(b, off, v, ep);
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (2 * (t + NT * i) < d) *reinterpret_cast<u32x2*>(row + 2 * (t + NT * i)) = u32x2{v[i][0], v[i][2]};
    __syncthreads();
  };
  // LayerNorm of `row` (instructions.js:451-550) in registers; gamma and beta only if the slabs do not carry them.
  const auto normalised = [&](f32x4 (&x)[NS], bool affine) {
    float sum = 0.f, q = 0.f;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      x[s] = *reinterpret_cast<const f32x4*>(row + SEG * s + 4 * lane);
      sum += (x[s][0] + x[s][1]) + (x[s][2] + x[s][3]);
    }
    const int e0l = 4 * opaque(lane);
    const float fd = (float)d, mean = wave_total(sum) / fd;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const float e0 = x[s][0] - mean, e1 = x[s][1] - mean, e2 = x[s][2] - mean, e3 = x[s][3] - mean;
      q += s < FULL || SEG * s + e0l < d ? (e0 * e0 + e1 * e1) + (e2 * e2 + e3 * e3) : 0.f;
    }
    const float stdev = sqrtf(wave_total(q) / fd + 1e-5f), rstd = 1.0f / stdev;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      const float r = s < FULL || SEG * s + e0l < d ? rstd : 0.f;  // (beyond d the weights are zero, and so is x, whatever the mean)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = quotient(x[s][e] - mean, stdev, r);
        x[s][e] = affine ? gam[s][e] * v + bet[s][e] : v;
      }
    }
  };
  // int8: a column's scale meets its finished sum, which may leave the range of fp32 where the scaled products and the result
  // do not (inputs of 1e35, scales of 1e-34). A wave with a sum that is not finite takes its sums again, of inputs times DOWN (4 d products
  // of up to 127 times the largest float stay finite), for those who finish such columns.
  constexpr float DOWN = 0x1p-24f, UP = 0x1p24f;
  const auto sums_of = [&](auto& sums, auto take, auto keep) {
    take(1.f);
    keep(false);
    if constexpr (I8) {
      float all = 0.f;
#pragma unroll
      for (const float v : sums) all += fabsf(v);
      if (__builtin_expect(!(all < INFINITY), 0)) {
#pragma unroll
        for (auto& wt : w) wt.v = opaque(wt.v);  // (unpacked again: the floats would have to be kept for this)
        take(DOWN);
        keep(true);
      }
    }
    __syncthreads();
  };
  const auto columns = [&](const f32x4 (&x)[NS], int nc, auto cw) {  // products to `out`
    float sums[decltype(cw)::value];
    sums_of(
        sums,
        [&](float f) {
#pragma unroll
          for (int j = 0; j < cw(); ++j) {
            sums[j] = 0.f;
#pragma unroll
            for (int s = 0; s < NS; ++s) sums[j] += dot4(w[j * NS + s].value(), f * x[s]);
          }
          wave_sums(sums);
        },
        [&](bool far) {
#pragma unroll
          for (int j = 0; j < cw(); ++j)
            if (lane == 0 && wave + NW * j < nc) (far ? far_out : out)[wave + NW * j] = sums[j];
        });
  };
  const auto segments = [&](const auto& x, auto cw) {  // partial sums of the projections to `part`
    float sums[NS];
    sums_of(
        sums,
        [&](float f) {
#pragma unroll
          for (int c = 0; c < NS; ++c) {
            sums[c] = 0.f;
#pragma unroll
            for (int j = 0; j < cw(); ++j) sums[c] += dot4(w[c * cw() + j].value(), f * x[j]);
          }
          wave_sums(sums);
        },
        [&](bool far) {
#pragma unroll
          for (int c = 0; c < NS; ++c)
            if (lane == 0) (far ? far_part : part)[wave][c] = sums[c];
        });
  };
  // This thread's column of `out`, or of a projection whose partial sums the first `waves` waves have.
  const auto finished_column = [&] {
    float v = out[tid];
    if constexpr (I8) {
      const float s = scale / 127.0f;
      if (__builtin_expect(fabsf(v) < INFINITY, 1)) v *= s;
      else v = far_out[tid] * s * UP;
    }
    return v + bias;
  };
  const auto finished_parts = [&](int waves) {
    float v = 0.f;
    for (int u = 0; u < waves; ++u) v += part[u][tid];
    if constexpr (I8) {
      const float s = scale / 127.0f;
      if (__builtin_expect(fabsf(v) < INFINITY, 1)) {
        v *= s;
      } else {
        v = 0.f;
        for (int u = 0; u < waves; ++u) v += fabsf(part[u][tid]) < INFINITY ? part[u][tid] * DOWN : far_part[u][tid];
        v = v * s * UP;
      }
    }
    return v + bias;
  };

  int tok = a0->tok ? a0->tok[0] : a0->tok_value;
  unsigned ep = a0->ebase;
  const int nsteps = a0->nsteps;
  request_A(0);
  for (int step = 0; step < nsteps; ++step) {
    ConstArgs* const as = fresh_args();
    const int pos = as->pos0 + step, n = pos + 1;
    // Slices of the context: 64 positions and more each, as many as the workgroups allow.
    int slices = (n + 63) >> 6;
    slices = slices > most ? most : slices;
    const int per = (n + slices - 1) / slices;
    slices = (n + per - 1) / per;
    const int head = wg % H, slice = wg / H;
    const bool attends = slice < slices, owner = slice == slices - 1;
    const int naps_att = as->delay[2] + (as->att_slope[0] * n >> 10), naps_others = as->delay[3] + (as->att_slope[1] * n >> 10);
    float res = 0.f;  // residual stream: column cC + tid
    {                 // the embedding (instructions.js:795-821)
      const float *te = as->wte + (size_t)tok * d, *pe = as->wpe + (size_t)pos * d;
      for (int i = 4 * tid; i < d; i += 4 * NT) *reinterpret_cast<f32x4*>(row + i) = *reinterpret_cast<const f32x4*>(te + i) + *reinterpret_cast<const f32x4*>(pe + i);
      if (tid < ncC) res = te[cC + tid] + pe[cC + tid];
      __syncthreads();
    }
    for (int li = 0; li < L; ++li, ep += 5) {
      // ---- c_attn: LN1, q/k/v ----
      if (ncA) {
        if (li) {
          nap(fresh_args()->delay[0]);
          gather_row(fresh_args()->bufR2, ep);
          if (bail) return;
        }
        f32x4 x[NS];
        normalised(x, I8);
        columns(x, ncA, Count<CWA>());
        if (tid < ncA) publish(fresh_args()->bufQKV + cA + tid, finished_column(), ep + 1);
      }
      // ---- attention of (head, slice) ----
      if (attends) {
        ConstArgs* const a = fresh_args();
        const int ctx = a->ctx, ol = opaque(lane), kp = 4 * (ol & (lpk - 1)), kg = ol >> lsh;  // this lane's elements and key
        const int first = slice * per, last = first + per < n ? first + per : n, key0 = first + wave * kpw + kg;
        float* Kc = fresh_args()->kv + ((size_t)2 * li * H + head) * ctx * hs;
        float* Vc = Kc + (size_t)H * ctx * hs;
        const __amdgpu_buffer_rsrc_t kb = buffer_of(Kc, (size_t)ctx * hs * 4), vb = buffer_of(Vc, (size_t)ctx * hs * 4);
        const bool in = kp < hs;
        f32x4 kf[R], vf[R];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int key = key0 + r * NW * kpw, o = in && key < last && key < pos ? 4 * (key * hs + kp) : OUT;
          kf[r] = load4<SC1>(kb, o);
          vf[r] = load4<SC1>(vb, o);
        }
        nap(fresh_args()->delay[1]);
        f32x4 q, kn, vn;
        {
          int off[6];
          u32x4 v[6];
#pragma unroll
          for (int i = 0; i < 6; ++i) off[i] = 8 * ((owner ? (i >> 1) * d : 0) + head * hs + (in ? kp : 0) + 2 * (i & 1));
          wt.words(buffer_of(fresh_args()->bufQKV, 24 * (size_t)d), off, v, ep + 1);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            q[i] = in ? __uint_as_float(v[i >> 1][2 * (i & 1)]) : 0.f;
            kn[i] = __uint_as_float(v[2 + (i >> 1)][2 * (i & 1)]);
            vn[i] = __uint_as_float(v[4 + (i >> 1)][2 * (i & 1)]);
          }
        }
        if (owner && wave == 0 && kg == 0 && in) {
          st_agent(Kc + (size_t)pos * hs + kp, kn);
          st_agent(Vc + (size_t)pos * hs + kp, vn);
        }
        float sc[R], m = -INFINITY, l = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const int key = key0 + r * NW * kpw;
          if (key == pos) kf[r] = kn, vf[r] = vn;
          sc[r] = dot4(q, kf[r]);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) sc[r] = key_sum(sc[r], lpk) * fresh_args()->scale;
#pragma unroll
        for (int r = 0; r < R; ++r)
          if (key0 + r * NW * kpw < last) m = fmaxf(m, sc[r]);
        m = across_keys(m, lpk, [](float x, float y) { return fmaxf(x, y); });
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
        const float base = m == -INFINITY ? 0.f : m;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          const float p = key0 + r * NW * kpw < last ? expf(sc[r] - base) : 0.f;
          l += p;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] += p * vf[r][e];
        }
        const auto add = [](float x, float y) { return x + y; };
        l = across_keys(l, lpk, add);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = across_keys(o[e], lpk, add);
        if (kg == 0 && in) *reinterpret_cast<f32x4*>(&heads[wave][kp]) = o;
        if (lane == 0) heads[wave][hs] = l, heads[wave][hs + 1] = m;
        __syncthreads();
        if (bail) return;
        if (tid < hs + 2) {
          float mw[NW], M = -INFINITY, v = 0.f;
#pragma unroll
          for (int u = 0; u < NW; ++u) {
            mw[u] = heads[u][hs + 1];
            M = fmaxf(M, mw[u]);
          }
          const int e = tid <= hs ? tid : 0;
#pragma unroll
          for (int u = 0; u < NW; ++u) v += (mw[u] == -INFINITY ? 0.f : expf(mw[u] - M)) * heads[u][e];
          publish(fresh_args()->bufATT + (size_t)(head * DG_SPLIT + slice) * (hs + 2) + tid, tid > hs ? M : v, ep + 2);
        }
      }
      // ---- attention c_proj + residual ----
      if (ncC) {
        request_C(li);
        nap(attends ? naps_att : naps_others);
        f32x4 x[1] = {{0.f, 0.f, 0.f, 0.f}};
        if (wave < S) {
          const int e0 = SEG * wave + 4 * opaque(lane), e = e0 < d ? e0 : 0, h = div_by(e, hs, rhs), words = hs + 2;
          const __amdgpu_buffer_rsrc_t b = buffer_of(fresh_args()->bufATT, 8 * (size_t)H * DG_SPLIT * words);
          const int at = 8 * (h * DG_SPLIT * words + (e - h * hs)), ml = 8 * (h * DG_SPLIT * words + hs);
          const auto merge = [&](auto most_slices) {
            constexpr int N = decltype(most_slices)::value;
            int off[3 * N];
            u32x4 v[3 * N];
#pragma unroll
            for (int s = 0; s < N; ++s) {
              const int there = 8 * words * (s < slices ? s : 0);
              off[3 * s] = at + there;
              off[3 * s + 1] = at + 16 + there;
              off[3 * s + 2] = ml + there;
            }
            wt.words(b, off, v, ep + 2);
            float M = -INFINITY, l = 0.f;
#pragma unroll
            for (int s = 0; s < N; ++s)
              if (s < slices) M = fmaxf(M, __uint_as_float(v[3 * s + 2][2]));
#pragma unroll
            for (int s = 0; s < N; ++s)
              if (s < slices) {
                const float ms = __uint_as_float(v[3 * s + 2][2]), f = ms == -INFINITY ? 0.f : expf(ms - M);
                l += f * __uint_as_float(v[3 * s + 2][0]);
#pragma unroll
                for (int i = 0; i < 4; ++i) x[0][i] += f * __uint_as_float(v[3 * s + (i >> 1)][2 * (i & 1)]);
              }
#pragma unroll
            for (int i = 0; i < 4; ++i) x[0][i] /= l;  // (beyond d: that of the first elements, its weights are zero)
          };
          if (slices <= 2) merge(Count<2>());
          else merge(Count<DG_SPLIT>());
        }
        segments(x, Count<1>());
        if (bail) return;
        if (tid < ncC) {
          res += finished_parts(S);
          publish(fresh_args()->bufR1 + cC + tid, res, ep + 3);
        }
      }
      // ---- c_fc: LN2, GELU ----
      if (ncD) {
        request_D(li);
        nap(fresh_args()->delay[4]);
        gather_row(fresh_args()->bufR1, ep + 3);
        if (bail) return;
        f32x4 x[NS];
        normalised(x, I8);
        columns(x, ncD, Count<CWD>());
        if (tid < ncD) publish(fresh_args()->bufH + cD + tid, gelu_ref(finished_column()), ep + 4);
      }
      // ---- mlp c_proj + residual ----
      if (ncC) {
        request_E(li);
        nap(fresh_args()->delay[5]);
        f32x4 x[CWD];
        int off[2 * CWD];
        u32x4 v[2 * CWD];
#pragma unroll
        for (int i = 0; i < 2 * CWD; ++i) {
          const int e = SEG * (wave + NW * (i >> 1)) + 4 * opaque(lane) + 2 * (i & 1);
          off[i] = e < 4 * d ? 8 * e : 8 * (e & 2);  // (beyond the row its weights are zero)
        }
        wt.words(buffer_of(fresh_args()->bufH, 32 * (size_t)d), off, v, ep + 4);
#pragma unroll
        for (int i = 0; i < 4 * CWD; ++i) x[i >> 2][i & 3] = __uint_as_float(v[i >> 1][2 * (i & 1)]);
        segments(x, Count<CWD>());
        if (bail) return;
        if (tid < ncC) {
          res += finished_parts(SH < NW ? SH : NW);
          publish(fresh_args()->bufR2 + cC + tid, res, ep + 5);
        }
      }
      if (li + 1 < L) request_A(li + 1);
    }

    // ---- final LayerNorm, vocabulary projection (instructions.js:849-856, 916-943) ----
    const bool ends = step + 1 == nsteps;
    {
      constexpr int RV = NS > 4 ? 2 : 4;  // table rows of a wave in flight
      const int v0 = wg * fresh_args()->rows_per_wg, v1 = v0 + fresh_args()->rows_per_wg < V ? v0 + fresh_args()->rows_per_wg : V;
      f32x4 t[RV][NS];
      const auto table = [&](int v) {
        const int o = 16 * opaque(lane);
#pragma unroll
        for (int i = 0; i < RV; ++i) {
          const bool in = v + i < v1;
          const __amdgpu_buffer_rsrc_t b = buffer_of(fresh_args()->wte + (size_t)(in ? v + i : 0) * d, 4 * (size_t)d);
#pragma unroll
          for (int s = 0; s < NS; ++s) t[i][s] = load4<0>(b, in ? o + 4 * SEG * s : OUT);
        }
      };
      table(v0 + RV * wave);
      request_ln(fresh_args()->lnf_g, fresh_args()->lnf_b);
      nap(fresh_args()->delay[0]);
      gather_row(fresh_args()->bufR2, ep);
      if (bail) return;
      f32x4 x[NS];
      normalised(x, true);
      float best = -INFINITY;
      int besti = 0x7fffffff;
#pragma unroll 1
      for (int v = v0 + RV * wave; v < v1; v += RV * NW) {
        float z[RV];
#pragma unroll
        for (int i = 0; i < RV; ++i) {
          z[i] = 0.f;
#pragma unroll
          for (int s = 0; s < NS; ++s) z[i] += dot4(t[i][s], x[s]);
        }
        table(v + RV * NW);
        wave_sums(z);
#pragma unroll
        for (int i = 0; i < RV; ++i)
          if (v + i < v1) {
            if (!SAMPLE && (z[i] > best || (besti == 0x7fffffff && z[i] == z[i]))) best = z[i], besti = v + i;  // (NaN: never)
            if ((SAMPLE || ends) && lane == 0) run[v + i - v0] = z[i];
          }
      }
      if (!SAMPLE && lane == 0) best_v[wave] = best, best_i[wave] = besti;
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the step's keys and values are where others read them)
      __syncthreads();
      if constexpr (SAMPLE) {
        if (wave == 0) {
          const int k = fresh_args()->top_k, n = v1 - v0;
          sel_key mine = 0;
          if (n <= 256) {
            sel_key keys[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int j = lane + 64 * i;
              keys[i] = j < n ? make_key(run[j], v0 + j) : 0;
            }
            mine = wave_firsts(keys, k, lane);
          } else {
            sel_key last = ~(sel_key)0;
            for (int r = 0; r < k; ++r) {
              sel_key best = 0;
              for (int j = lane; j < n; j += 64) {
                const sel_key key = make_key(run[j], v0 + j);
                best = key < last && key > best ? key : best;
              }
              last = wave_first(best);
              if (lane == r) mine = last;
            }
          }
          if (lane < k) {  // the r-th of all workgroups side by side
            const u32x4 pk = {(unsigned)mine, ep + 1, (unsigned)(mine >> 32), ep + 1};
            u64* to = fresh_args()->bufAM + 2 * (size_t)G * (PD_TOPK * (step & 1) + lane) + 2 * wg;
            asm volatile("global_store_dwordx4 %0, %1, off sc1" : : "v"(to), "v"(pk) : "memory");
          }
        }
      } else if (tid == 0) {
        for (int u = 1; u < NW; ++u) {
          const float v = best_v[u];
          const int i = best_i[u];
          if (i != 0x7fffffff && (besti == 0x7fffffff || v > best || (v == best && i < besti))) best = v, besti = i;
        }
        const u32x4 pk = {__float_as_uint(best), ep + 1, (unsigned)besti, ep + 1};
        u64* to = fresh_args()->bufAM + 2 * (size_t)(G * (step & 1) + wg);
        asm volatile("global_store_dwordx4 %0, %1, off sc1" : : "v"(to), "v"(pk) : "memory");
      }
      if (ends)
        for (int i = tid; i < v1 - v0; i += NT) {
          fresh_args()->logits[v0 + i] = run[i];
          if (fresh_args()->host_logits) fresh_args()->host_logits[v0 + i] = run[i];
        }
      if (ends && wg) return;
    }
    if (!ends) request_A(0);
    if constexpr (SAMPLE) {
      // ---- the top_k first of all workgroups' candidates, cpuSoftmax in float64 and sampleFromDistribution (globals.js:47-74) ----
      const int k = fresh_args()->top_k;
      const double rnd = fresh_args()->u ? fresh_args()->u[step] : fresh_args()->u_arg[step];
      nap(fresh_args()->delay[6]);
      const auto gather = [&](auto per_thread) {
        constexpr int N = decltype(per_thread)::value;
        int off[N];
        u32x4 v[N];
        sel_key keys[N];
        const int t = opaque(tid);
#pragma unroll
        for (int i = 0; i < N; ++i) off[i] = 16 * (t + NT * i < G * k ? t + NT * i : t);
        wt.words(buffer_of(fresh_args()->bufAM + 2 * (size_t)G * PD_TOPK * (step & 1), 16 * (size_t)G * PD_TOPK), off, v, ep + 1);
#pragma unroll
        for (int i = 0; i < N; ++i) keys[i] = t + NT * i < G * k ? (sel_key)v[i][2] << 32 | v[i][0] : 0;
        const sel_key mine = wave_firsts(keys, k, lane);
        if (lane < PD_TOPK) firsts[wave * PD_TOPK + lane] = mine;
      };
      if (k <= 2) gather(Count<1>());
      else if (k <= 4) gather(Count<2>());
      else gather(Count<4>());
      __syncthreads();
      if (bail) return;
      static_assert(NW * PD_TOPK == 64 && 4 * NT == PD_TOPK * G, "a key per lane, four words a thread");
      const sel_key all[1] = {firsts[lane]};
      const sel_key mine = wave_firsts(all, k, lane);
      // lane r: the r-th; sums in the reference's order on every lane
      const unsigned first = __builtin_amdgcn_readfirstlane((unsigned)(mine >> 32));
      const double mx = (double)key_value((sel_key)first << 32);
      const double e = exp(((double)key_value(mine) - mx) / fresh_args()->temperature);
      double sum = 0.0;
      for (int r = 0; r < k; ++r) sum += wave_read(e, r);
      const double p = e / sum;
      double cum = 0.0;
      int pick = -1;
      for (int r = 0; r < k && pick < 0; ++r) {
        cum += wave_read(p, r);
        if (rnd < cum) pick = r;
      }
      tok = __builtin_amdgcn_readfirstlane(__shfl(key_index(mine), pick < 0 ? k - 1 : pick));
      tok = tok >= 0 && tok < V ? tok : 0;
    } else {
      // ---- the arg-max of all workgroups (lowest index of equal ones) ----
      if (wave < G / 64) {
        nap(fresh_args()->delay[6]);
        int off[1] = {16 * opaque(tid)};
        u32x4 v[1];
        wt.words(buffer_of(fresh_args()->bufAM + 2 * (size_t)G * (step & 1), 16 * (size_t)G), off, v, ep + 1);
        float best = __uint_as_float(v[0][0]);
        int besti = (int)v[0][2];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          const float ov = __shfl_xor(best, o);
          const int oi = __shfl_xor(besti, o);
          if (oi != 0x7fffffff && (besti == 0x7fffffff || ov > best || (ov == best && oi < besti))) best = ov, besti = oi;
        }
        if (lane == 0) best_v[wave] = best, best_i[wave] = besti;
      }
      __syncthreads();
      if (bail) return;
      {
        float best = best_v[0];
        int besti = best_i[0];
        for (int u = 1; u < G / 64; ++u) {
          const float v = best_v[u];
          const int i = best_i[u];
          if (i != 0x7fffffff && (besti == 0x7fffffff || v > best || (v == best && i < besti))) best = v, besti = i;
        }
        tok = __builtin_amdgcn_readfirstlane(besti < V ? besti : 0);
      }
    }
    ep += 1;
    if (wg == 0 && tid == 0) {
      fresh_args()->out_tok[step] = tok;
      if (fresh_args()->host_ids) fresh_args()->host_ids[step] = tok;
      if (ends && fresh_args()->host_done) *fresh_args()->host_done = 0;
    }
  }
}

constexpr size_t RUN_LDS = 84 * 1024;  // more than half of a compute unit's, so that exactly one workgroup lives on each
constexpr size_t MAX_LDS = 128 * 1024;

size_t run_bytes(int V) { const size_t n = 4 * (size_t)((V + G - 1) / G); return n > RUN_LDS ? n : RUN_LDS; }

template <bool I8, int NS, int R, bool SAMPLE>
hipError_t launch_r(const PersistentArgs& a, hipStream_t s) {
  static bool enabled = false;  // dynamic LDS size already raised
  if (!enabled) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(decode_generic_kernel<I8, NS, R, SAMPLE>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)MAX_LDS);
    if (e != hipSuccess) return e;
    enabled = true;
  }
  decode_generic_kernel<I8, NS, R, SAMPLE><<<G, NT, run_bytes(a.V), s>>>(a);
  return hipGetLastError();
}
template <bool I8, int NS>
hipError_t launch_ns(const PersistentArgs& a, hipStream_t s) {
  if (a.top_k > 1) return a.d / a.H <= 64 ? launch_r<I8, NS, 4, true>(a, s) : launch_r<I8, NS, 8, true>(a, s);
  return a.d / a.H <= 64 ? launch_r<I8, NS, 4, false>(a, s) : launch_r<I8, NS, 8, false>(a, s);
}
template <bool I8>
hipError_t launch_any(const PersistentArgs& a, hipStream_t s) {
  if (a.d <= 256) return launch_ns<I8, 1>(a, s);
  if (a.d <= 512) return launch_ns<I8, 2>(a, s);
  if (a.d <= 768) return launch_ns<I8, 3>(a, s);
  if (a.d <= 1024) return launch_ns<I8, 4>(a, s);
  if (a.d <= 1280) return launch_ns<I8, 5>(a, s);
  return launch_ns<I8, 7>(a, s);
}

}  // namespace

bool decode_generic_supports(int d, int H, int hs, int ctx, int V, int compute_units) {
  if (compute_units < G || d % 8 || hs % 4 || hs > 128 || d > 1792 || H * hs != d || H > G || run_bytes(V) > MAX_LDS) return false;
  // (every width and dtype of this range, at short and long contexts, is faster than with launches: the figures above)
  // a slice's keys fit the registers of its workgroup
  const int lpk = hs <= 16 ? 4 : hs <= 32 ? 8 : hs <= 64 ? 16 : 32, most = H * DG_SPLIT <= G ? DG_SPLIT : G / H;
  return ctx <= most * (hs <= 64 ? 4 : 8) * NW * (64 / lpk);
}

hipError_t launch_decode_generic(const PersistentArgs& a, hipStream_t s) {
  if (!decode_generic_supports(a.d, a.H, a.d / a.H, a.ctx, a.V, G) || a.nsteps < 1 || a.top_k < 1 || a.top_k > PD_TOPK || a.top_k > a.V || a.pos0 + a.nsteps > a.ctx) return hipErrorInvalidValue;
  return a.weight_dtype == 1 ? launch_any<true>(a, s) : launch_any<false>(a, s);
}

}  // namespace wgpt
