// Per-block HIP kernels for gfx950 (wave64). One kernel family per instruction
// block of the reference (instructions.js); the arithmetic each one reproduces is
// cited at the kernel. Summation orders differ from the WGSL (lanes split the
// reduction and combine by wave shuffles), which stays inside the fp32 tolerance.
#include "kernels.h"

#include <algorithm>
#include <type_traits>

#include "gemm_split.h"
#include "pair_f16.h"
#include "select_key.h"

namespace wgpt {

namespace {

constexpr int WG = 256;     // threads per workgroup for every kernel here
constexpr int NWAVE = WG / 64;

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}

// Sum over a 256-thread workgroup; `sh` holds NWAVE floats. Every thread gets the result.
__device__ __forceinline__ float block_sum(float v, float* sh) {
  v = wave_sum(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  v = (sh[0] + sh[1]) + (sh[2] + sh[3]);
  __syncthreads();
  return v;
}

__device__ __forceinline__ float block_max(float v, float* sh) {
  v = wave_max(v);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  v = fmaxf(fmaxf(sh[0], sh[1]), fmaxf(sh[2], sh[3]));
  __syncthreads();
  return v;
}

// GELU of the reference, instructions.js:718-727: tanh form, exact 0 below -10,
// identity above 10; x^3 as x*x*x.
__device__ __forceinline__ float gelu_ref(float x) {
  const float x3 = x * x * x;
  const float cdf = 0.5f * (1.0f + tanhf(0.7978845608f * (x + 0.044715f * x3)));
  float r = x * cdf;
  r = x < -10.0f ? 0.0f : r;
  r = x > 10.0f ? x : r;
  return r;
}

// The same for a slab word, whose four bytes are consecutive k of ONE column (scale in every component of sc).
__device__ __forceinline__ float4 unpack_i8x4_k(int32_t word, const float4& sc);

__device__ __forceinline__ float4 ld4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ void st4(float* p, float4 v) { *reinterpret_cast<float4*>(p) = v; }

__device__ __forceinline__ void fma4(float4& acc, float a, const float4& w) {
  acc.x += a * w.x;
  acc.y += a * w.y;
  acc.z += a * w.z;
  acc.w += a * w.w;
}

// unpackInt8x4, other/int8-gemm.js:126-132: sign-extend each byte, then
// f32(b) / 127.0 * scale with a rounding after the divide and after the multiply.
__device__ __forceinline__ float4 unpack_i8x4(int32_t word, const float4& sc) {
  const int b0 = (word << 24) >> 24;
  const int b1 = (word << 16) >> 24;
  const int b2 = (word << 8) >> 24;
  const int b3 = word >> 24;
  float4 r;
  r.x = __fdiv_rn((float)b0, 127.0f) * sc.x;
  r.y = __fdiv_rn((float)b1, 127.0f) * sc.y;
  r.z = __fdiv_rn((float)b2, 127.0f) * sc.z;
  r.w = __fdiv_rn((float)b3, 127.0f) * sc.w;
  return r;
}
__device__ __forceinline__ float4 unpack_i8x4_k(int32_t word, const float4& sc) { return unpack_i8x4(word, sc); }

// ---------------------------------------------------------------------------
// FastMatMulBlock for M <= 4 (batch-1 decode): C = A . W + bias,
// instructions.js:248-314. W is [K,N] row-major as the reference keeps it.
// Stage 1: a workgroup owns a 64-column x 64-row tile of W; 16 lanes read one
// 256-byte row segment as float4s, the 16 lane groups take rows k0+ty, +16, ...
// and combine through LDS. Stage 2 sums the K/64 partials in ascending order,
// adds the bias last (as the shader does) and applies the epilogue.
// ---------------------------------------------------------------------------
template <int R>
__global__ __launch_bounds__(WG) void gemv_kn_partial(int N, int K, const float* __restrict__ A, int lda,
                                                       const float* __restrict__ W, int ldw, float* __restrict__ part) {
  __shared__ float4 red[R][16][16];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int n0 = blockIdx.x * 64 + tx * 4;
  const int k0 = blockIdx.y * GEMV_KCHUNK;
  float4 acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (n0 < N) {
#pragma unroll
    for (int i = 0; i < GEMV_KCHUNK / 16; ++i) {
      const int k = k0 + ty + 16 * i;
      if (k < K) {
        const float4 w = ld4(W + (size_t)k * ldw + n0);
#pragma unroll
        for (int r = 0; r < R; ++r) fma4(acc[r], A[(size_t)r * lda + k], w);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) red[r][ty][tx] = acc[r];
  __syncthreads();
  if (ty < R && n0 < N) {
    float4 s = red[ty][0][tx];
#pragma unroll
    for (int j = 1; j < 16; ++j) {
      const float4 v = red[ty][j][tx];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    st4(part + ((size_t)blockIdx.y * R + ty) * N + n0, s);
  }
}

// Sum of S partial sums, `stride` floats apart, in ascending order, U of them requested at a time: one after the other each is
// a memory round trip (reduce_ln_kernel, 128 rows of 768 in 8 slices: 5.6 -> 5.2 us; 345M prompt of 512: 3.47 -> 3.25 ms).
template <int U>
__device__ __forceinline__ float4 sum_slices_by(const float* p, size_t stride, int S) {
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s0 = 0; s0 < S; s0 += U) {
    float4 v[U];
#pragma unroll
    for (int j = 0; j < U; ++j) v[j] = ld4(p + (size_t)(s0 + j < S ? s0 + j : S - 1) * stride);
#pragma unroll
    for (int j = 0; j < U; ++j)
      if (s0 + j < S) {
        s.x += v[j].x; s.y += v[j].y; s.z += v[j].z; s.w += v[j].w;
      }
  }
  return s;
}
__device__ __forceinline__ float4 sum_slices(const float* p, size_t stride, int S) {
  return S <= 2 ? sum_slices_by<2>(p, stride, S) : S <= 4 ? sum_slices_by<4>(p, stride, S) : sum_slices_by<8>(p, stride, S);
}

// With kv.Kc set, C is a [M, 3d] q/k/v matrix whose key and value columns also go to the cache [H][ctx][hs].
__global__ __launch_bounds__(WG) void gemv_reduce(int M, int N, int S, const float* __restrict__ part,
                                                   const float* __restrict__ bias, float* C, int ldc, int epi,
                                                   const float* resid, KvAfter kv = KvAfter{nullptr, nullptr, 0, 0, 0, 0}) {
  const int n4 = N >> 2;
  const int idx = blockIdx.x * WG + threadIdx.x;
  if (idx >= M * n4) return;
  const int r = idx / n4, n0 = (idx - r * n4) * 4;
  float4 s = sum_slices(part + (size_t)r * N + n0, (size_t)M * N, S);
  if (bias) {
    const float4 b = ld4(bias + n0);
    s.x += b.x; s.y += b.y; s.z += b.z; s.w += b.w;
  }
  if (epi == EPI_GELU) {
    s.x = gelu_ref(s.x); s.y = gelu_ref(s.y); s.z = gelu_ref(s.z); s.w = gelu_ref(s.w);
  } else if (epi == EPI_RESIDUAL) {
    const float4 q = ld4(resid + (size_t)r * ldc + n0);
    s.x += q.x; s.y += q.y; s.z += q.z; s.w += q.w;
  }
  st4(C + (size_t)r * ldc + n0, s);
  if (kv.Kc && n0 >= kv.d) {
    const int which = n0 >= 2 * kv.d, c = n0 - (1 + which) * kv.d, h = c / kv.hs, e = c - h * kv.hs;
    st4((which ? kv.Vc : kv.Kc) + ((size_t)h * kv.ctx + kv.pos0 + r) * kv.hs + e, s);
  }
}

// gemv_reduce for the many slices of a matrix-vector product (S = K / 64): sixteen threads share an output
// float4, thread ty summing slices ty, ty + 16, ... (loads in flight together instead of S in a row), the
// sixteen sums combined in ascending ty by the first of them. Same result for every run; bias last.
__global__ __launch_bounds__(WG) void gemv_reduce_wide(int M, int N, int S, const float* __restrict__ part,
                                                        const float* __restrict__ bias, float* C, int ldc, int epi,
                                                        const float* resid) {
  __shared__ float4 red[16][16];
  const int n4 = N >> 2;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int idx = blockIdx.x * 16 + tx;
  const bool live = idx < M * n4;
  const int r = live ? idx / n4 : 0, n0 = live ? (idx - r * n4) * 4 : 0;
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live) {
#pragma unroll 4
    for (int sp = ty; sp < S; sp += 16) {
      const float4 v = ld4(part + ((size_t)sp * M + r) * N + n0);
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
  }
  red[ty][tx] = s;
  __syncthreads();
  if (ty != 0 || !live) return;
#pragma unroll
  for (int j = 1; j < 16; ++j) {
    const float4 v = red[j][tx];
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  if (bias) {
    const float4 b = ld4(bias + n0);
    s.x += b.x; s.y += b.y; s.z += b.z; s.w += b.w;
  }
  if (epi == EPI_GELU) {
    s.x = gelu_ref(s.x); s.y = gelu_ref(s.y); s.z = gelu_ref(s.z); s.w = gelu_ref(s.w);
  } else if (epi == EPI_RESIDUAL) {
    const float4 q = ld4(resid + (size_t)r * ldc + n0);
    s.x += q.x; s.y += q.y; s.z += q.z; s.w += q.w;
  }
  st4(C + (size_t)r * ldc + n0, s);
}

// gemv_reduce of one row followed by the LayerNorm of that row (layernorm_kernel's arithmetic and order of
// operations, thread t holding the float4 t, t + WG, ... of the row): C gets the finished row, ln_out its
// normalisation. One workgroup per row; N a multiple of 4, at most 4 * WG * REDUCE_LN_MAXV.
constexpr int REDUCE_LN_MAXV = 4;
__global__ __launch_bounds__(WG) void reduce_ln_kernel(int M, int N, int S, const float* __restrict__ part,
                                                        const float* __restrict__ bias, float* C, int ldc, int epi,
                                                        const float* resid, const float* __restrict__ gamma,
                                                        const float* __restrict__ beta, float* __restrict__ ln_out, int ldo) {
  __shared__ float sh[NWAVE];
  const int r = blockIdx.x, n4 = N >> 2;
  float4 v[REDUCE_LN_MAXV], gpre[REDUCE_LN_MAXV], bpre[REDUCE_LN_MAXV];
  float sum = 0.f;
#pragma unroll
  for (int j = 0; j < REDUCE_LN_MAXV; ++j) {
    const int i = threadIdx.x + j * WG;
    v[j] = make_float4(0.f, 0.f, 0.f, 0.f);
    gpre[j] = bpre[j] = v[j];
    if (i < n4) {
      const int n0 = 4 * i;
      // (requested with the partial sums: behind the two reductions they would be a memory round trip of their own)
      gpre[j] = ld4(gamma + n0);
      bpre[j] = ld4(beta + n0);
      float4 a = sum_slices(part + (size_t)r * N + n0, (size_t)M * N, S);
      if (bias) {
        const float4 b = ld4(bias + n0);
        a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
      }
      if (epi == EPI_GELU) {
        a.x = gelu_ref(a.x); a.y = gelu_ref(a.y); a.z = gelu_ref(a.z); a.w = gelu_ref(a.w);
      } else if (epi == EPI_RESIDUAL) {
        const float4 q = ld4(resid + (size_t)r * ldc + n0);
        a.x += q.x; a.y += q.y; a.z += q.z; a.w += q.w;
      }
      st4(C + (size_t)r * ldc + n0, a);
      v[j] = a;
      sum += (a.x + a.y) + (a.z + a.w);
    }
  }
  const float mean = block_sum(sum, sh) / (float)N;
  float q = 0.f;
#pragma unroll
  for (int j = 0; j < REDUCE_LN_MAXV; ++j) {
    if (threadIdx.x + j * WG < n4) {
      const float a = v[j].x - mean, b = v[j].y - mean, c = v[j].z - mean, d = v[j].w - mean;
      q += (a * a + b * b) + (c * c + d * d);
    }
  }
  const float var = block_sum(q, sh) / (float)N;
  const float stdev = sqrtf(var + 1e-5f);
#pragma unroll
  for (int j = 0; j < REDUCE_LN_MAXV; ++j) {
    const int i = threadIdx.x + j * WG;
    if (i < n4) {
      const float4 g = gpre[j], b = bpre[j];
      float4 o;
      o.x = g.x * ((v[j].x - mean) / stdev) + b.x;
      o.y = g.y * ((v[j].y - mean) / stdev) + b.y;
      o.z = g.z * ((v[j].z - mean) / stdev) + b.z;
      o.w = g.w * ((v[j].w - mean) / stdev) + b.w;
      st4(ln_out + (size_t)r * ldo + 4 * i, o);
    }
  }
}

// int8 weight-only stage 1 (other/int8-gemm.js:156-210 at M <= 4): a wave reads
// 64 consecutive words (256 columns) of one row; 4 waves take rows k0+ty, +4, ...
template <int R>
__global__ __launch_bounds__(WG) void gemv_kn_i8_partial(int N, int K, const float* __restrict__ A, int lda,
                                                          const int32_t* __restrict__ Wq, int ldwq,
                                                          const float* __restrict__ scale, float* __restrict__ part) {
  __shared__ float4 red[R][NWAVE][64];
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  const int n0 = blockIdx.x * 256 + tx * 4;
  const int k0 = blockIdx.y * GEMV_KCHUNK;
  float4 acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (n0 < N) {
    const float4 sc = ld4(scale + n0);
#pragma unroll 4
    for (int i = 0; i < GEMV_KCHUNK / NWAVE; ++i) {
      const int k = k0 + ty + NWAVE * i;
      if (k < K) {
        const float4 w = unpack_i8x4(Wq[(size_t)k * ldwq + (n0 >> 2)], sc);
#pragma unroll
        for (int r = 0; r < R; ++r) fma4(acc[r], A[(size_t)r * lda + k], w);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) red[r][ty][tx] = acc[r];
  __syncthreads();
  if (ty < R && n0 < N) {
    float4 s = red[ty][0][tx];
#pragma unroll
    for (int j = 1; j < NWAVE; ++j) {
      const float4 v = red[ty][j][tx];
      s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
    }
    st4(part + ((size_t)blockIdx.y * R + ty) * N + n0, s);
  }
}

__global__ __launch_bounds__(WG) void dequant_i8_kernel(int K, int N, const int32_t* __restrict__ Wq, int ldwq,
                                                         const float* __restrict__ scale, float* __restrict__ W, int ldw) {
  const int n4 = N >> 2;
  const size_t idx = (size_t)blockIdx.x * WG + threadIdx.x;
  if (idx >= (size_t)K * n4) return;
  const int k = (int)(idx / n4), w = (int)(idx - (size_t)k * n4);
  st4(W + (size_t)k * ldw + 4 * w, unpack_i8x4(Wq[(size_t)k * ldwq + w], ld4(scale + 4 * w)));
}

// ResidualBlock, instructions.js:381-382
__global__ __launch_bounds__(WG) void residual_kernel(size_t n4, const float* a, const float* b, float* out) {
  const size_t i = (size_t)blockIdx.x * WG + threadIdx.x;
  if (i >= n4) return;
  const float4 x = ld4(a + 4 * i), y = ld4(b + 4 * i);
  st4(out + 4 * i, make_float4(x.x + y.x, x.y + y.y, x.z + y.z, x.w + y.w));
}

// GeluBlock, instructions.js:718-746
__global__ __launch_bounds__(WG) void gelu_kernel(size_t n4, const float* x, float* out) {
  const size_t i = (size_t)blockIdx.x * WG + threadIdx.x;
  if (i >= n4) return;
  const float4 v = ld4(x + 4 * i);
  st4(out + 4 * i, make_float4(gelu_ref(v.x), gelu_ref(v.y), gelu_ref(v.z), gelu_ref(v.w)));
}

// LayerNormBlock: stats pass + norm pass of instructions.js:451-550 in one kernel,
// one workgroup per row. mean = sum/N; var = sum((x-mean)^2)/N; stdev = sqrt(var + 1e-5);
// out = gamma * ((x - mean) / stdev) + beta with a true division.
__global__ __launch_bounds__(WG) void layernorm_kernel(int N, const float* __restrict__ x, int ldx,
                                                        const float* __restrict__ gamma, const float* __restrict__ beta,
                                                        float* __restrict__ out, int ldo) {
  __shared__ float sh[NWAVE];
  const float* xr = x + (size_t)blockIdx.x * ldx;
  float* orow = out + (size_t)blockIdx.x * ldo;
  const int n4 = N >> 2;
  float s = 0.f;
  for (int i = threadIdx.x; i < n4; i += WG) {
    const float4 v = ld4(xr + 4 * i);
    s += (v.x + v.y) + (v.z + v.w);
  }
  const float mean = block_sum(s, sh) / (float)N;
  float q = 0.f;
  for (int i = threadIdx.x; i < n4; i += WG) {
    const float4 v = ld4(xr + 4 * i);
    const float a = v.x - mean, b = v.y - mean, c = v.z - mean, d = v.w - mean;
    q += (a * a + b * b) + (c * c + d * d);
  }
  const float var = block_sum(q, sh) / (float)N;
  const float stdev = sqrtf(var + 1e-5f);
  for (int i = threadIdx.x; i < n4; i += WG) {
    const float4 v = ld4(xr + 4 * i), g = ld4(gamma + 4 * i), b = ld4(beta + 4 * i);
    float4 o;
    o.x = g.x * ((v.x - mean) / stdev) + b.x;
    o.y = g.y * ((v.y - mean) / stdev) + b.y;
    o.z = g.z * ((v.z - mean) / stdev) + b.z;
    o.w = g.w * ((v.w - mean) / stdev) + b.w;
    st4(orow + 4 * i, o);
  }
}

// SoftmaxBlock, instructions.js:618-663: max from -3.402823e38, sum of exp(x - max),
// out = exp(x - max) / sum with the exponential recomputed and a true division.
// TRANSPOSE: the store of instructions.js:594 with `transpose` set: element i of row r goes to out[i * M + r].
template <bool TRANSPOSE>
__global__ __launch_bounds__(WG) void softmax_kernel(int M, int N, const float* __restrict__ x, float* __restrict__ out) {
  __shared__ float sh[NWAVE];
  const float* xr = x + (size_t)blockIdx.x * N;
  float* orow = out + (size_t)blockIdx.x * N;
  float m = -3.402823e+38f;
  for (int i = threadIdx.x; i < N; i += WG) m = fmaxf(m, xr[i]);
  m = block_max(m, sh);
  float s = 0.f;
  for (int i = threadIdx.x; i < N; i += WG) s += expf(xr[i] - m);
  s = block_sum(s, sh);
  for (int i = threadIdx.x; i < N; i += WG) {
    const float v = expf(xr[i] - m) / s;
    if (TRANSPOSE) out[(size_t)i * M + blockIdx.x] = v;
    else orow[i] = v;
  }
}

// out[c * rows + r] = in[r * cols + c] through a 32 x 32 tile of LDS (the host-side transpose of globals.js:80-94).
__global__ __launch_bounds__(256) void transpose_kernel(int rows, int cols, const float* __restrict__ in, float* __restrict__ out) {
  __shared__ float tile[32][33];
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  for (int k = ty; k < 32; k += 8)
    if (r0 + k < rows && c0 + tx < cols) tile[k][tx] = in[(size_t)(r0 + k) * cols + c0 + tx];
  __syncthreads();
  for (int k = ty; k < 32; k += 8)
    if (c0 + k < cols && r0 + tx < rows) out[(size_t)(c0 + k) * rows + r0 + tx] = tile[tx][k];
}

// EmbedBlock, instructions.js:795-821: gather + positional add in one pass.
__global__ __launch_bounds__(WG) void embed_kernel(const int32_t* __restrict__ idx, int d, int pos0,
                                                    const float* __restrict__ wte, const float* __restrict__ wpe,
                                                    float* __restrict__ out, const int* __restrict__ pos_dev = nullptr) {
  const int i = blockIdx.x;
  if (pos_dev) pos0 = *pos_dev;
  const size_t tok = (size_t)idx[i];
  const float* e = wte + tok * d;
  const float* p = wpe + (size_t)(pos0 + i) * d;
  for (int c = threadIdx.x; c < (d >> 2); c += WG) {
    const float4 a = ld4(e + 4 * c), b = ld4(p + 4 * c);
    st4(out + (size_t)i * d + 4 * c, make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w));
  }
}

// DeEmbedBlock, instructions.js:916-943, on the un-chunked, un-transposed wte[V,d]:
// row-major wte already has the contraction index contiguous, so a wave streams
// whole rows with 128-bit loads and reduces by shuffles. 4 rows per wave in flight.
constexpr int VOCAB_ROWS_PER_WAVE = 4;
__global__ __launch_bounds__(WG) void vocab_gemv_kernel(int V, int d, const float* __restrict__ x,
                                                         const float* __restrict__ wte, float* __restrict__ logits) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  for (int c = threadIdx.x; c < (d >> 2); c += WG) st4(xs + 4 * c, ld4(x + 4 * c));
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int v0 = (blockIdx.x * NWAVE + wave) * VOCAB_ROWS_PER_WAVE;
  float acc[VOCAB_ROWS_PER_WAVE];
#pragma unroll
  for (int r = 0; r < VOCAB_ROWS_PER_WAVE; ++r) acc[r] = 0.f;
  for (int c = lane; c < (d >> 2); c += 64) {
    const float4 xv = ld4(xs + 4 * c);
#pragma unroll
    for (int r = 0; r < VOCAB_ROWS_PER_WAVE; ++r) {
      if (v0 + r < V) {
        const float4 w = ld4(wte + (size_t)(v0 + r) * d + 4 * c);
        acc[r] += (xv.x * w.x + xv.y * w.y) + (xv.z * w.z + xv.w * w.w);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < VOCAB_ROWS_PER_WAVE; ++r) {
    const float s = wave_sum(acc[r]);
    if (lane == 0 && v0 + r < V) logits[v0 + r] = s;
  }
}

// AttentionBlock's formatQ + fusedWeights + softmax + attentionValues
// (instructions.js:1129-1136, 1167-1176, 618-663, 1205-1212) for one (head, query
// row) per workgroup, reading K and V rows 0..p of head h at Kc + h*hstride + j*ldkv. Masked
// positions j > p get weight exactly 0 in the reference (exp(-1e9 - max) underflows),
// so they are skipped rather than multiplied by zero.
__global__ __launch_bounds__(WG) void attention_kernel(int pos0, int hs, int lpk, float scale, const float* __restrict__ q,
                                                        int ldq, const float* __restrict__ Kc, const float* __restrict__ Vc,
                                                        size_t hstride, int ldkv, float* __restrict__ out, int ldo, PairRows pairs) {
  extern __shared__ __attribute__((aligned(16))) float scores[];
  __shared__ __attribute__((aligned(16))) float qs[256];  // read as float4
  __shared__ float red[1024];
  __shared__ float sh[NWAVE];
  const int h = blockIdx.x, i = blockIdx.y;
  const int nkeys = pos0 + i + 1;
  const int tid = threadIdx.x;
  if (tid < hs) qs[tid] = q[(size_t)i * ldq + h * hs + tid];
  __syncthreads();
  const int sub = tid & (lpk - 1), grp = tid / lpk, ngrp = WG / lpk;
  const bool act = sub * 4 < hs;
  const float4 qv = act ? ld4(qs + sub * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
  const float* kbase = Kc + h * hstride + sub * 4;
  const float* vbase = Vc + h * hstride + sub * 4;
  // eight key rows per lane group requested before the first is used: one after the other, the ~24 rounds of a
  // 380-key context each waited a full memory round trip
  for (int j0 = 0; j0 < nkeys; j0 += 8 * ngrp) {
    float4 kv[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int j = j0 + u * ngrp + grp;
      kv[u] = (act && j < nkeys) ? ld4(kbase + (size_t)j * ldkv) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int j = j0 + u * ngrp + grp;
      float part = (qv.x * kv[u].x + qv.y * kv[u].y) + (qv.z * kv[u].z + qv.w * kv[u].w);
      for (int off = lpk >> 1; off > 0; off >>= 1) part += __shfl_xor(part, off);
      if (sub == 0 && j < nkeys) scores[j] = part * scale;
    }
  }
  __syncthreads();
  float m = -3.402823e+38f;
  for (int j = tid; j < nkeys; j += WG) m = fmaxf(m, scores[j]);
  m = block_max(m, sh);
  float s = 0.f;
  for (int j = tid; j < nkeys; j += WG) {
    const float e = expf(scores[j] - m);
    scores[j] = e;
    s += e;
  }
  s = block_sum(s, sh);
  for (int j = tid; j < nkeys; j += WG) scores[j] = scores[j] / s;
  __syncthreads();
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  if (act) {
    int j = grp;
    for (; j + 7 * ngrp < nkeys; j += 8 * ngrp) {
      float4 vv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) vv[u] = ld4(vbase + (size_t)(j + u * ngrp) * ldkv);
#pragma unroll
      for (int u = 0; u < 8; ++u) fma4(acc, scores[j + u * ngrp], vv[u]);
    }
    for (; j < nkeys; j += ngrp) fma4(acc, scores[j], ld4(vbase + (size_t)j * ldkv));
    st4(red + grp * hs + sub * 4, acc);
  }
  __syncthreads();
  if (tid < hs) {
    float o = 0.f;
    for (int g = 0; g < ngrp; ++g) o += red[g * hs + tid];
    if (pairs.rows) put_pair(pairs.rows, pairs.K16, i, h * hs + tid, o * pairs.scale);
    else out[(size_t)i * ldo + h * hs + tid] = o;
  }
}


// Prefill attention for head size 64 with K and V tiled through LDS: one workgroup
// per (head, block of 16 query rows). Keys are visited in tiles of 64: the K and V
// rows of the tile are staged in LDS once and shared by the 16 queries (the
// per-query kernel above re-reads every row from L2 for every query). Thread
// (q = tid/16, c = tid%16): scores of query q for keys c, c+16, c+32, c+48 of the
// tile (q row in registers, K rows from LDS), running softmax over tiles, then the
// four output columns 4c..4c+3 of query q (weights through LDS, V rows from LDS).
// Arithmetic as the reference up to re-association: scale after the dot
// (instructions.js:1176), masked keys contribute nothing, exp(x - max) / sum.
constexpr int ATQ = 16, ATK = 64, AHS = 64, AKS = AHS + 4;  // row stride of the staged tiles (bank spread)
__device__ __forceinline__ float row16_allsum(float v) {
  v += __shfl_xor(v, 8);
  v += __shfl_xor(v, 4);
  v += __shfl_xor(v, 2);
  v += __shfl_xor(v, 1);
  return v;
}
__device__ __forceinline__ float row16_allmax(float v) {
  v = fmaxf(v, __shfl_xor(v, 8));
  v = fmaxf(v, __shfl_xor(v, 4));
  v = fmaxf(v, __shfl_xor(v, 2));
  v = fmaxf(v, __shfl_xor(v, 1));
  return v;
}

__global__ __launch_bounds__(WG) void attention_tile_kernel(int Tq, int pos0, float scale, const float* __restrict__ q, int ldq,
                                                             const float* __restrict__ Kc, const float* __restrict__ Vc,
                                                             size_t hstride, int ldkv, float* __restrict__ out, int ldo) {
  __shared__ float Ks[ATK * AKS];
  __shared__ float Vs[ATK * AKS];
  __shared__ float Ps[ATQ * ATK];
  const int h = blockIdx.x, i0 = blockIdx.y * ATQ;
  const int tid = threadIdx.x, qi = tid >> 4, c = tid & 15;
  const int i = i0 + qi;                 // query row of this thread (may be >= Tq in the last block)
  const int p = pos0 + i;                // its absolute position: keys 0..p are visible
  const int pmax = pos0 + (i0 + ATQ - 1 < Tq - 1 ? i0 + ATQ - 1 : Tq - 1);
  float4 qr[AHS / 4];
#pragma unroll
  for (int k = 0; k < AHS / 4; ++k)
    qr[k] = i < Tq ? ld4(q + (size_t)i * ldq + h * AHS + 4 * k) : make_float4(0.f, 0.f, 0.f, 0.f);
  const float* kbase = Kc + h * hstride;
  const float* vbase = Vc + h * hstride;
  float m = -INFINITY, l = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int j0 = 0; j0 <= pmax; j0 += ATK) {
    __syncthreads();  // previous tile fully consumed
    // stage the tile: 64 rows x 16 float4, 256 threads x 4
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = (tid >> 4) + 16 * r, col4 = tid & 15;
      float4 kv = make_float4(0.f, 0.f, 0.f, 0.f), vv = kv;
      if (j0 + row <= pmax) {
        kv = ld4(kbase + (size_t)(j0 + row) * ldkv + 4 * col4);
        vv = ld4(vbase + (size_t)(j0 + row) * ldkv + 4 * col4);
      }
      st4(Ks + row * AKS + 4 * col4, kv);
      st4(Vs + row * AKS + 4 * col4, vv);
    }
    __syncthreads();
    // scores of keys c, c+16, c+32, c+48
    float sc[4];
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float* kr = Ks + (c + 16 * r) * AKS;
      float a = 0.f;
#pragma unroll
      for (int k = 0; k < AHS / 4; ++k) {
        const float4 kv = ld4(kr + 4 * k);
        a += (qr[k].x * kv.x + qr[k].y * kv.y) + (qr[k].z * kv.z + qr[k].w * kv.w);
      }
      sc[r] = (j0 + c + 16 * r <= p) ? a * scale : -INFINITY;
      tmax = fmaxf(tmax, sc[r]);
    }
    tmax = row16_allmax(tmax);
    const float mnew = fmaxf(m, tmax);
    // rows beyond Tq and fully masked tiles keep m = -inf: guard the exponentials
    const float corr = mnew > -INFINITY ? expf(m - mnew) : 1.f;
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float pr = sc[r] > -INFINITY ? expf(sc[r] - mnew) : 0.f;
      Ps[qi * ATK + c + 16 * r] = pr;
      psum += pr;
    }
    psum = row16_allsum(psum);
    l = l * corr + psum;
    m = mnew;
    o.x *= corr; o.y *= corr; o.z *= corr; o.w *= corr;
    __syncthreads();  // weights of the tile visible (only this query's 16 lanes wrote them, but waves differ in pace)
    const float* pr = Ps + qi * ATK;
    const float* vr = Vs + 4 * c;
#pragma unroll 8
    for (int j = 0; j < ATK; ++j) fma4(o, pr[j], ld4(vr + j * AKS));
  }
  if (i < Tq) st4(out + (size_t)i * ldo + h * AHS + 4 * c, make_float4(o.x / l, o.y / l, o.z / l, o.w / l));
}

// ---------------------------------------------------------------------------
// Prefill attention on the matrix cores (head size 64, at least 32 queries).
// A workgroup owns 32 queries of one head; its four or eight waves split the visible keys
// into contiguous runs of 32-key tiles and are merged at the end (flash-decoding).
// Everything is computed transposed, S^T = K Q^T and O^T = V^T P^T, with
// v_mfma_f32_32x32x2_f32: an accumulator then holds, per lane, 16 keys (or output
// dimensions) of ONE query (column l % 32), so the softmax over keys is a reduction
// over a lane's own registers plus one exchange with lane l ^ 32, the rescaling of
// O by exp(m_old - m_new) is a per-lane scalar, and the probabilities are already
// in the operand layout of the second product:
//   accumulator register r of lane l is row (r/4)*8 + (l/32)*4 + r%4, column l%32;
//   operand lane l supplies A[row l%32][k l/32] and B[k l/32][col l%32] per step.
// The contraction index of either product may be visited in any order as long as
// both operands agree: QK^T steps through dimension (l/32)*32 + i at step i (each
// lane's 32 dimensions are contiguous in memory), PV through key
// (i/4)*8 + (l/32)*4 + i%4 at step i (exactly the key that register i holds).
// Scores are scaled by folding 1/sqrt(hs) into Q.
// ---------------------------------------------------------------------------
constexpr int AMQ = 32;        // queries per workgroup
constexpr int AMK = 32;        // keys per tile
constexpr int AMKST = AHS + 4; // row stride of a staged K tile (conflict-free 128-bit reads by 32 rows)
constexpr int AM_WAVE_FLOATS = AMK * AMKST + AMK * AHS;  // K tile + V tile of one wave
constexpr int AMOST = AMQ + 1; // row stride of a wave's O^T[dim][query] in the merge

typedef float f32x16 __attribute__((ext_vector_type(16)));

template <int NWV>
__global__ __launch_bounds__(NWV * 64) void attention_mfma_kernel(int Tq, int pos0, float scale, const float* __restrict__ q, int ldq,
                                                             const float* __restrict__ Kc, const float* __restrict__ Vc,
                                                             size_t hstride, int ldkv, float* __restrict__ out, int ldo) {
  extern __shared__ __attribute__((aligned(16))) float am_lds[];
  const int h = blockIdx.x, q0 = blockIdx.y * AMQ;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l32 = lane & 31, hh = lane >> 5;
  float* Ks = am_lds + wave * AM_WAVE_FLOATS;
  float* Vs = Ks + AMK * AMKST;
  const float* kbase = Kc + h * hstride;
  const float* vbase = Vc + h * hstride;
  const int qrow = q0 + l32;                 // this lane's query (may be >= Tq in the last block)
  const int qpos = pos0 + qrow;              // keys 0..qpos are visible to it
  const int qlast = q0 + AMQ - 1 < Tq - 1 ? q0 + AMQ - 1 : Tq - 1;
  const int nkeys = pos0 + qlast + 1;        // keys any query of the block sees
  const int nt = (nkeys + AMK - 1) / AMK;
  const int per = (nt + NWV - 1) / NWV;
  const int tb = wave * per;
  const int te = tb + per < nt ? tb + per : nt;

  float qf[32];  // scaled Q[qrow][hh*32 + i]
  {
    const float* qp = q + (size_t)(qrow < Tq ? qrow : Tq - 1) * ldq + h * AHS + hh * 32;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float4 v = ld4(qp + 4 * j);
      qf[4 * j] = v.x * scale; qf[4 * j + 1] = v.y * scale; qf[4 * j + 2] = v.z * scale; qf[4 * j + 3] = v.w * scale;
    }
  }
  float m = -INFINITY, lsum = 0.f;
  f32x16 o0, o1;
#pragma unroll
  for (int r = 0; r < 16; ++r) { o0[r] = 0.f; o1[r] = 0.f; }

  // the tile after the current one is already on its way from memory while the current one is multiplied.
  // The loads are unconditional (a load under a branch is waited for where the paths join, which would undo the
  // overlap): rows past the last key repeat it; no query of the block sees them, so their weights are exactly 0
  // and the repeated values only have to be finite.
  float4 kreg[8], vreg[8];
  auto fetch = [&](int t) {
    const int k0 = t * AMK;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int f = lane + 64 * j, row = f >> 4, c4 = f & 15;
      const int key = k0 + row < nkeys ? k0 + row : nkeys - 1;
      kreg[j] = ld4(kbase + (size_t)key * ldkv + 4 * c4);
      vreg[j] = ld4(vbase + (size_t)key * ldkv + 4 * c4);
    }
  };
  fetch(tb);
  for (int t = tb; t < te; ++t) {
    const int k0 = t * AMK;
    // stage the K and V tiles of this wave: 32 rows x 16 float4 each, 8 per lane
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int f = lane + 64 * j, row = f >> 4, c4 = f & 15;
      st4(Ks + row * AMKST + 4 * c4, kreg[j]);
      st4(Vs + row * AHS + 4 * c4, vreg[j]);
    }
    fetch(t + 1);
    __builtin_amdgcn_wave_barrier();  // the tiles are private to the wave: LDS operations of a wave complete in order
    // S^T[key][query] = sum_dim K[key][dim] Q[query][dim]
    f32x16 sacc;
#pragma unroll
    for (int r = 0; r < 16; ++r) sacc[r] = 0.f;
    {
      const float* kr = Ks + l32 * AMKST + hh * 32;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float4 kv = ld4(kr + 4 * j);
        sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.x, qf[4 * j], sacc, 0, 0, 0);
        sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.y, qf[4 * j + 1], sacc, 0, 0, 0);
        sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.z, qf[4 * j + 2], sacc, 0, 0, 0);
        sacc = __builtin_amdgcn_mfma_f32_32x32x2f32(kv.w, qf[4 * j + 3], sacc, 0, 0, 0);
      }
    }
    // causal mask and the running maximum of this lane's query
    float tmax = -INFINITY;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int key = k0 + (r >> 2) * 8 + hh * 4 + (r & 3);
      sacc[r] = key <= qpos ? sacc[r] : -INFINITY;
      tmax = fmaxf(tmax, sacc[r]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32));
    const float mnew = fmaxf(m, tmax);
    // a query with no visible key so far keeps m = -inf: guard the exponentials
    const float corr = mnew > -INFINITY ? __expf(m - mnew) : 1.f;
    float psum = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const float pr = sacc[r] > -INFINITY ? __expf(sacc[r] - mnew) : 0.f;
      sacc[r] = pr;
      psum += pr;
    }
    lsum = lsum * corr + psum;
    m = mnew;
#pragma unroll
    for (int r = 0; r < 16; ++r) { o0[r] *= corr; o1[r] *= corr; }
    // O^T[dim][query] += sum_key V[key][dim] P[query][key]; step i visits the key of register i
    {
      const float* vr = Vs + hh * 4 * AHS + l32;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const float* vk = vr + ((i >> 2) * 8 + (i & 3)) * AHS;
        o0 = __builtin_amdgcn_mfma_f32_32x32x2f32(vk[0], sacc[i], o0, 0, 0, 0);
        o1 = __builtin_amdgcn_mfma_f32_32x32x2f32(vk[32], sacc[i], o1, 0, 0, 0);
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
  lsum += __shfl_xor(lsum, 32);  // the two halves of a column saw disjoint keys, the same maximum

  // merge of the four waves: each leaves O^T (64 x 32), m and l of its key run in its own LDS region
  float* Om = am_lds + wave * AM_WAVE_FLOATS;  // [AHS][AMOST], then m[AMQ], l[AMQ]
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int dim = (r >> 2) * 8 + hh * 4 + (r & 3);
    Om[dim * AMOST + l32] = o0[r];
    Om[(dim + 32) * AMOST + l32] = o1[r];
  }
  if (hh == 0) {
    Om[AHS * AMOST + l32] = m;
    Om[AHS * AMOST + AMQ + l32] = lsum;
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < AMQ * AHS / (NWV * 64); ++j) {
    const int e = tid + NWV * 64 * j, qi = e >> 6, dim = e & 63;
    float mw[NWV], M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      mw[w] = am_lds[w * AM_WAVE_FLOATS + AHS * AMOST + qi];
      M = fmaxf(M, mw[w]);
    }
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      const float f = mw[w] > -INFINITY ? __expf(mw[w] - M) : 0.f;
      num += am_lds[w * AM_WAVE_FLOATS + dim * AMOST + qi] * f;
      den += am_lds[w * AM_WAVE_FLOATS + AHS * AMOST + AMQ + qi] * f;
    }
    if (q0 + qi < Tq) out[(size_t)(q0 + qi) * ldo + h * AHS + dim] = num / den;
  }
}

// ---------------------------------------------------------------------------
// One decode token with one launch per block of the layer (the path of every model shape, replayable as a HIP
// graph: nothing in a launch depends on the position except through *pos).
//
// gemv_slab_kernel: FastMatMulBlock at M = 1 (instructions.js:248-314) in ONE launch and one pass. The weights
// are read from the decode slabs, in which the K values of a column are contiguous (segments of 256: 64 lanes x
// float4, or x one word of four int8; K zero-padded to S segments): a wave owns R whole columns, so a dot product
// never leaves its wave, no partial sums pass through memory and the sum has one fixed order. Every workgroup
// first builds the input row in LDS, with the LayerNormBlock in front of the product applied on the way
// (instructions.js:451-550: layernorm_kernel's order of operations; each workgroup repeats the two reductions
// over the few KB of the row rather than wait for a separate launch). fp32 slabs of c_attn and c_fc hold
// diag(gamma) W and their bias holds bias + beta W, so for them the row is only normalised (ROW_NORMALISE);
// int8 slabs take the full LayerNorm (ROW_LAYERNORM). int8 weights are dequantised one by one as the shader does,
// float(q) / 127.0f * scale[n] (other/int8-gemm.js:126-132). Bias last, then GELU or the residual add; the key
// and value columns of a q/k/v row also go to cache row *pos.
// ---------------------------------------------------------------------------
enum { ROW_PLAIN = 0, ROW_NORMALISE = 1, ROW_LAYERNORM = 2, ROW_MERGE = 3 };
struct GemvSlabArgs {
  int N, K, S;
  const void* slab;
  const float* scale;   // int8: per column
  const float* x;       // [K]
  int row_mode;
  const float* gamma;
  const float* beta;
  const float* bias;
  int epi;
  const float* resid;   // [N], may alias C
  float* C;             // [N]
  float* Kc;            // null: no cache scatter
  float* Vc;
  int d, hs, ctx;
  const int* pos;
  int nslice;           // ROW_MERGE: x holds [K / mhs][nslice][mhs + 4] attention slices, of which the first nmerge are read
  int mhs;
  int nmerge;
};

typedef float nt_f32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ float4 ld4_stream(const float4* p) {  // read once per token: keep it out of the way of the row and the cache
  const nt_f32x4 t = __builtin_nontemporal_load(reinterpret_cast<const nt_f32x4*>(p));
  return make_float4(t.x, t.y, t.z, t.w);
}

template <int R, bool I8>
__global__ __launch_bounds__(WG) void gemv_slab_kernel(GemvSlabArgs a) {
  // segments of a column requested at a time (two register sets of this many): sized so that the kernel stays within
  // 128 registers and two workgroups fit a compute unit (grids of 300-400 workgroups then run in one round)
  constexpr int CH = (!I8 && R > 1) ? 4 : 8;
  extern __shared__ __attribute__((aligned(16))) float xs[];  // [S * 256]
  __shared__ float sh[NWAVE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int k4 = a.K >> 2, s64 = a.S * 64;
  // This wave's columns (beyond N: the last one again, never stored) and the first chunk of their weights, which
  // do not depend on the row: requested before the row is built, so that they travel during the LayerNorm.
  const int col0 = (blockIdx.x * NWAVE + wave) * R;
  typedef typename std::conditional<I8, int32_t, float4>::type Item;
  const Item* base[R];
  float4 sc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int col = col0 + r < a.N ? col0 + r : a.N - 1;
    base[r] = static_cast<const Item*>(a.slab) + (size_t)col * a.S * 64 + lane;
    if (I8) {
      const float s = a.scale[col];
      sc[r] = make_float4(s, s, s, s);
    }
  }
  // What the epilogue adds is requested now as well: a load behind the dot products would be one more memory round
  // trip at the end of a kernel that consists of little else. (resid may be C itself: column n is read and written
  // by its owner only.)
  float ebias[R], eres[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int col = col0 + r < a.N ? col0 + r : a.N - 1;
    ebias[r] = a.bias ? a.bias[col] : 0.f;
    eres[r] = a.epi == EPI_RESIDUAL ? a.resid[col] : 0.f;
  }
  const int kvpos = a.Kc ? *a.pos : 0;
  // ... and the LayerNorm parameters of this thread's first two float4 of the row (int8 slabs do not carry them)
  float4 gpre[2], bpre[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    gpre[p] = bpre[p] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (a.row_mode == ROW_LAYERNORM) {
      const int i = tid + WG * p < k4 ? tid + WG * p : k4 - 1;
      gpre[p] = ld4(a.gamma + 4 * i);
      bpre[p] = ld4(a.beta + 4 * i);
    }
  }
  Item w0[R][CH], w1[R][CH];
  auto request = [&](Item (&w)[R][CH], int c0) {
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < CH; ++j) {
        // unconditional: a segment beyond S repeats the last one and meets zeros
        const int seg = c0 + j < a.S ? c0 + j : a.S - 1;
        if constexpr (I8) w[r][j] = __builtin_nontemporal_load(base[r] + (size_t)seg * 64);
        else w[r][j] = ld4_stream(base[r] + (size_t)seg * 64);
      }
  };
  request(w0, 0);

  float s1 = 0.f;
  if (a.row_mode == ROW_MERGE) {
    // the row is the attention output, still in slices of the context: (o[hs] unnormalised, max, sum) per head and
    // slice, combined here as attention_decode_slice_kernel's header describes
    const int stride = a.mhs + 4;
    for (int i = tid; i < s64; i += WG) {
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (i < k4) {
        const int h = (4 * i) / a.mhs, e = 4 * i - h * a.mhs;
        const float* ph = a.x + (size_t)h * a.nslice * stride;
        // eight slices at a time, everything requested before anything is used: one round trip, not one per slice
        float mx = -3.402823e+38f, den = 0.f;
        for (int s0 = 0; s0 < a.nmerge; s0 += 8) {
          float mv[8], lv[8];
          float4 ov[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int sl = s0 + j < a.nmerge ? s0 + j : a.nmerge - 1;
            mv[j] = ph[sl * stride + a.mhs];
            lv[j] = ph[sl * stride + a.mhs + 1];
            ov[j] = ld4(ph + sl * stride + e);
          }
          float mnew = mx;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (s0 + j < a.nmerge) mnew = fmaxf(mnew, mv[j]);
          const float keep = expf(mx - mnew);  // rescales what earlier groups of eight have left
          den *= keep;
          v = make_float4(v.x * keep, v.y * keep, v.z * keep, v.w * keep);
          mx = mnew;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (s0 + j < a.nmerge) {
              const float w = expf(mv[j] - mx);
              den += w * lv[j];
              fma4(v, w, ov[j]);
            }
        }
        v = make_float4(v.x / den, v.y / den, v.z / den, v.w / den);
      }
      st4(xs + 4 * i, v);
    }
  } else {
    for (int i = tid; i < s64; i += WG) {
      const float4 v = i < k4 ? ld4(a.x + 4 * i) : make_float4(0.f, 0.f, 0.f, 0.f);
      st4(xs + 4 * i, v);
      s1 += (v.x + v.y) + (v.z + v.w);
    }
  }
  if (a.row_mode == ROW_NORMALISE || a.row_mode == ROW_LAYERNORM) {
    const float mean = block_sum(s1, sh) / (float)a.K;
    float q = 0.f;
    for (int i = tid; i < k4; i += WG) {
      const float4 v = ld4(xs + 4 * i);
      const float e0 = v.x - mean, e1 = v.y - mean, e2 = v.z - mean, e3 = v.w - mean;
      q += (e0 * e0 + e1 * e1) + (e2 * e2 + e3 * e3);
    }
    const float var = block_sum(q, sh) / (float)a.K;
    const float stdev = sqrtf(var + 1e-5f);
    for (int i = tid, p = 0; i < k4; i += WG, ++p) {
      const float4 v = ld4(xs + 4 * i);
      float4 o = make_float4((v.x - mean) / stdev, (v.y - mean) / stdev, (v.z - mean) / stdev, (v.w - mean) / stdev);
      if (a.row_mode == ROW_LAYERNORM) {
        const float4 g = p == 0 ? gpre[0] : (p == 1 ? gpre[1] : ld4(a.gamma + 4 * i));
        const float4 b = p == 0 ? bpre[0] : (p == 1 ? bpre[1] : ld4(a.beta + 4 * i));
        o = make_float4(g.x * o.x + b.x, g.y * o.y + b.y, g.z * o.z + b.z, g.w * o.w + b.w);
      }
      st4(xs + 4 * i, o);
    }
  }
  __syncthreads();
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.f;
  auto contract = [&](const Item (&w)[R][CH], int c0) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      float4 xv = make_float4(0.f, 0.f, 0.f, 0.f);
      if (c0 + j < a.S) xv = ld4(xs + (c0 + j) * 256 + lane * 4);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float4 wv;
        if constexpr (I8) wv = unpack_i8x4_k(w[r][j], sc[r]);
        else wv = w[r][j];
        acc[r] += (wv.x * xv.x + wv.y * xv.y) + (wv.z * xv.z + wv.w * xv.w);
      }
    }
  };
  for (int c0 = 0; c0 < a.S; c0 += 2 * CH) {
    if (c0 + CH < a.S) request(w1, c0 + CH);
    contract(w0, c0);
    if (c0 + CH < a.S) {
      if (c0 + 2 * CH < a.S) request(w0, c0 + 2 * CH);
      contract(w1, c0 + CH);
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    float v = wave_sum(acc[r]);
    const int n = col0 + r;
    if (lane == 0 && n < a.N) {
      if (a.bias) v += ebias[r];
      if (a.epi == EPI_GELU) v = gelu_ref(v);
      else if (a.epi == EPI_RESIDUAL) v += eres[r];
      a.C[n] = v;
      if (a.Kc && n >= a.d) {
        const int which = n >= 2 * a.d, c = n - (1 + which) * a.d, h = c / a.hs, e = c - h * a.hs;
        (which ? a.Vc : a.Kc)[((size_t)h * a.ctx + kvpos) * a.hs + e] = v;
      }
    }
  }
}

// Attention of ONE query (the token being decoded, at cache position *pos) per head: formatQ + fusedWeights +
// softmax + attentionValues of instructions.js:1129-1212 as attention_kernel computes them, arranged for the
// latency of a single dependent chain: a workgroup per head requests the first 16 key rows AND value rows of each
// of its lane groups (256 positions at head size 64) before anything else, so a context of up to 256 positions
// costs one memory round trip; longer contexts continue in batches of the same size.
__global__ __launch_bounds__(WG) void attention_decode_kernel(int hs, int lpk, int ctx, float scale, const float* __restrict__ q,
                                                               const float* __restrict__ Kc, const float* __restrict__ Vc,
                                                               size_t hstride, float* __restrict__ out, const int* __restrict__ pos) {
  constexpr int U = 16;
  extern __shared__ __attribute__((aligned(16))) float scores[];
  __shared__ float red[1024];
  __shared__ float sh[NWAVE];
  const int h = blockIdx.x, tid = threadIdx.x;
  const int sub = tid & (lpk - 1), grp = tid / lpk, ngrp = WG / lpk;
  const bool act = sub * 4 < hs;
  const float* kbase = Kc + h * hstride + (act ? sub * 4 : 0);
  const float* vbase = Vc + h * hstride + (act ? sub * 4 : 0);
  // The first batch is requested before the position is known (rows up to the end of the cache exist; those
  // beyond the context hold finite leftovers and are not used): its round trip overlaps that of *pos.
  const float4 qv = act ? ld4(q + h * hs + sub * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
  float4 k0[U], v0[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int j = u * ngrp + grp;
    j = j < ctx ? j : ctx - 1;
    k0[u] = ld4(kbase + (size_t)j * hs);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int j = u * ngrp + grp;
    j = j < ctx ? j : ctx - 1;
    v0[u] = ld4(vbase + (size_t)j * hs);
  }
  const int nkeys = *pos + 1;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = u * ngrp + grp;
    float part = (qv.x * k0[u].x + qv.y * k0[u].y) + (qv.z * k0[u].z + qv.w * k0[u].w);
    for (int off = lpk >> 1; off > 0; off >>= 1) part += __shfl_xor(part, off);
    if (sub == 0 && j < nkeys) scores[j] = part * scale;
  }
  for (int j0 = U * ngrp; j0 < nkeys; j0 += U * ngrp) {
    float4 kv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int j = j0 + u * ngrp + grp;
      j = j < nkeys ? j : nkeys - 1;
      kv[u] = ld4(kbase + (size_t)j * hs);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + u * ngrp + grp;
      float part = (qv.x * kv[u].x + qv.y * kv[u].y) + (qv.z * kv[u].z + qv.w * kv[u].w);
      for (int off = lpk >> 1; off > 0; off >>= 1) part += __shfl_xor(part, off);
      if (sub == 0 && j < nkeys) scores[j] = part * scale;
    }
  }
  __syncthreads();
  float m = -3.402823e+38f;
  for (int j = tid; j < nkeys; j += WG) m = fmaxf(m, scores[j]);
  m = block_max(m, sh);
  float s = 0.f;
  for (int j = tid; j < nkeys; j += WG) {
    const float e = expf(scores[j] - m);
    scores[j] = e;
    s += e;
  }
  s = block_sum(s, sh);
  for (int j = tid; j < nkeys; j += WG) scores[j] = scores[j] / s;
  __syncthreads();
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int j = u * ngrp + grp;
    if (j < nkeys) fma4(acc, scores[j], v0[u]);
  }
  for (int j0 = U * ngrp; j0 < nkeys; j0 += U * ngrp) {
    float4 vv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      int j = j0 + u * ngrp + grp;
      j = j < nkeys ? j : nkeys - 1;
      vv[u] = ld4(vbase + (size_t)j * hs);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = j0 + u * ngrp + grp;
      if (j < nkeys) fma4(acc, scores[j], vv[u]);
    }
  }
  if (act) st4(red + grp * hs + sub * 4, acc);
  __syncthreads();
  if (tid < hs) {
    float o = 0.f;
    for (int g = 0; g < ngrp; ++g) o += red[g * hs + tid];
    out[h * hs + tid] = o;
  }
}

// The same attention with the cache cut into fixed slices of ADS_ROWS x WG / lanes-per-key positions (64 at head size
// 64), a workgroup per (head, slice): the rows of a slice are one small request per lane group, so a context of any
// length is one memory round trip, spread over as many compute units as it has slices (one workgroup per head
// streaming a whole context is bound by what a single compute unit can fetch: 10 us at 150 positions, 25 us at 550).
// A slice up to the position the caller expects (spec_pos, the host's knowledge of *pos) requests its rows before it
// has read *pos; the others read *pos first and leave at once if they lie beyond the context. A slice leaves
// (sum_j e_j v_j, m, sum_j e_j) with e_j = exp(score_j - m), m its own maximum (flash-decoding); one beyond the
// context leaves (0, -FLT_MAX, 0). The consumer (gemv_slab_kernel, ROW_MERGE) combines them:
// out = sum_s w_s o_s / sum_s w_s l_s with w_s = exp(m_s - max_s m_s), which is softmax(scores) . V of
// instructions.js:1129-1212 in another order of summation.
constexpr int ADS_ROWS = 4;
__global__ __launch_bounds__(WG) void attention_decode_slice_kernel(int hs, int lpk, int ctx, float scale, const float* __restrict__ q,
                                                                     const float* __restrict__ Kc, const float* __restrict__ Vc,
                                                                     size_t hstride, float* __restrict__ part, const int* __restrict__ pos,
                                                                     int spec_pos) {
  constexpr int U = ADS_ROWS;
  extern __shared__ __attribute__((aligned(16))) float scores[];  // [U * WG / lpk]
  __shared__ float red[1024];
  __shared__ float sh[NWAVE];
  const int h = blockIdx.x, sl = blockIdx.y, nsl = gridDim.y, tid = threadIdx.x;
  const int sub = tid & (lpk - 1), grp = tid / lpk, ngrp = WG / lpk;
  const int j_lo = sl * U * ngrp;
  const bool act = sub * 4 < hs;
  const float* kbase = Kc + h * hstride + (act ? sub * 4 : 0);
  const float* vbase = Vc + h * hstride + (act ? sub * 4 : 0);
  // An expected slice requests its rows before the position is known (rows up to the end of the cache exist), as
  // attention_decode_kernel does. The others look at the position first: most of them are beyond the context most of
  // the time, and their rows would be most of the launch's traffic for nothing.
  const float4 qv = act ? ld4(q + h * hs + sub * 4) : make_float4(0.f, 0.f, 0.f, 0.f);  // (first: nothing below may wait for it)
  const bool spec = j_lo <= spec_pos;  // the caller expects this slice to have positions
  int n_here = 0;
  if (!spec) n_here = min(*pos + 1 - j_lo, U * ngrp);
  float* dst = part + ((size_t)h * nsl + sl) * (hs + 4);
  if (!spec && n_here <= 0) {
    if (tid < hs) dst[tid] = 0.f;
    if (tid == 0) {
      dst[hs] = -3.402823e+38f;
      dst[hs + 1] = 0.f;
    }
    return;
  }
  float4 k0[U], v0[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int j = j_lo + u * ngrp + grp;
    j = j < ctx ? j : ctx - 1;
    k0[u] = ld4(kbase + (size_t)j * hs);
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    int j = j_lo + u * ngrp + grp;
    j = j < ctx ? j : ctx - 1;
    v0[u] = ld4(vbase + (size_t)j * hs);
  }
  if (spec) {
    n_here = min(*pos + 1 - j_lo, U * ngrp);  // positions of this slice inside the context
    if (n_here <= 0) {                        // (the caller's expectation was wrong)
      if (tid < hs) dst[tid] = 0.f;
      if (tid == 0) {
        dst[hs] = -3.402823e+38f;
        dst[hs + 1] = 0.f;
      }
      return;
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int jl = u * ngrp + grp;
    float p = (qv.x * k0[u].x + qv.y * k0[u].y) + (qv.z * k0[u].z + qv.w * k0[u].w);
    for (int off = lpk >> 1; off > 0; off >>= 1) p += __shfl_xor(p, off);
    if (sub == 0 && jl < n_here) scores[jl] = p * scale;
  }
  __syncthreads();
  float m = -3.402823e+38f;
  for (int j = tid; j < n_here; j += WG) m = fmaxf(m, scores[j]);
  m = block_max(m, sh);
  float l = 0.f;
  for (int j = tid; j < n_here; j += WG) {
    const float e = expf(scores[j] - m);
    scores[j] = e;
    l += e;
  }
  l = block_sum(l, sh);
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int jl = u * ngrp + grp;
    if (jl < n_here) fma4(acc, scores[jl], v0[u]);
  }
  if (act) st4(red + grp * hs + sub * 4, acc);
  __syncthreads();
  if (tid < hs) {
    float o = 0.f;
    for (int g = 0; g < ngrp; ++g) o += red[g * hs + tid];
    dst[tid] = o;
  }
  if (tid == 0) {
    dst[hs] = m;
    dst[hs + 1] = l;
  }
}

// The final LayerNormBlock (model.js:224) and DeEmbedBlock (instructions.js:916-943) of a decode token in one
// launch: every workgroup normalises the row itself while staging it (layernorm_kernel's order of operations), then
// vocab_gemv_kernel's rows; the first workgroup finally advances the cache position, if the caller passes one (nothing
// later in the token reads it).
__global__ __launch_bounds__(WG) void vocab_gemv_ln_kernel(int V, int d, const float* __restrict__ x, const float* __restrict__ gamma,
                                                            const float* __restrict__ beta, const float* __restrict__ wte,
                                                            float* __restrict__ logits, int* pos) {
  extern __shared__ __attribute__((aligned(16))) float xs[];
  __shared__ float sh[NWAVE];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int v0 = (blockIdx.x * NWAVE + wave) * VOCAB_ROWS_PER_WAVE;
  const int n4 = d >> 2;
  // Everything that does not depend on the row is requested first, so that it travels during the LayerNorm: the first
  // two sweeps of this wave's table rows, and the LayerNorm parameters of this thread's first two float4 of the row.
  constexpr int PRE = 2;
  float4 wpre[PRE][VOCAB_ROWS_PER_WAVE], gpre[PRE], bpre[PRE];
#pragma unroll
  for (int p = 0; p < PRE; ++p) {
    const int c = lane + 64 * p < n4 ? lane + 64 * p : n4 - 1;
#pragma unroll
    for (int r = 0; r < VOCAB_ROWS_PER_WAVE; ++r) {
      const int row = v0 + r < V ? v0 + r : V - 1;
      wpre[p][r] = ld4(wte + (size_t)row * d + 4 * c);
    }
    const int ct = (int)threadIdx.x + WG * p < n4 ? (int)threadIdx.x + WG * p : n4 - 1;
    gpre[p] = ld4(gamma + 4 * ct);
    bpre[p] = ld4(beta + 4 * ct);
  }
  float s1 = 0.f;
  for (int c = threadIdx.x; c < n4; c += WG) {
    const float4 v = ld4(x + 4 * c);
    st4(xs + 4 * c, v);
    s1 += (v.x + v.y) + (v.z + v.w);
  }
  const float mean = block_sum(s1, sh) / (float)d;
  float q = 0.f;
  for (int c = threadIdx.x; c < n4; c += WG) {
    const float4 v = ld4(xs + 4 * c);
    const float e0 = v.x - mean, e1 = v.y - mean, e2 = v.z - mean, e3 = v.w - mean;
    q += (e0 * e0 + e1 * e1) + (e2 * e2 + e3 * e3);
  }
  const float var = block_sum(q, sh) / (float)d;
  const float stdev = sqrtf(var + 1e-5f);
  for (int c = threadIdx.x, p = 0; c < n4; c += WG, ++p) {
    const float4 v = ld4(xs + 4 * c);
    const float4 g = p == 0 ? gpre[0] : (p == 1 ? gpre[1] : ld4(gamma + 4 * c));
    const float4 b = p == 0 ? bpre[0] : (p == 1 ? bpre[1] : ld4(beta + 4 * c));
    st4(xs + 4 * c, make_float4(g.x * ((v.x - mean) / stdev) + b.x, g.y * ((v.y - mean) / stdev) + b.y,
                                g.z * ((v.z - mean) / stdev) + b.z, g.w * ((v.w - mean) / stdev) + b.w));
  }
  __syncthreads();
  float acc[VOCAB_ROWS_PER_WAVE];
#pragma unroll
  for (int r = 0; r < VOCAB_ROWS_PER_WAVE; ++r) acc[r] = 0.f;
#pragma unroll
  for (int p = 0; p < PRE; ++p) {
    const int c = lane + 64 * p;
    if (c < n4) {
      const float4 xv = ld4(xs + 4 * c);
#pragma unroll
      for (int r = 0; r < VOCAB_ROWS_PER_WAVE; ++r) {
        const float4 w = wpre[p][r];
        if (v0 + r < V) acc[r] += (xv.x * w.x + xv.y * w.y) + (xv.z * w.z + xv.w * w.w);
      }
    }
  }
  for (int c = lane + 64 * PRE; c < n4; c += 64) {
    const float4 xv = ld4(xs + 4 * c);
#pragma unroll
    for (int r = 0; r < VOCAB_ROWS_PER_WAVE; ++r) {
      if (v0 + r < V) {
        const float4 w = ld4(wte + (size_t)(v0 + r) * d + 4 * c);
        acc[r] += (xv.x * w.x + xv.y * w.y) + (xv.z * w.z + xv.w * w.w);
      }
    }
  }
#pragma unroll
  for (int r = 0; r < VOCAB_ROWS_PER_WAVE; ++r) {
    const float sum = wave_sum(acc[r]);
    if (lane == 0 && v0 + r < V) logits[v0 + r] = sum;
  }
  if (pos && blockIdx.x == 0 && threadIdx.x == 0) *pos += 1;
}

// Token selection of GPT.generate (model.js:81-85) on the device:
//   selectTopK (globals.js:66-74): stable descending sort of (value, index), first k;
//   cpuSoftmax (globals.js:59-64) of those k logits in float64:
//     exp((x - max) / temperature), summed left to right, divided by the sum;
//   sampleFromDistribution (globals.js:47-57): first i with u < p_0 + .. + p_i, else k - 1;
//     u is the caller's uniform draw in [0, 1) (the reference's Math.random()).
// The chosen id goes to tok[0] (input of the next decode step) and out[slot]; ids/probs
// (optional) receive the k selected indices and their probabilities.

// One workgroup. A bound below which the k largest logits cannot lie is the k-th largest of the threads' maxima, or a little
// less; the logits not below it are k candidates or some more (normal logits, V = 50257, k = 40: about 60), and only they are
// sorted: by counting, for each, the larger ones, or with a bitonic network when they are many. Reading the logits is 4 us of
// a launch (58 KB/us is what a compute unit gets): 13 us for V = 50257 and k = 40, where k rounds of a workgroup-wide arg-max
// took 165.
// Logits that leave more candidates than LDS holds (long runs of equal values) get the exact bound first, one bit at a time.
constexpr int SAMPLE_CAND = 8192, SAMPLE_RANK = 256;
template <bool REG>  // REG: V <= 65536, a thread's logits stay in registers between the two looks at them
__global__ __launch_bounds__(1024) void sample_topk_kernel(int V, int k, double temperature, const double* __restrict__ u,
                                                            const float* __restrict__ logits, int32_t* tok, int32_t* out, int slot,
                                                            int32_t* ids, double* probs) {
  extern __shared__ __attribute__((aligned(16))) sel_key cand[];  // [SAMPLE_CAND]
  __shared__ double ev[SAMPLE_MAX_K];
  __shared__ double total;
  __shared__ float bound;
  __shared__ int count;
  const int tid = threadIdx.x, lane = tid & 63;
  if (k > V) k = V;
  constexpr int RJ = REG ? 16 : 1;
  float4 mine[RJ];
  const auto fetch = [&](int j) {  // logits 4 (tid + 1024 j) ..
    const int i = 4 * (tid + 1024 * j);
    if (i + 3 < V) return ld4(logits + i);
    return make_float4(i < V ? logits[i] : NAN, i + 1 < V ? logits[i + 1] : NAN, i + 2 < V ? logits[i + 2] : NAN, NAN);
  };
  // f(value, index) for every logit of this thread (and NAN for places beyond the last)
  const auto each = [&](auto f) {
    const auto four = [&](const float4& v, int j) {
      const int i = 4 * (tid + 1024 * j);
      f(v.x, i);
      f(v.y, i + 1);
      f(v.z, i + 2);
      f(v.w, i + 3);
    };
    if constexpr (REG) {
#pragma unroll
      for (int j = 0; j < RJ; ++j) four(mine[j], j);
    } else {
      for (int j = 0; 4096 * j < V; ++j) four(fetch(j), j);
    }
  };
  if constexpr (REG) {
#pragma unroll
    for (int j = 0; j < RJ; ++j) mine[j] = fetch(j);
  }
  if (tid == 0) count = 0;
  float top = -INFINITY;
  each([&](float v, int) { top = fmaxf(top, v); });
  unsigned* tops = reinterpret_cast<unsigned*>(cand);
  tops[tid] = order_bits(top);
  __syncthreads();
  if (tid < 64) {
    unsigned m[16], least = 0u;
#pragma unroll
    for (int j = 0; j < 16; ++j) m[j] = tops[lane + 64 * j];
    for (int bit = 31; bit >= 0; --bit) {
      const unsigned trial = least | 1u << bit;
      int n = 0;
#pragma unroll
      for (int j = 0; j < 16; ++j) n += __popcll(__ballot(m[j] >= trial));
      if (n < k) continue;
      least = trial;
      if (n <= k + k / 2 + 16 && n < 512) break;  // near enough
    }
    // (the bits of -infinity are the least that a maximum has; with a shorter prefix every logit is a candidate)
    const unsigned low = order_bits(-INFINITY);
    if (tid == 0) bound = key_value((sel_key)(least < low ? low : least) << 32);
  }
  __syncthreads();
  const float least = bound;
  each([&](float v, int i) {
    if (v >= least) {
      const int at = atomicAdd(&count, 1);
      if (at < SAMPLE_CAND) cand[at] = make_key(v, i);
    }
  });
  __syncthreads();
  if (count > SAMPLE_CAND || count < k) {  // (fewer than k: NaN among the logits)
    // the exact k-th largest key, from its highest bit down: keys are distinct, so exactly k are not below it
    sel_key exact = 0;
    for (int bit = 63; bit >= 0; --bit) {
      const sel_key trial = exact | (sel_key)1 << bit;
      int n = 0;
      each([&](float v, int i) { n += i < V && make_key(v, i) >= trial; });
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off);
      __syncthreads();
      if (tid == 0) count = 0;
      __syncthreads();
      if (lane == 0) atomicAdd(&count, n);
      __syncthreads();
      if (count >= k) exact = trial;
    }
    __syncthreads();
    if (tid == 0) count = 0;
    __syncthreads();
    each([&](float v, int i) {
      if (i < V && make_key(v, i) >= exact) cand[atomicAdd(&count, 1)] = make_key(v, i);
    });
    __syncthreads();
  }
  const int n = count;
  if (n <= SAMPLE_RANK) {
    const sel_key x = tid < n ? cand[tid] : 0;
    int rank = 0;
    if (tid < n)
      for (int i = 0; i < n; ++i) rank += cand[i] > x;
    __syncthreads();
    if (tid < n) cand[rank] = x;
  } else {
    int size2 = 512;
    while (size2 < n) size2 <<= 1;
    for (int i = n + tid; i < size2; i += 1024) cand[i] = 0;
    __syncthreads();
    for (int size = 2; size <= size2; size <<= 1)
      for (int j = size >> 1; j > 0; j >>= 1) {
        for (int p = tid; p < size2 / 2; p += 1024) {
          const int a = 2 * p - (p & (j - 1)), b = a + j;
          const sel_key x = cand[a], y = cand[b];
          if ((y > x) == ((a & size) == 0)) {
            cand[a] = y;
            cand[b] = x;
          }
        }
        __syncthreads();
      }
  }
  __syncthreads();
  const double mx = (double)key_value(cand[0]);
  if (tid < k) ev[tid] = exp(((double)key_value(cand[tid]) - mx) / temperature);
  __syncthreads();
  if (tid < 64) {  // left to right, as cpuSoftmax adds them
    double sum = 0.0;
    for (int base = 0; base < k; base += 64) {
      const double mine64 = base + lane < k ? ev[base + lane] : 0.0;
      const int m = k - base < 64 ? k - base : 64;
      for (int i = 0; i < m; ++i) sum += wave_read(mine64, i);
    }
    if (tid == 0) total = sum;
  }
  __syncthreads();
  if (tid < k) {
    const double p = ev[tid] / total;
    ev[tid] = p;
    if (probs) probs[tid] = p;
    if (ids) ids[tid] = key_index(cand[tid]);
  }
  __syncthreads();
  if (tid < 64) {
    const double rnd = *u;
    double cum = 0.0;
    int pick = -1;
    for (int base = 0; base < k && pick < 0; base += 64) {
      const double mine64 = base + lane < k ? ev[base + lane] : 0.0;
      const int m = k - base < 64 ? k - base : 64;
      for (int i = 0; i < m && pick < 0; ++i) {
        cum += wave_read(mine64, i);
        if (rnd < cum) pick = base + i;
      }
    }
    if (pick < 0) pick = k - 1;
    if (tid == 0) {
      tok[0] = key_index(cand[pick]);
      if (out) out[slot] = key_index(cand[pick]);
    }
  }
}

// Greedy selection: selectTopK with top_k = 1 (globals.js:66-74) is a stable
// descending sort, i.e. the largest logit with the lowest index on ties.
__global__ __launch_bounds__(1024) void argmax_kernel(int V, const float* __restrict__ logits, int32_t* tok, int32_t* out,
                                                       int slot) {
  __shared__ float bv[1024];
  __shared__ int bi[1024];
  float best = -INFINITY;
  int besti = 0x7fffffff;
  // eight loads in flight per thread (one after the other, V = 50257 took 16 us); ascending i, so ties keep the lowest index
  for (int i0 = threadIdx.x; i0 < V; i0 += 8 * 1024) {
    float v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = i0 + u * 1024 < V ? logits[i0 + u * 1024] : 0.f;
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const int i = i0 + u * 1024;
      if (i < V && (v[u] > best || (besti == 0x7fffffff && v[u] == v[u]))) {  // (NaN: never)
        best = v[u];
        besti = i;
      }
    }
  }
  bv[threadIdx.x] = best;
  bi[threadIdx.x] = besti;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) {
      const float ov = bv[threadIdx.x + s];
      const int oi = bi[threadIdx.x + s];
      const float cv = bv[threadIdx.x];
      const int ci = bi[threadIdx.x];
      if (oi != 0x7fffffff && (ci == 0x7fffffff || ov > cv || (ov == cv && oi < ci))) {
        bv[threadIdx.x] = ov;
        bi[threadIdx.x] = oi;
      }
    }
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    const int first = bi[0] < V ? bi[0] : 0;
    tok[0] = first;
    if (out) out[slot] = first;
  }
}

inline unsigned cdiv(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

}  // namespace

// second pass of a matrix-vector product: slices side by side (up to sixteen slices the sum is still in ascending order)
static void launch_gemv_reduce(int M, int N, int S, const float* workspace, const float* bias, float* C, int ldc, int epi,
                               const float* resid, hipStream_t s) {
  if (S >= 4) gemv_reduce_wide<<<cdiv((size_t)M * (N >> 2), 16), WG, 0, s>>>(M, N, S, workspace, bias, C, ldc, epi, resid);
  else gemv_reduce<<<cdiv((size_t)M * (N >> 2), WG), WG, 0, s>>>(M, N, S, workspace, bias, C, ldc, epi, resid);
}

size_t gemv_workspace_floats(int M, int N, int K) {
  return (size_t)cdiv(K, GEMV_KCHUNK) * (size_t)(M < 1 ? 1 : M) * (size_t)N;
}

hipError_t launch_gemv_kn(int M, int N, int K, const float* A, int lda, const float* W, int ldw, const float* bias,
                          float* C, int ldc, int epi, const float* resid, float* workspace, hipStream_t s) {
  const int S = cdiv(K, GEMV_KCHUNK);
  const dim3 grid(cdiv(N, 64), S);
  switch (M) {
    case 1: gemv_kn_partial<1><<<grid, WG, 0, s>>>(N, K, A, lda, W, ldw, workspace); break;
    case 2: gemv_kn_partial<2><<<grid, WG, 0, s>>>(N, K, A, lda, W, ldw, workspace); break;
    case 3: gemv_kn_partial<3><<<grid, WG, 0, s>>>(N, K, A, lda, W, ldw, workspace); break;
    case 4: gemv_kn_partial<4><<<grid, WG, 0, s>>>(N, K, A, lda, W, ldw, workspace); break;
    default: return hipErrorInvalidValue;
  }
  launch_gemv_reduce(M, N, S, workspace, bias, C, ldc, epi, resid, s);
  return hipGetLastError();
}

hipError_t launch_gemv_kn_i8(int M, int N, int K, const float* A, int lda, const int32_t* Wq, int ldwq,
                             const float* scale, const float* bias, float* C, int ldc, int epi, const float* resid,
                             float* workspace, hipStream_t s) {
  const int S = cdiv(K, GEMV_KCHUNK);
  const dim3 grid(cdiv(N, 256), S);
  switch (M) {
    case 1: gemv_kn_i8_partial<1><<<grid, WG, 0, s>>>(N, K, A, lda, Wq, ldwq, scale, workspace); break;
    case 2: gemv_kn_i8_partial<2><<<grid, WG, 0, s>>>(N, K, A, lda, Wq, ldwq, scale, workspace); break;
    case 3: gemv_kn_i8_partial<3><<<grid, WG, 0, s>>>(N, K, A, lda, Wq, ldwq, scale, workspace); break;
    case 4: gemv_kn_i8_partial<4><<<grid, WG, 0, s>>>(N, K, A, lda, Wq, ldwq, scale, workspace); break;
    default: return hipErrorInvalidValue;
  }
  launch_gemv_reduce(M, N, S, workspace, bias, C, ldc, epi, resid, s);
  return hipGetLastError();
}

hipError_t launch_dequant_i8(int K, int N, const int32_t* Wq, int ldwq, const float* scale, float* W, int ldw, hipStream_t s) {
  dequant_i8_kernel<<<cdiv((size_t)K * (N >> 2), WG), WG, 0, s>>>(K, N, Wq, ldwq, scale, W, ldw);
  return hipGetLastError();
}

size_t gemm_workspace_floats(int M, int N) { return (size_t)8 * M * N; }

namespace {
// Second pass of a split-K product: ordered sum of the S partial matrices, bias, epilogue; with `ln` the
// LayerNorm of the finished rows in the same kernel.
void finish_split(int M, int N, int S, const float* workspace, const float* bias, float* C, int ldc, int epi, const float* resid,
                  const LnAfter* ln, const KvAfter* kv, hipStream_t s) {
  if (kv) {
    gemv_reduce<<<cdiv((size_t)M * (N >> 2), WG), WG, 0, s>>>(M, N, S, workspace, bias, C, ldc, epi, resid, *kv);
    if (ln) layernorm_kernel<<<M, WG, 0, s>>>(N, C, ldc, ln->gamma, ln->beta, ln->out, ln->ldo);
    return;
  }
  if (ln && (N & 3) == 0 && N <= 4 * WG * REDUCE_LN_MAXV) {
    reduce_ln_kernel<<<M, WG, 0, s>>>(M, N, S, workspace, bias, C, ldc, epi, resid, ln->gamma, ln->beta, ln->out, ln->ldo);
    return;
  }
  gemv_reduce<<<cdiv((size_t)M * (N >> 2), WG), WG, 0, s>>>(M, N, S, workspace, bias, C, ldc, epi, resid);
  if (ln) layernorm_kernel<<<M, WG, 0, s>>>(N, C, ldc, ln->gamma, ln->beta, ln->out, ln->ldo);
}

constexpr size_t GEMM_BYTES = ((size_t)1 << 31) - 4096;  // of A or W that a launch reaches: its offsets have 32 bits and a sign
// Rows of W that a launch takes (a multiple of four, or all K), ldw words of four bytes apart; 0: not even four
int gemm_rows_of_w(int K, int ldw) {
  return (int)std::min<size_t>((size_t)K, std::min(GEMM_BYTES / (sizeof(float) * (size_t)ldw), GEMM_BYTES / sizeof(float)) / 4 * 4);
}

// C = epi(A . W + bias) on the matrix cores; W fp32 [K, ldw], or words of four int8 with a scale per column
// (blocked: in the order of launch_block_weights). K from gemm_rows_of_w.
hipError_t run_gemm(int M, int N, int K, const float* A, int lda, const void* W, int ldw, const float* wscale, const float* bias,
                    float* C, int ldc, int epi, const float* resid, float* workspace, const LnAfter* ln, const KvAfter* kv, bool blocked, hipStream_t s) {
  const bool i8 = wscale != nullptr;
  SplitGemmArgs a{};
  a.N = N; a.K = K; a.lda = lda; a.W = W; a.ldw = ldw; a.blocked = blocked; a.wscale = wscale; a.bias = bias; a.epi = epi; a.ldc = ldc;
  if (kv) { a.Kc = kv->Kc; a.Vc = kv->Vc; a.d = kv->d; a.hs = kv->hs; a.ctx = kv->ctx; }
  // the kernels address A with 32-bit offsets: very tall matrices go in runs of rows, of which the last has K columns
  const int rows = (int)std::min<size_t>((size_t)M, 1 + (GEMM_BYTES - sizeof(float) * (size_t)K) / (sizeof(float) * (size_t)lda));
  for (int m0 = 0; m0 < M; m0 += rows) {
    const int m = std::min(rows, M - m0);
    const SplitPlan p = plan_gemm_split(m, N, K, i8, blocked, ln != nullptr, workspace != nullptr);
    a.M = m;
    a.A = A + (size_t)m0 * lda;
    a.C = C + (size_t)m0 * ldc;
    a.resid = resid ? resid + (size_t)m0 * ldc : nullptr;
    a.pos0 = kv ? kv->pos0 + m0 : 0;
    a.part = p.S > 1 ? workspace : nullptr;
    const hipError_t e = launch_gemm_split(p, a, i8, s);
    if (e != hipSuccess) return e;
    KvAfter kv2;
    if (kv) { kv2 = *kv; kv2.pos0 = a.pos0; }
    LnAfter ln2;
    if (ln) { ln2 = *ln; ln2.out = ln->out + (size_t)m0 * ln->ldo; }
    if (p.S > 1) finish_split(m, N, p.S, workspace, bias, a.C, ldc, epi, a.resid, ln ? &ln2 : nullptr, kv ? &kv2 : nullptr, s);
    else if (ln) layernorm_kernel<<<m, WG, 0, s>>>(N, a.C, ldc, ln2.gamma, ln2.beta, ln2.out, ln2.ldo);
  }
  return hipGetLastError();
}

// Rows of W so long that not even four are in reach (134 M columns, four times as many of int8): the matrix-vector kernels, a
// few rows of A at a time, in the workspace of the product.
template <typename F>
hipError_t gemv_by_rows(int M, int N, int K, const float* workspace, F launch) {
  const int most = std::min(M, GEMV_MAX_ROWS);
  if (!workspace || gemv_workspace_floats(most, N, K) > gemm_workspace_floats(M, N)) return hipErrorInvalidValue;
  for (int m0 = 0; m0 < M; m0 += most) {
    const hipError_t e = launch(m0, std::min(most, M - m0));
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}
}  // namespace

hipError_t launch_gemm(int M, int N, int K, const float* A, int lda, const float* W, int ldw, const float* bias,
                       float* C, int ldc, int epi, const float* resid, float* workspace, hipStream_t s, const LnAfter* ln,
                       const KvAfter* kv, bool blocked) {
  // a larger W goes in runs of rows whose products are added up
  const int rows = gemm_rows_of_w(K, ldw);
  if (rows >= K) return run_gemm(M, N, K, A, lda, W, ldw, nullptr, bias, C, ldc, epi, resid, workspace, ln, kv, blocked, s);
  if (blocked || epi != EPI_NONE || ln || kv) return hipErrorInvalidValue;
  if (rows == 0) return gemv_by_rows(M, N, K, workspace, [&](int m0, int m) {
    return launch_gemv_kn(m, N, K, A + (size_t)m0 * lda, lda, W, ldw, bias, C + (size_t)m0 * ldc, ldc, EPI_NONE, nullptr, workspace, s);
  });
  for (int k0 = 0; k0 < K; k0 += rows) {
    const hipError_t e = run_gemm(M, N, std::min(rows, K - k0), A + k0, lda, W + (size_t)k0 * ldw, ldw, nullptr,
                                  k0 + rows >= K ? bias : nullptr, C, ldc, k0 ? EPI_RESIDUAL : EPI_NONE, k0 ? C : nullptr, workspace, nullptr, nullptr, false, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_gemm_i8(int M, int N, int K, const float* A, int lda, const int32_t* Wq, int ldwq, const float* scale,
                          const float* bias, float* C, int ldc, int epi, const float* resid, float* workspace, hipStream_t s,
                          const LnAfter* ln, const KvAfter* kv, bool blocked) {
  const int rows = gemm_rows_of_w(K, ldwq);
  if (rows >= K) return run_gemm(M, N, K, A, lda, Wq, ldwq, scale, bias, C, ldc, epi, resid, workspace, ln, kv, blocked, s);
  if (blocked || epi != EPI_NONE || ln || kv) return hipErrorInvalidValue;
  if (rows == 0) return gemv_by_rows(M, N, K, workspace, [&](int m0, int m) {
    return launch_gemv_kn_i8(m, N, K, A + (size_t)m0 * lda, lda, Wq, ldwq, scale, bias, C + (size_t)m0 * ldc, ldc, EPI_NONE, nullptr, workspace, s);
  });
  for (int k0 = 0; k0 < K; k0 += rows) {
    const hipError_t e = run_gemm(M, N, std::min(rows, K - k0), A + k0, lda, Wq + (size_t)k0 * ldwq, ldwq, scale,
                                  k0 + rows >= K ? bias : nullptr, C, ldc, k0 ? EPI_RESIDUAL : EPI_NONE, k0 ? C : nullptr, workspace, nullptr, nullptr, false, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t launch_residual(size_t n4, const float* a, const float* b, float* out, hipStream_t s) {
  residual_kernel<<<cdiv(n4, WG), WG, 0, s>>>(n4, a, b, out);
  return hipGetLastError();
}

hipError_t launch_gelu(size_t n4, const float* x, float* out, hipStream_t s) {
  gelu_kernel<<<cdiv(n4, WG), WG, 0, s>>>(n4, x, out);
  return hipGetLastError();
}

hipError_t launch_layernorm(int M, int N, const float* x, int ldx, const float* gamma, const float* beta, float* out, int ldo,
                            hipStream_t s) {
  layernorm_kernel<<<M, WG, 0, s>>>(N, x, ldx, gamma, beta, out, ldo);
  return hipGetLastError();
}

hipError_t launch_transpose(int rows, int cols, const float* in, float* out, hipStream_t s) {
  transpose_kernel<<<dim3((unsigned)((cols + 31) / 32), (unsigned)((rows + 31) / 32)), 256, 0, s>>>(rows, cols, in, out);
  return hipGetLastError();
}

hipError_t launch_softmax(int M, int N, const float* x, float* out, bool transpose, hipStream_t s) {
  if (transpose) softmax_kernel<true><<<M, WG, 0, s>>>(M, N, x, out);
  else softmax_kernel<false><<<M, WG, 0, s>>>(M, N, x, out);
  return hipGetLastError();
}

hipError_t launch_embed(const int32_t* idx, int T, int d, int pos0, const float* wte, const float* wpe, float* out, hipStream_t s) {
  embed_kernel<<<T, WG, 0, s>>>(idx, d, pos0, wte, wpe, out);
  return hipGetLastError();
}

hipError_t launch_vocab_gemv(int V, int d, const float* x, const float* wte, float* logits, hipStream_t s) {
  const int rows_per_wg = NWAVE * VOCAB_ROWS_PER_WAVE;
  vocab_gemv_kernel<<<cdiv(V, rows_per_wg), WG, sizeof(float) * d, s>>>(V, d, x, wte, logits);
  return hipGetLastError();
}

// Where the split operands pay for the pass that makes them (two launches; MI355X, us saved per call against the kernels
// below). Head size 64 has a matrix kernel of its own: from 700 rows 4 to 8 us at 2 to 25 heads, at 600 rows 4 at 2 heads but
// -0.3 at 25. The other sizes have a workgroup per query, which reads all keys: 12 heads x 48 at 128 rows -2.5, at 192 4.1, at
// 943 98; 12 x 32 at 192 3.4, 2 x 32 -0.4; above 96 the operands of a wave take half the registers: 1 x 128 at 192 rows -2.3,
// at 256 0.1, at 320 0.8, 8 x 128 -2.8, 3.1, 9.5. Sizes up to 16 are padded to 32 dimensions and need several heads for their
// work to be more than the launches: 12 x 8 at 192 rows 1.8, 2 x 8 -0.7, at 1024 -2.0, at 2048 4.4.
static bool attention_splits(int Tq, int pos0, int H, int hs) {
  if (hs > 128 || (hs & 3) || H > 65535 || pos0 + Tq > 12288) return false;
  if (hs <= 16 && (size_t)H * Tq < 12 * 192) return false;
  return Tq >= (hs == AHS ? 700 : hs > 96 ? 256 : 192);
}

size_t attention_workspace_bytes(int Tq, int pos0, int H, int hs) {
  return attention_splits(Tq, pos0, H, hs) ? attention_split_bytes(Tq, pos0, H, hs) : 0;
}

hipError_t launch_attention(int Tq, int pos0, int H, int hs, float scale, const float* q, int ldq, const float* Kc,
                            const float* Vc, size_t hstride, int ldkv, float* out, int ldo, void* ws, hipStream_t s, const PairRows* pairs) {
  if (ws && attention_splits(Tq, pos0, H, hs)) return launch_attention_split(Tq, pos0, H, hs, scale, q, ldq, Kc, Vc, hstride, ldkv, out, ldo, ws, s, pairs);
  // a block of 32 queries per workgroup on the matrix cores
  if (!pairs && hs == AHS && Tq >= AMQ) {
    static_assert(AHS * AMOST + 2 * AMQ <= AM_WAVE_FLOATS, "merge area must fit a wave's tile area");
    // eight waves once the longest query block has more than eight key tiles
    const bool wide = cdiv(pos0 + Tq, AMK) > 8;
    const size_t lds = sizeof(float) * (wide ? 8 : 4) * AM_WAVE_FLOATS;
    static bool enabled = false;
    if (!enabled) {
      hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_mfma_kernel<4>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)(sizeof(float) * 4 * AM_WAVE_FLOATS));
      if (e == hipSuccess)
        e = hipFuncSetAttribute(reinterpret_cast<const void*>(attention_mfma_kernel<8>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)(sizeof(float) * 8 * AM_WAVE_FLOATS));
      if (e != hipSuccess) return e;
      enabled = true;
    }
    if (wide) attention_mfma_kernel<8><<<dim3(H, cdiv(Tq, AMQ)), 512, lds, s>>>(Tq, pos0, scale, q, ldq, Kc, Vc, hstride, ldkv, out, ldo);
    else attention_mfma_kernel<4><<<dim3(H, cdiv(Tq, AMQ)), 256, lds, s>>>(Tq, pos0, scale, q, ldq, Kc, Vc, hstride, ldkv, out, ldo);
    return hipGetLastError();
  }
  // enough (head, query block) workgroups to fill the GPU; else one workgroup per query row
  if (!pairs && hs == AHS && Tq >= ATQ && H * cdiv(Tq, ATQ) >= 128) {
    attention_tile_kernel<<<dim3(H, cdiv(Tq, ATQ)), WG, 0, s>>>(Tq, pos0, scale, q, ldq, Kc, Vc, hstride, ldkv, out, ldo);
    return hipGetLastError();
  }
  int lpk = 1;
  while (lpk * 4 < hs) lpk <<= 1;
  if (lpk > 64 || hs > 256 || (hs & 3)) return hipErrorInvalidValue;
  const size_t smem = sizeof(float) * (size_t)(pos0 + Tq);
  if (smem > 48 * 1024) return hipErrorInvalidValue;
  attention_kernel<<<dim3(H, Tq), WG, smem, s>>>(pos0, hs, lpk, scale, q, ldq, Kc, Vc, hstride, ldkv, out, ldo, pairs ? *pairs : PairRows{});
  return hipGetLastError();
}

hipError_t launch_sample_topk(int V, int k, double temperature, const double* u, const float* logits, int32_t* tok,
                              int32_t* out, int slot, int32_t* ids, double* probs, hipStream_t s) {
  if (V < 1 || V > SAMPLE_MAX_V || k < 1 || k > SAMPLE_MAX_K) return hipErrorInvalidValue;
  constexpr size_t lds = sizeof(sel_key) * SAMPLE_CAND;
  const auto kernel = V <= 65536 ? sample_topk_kernel<true> : sample_topk_kernel<false>;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return e;
  kernel<<<1, 1024, lds, s>>>(V, k, temperature, u, logits, tok, out, slot, ids, probs);
  return hipGetLastError();
}

hipError_t launch_gemv_slab(int N, int K, const void* slab, bool int8, const float* scale, const float* x, int row_mode,
                            const float* gamma, const float* beta, const float* bias, float* C, int epi, const float* resid,
                            const KvAfter* kv, const int* pos, hipStream_t s, const AttnSlices* merge) {
  if ((K & 3) || N < 1) return hipErrorInvalidValue;
  if (merge && (row_mode != GEMV_ROW_PLAIN || merge->nslice < 1 || merge->nmerge < 1 || merge->nmerge > merge->nslice || merge->hs < 4 ||
                (merge->hs & 3) || K % merge->hs))
    return hipErrorInvalidValue;
  const int S = cdiv(K, 256);
  const size_t lds = sizeof(float) * (size_t)S * 256;
  if (lds > 48 * 1024) return hipErrorInvalidValue;
  GemvSlabArgs a{N, K, S, slab, scale, merge ? merge->part : x, merge ? (int)ROW_MERGE : row_mode, gamma, beta, bias, epi, resid, C,
                 kv ? kv->Kc : nullptr, kv ? kv->Vc : nullptr, kv ? kv->d : 0, kv ? kv->hs : 1, kv ? kv->ctx : 0, pos,
                 merge ? merge->nslice : 0, merge ? merge->hs : 1, merge ? merge->nmerge : 0};
  if (int8) {
    if (N >= 4096) gemv_slab_kernel<4, true><<<cdiv(N, NWAVE * 4), WG, lds, s>>>(a);
    else gemv_slab_kernel<2, true><<<cdiv(N, NWAVE * 2), WG, lds, s>>>(a);
  } else {
    if (N >= 2048) gemv_slab_kernel<2, false><<<cdiv(N, NWAVE * 2), WG, lds, s>>>(a);
    else gemv_slab_kernel<1, false><<<cdiv(N, NWAVE), WG, lds, s>>>(a);
  }
  return hipGetLastError();
}

hipError_t launch_embed_at(const int32_t* tok, int d, const int* pos, const float* wte, const float* wpe, float* x, hipStream_t s) {
  embed_kernel<<<1, WG, 0, s>>>(tok, d, 0, wte, wpe, x, pos);
  return hipGetLastError();
}

hipError_t launch_attention_decode(int H, int hs, int ctx, float scale, const float* q, const float* Kc, const float* Vc, float* out,
                                   const int* pos, hipStream_t s) {
  int lpk = 1;
  while (lpk * 4 < hs) lpk <<= 1;
  if (lpk > 64 || hs > 256 || (hs & 3)) return hipErrorInvalidValue;
  const size_t smem = sizeof(float) * (size_t)ctx;  // scores of the longest context: the launch is the same at every position
  if (smem > 48 * 1024) return hipErrorInvalidValue;
  attention_decode_kernel<<<H, WG, smem, s>>>(hs, lpk, ctx, scale, q, Kc, Vc, (size_t)ctx * hs, out, pos);
  return hipGetLastError();
}

int attention_decode_slice_positions(int hs) {
  int lpk = 1;
  while (lpk * 4 < hs) lpk <<= 1;
  return lpk > 64 ? 0 : ADS_ROWS * (WG / lpk);
}

int attention_decode_slices(int hs, int ctx) {
  const int p = attention_decode_slice_positions(hs);
  return p ? cdiv(ctx, p) : 0;
}

hipError_t launch_attention_decode_slices(int H, int hs, int ctx, float scale, const float* q, const float* Kc, const float* Vc,
                                          const AttnSlices* out, const int* pos, int spec_pos, hipStream_t s) {
  int lpk = 1;
  while (lpk * 4 < hs) lpk <<= 1;
  if (lpk > 64 || hs > 256 || (hs & 3) || !out || out->hs != hs || out->nslice != attention_decode_slices(hs, ctx)) return hipErrorInvalidValue;
  const size_t smem = sizeof(float) * ADS_ROWS * (WG / lpk);
  attention_decode_slice_kernel<<<dim3(H, out->nslice), WG, smem, s>>>(hs, lpk, ctx, scale, q, Kc, Vc, (size_t)ctx * hs, out->part, pos,
                                                                       spec_pos);
  return hipGetLastError();
}

hipError_t launch_vocab_gemv_ln(int V, int d, const float* x, const float* gamma, const float* beta, const float* wte, float* logits,
                                int* pos, hipStream_t s) {
  const int rows_per_wg = NWAVE * VOCAB_ROWS_PER_WAVE;
  vocab_gemv_ln_kernel<<<cdiv(V, rows_per_wg), WG, sizeof(float) * d, s>>>(V, d, x, gamma, beta, wte, logits, pos);
  return hipGetLastError();
}

hipError_t launch_argmax(int V, const float* logits, int32_t* tok, int32_t* out, int slot, hipStream_t s) {
  argmax_kernel<<<1, 1024, 0, s>>>(V, logits, tok, out, slot);
  return hipGetLastError();
}

}  // namespace wgpt
