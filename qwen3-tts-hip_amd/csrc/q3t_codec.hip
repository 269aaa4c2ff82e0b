// gfx950 kernels of the codec decoder (codec frames -> 24 kHz audio) besides its matrix-core
// GEMMs (launch_gemm) and convolutions: RVQ gather, depthwise causal conv, LayerNorm, causal
// attention with RoPE, and the last convolution.  Activations are time-major [T][C] fp32; a "padded"
// buffer starts with zero rows so that causal convolutions read rows before time 0 as zeros.
#include "q3t_codec.h"
#include "q3t_bf16x3.h"

#include <float.h>
#include <math.h>

namespace q3t {
namespace {

__device__ __forceinline__ float wave_sum64(float v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// E[t][0, D) = first[codes[t][0] mod V]; E[t][D, 2D) = sum over groups g = 1 .. G-1 (in that
// order) of rest[g-1][codes[t][g] mod V] (codec_rvq_project_f32's gathers, kernels.rs:454-495).
__global__ void k_codec_rvq(const int32_t *codes, int groups, const float *first, const float *rest, int V, int D,
                            float *E) {
  const int t = blockIdx.x;
  const int32_t *c = codes + (size_t)t * groups;
  auto wrap = [&](int32_t code) { return ((code % V) + V) % V; };
  for (int d = threadIdx.x; d < D; d += blockDim.x) {
    E[(size_t)t * 2 * D + d] = first[(size_t)wrap(c[0]) * D + d];
    float r = 0.f;
    for (int g = 1; g < groups; ++g) r += rest[((size_t)(g - 1) * V + wrap(c[g])) * D + d];
    E[(size_t)t * 2 * D + D + d] = r;
  }
}

// alpha := exp(alpha), beta := 1 / (exp(beta) + 1e-9), once at load: the per-channel factors of
// every Snake (codec_snake_beta_f32, kernels.rs:692-710).
__global__ void k_codec_snake_prep(float *alpha, float *beta, int C) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= C) return;
  alpha[c] = expf(alpha[c]);
  beta[c] = 1.0f / (expf(beta[c]) + 1.0e-9f);
}

// ConvNeXt's depthwise causal convolution, 7 taps, rows before time 0 zeros
// (codec_depthwise_causal_conv1d_f32, kernels.rs:642-667), and the LayerNorm of its rows
// (codec_layernorm_f32, kernels.rs:582-612): variance E[x^2] - mean^2, clamped at 0.  A 256-thread
// workgroup per row of 1,024 channels, a thread's four channels 256 apart and in registers between
// the two.  Latency-bound: two kernels and a memset of the rows before time 0 were three launches of
// ~4 us each.
constexpr int kDwC = 1024, kDwK = 7;

__global__ __launch_bounds__(256) void k_codec_dwconv_norm(const float *x, const float *w, const float *wb,
                                                           const float *g, const float *b, float eps, float *out) {
  constexpr int N = kDwC / 256;
  __shared__ float ps[4], pq[4];
  const int tid = threadIdx.x, t = blockIdx.x;
  float v[N], s = 0.f, q = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int c = tid + 256 * i;
    v[i] = wb[c];
#pragma unroll
    for (int j = 0; j < kDwK; ++j) {
      const int r = t - (kDwK - 1) + j;
      const float e = x[(size_t)max(r, 0) * kDwC + c];
      v[i] += (r >= 0 ? e : 0.f) * w[c * kDwK + j];
    }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) {
    s += v[i];
    q += v[i] * v[i];
  }
  s = wave_sum64(s);
  q = wave_sum64(q);
  if ((tid & 63) == 0) {
    ps[tid >> 6] = s;
    pq[tid >> 6] = q;
  }
  __syncthreads();
  const float mean = (((ps[0] + ps[1]) + ps[2]) + ps[3]) / (float)kDwC;
  const float var = fmaxf((((pq[0] + pq[1]) + pq[2]) + pq[3]) / (float)kDwC - mean * mean, 0.f);
  const float inv = rsqrtf(var + eps);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int c = tid + 256 * i;
    out[(size_t)t * kDwC + c] = (v[i] - mean) * inv * g[c] + b[c];
  }
}

// Causal attention over rows 0..t for query row t and head h: rotate-half RoPE on q and k
// (position = row, cos/sin table [T][32]; rope_bhsd_f32, kernels.rs:40-77), scores scaled by
// `scale`, softmax, weighted sum of V (attention_scores_causal_f32 + masked softmax + apply_value,
// kernels.rs:980-1040).  qkv rows: [q heads | k heads | v heads] x 64 dims, not rotated.
//
// One workgroup per (head, 16 query rows), longest first, on v_mfma_f32_16x16x4_f32 (fp32 products
// and sums); its four waves take every fourth 16-key tile with an online softmax each, the next
// tile in flight, and merge through LDS in wave order (k_attn_prefill's scheme at 64 dims).  Lane
// (li, kk) holds dims 8 kk .. + 7 and 32 + 8 kk .. + 7 of key and query row li, the two halves of
// 8 rotation pairs, so RoPE needs no exchange and no pass of its own; scores of keys 4 kk + e for
// query li; and dims 16 kk .. + 15 of the output of query li (value rows are read 4 dims a lane).
// Bound: the latency of a tile's chain, T / 64 tiles a wave.  One workgroup per query row on the
// vector units, with a RoPE launch before it, took 69 + 4 us at T = 240.
__global__ __launch_bounds__(256, 2) void k_codec_attention(const float *qkv, int T, int ld, int heads,
                                                            const float2 *table, float scale, float *out, int ldo) {
  constexpr int W = 4;
  __shared__ float mo[W][16][64];
  __shared__ float mm[W][16], ml[W][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, li = lane & 15, kk = lane >> 4;
  const int h = blockIdx.x, q0 = 16 * ((int)gridDim.y - 1 - (int)blockIdx.y), Q = heads * 64;
  const int nkt = (min(q0 + 16, T) + 15) / 16;

  struct Rows {  // a row's 16 dims, their 8 rotations, and (keys) 4 value rows of 4 dims
    f32x4_t x[4], cs[4], v[4];
  };
  auto load_row = [&](int r, int col, Rows &o) {
    const f32x4_t *p = reinterpret_cast<const f32x4_t *>(qkv + (size_t)r * ld + col + 8 * kk);
    o.x[0] = p[0]; o.x[1] = p[1]; o.x[2] = p[8]; o.x[3] = p[9];
    const f32x4_t *c = reinterpret_cast<const f32x4_t *>(table + (size_t)r * 32 + 8 * kk);
#pragma unroll
    for (int i = 0; i < 4; ++i) o.cs[i] = c[i];
  };
  auto rotate = [](const Rows &o, float *y) {  // y[i], y[8 + i]: pair i
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float p = o.x[i >> 2][i & 3], q = o.x[2 + (i >> 2)][i & 3];
      const float cos = o.cs[i >> 1][2 * (i & 1)], sin = o.cs[i >> 1][2 * (i & 1) + 1];
      y[i] = p * cos - q * sin;
      y[8 + i] = q * cos + p * sin;
    }
  };
  auto load_tile = [&](int kt, Rows &o) {
    load_row(min(16 * kt + li, T - 1), Q + h * 64, o);
#pragma unroll
    for (int s = 0; s < 4; ++s)
      o.v[s] = *reinterpret_cast<const f32x4_t *>(qkv + (size_t)min(16 * kt + 4 * kk + s, T - 1) * ld + 2 * Q + h * 64 +
                                                  4 * li);
  };
  Rows cur, nxt;
  if (wave < nkt) load_tile(wave, cur);
  float q[16];
  {
    Rows r;
    load_row(min(q0 + li, T - 1), h * 64, r);
    rotate(r, q);
  }
  f32x4_t o[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) o[t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -FLT_MAX, l = 0.f;
  const int qrow = q0 + li;
  for (int kt = wave; kt < nkt; kt += W) {
    if (kt + W < nkt) load_tile(kt + W, nxt);
    float k[16];
    rotate(cur, k);
    f32x4_t st = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 16; ++s) st = __builtin_amdgcn_mfma_f32_16x16x4f32(k[s], q[s], st, 0, 0, 0);
    float p[4], mt = -FLT_MAX;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p[e] = 16 * kt + 4 * kk + e <= qrow ? st[e] * scale : -FLT_MAX;
      mt = fmaxf(mt, p[e]);
    }
    mt = fmaxf(mt, __shfl_xor(mt, 16, 64));
    mt = fmaxf(mt, __shfl_xor(mt, 32, 64));
    const float m_new = fmaxf(m_run, mt), corr = expf(m_run - m_new);
    float ps = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      p[e] = p[e] == -FLT_MAX ? 0.f : expf(p[e] - m_new);
      ps += p[e];
    }
    l = l * corr + ps;
    m_run = m_new;
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] *= corr;
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int t = 0; t < 4; ++t) o[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(cur.v[s][t], p[s], o[t], 0, 0, 0);
    cur = nxt;
  }
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (kk == 0) {
    mm[wave][li] = m_run;
    ml[wave][li] = l;
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int e = 0; e < 4; ++e) mo[wave][4 * e + t][lane] = o[t][e];
  __syncthreads();
  if (qrow >= T) return;
  float m = mm[0][li];
#pragma unroll
  for (int w = 1; w < W; ++w) m = fmaxf(m, mm[w][li]);
  float lsum = 0.f, r[4] = {};
#pragma unroll
  for (int w = 0; w < W; ++w) {  // a wave without a tile has m = -FLT_MAX, l = 0: weight 0
    const float f = expf(mm[w][li] - m);
    lsum += ml[w][li] * f;
#pragma unroll
    for (int t = 0; t < 4; ++t) r[t] += mo[w][4 * wave + t][lane] * f;
  }
  const float inv = 1.0f / lsum;
  *reinterpret_cast<float4 *>(out + (size_t)qrow * ldo + h * 64 + 16 * kk + 4 * wave) =
      make_float4(r[0] * inv, r[1] * inv, r[2] * inv, r[3] * inv);
}

// Last convolution, 96 channels and 7 taps to one, + clamp to [-1, 1]: out[t] = clamp(b + sum_j P[t - 6 + j][j])
// with P[t][j] = sum_c x[t][c] w[j][c], rows before time 0 zeros (kernels.rs:742-770, 903-918).
//
// What bounds it: reading x.  The products over channels are a GEMM with the taps as (seven of sixteen)
// columns on v_mfma_f32_16x16x4_f32 (fp32 products and sums; 1.4 GFLOP at 240 frames, ~10 us), whose
// operand is x as it lies in memory: lane (li, kk) loads 16 bytes of row li per 16 channels and their
// four k's.  Only the seven sums a row go through LDS, to be added along the diagonal.  A thread per
// output with the rows staged in LDS, 672 dependent products each and a wave per SIMD for want of LDS,
// took 128 us at 240 frames (177 MB, 35 us at the copy rate) and 13 at 6.
// A wave takes two 16-row tiles, all twelve loads in flight; a block's 128 rows give 122 outputs.
constexpr int kFinalC = 96, kFinalK = 7, kFinalRows = 128, kFinalOut = kFinalRows - kFinalK + 1;

__global__ __launch_bounds__(256) void k_codec_final(const float *x, const float *w, const float *b, int T,
                                                     float *out) {
  constexpr int NC = kFinalC / 16, RT = 2;
  __shared__ float P[kFinalK][kFinalRows + 4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kk = lane >> 4;
  const int t0 = blockIdx.x * kFinalOut;
  f32x4_t xv[RT][NC], wv[NC];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int g = t0 - (kFinalK - 1) + 16 * (RT * wave + t) + li;
    const float *src = x + (size_t)min(max(g, 0), T - 1) * kFinalC + 4 * kk;
#pragma unroll
    for (int c = 0; c < NC; ++c) xv[t][c] = *reinterpret_cast<const f32x4_t *>(src + 16 * c);
    if (g < 0) {
#pragma unroll
      for (int c = 0; c < NC; ++c) xv[t][c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
  }
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    wv[c] = *reinterpret_cast<const f32x4_t *>(w + min(li, kFinalK - 1) * kFinalC + 16 * c + 4 * kk);
    if (li >= kFinalK) wv[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    f32x4_t acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[t][c][s], wv[c][s], acc, 0, 0, 0);
    // lane (li, kk) holds rows 4 kk .. + 3 of column li
    if (li < kFinalK) *reinterpret_cast<f32x4_t *>(&P[li][16 * (RT * wave + t) + 4 * kk]) = acc;
  }
  __syncthreads();
  const int t = t0 + tid;
  if (tid >= kFinalOut || t >= T) return;
  float s = b[0];
#pragma unroll
  for (int j = 0; j < kFinalK; ++j) s += P[j][tid + j];
  out[t] = fminf(fmaxf(s, -1.0f), 1.0f);
}

unsigned blocks_for(size_t n, unsigned threads) { return (unsigned)((n + threads - 1) / threads); }

}  // namespace

hipError_t launch_codec_rvq(const int32_t *codes, int frames, int groups, const float *first, const float *rest,
                            int V, int D, float *E, hipStream_t s) {
  if (frames <= 0 || groups < 2 || V <= 0 || D <= 0) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_codec_rvq, dim3(frames), dim3(256), 0, s, codes, groups, first, rest, V, D, E);
  return hipGetLastError();
}

hipError_t launch_codec_snake_prep(float *alpha, float *beta, int C, hipStream_t s) {
  if (C <= 0 || !alpha || !beta) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_codec_snake_prep, dim3((C + 255) / 256), dim3(256), 0, s, alpha, beta, C);
  return hipGetLastError();
}

hipError_t launch_codec_dwconv_norm(const float *x, const float *w, const float *wb, const float *g, const float *b,
                                    int T, int C, int K, float eps, float *out, hipStream_t s) {
  if (T <= 0 || C != kDwC || K != kDwK) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_codec_dwconv_norm, dim3(T), dim3(256), 0, s, x, w, wb, g, b, eps, out);
  return hipGetLastError();
}

hipError_t launch_codec_attention(const float *qkv, int T, int ld, int heads, const float2 *table, float scale,
                                  float *out, int ldo, hipStream_t s) {
  if (T <= 0 || T > kCodecMaxAttnRows || heads <= 0 || ld < 3 * heads * 64 || ld % 4 || ldo < heads * 64 || ldo % 4)
    return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_codec_attention, dim3(heads, (T + 15) / 16), dim3(256), 0, s, qkv, T, ld, heads, table, scale,
                     out, ldo);
  return hipGetLastError();
}

hipError_t launch_codec_final(const float *x, const float *w, const float *b, int T, int C, int K, float *out,
                              hipStream_t s) {
  auto aligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (T <= 0 || C != kFinalC || K != kFinalK || !aligned(x) || !aligned(w)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_codec_final, dim3(blocks_for(T, kFinalOut)), dim3(256), 0, s, x, w, b, T, out);
  return hipGetLastError();
}

}  // namespace q3t
