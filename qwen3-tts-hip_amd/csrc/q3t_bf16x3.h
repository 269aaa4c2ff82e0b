// Device helpers shared by the kernels: wave sums, the block order of a tiled grid, the three-term bf16
// form of an fp32 value, and the codec's Snake activation.
#pragma once

#include <hip/hip_runtime.h>

namespace q3t {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

// Cross-lane reductions on DPP (data-parallel primitives: VALU lane permutes, no LDS round
// trip).  Each step adds a permuted copy: quad_perm [1,0,3,2] and [2,3,0,1] (quads),
// row_half_mirror and row_mirror (rows of 16), then row_bcast:15 / row_bcast:31 fold the
// four rows into lane 63.  The order is fixed, so results are deterministic.
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ float dpp_f(float v, float fill) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, fill), __builtin_bit_cast(int, v),
                                                               CTRL, ROWS, 0xf, false));
}

// Sum over each row of 16 lanes, in every lane of the row.
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_f<0xB1>(v, 0.f);
  v += dpp_f<0x4E>(v, 0.f);
  v += dpp_f<0x141>(v, 0.f);
  v += dpp_f<0x140>(v, 0.f);
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
  v = row16_sum(v);
  v += dpp_f<0x142, 0xa>(v, 0.f);
  v += dpp_f<0x143, 0xc>(v, 0.f);
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Row block mb and column block nb of this workgroup, nbx column blocks a row block, all on grid x (y ends
// at 65,535 blocks, which a codec decode of 2,185 frames passes).  Few column blocks: each XCD
// (workgroup id % 8) takes a contiguous range of row-major block tiles, so that its L2 reads only its own
// rows, once for all column blocks.
__device__ __forceinline__ void block_tile(int nbx, int &mb, int &nb) {
  int t = blockIdx.x;
  if (nbx <= 8) {
    const int total = gridDim.x, xcd = t % 8, local = t / 8, C = (total + 7) / 8, r = total % 8;
    t = (r == 0 || xcd < r) ? xcd * C + local : r * C + (xcd - r) * (C - 1) + local;
  }
  mb = t / nbx;
  nb = t % nbx;
}

// x = hi + mid + lo, each bf16, exactly: hi is the upper half of x (its top 8 significant bits), x -
// hi is exact in fp32 and holds the other 16, mid is the upper half of that and lo the rest.  Every
// product with a bf16 weight is then exact, and a GEMM matches an fp32 product up to the order of
// the fp32 additions.  Halves are cut off by a mask and packed in pairs by a byte permute: 5.5
// full-rate operations an element.  Rounding to nearest instead (v_cvt_pk_bf16_f32 and back) takes
// as many, but the conversion issues at about a fifth of the rate: 1.8 times the time for the first
// term.  Not contracted: the residual is taken from the rounded x even where x is a product computed
// just before (otherwise the compiler may fuse that product into x - hi).
template <int N, typename V>
__device__ __forceinline__ void split_bf16_nc(const float *x, V &hi, V &mid, V &lo) {
#pragma clang fp contract(off)
  uint32_t h[N / 2], m[N / 2], l[N / 2];
  auto upper = [](float v) { return __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) & 0xffff0000u); };
  auto pair = [](float a, float b) {  // upper half of a, then of b
    return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
  };
#pragma unroll
  for (int e = 0; e < N; e += 2) {
    const float r0 = x[e] - upper(x[e]), r1 = x[e + 1] - upper(x[e + 1]);
    const float s0 = r0 - upper(r0), s1 = r1 - upper(r1);
    h[e / 2] = pair(x[e], x[e + 1]);
    m[e / 2] = pair(r0, r1);
    l[e / 2] = pair(s0, s1);
  }
  __builtin_memcpy(&hi, h, sizeof hi);
  __builtin_memcpy(&mid, m, sizeof mid);
  __builtin_memcpy(&lo, l, sizeof lo);
}
__device__ __forceinline__ void split_bf16x8_nc(const float *x, bf16x8_t &hi, bf16x8_t &mid, bf16x8_t &lo) {
  split_bf16_nc<8>(x, hi, mid, lo);
}

// The same value in three terms rounded to nearest, the form of the GEMMs (the sums of a GEMM depend
// on the terms in their last bits).  The conversion issues at about a fifth of the rate of the mask and
// permute above.
__device__ __forceinline__ void split_bf16x8_rn(const float *x, bf16x8_t &hi, bf16x8_t &mid, bf16x8_t &lo) {
#pragma clang fp contract(off)
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const f32x2_t v = {x[e], x[e + 1]};
    const bf16x2_t h = __builtin_convertvector(v, bf16x2_t);
    const f32x2_t r1 = v - __builtin_convertvector(h, f32x2_t);
    const bf16x2_t m = __builtin_convertvector(r1, bf16x2_t);
    const f32x2_t r2 = r1 - __builtin_convertvector(m, f32x2_t);
    const bf16x2_t l = __builtin_convertvector(r2, bf16x2_t);
    hi[e] = h[0]; hi[e + 1] = h[1];
    mid[e] = m[0]; mid[e + 1] = m[1];
    lo[e] = l[0]; lo[e + 1] = l[1];
  }
}

// Of a product x g: the first term is the rounded product's, the others hold what the exact product has
// past it.
__device__ __forceinline__ void split_bf16x8_rn_mul(const float *x, const float *g, bf16x8_t &hi, bf16x8_t &mid,
                                                    bf16x8_t &lo) {
#pragma clang fp contract(off)
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const f32x2_t v = {x[e] * g[e], x[e + 1] * g[e + 1]};
    const bf16x2_t h = __builtin_convertvector(v, bf16x2_t);
    const f32x2_t hf = __builtin_convertvector(h, f32x2_t);
    const f32x2_t r1 = {__builtin_fmaf(x[e], g[e], -hf[0]), __builtin_fmaf(x[e + 1], g[e + 1], -hf[1])};
    const bf16x2_t m = __builtin_convertvector(r1, bf16x2_t);
    const f32x2_t r2 = r1 - __builtin_convertvector(m, f32x2_t);
    const bf16x2_t l = __builtin_convertvector(r2, bf16x2_t);
    hi[e] = h[0]; hi[e + 1] = h[1];
    mid[e] = m[0]; mid[e + 1] = m[1];
    lo[e] = l[0]; lo[e + 1] = l[1];
  }
}

// Snake: v + sin(v ea)^2 ib, with the per-channel tables ea = exp(alpha), ib = 1 / (exp(beta) +
// 1e-9) (codec_snake_beta_f32, kernels.rs:692-710).
//
// sin^2 has period pi, so y = v ea is reduced by n = rint(y / pi) to r = y - n pi in
// [-pi/2, pi/2] (pi in two fp32 parts, each step one fma) and the sign of sin(r) does not
// matter; sin(r) is an odd polynomial of degree 11 (least-squares minimax fit of the relative
// error over |r| <= 1.62, 3.5e-11 before rounding).  Straight-line code of 14 operations: the
// library's sinf takes data-dependent branches for its range reduction, which a matrix-core
// kernel's prologue or epilogue cannot hide.  Against fp64 over N(0, 1) and N(0, 100) arguments
// sin(r) is within 1.2e-7 absolute, 2e-8 rms (a correctly rounded sine: 6e-8, 1.5e-8).  The
// reduction holds while n is an exact small integer; past kSnakeFast the caller takes snake_any.
constexpr float kSnakeFast = 65536.0f;

__device__ __forceinline__ float snake_fast(float v, float y, float ib) {
  const float n = __builtin_rintf(y * 3.183098733e-01f);
  float r = __builtin_fmaf(n, -3.141592741e+00f, y);
  r = __builtin_fmaf(n, 8.742277657e-08f, r);
  const float z = r * r;
  float p = __builtin_fmaf(z, -2.381510633e-08f, 2.752115961e-06f);
  p = __builtin_fmaf(z, p, -1.984078554e-04f);
  p = __builtin_fmaf(z, p, 8.333330043e-03f);
  p = __builtin_fmaf(z, p, -1.666666716e-01f);
  const float s = __builtin_fmaf(r * z, p, r);
  return __builtin_fmaf(s * s, ib, v);
}

__device__ __forceinline__ float snake_any(float v, float y, float ib) {
  const float s = sinf(y);
  return __builtin_fmaf(s * s, ib, v);
}

// Snake of N values in place (any magnitude): the library sine only where some |y| is past the
// fast form's range.  A NaN goes through either form as a NaN.
template <int N>
__device__ __forceinline__ void snake_n(float *v, const float *ea, const float *ib) {
  float big = 0.f;
  float x[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float y = v[i] * ea[i];
    big = fmaxf(big, fabsf(y));
    x[i] = snake_fast(v[i], y, ib[i]);
  }
  if (__builtin_expect(!(big < kSnakeFast), 0)) {
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = snake_any(v[i], v[i] * ea[i], ib[i]);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = x[i];
}

}  // namespace q3t
