// Matrix-core GEMM for many rows (prompt prefill, text projection, codec linears and table builds):
// Y[M][N] = f(X[M][K] . W[N][K]^T), bf16 weights in packed order (GemmArgs::w_packed), fp32
// activations as three exact bf16 terms, fp32 accumulation; optional RMSNorm of the rows.
//
// The order of the additions is part of what a GEMM returns (launch_gemm), whichever kernel computes it:
// tokens are argmaxes or draws over logits, a stream of a few hundred frames comes across logits that
// are equal to a bit or two, and a sum in another order then turns its codes from there on.
#include "q3t_kernels.h"

#include <algorithm>
#include <type_traits>

#include "q3t_bf16x3.h"

namespace q3t {
namespace {

// The epilogues for four consecutive columns of a row: v the sums, r / b / c / c2 the operands
// (residual, bias, scale or Snake tables).
template <int EPI>
__device__ __forceinline__ void tile_epilogue(const GemmArgs &a, float *v, const float *r, const float *b, const float *c,
                                              const float *c2) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if constexpr (EPI == EPI_RESIDUAL) v[e] = r[e] + v[e];
    if constexpr (EPI == EPI_BIAS) v[e] = v[e] + b[e];
    if constexpr (EPI == EPI_AFFINE_RES) {
      if (a.bias) v[e] = v[e] + b[e];
      if (a.scale) v[e] = v[e] * c[e];
      v[e] = r[e] + v[e];
    }
    if constexpr (EPI == EPI_BIAS_GELU) {
      v[e] = v[e] + b[e];
      v[e] = 0.5f * v[e] * (1.0f + erff(v[e] * 0.7071067811865476f));
    }
    if constexpr (EPI == EPI_BIAS_SILU) {
      v[e] = v[e] + b[e];
      v[e] = v[e] / (1.0f + expf(-v[e]));
    }
    if constexpr (EPI == EPI_RES_SNAKE) v[e] = r[e] + (v[e] + b[e]);
  }
  if constexpr (EPI == EPI_RES_SNAKE) snake_n<4>(v, c, c2);
}

// 1 / rms of rows r0 .. r0 + rows - 1 (past the last row: of the last), into inv[rows], by all waves:
// lane sums of every 64th square, then wave_sum.  RB rows a wave and 512 columns a round: two round
// trips to the L2 for rows of 1,024.  A launch of its own per norm costs what the round trips do
// and the gap before it.
template <int RB>
__device__ __forceinline__ void rows_inv_rms(const GemmArgs &a, int r0, int rows, int wave, int waves, int lane,
                                             float *inv) {
  constexpr int U = 8;
  for (int r = wave; r < rows; r += RB * waves) {
    const float *x[RB];
    float ss[RB] = {};
#pragma unroll
    for (int i = 0; i < RB; ++i) x[i] = a.X + (size_t)min(r0 + min(r + i * waves, rows - 1), a.M - 1) * a.ldx;
    int k0 = 0;
    for (; k0 + 64 * U <= a.K; k0 += 64 * U) {
      float v[RB][U];
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int e = 0; e < U; ++e) v[i][e] = (x[i] + k0)[lane + 64 * e];
      __builtin_amdgcn_sched_barrier(0);  // every load before the first sum
#pragma unroll
      for (int e = 0; e < U; ++e)
#pragma unroll
        for (int i = 0; i < RB; ++i) ss[i] = __builtin_fmaf(v[i][e], v[i][e], ss[i]);
    }
    for (int k = k0 + lane; k < a.K; k += 64)
#pragma unroll
      for (int i = 0; i < RB; ++i) ss[i] = __builtin_fmaf(x[i][k], x[i][k], ss[i]);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const float w = wave_sum(ss[i]);
      s = lane == i ? w : s;
    }
    if (lane < RB && r + lane * waves < rows) inv[r + lane * waves] = 1.0f / sqrtf(s / (float)a.K + a.eps);
  }
}

// Block tile 32 rows x 64 CT packed weight rows (SwiGLU: 64 gate rows and the matching up rows), four
// waves side by side, per K group.  What bounds it: per CU, loading X and the weights (64 bytes a
// clock) and splitting X (~9 vector operations an element) take as long as the matrix cores do with
// what is loaded (three MFMAs a product), so all three have to run at once, and a block's own chain
// of k steps must never wait.  Hence:
//   * Everything is loaded well ahead of use: the weights, straight from global memory in
//     matrix-core order (1 KiB contiguous per 16 columns and step, read by one wave only), in a ring
//     of four k steps; X two 64-wide chunks ahead in registers.  Addresses are uniform and the loads
//     are outside of every branch.
//   * X is split into its three terms once per block, into LDS planes of [step][row][4 slots of
//     16 bytes], slots xor-ed with (row / 2) % 4 (any 8 rows of a slot in distinct bank columns),
//     double buffered: one barrier per 64 k.
//   * 32 rows rather than 64: four waves a SIMD from different blocks, so that one
//     block's splitting runs under another's matrix-core work, and finer shares of the CUs.
//   * The weight tile is the A operand: a lane ends with four consecutive columns of one row, so
//     loads and stores of the epilogue are 16 bytes wide.
//   * PARTS (GemmArgs::k_parts above one): each part's sum is a chain of its own; the parts' sums are
//     added in part order.  KG = 2: two such groups of waves in a block take the parts' first and
//     second half; the second's sums wait in LDS, one image a part.
//   * TAIL: a group's k steps are not whole pairs of chunks; what is missing is staged as zeros and
//     not multiplied.
template <int EPI, bool NORM, int KG, int CT, bool TAIL, bool PARTS>
__global__ __launch_bounds__(256 * KG, 2) void k_gemm_tile(GemmArgs a, int vec) {
  constexpr bool SW = EPI == EPI_SWIGLU;
  static_assert(KG == 1 || PARTS, "the groups take whole parts");
  static_assert(!SW || CT == 2, "a gate tile and its up tile");
  constexpr int BM = 32, BW = 64 * CT;
  constexpr int RT = 2, OT = SW ? 1 : CT;             // row and output tiles per wave, CT weight tiles
  constexpr int PLANE = 2 * BM * 4, BUF = 3 * PLANE;  // 16-byte units of a term, of a staging buffer
  extern __shared__ bf16x8_t lds[];                   // [KG][2][BUF], row scales [BM], KG = 2: images
  const int tid = threadIdx.x & 255, lane = tid & 63, li = lane & 15, kb = lane >> 4;
  const int gwave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform for the compiler too
  const int grp = KG > 1 ? gwave >> 2 : 0, wave = gwave & 3;
  bf16x8_t *xs = lds + grp * 2 * BUF;
  float *rinv = reinterpret_cast<float *>(lds + KG * 2 * BUF);
  f32x4_t *image = reinterpret_cast<f32x4_t *>(rinv + BM) + tid;  // [part - half][RT * CT][256]

  int mb, nb;
  block_tile((a.N + (SW ? BW / 2 : BW) - 1) / (SW ? BW / 2 : BW), mb, nb);
  const int m0 = mb * BM;
  const int n0 = nb * (SW ? BW / 2 : BW) + wave * OT * 16;  // this wave's first output column
  // k steps [s0, s1) of 32 for this group, parts [part, ..), worked on in pairs of 64-wide chunks (four
  // steps)
  const int steps = a.K / 32, parts = PARTS ? a.k_parts : 1, half = (parts + 1) / 2, mid = steps * half / parts;
  const int s0 = KG > 1 && grp ? mid : 0, s1 = KG > 1 && !grp ? mid : steps;
  int part = KG > 1 && grp ? half : 0, bound = steps * (part + 1) / parts;
  // of the longer group: every wave meets every barrier
  const int pairs = ((KG > 1 ? max(mid, steps - mid) : steps) + 3) / 4;

  // X: this thread stages row (tid % 128) / 4, k = 8 (tid % 4) .. + 7 of step tid / 128 of a chunk.
  // Addresses are a uniform base (step) plus a 32-bit offset in the block.
  const int srow = (tid & 127) >> 2, slot = tid & 3, sp = tid >> 7;
  const float *xb = a.X + (size_t)m0 * a.ldx;
  const uint32_t xo = (uint32_t)min(srow, a.M - 1 - m0) * (uint32_t)a.ldx + 8 * slot, go = 8 * slot;
  f32x4_t xr[2][2], gr[NORM ? 2 : 1][2];  // [set][half]
  auto xload = [&](int st0, auto set) {
    constexpr int SET = decltype(set)::value;
    const int st = min(st0, s1 - 1);
    const uint32_t up = st0 + 1 < s1 ? 32u * (uint32_t)sp : 0u;  // the second step, if there is one
    const float *xs0 = xb + 32 * st, *gs0 = NORM ? a.gamma + 32 * st : nullptr;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      xr[SET][h] = *reinterpret_cast<const f32x4_t *>(xs0 + (xo + up + 4 * h));
      if constexpr (NORM) gr[SET][h] = *reinterpret_cast<const f32x4_t *>(gs0 + (go + up + 4 * h));
    }
  };
  float rs = 1.f;
  auto xstore = [&](int st0, auto set) {  // to the buffer of the same number
    constexpr int SET = decltype(set)::value;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = xr[SET][e >> 2][e & 3];
    if constexpr (TAIL) {
      const bool in = st0 + sp < s1;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = in ? v[e] : 0.f;
    }
    if constexpr (NORM) {
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (v[e] * rs) * gr[SET][e >> 2][e & 3];
    }
    bf16x8_t hi, mid, lo;
    split_bf16x8_rn(v, hi, mid, lo);
    bf16x8_t *dst = xs + SET * BUF + (sp * BM + srow) * 4 + (slot ^ ((srow >> 1) & 3));
    dst[0] = lo;
    dst[PLANE] = mid;
    dst[2 * PLANE] = hi;
  };

  // Weight tiles of this wave (a partial last block repeats the last tile; nothing of it is stored)
  const int ntile = (a.N + 15) / 16;
  const uint16_t *wp[CT];
#pragma unroll
  for (int u = 0; u < CT; ++u) {
    const int t = min(n0 / 16 + (SW ? u % OT : u), ntile - 1) + (SW && u >= OT ? ntile : 0);
    wp[u] = a.W + (size_t)t * steps * 512;
  }
  bf16x8_t w[4][CT];  // ring over k steps
  auto wload = [&](int st, auto at) {
#pragma unroll
    for (int u = 0; u < CT; ++u)
      w[decltype(at)::value][u] = *reinterpret_cast<const bf16x8_t *>(wp[u] + (size_t)min(st, s1 - 1) * 512 + lane * 8u);
  };

  f32x4_t acc[RT][CT], tot[PARTS ? RT : 1][PARTS ? CT : 1];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int u = 0; u < CT; ++u) {
      acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if constexpr (PARTS) tot[t][u] = f32x4_t{-0.f, -0.f, -0.f, -0.f};  // -0 + v = v, -0 too
    }

  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};
  constexpr std::integral_constant<int, 2> I2{};
  constexpr std::integral_constant<int, 3> I3{};
  const bf16x8_t *fsrc = xs + li * 4 + (kb ^ ((li >> 1) & 3));
  // step st = step p of the chunk in buffer SET, weights in ring slot 2 SET + p
  auto mma = [&](auto set, auto step, int st) {
    constexpr int SET = decltype(set)::value, PS = decltype(step)::value;
    if (TAIL && st >= s1) return;
#pragma unroll
    for (int q = 0; q < 3; ++q) {  // lo, mid, hi
      bf16x8_t x[RT];
#pragma unroll
      for (int t = 0; t < RT; ++t) x[t] = fsrc[SET * BUF + q * PLANE + PS * BM * 4 + 64 * t];
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int u = 0; u < CT; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[2 * SET + PS][u], x[t], acc[t][u], 0, 0, 0);
    }
    if constexpr (PARTS) {
      if (st + 1 == bound) {  // the part's sum is whole
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
          for (int u = 0; u < CT; ++u) {
            if (KG > 1 && grp) image[((part - half) * RT * CT + t * CT + u) * 256] = acc[t][u];
            else tot[t][u] += acc[t][u];
            acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
          }
        ++part;
        bound = steps * (part + 1) / parts;
      }
    }
  };

  wload(s0, I0);
  wload(s0 + 1, I1);
  wload(s0 + 2, I2);
  wload(s0 + 3, I3);
  if constexpr (NORM) {
    __builtin_amdgcn_sched_barrier(0);
    rows_inv_rms<BM / (4 * KG)>(a, m0, BM, gwave, 4 * KG, lane, rinv);
    __syncthreads();
    rs = rinv[srow];
  }
  xload(s0, I0);
  xload(s0 + 2, I1);
  xstore(s0, I0);
  __syncthreads();
  // Entering a pair: chunk st in buffer 0, chunk st + 2 in register set 1, weights of st .. st + 3.
  for (int i = 0, st = s0; i < pairs; ++i, st += 4) {
    xload(st + 4, I0);
    __builtin_amdgcn_sched_barrier(0);
    mma(I0, I0, st);
    wload(st + 4, I0);
    mma(I0, I1, st + 1);
    wload(st + 5, I1);
    __builtin_amdgcn_sched_barrier(0);
    xstore(st + 2, I1);
    __syncthreads();
    xload(st + 6, I1);
    __builtin_amdgcn_sched_barrier(0);
    mma(I1, I0, st + 2);
    wload(st + 6, I2);
    mma(I1, I1, st + 3);
    wload(st + 7, I3);
    __builtin_amdgcn_sched_barrier(0);
    xstore(st + 4, I0);
    __syncthreads();
  }

  if constexpr (KG > 1) {  // every image was written before the loop's last barrier
    if (grp) return;
    for (int p = half; p < parts; ++p)
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int u = 0; u < CT; ++u) tot[t][u] += image[((p - half) * RT * CT + t * CT + u) * 256];
  }

  // Lane (li, kb) holds columns 4 kb .. + 3 of row li of each tile.  Every operand is loaded before
  // the first store (Y may be the residual: each element is read and written by one lane only).
  constexpr bool RES = EPI == EPI_RESIDUAL || EPI == EPI_AFFINE_RES || EPI == EPI_RES_SNAKE;
  constexpr bool BIAS = EPI == EPI_BIAS || EPI == EPI_AFFINE_RES || EPI == EPI_BIAS_GELU ||
                        EPI == EPI_BIAS_SILU || EPI == EPI_RES_SNAKE;
  auto quad = [&](const float *p, int n, bool on) -> f32x4_t {  // columns n .. n + 3 of a row at p
    f32x4_t r{0.f, 0.f, 0.f, 0.f};
    if (!on) return r;
    if (vec) return n < a.N ? *reinterpret_cast<const f32x4_t *>(p + n) : r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = n + e < a.N ? p[n + e] : 0.f;
    return r;
  };
  f32x4_t rv[RES ? RT : 1][RES ? OT : 1], bv[OT], cv[OT], c2v[OT];
#pragma unroll
  for (int u = 0; u < OT; ++u) {
    const int n = n0 + 16 * u + 4 * kb;
    if constexpr (BIAS) bv[u] = quad(a.bias, n, EPI != EPI_AFFINE_RES || a.bias);
    if constexpr (EPI == EPI_AFFINE_RES) cv[u] = quad(a.scale, n, a.scale);
    if constexpr (EPI == EPI_RES_SNAKE) {
      cv[u] = quad(a.snake_a, n, true);
      c2v[u] = quad(a.snake_b, n, true);
    }
    if constexpr (RES) {
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const int m = min(m0 + 16 * t + li, a.M - 1);
        rv[t][u] = quad(a.res + (size_t)m * a.ldr, n, true);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int m = m0 + 16 * t + li;
#pragma unroll
    for (int u = 0; u < OT; ++u) {
      const int n = n0 + 16 * u + 4 * kb;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if constexpr (PARTS) v[e] = tot[t][u][e];
        else v[e] = acc[t][u][e];
        if constexpr (SW) {
          float up;
          if constexpr (PARTS) up = tot[t][u + OT][e];
          else up = acc[t][u + OT][e];
          v[e] = v[e] / (1.0f + expf(-v[e])) * up;
        }
      }
      float r[4], b[4], c[4], c2[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        r[e] = RES ? rv[RES ? t : 0][RES ? u : 0][e] : 0.f;
        b[e] = BIAS ? bv[u][e] : 0.f;
        c[e] = EPI == EPI_AFFINE_RES || EPI == EPI_RES_SNAKE ? cv[u][e] : 1.f;
        c2[e] = EPI == EPI_RES_SNAKE ? c2v[u][e] : 1.f;
      }
      tile_epilogue<EPI>(a, v, r, b, c, c2);
      if (m >= a.M || n >= a.N) continue;
      float *y = a.Y + (size_t)m * a.ldy + n;
      if (vec) {
        *reinterpret_cast<f32x4_t *>(y) = f32x4_t{v[0], v[1], v[2], v[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < a.N) y[e] = v[e];
      }
    }
  }
}

// Few rows: a workgroup per 16-column tile (SwiGLU: a gate tile and its up tile) and MT tiles of 16 rows.
// A wave's job is one K part (GemmArgs::k_parts): it issues the loads of PS k steps together, weights and X
// straight from global memory in matrix-core order, and leaves its sums in LDS, where the
// parts are added in part order.  With so few rows a launch lasts as long as one workgroup: one memory
// round trip or two, plus what its CU can load (64 bytes a clock, rows x K x 4 of X above all) and split.
// So the columns are spread as thin as the matrix cores take them, over every CU, nothing is waited
// for between a wave's loads, and no second launch adds up the parts.
constexpr int rows_waves(int MT) { return MT == 1 ? 16 : 8; }  // at most: registers for the loads in flight

template <int EPI, bool NORM, int MT>
__global__ __launch_bounds__(64 * rows_waves(MT)) void k_gemm_rows(GemmArgs a, int vec) {
  constexpr bool SW = EPI == EPI_SWIGLU;
  constexpr int T = SW ? 2 : 1, PS = MT > 1 ? 6 : SW ? 3 : NORM ? 4 : 6;
  constexpr bool RES = EPI == EPI_RESIDUAL || EPI == EPI_AFFINE_RES || EPI == EPI_RES_SNAKE;
  constexpr bool BIAS = EPI == EPI_BIAS || EPI == EPI_AFFINE_RES || EPI == EPI_BIAS_GELU ||
                        EPI == EPI_BIAS_SILU || EPI == EPI_RES_SNAKE;
  extern __shared__ f32x4_t part[];  // [k_parts][MT * T][64], then row scales [16 MT]
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, kb = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = blockDim.x >> 6;
  const int ntile = (a.N + 15) / 16, steps = a.K / 32, parts = a.k_parts;
  const int r0 = 16 * MT * blockIdx.y;  // first row
  float *rinv = reinterpret_cast<float *>(part + parts * MT * T * 64);

  // This thread's four outputs (threads below 64 MT): row om, columns on .. on + 3; operands first
  const int ot = min(tid >> 6, MT - 1), om = r0 + 16 * ot + li, on = blockIdx.x * 16 + 4 * kb, cm = min(om, a.M - 1);
  auto quad = [&](const float *p, bool have) -> f32x4_t {
    f32x4_t r{0.f, 0.f, 0.f, 0.f};
    if (!have) return r;
    if (vec) return on < a.N ? *reinterpret_cast<const f32x4_t *>(p + on) : r;
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = on + e < a.N ? p[on + e] : 0.f;
    return r;
  };
  f32x4_t rv{}, bv{}, cv{}, c2v{};
  if (tid < 64 * MT) {
    if constexpr (RES) rv = quad(a.res + (size_t)cm * a.ldr, true);
    if constexpr (BIAS) bv = quad(a.bias, EPI != EPI_AFFINE_RES || a.bias);
    if constexpr (EPI == EPI_AFFINE_RES) cv = quad(a.scale, a.scale);
    if constexpr (EPI == EPI_RES_SNAKE) {
      cv = quad(a.snake_a, true);
      c2v = quad(a.snake_b, true);
    }
  }

  const uint16_t *wp[T];
#pragma unroll
  for (int u = 0; u < T; ++u) wp[u] = a.W + (size_t)(blockIdx.x + u * ntile) * steps * 512 + lane * 8;
  bf16x8_t w[PS][T];
  auto wload = [&](int p0, int s1) {
#pragma unroll
    for (int i = 0; i < PS; ++i)
#pragma unroll
      for (int u = 0; u < T; ++u)
        w[i][u] = *reinterpret_cast<const bf16x8_t *>(wp[u] + (size_t)min(p0 + i, s1 - 1) * 512);
  };
  const float *xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = a.X + (size_t)min(r0 + 16 * t + li, a.M - 1) * a.ldx + 8 * kb;
  f32x4_t x[PS][MT][2];
  auto xload = [&](int p0, int s1) {
#pragma unroll
    for (int i = 0; i < PS; ++i)
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          x[i][t][h] = *reinterpret_cast<const f32x4_t *>(xp[t] + 32 * min(p0 + i, s1 - 1) + 4 * h);
  };
  // A wave's parts, PS steps at a time.  The first loads are under way before the norm's: together the waves'
  // cover X or most of it, and the norm finds it in the L2.  A wave past the last part loads as the last
  // does, and works on none.
  int z = min(wave, parts - 1), p0 = steps * z / parts, s1 = steps * (z + 1) / parts;
  wload(p0, s1);
  xload(p0, s1);
  float rs[MT];
  if constexpr (NORM) {
    __builtin_amdgcn_sched_barrier(0);
    rows_inv_rms<16 * MT / rows_waves(MT)>(a, r0, 16 * MT, wave, waves, lane, rinv);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < MT; ++t) rs[t] = rinv[16 * t + li];
  }
  f32x4_t acc[MT][T];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < T; ++u) acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  z = wave;
  while (z < parts) {
    f32x4_t g[NORM ? PS : 1][2];
    if constexpr (NORM) {
#pragma unroll
      for (int i = 0; i < PS; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h)
          g[i][h] = *reinterpret_cast<const f32x4_t *>(a.gamma + 32 * min(p0 + i, s1 - 1) + 8 * kb + 4 * h);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < PS; ++i) {
      if (p0 + i >= s1) break;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[e] = x[i][t][e >> 2][e & 3];
          if constexpr (NORM) v[e] = (v[e] * rs[t]) * g[i][e >> 2][e & 3];
        }
        bf16x8_t hi, mid, lo;
        split_bf16x8_rn(v, hi, mid, lo);
#pragma unroll
        for (int u = 0; u < T; ++u) {
          acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][u], lo, acc[t][u], 0, 0, 0);
          acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][u], mid, acc[t][u], 0, 0, 0);
          acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][u], hi, acc[t][u], 0, 0, 0);
        }
      }
    }
    p0 += PS;
    if (p0 >= s1) {
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int u = 0; u < T; ++u) {
          part[((z * MT + t) * T + u) * 64 + lane] = acc[t][u];
          acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        }
      z += waves;
      if (z >= parts) break;
      p0 = steps * z / parts;
      s1 = steps * (z + 1) / parts;
    }
    wload(p0, s1);
    xload(p0, s1);
  }
  __syncthreads();
  if (tid >= 64 * MT) return;
  float v[4], up[4];
  {
    f32x4_t s[T];
#pragma unroll
    for (int u = 0; u < T; ++u) s[u] = part[(ot * T + u) * 64 + lane];
    for (int z = 1; z < parts; ++z)
#pragma unroll
      for (int u = 0; u < T; ++u) s[u] += part[((z * MT + ot) * T + u) * 64 + lane];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = s[0][e];
      up[e] = s[T - 1][e];
    }
  }
  if (om >= a.M || on >= a.N) return;
  float *y = a.Y + (size_t)om * a.ldy + on;
  if constexpr (SW) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = v[e] / (1.0f + expf(-v[e])) * up[e];
  } else {
    float r[4], b[4], c[4], c2[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      r[e] = rv[e];
      b[e] = bv[e];
      c[e] = cv[e];
      c2[e] = c2v[e];
    }
    tile_epilogue<EPI>(a, v, r, b, c, c2);
  }
  if (vec) {
    *reinterpret_cast<f32x4_t *>(y) = f32x4_t{v[0], v[1], v[2], v[3]};
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (on + e < a.N) y[e] = v[e];
  }
}

// 16-byte accesses of the epilogue's operands.
int gemm_vec(const GemmArgs &a) {
  auto aligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  return a.N % 4 == 0 && a.ldy % 4 == 0 && (!a.res || a.ldr % 4 == 0) && aligned(a.Y) && aligned(a.res) &&
         aligned(a.bias) && aligned(a.scale) && aligned(a.snake_a) && aligned(a.snake_b);
}

template <int EPI, bool NORM, int MT>
hipError_t rows_launch(const GemmArgs &a, hipStream_t s) {
  constexpr int T = EPI == EPI_SWIGLU ? 2 : 1;
  const dim3 grid((a.N + 15) / 16, (a.M + 16 * MT - 1) / (16 * MT));
  // all waves for the norm; else as many as give them the same number of parts, one for each tile of outputs
  const int rounds = (a.k_parts + rows_waves(MT) - 1) / rows_waves(MT);
  const int waves = NORM ? rows_waves(MT) : std::max((a.k_parts + rounds - 1) / rounds, MT);
  const size_t lds = (size_t)a.k_parts * MT * T * 1024 + (NORM ? 16 * MT * 4 : 0);
  hipLaunchKernelGGL((k_gemm_rows<EPI, NORM, MT>), grid, dim3(64 * waves), lds, s, a, gemm_vec(a));
  return hipGetLastError();
}

template <int EPI, bool NORM, int KG, int CT, bool TAIL, bool PARTS>
hipError_t tile_launch(const GemmArgs &a, hipStream_t s) {
  const int out = EPI == EPI_SWIGLU ? 64 : 64 * CT;
  const dim3 grid((unsigned)((a.N + out - 1) / out * (int64_t)((a.M + 31) / 32)));
  const size_t lds = (size_t)KG * 2 * 3 * 2 * 32 * 64 + 32 * 4 + (KG > 1 ? (size_t)(a.k_parts / 2) * CT * 8192 : 0);
  hipLaunchKernelGGL((k_gemm_tile<EPI, NORM, KG, CT, TAIL, PARTS>), grid, dim3(256 * KG), lds, s, a, gemm_vec(a));
  return hipGetLastError();
}

// One K part: no groups.  Parts: two groups a block where there are fewer blocks than CUs, of 64 columns
// where those find a CU each (O and down of the 1.7B shape at 137 rows, 80 blocks of 128 columns: 30 -> 25 us;
// O and down of the 0.6B shape at 521 rows, 136 blocks: 23 -> 25, QKV at 137 rows, 160 blocks: 22 -> 27).  16 parts of 128
// columns leave no LDS for the second group's sums.
template <int EPI, bool NORM>
hipError_t tile_parts(const GemmArgs &a, hipStream_t s) {
  if (a.k_parts == 1)
    return a.K % 128 == 0 ? tile_launch<EPI, NORM, 1, 2, false, false>(a, s)
                          : tile_launch<EPI, NORM, 1, 2, true, false>(a, s);
  constexpr int out = EPI == EPI_SWIGLU ? 64 : 128;
  const int64_t blocks = (int64_t)((a.N + out - 1) / out) * ((a.M + 31) / 32);
  if constexpr (EPI != EPI_SWIGLU)
    if (2 * blocks <= 256) return tile_launch<EPI, NORM, 2, 1, true, true>(a, s);
  if (blocks < 256 && a.k_parts <= 12) return tile_launch<EPI, NORM, 2, 2, true, true>(a, s);
  return tile_launch<EPI, NORM, 1, 2, true, true>(a, s);
}

// One row tile, or few 16 x 16 output tiles (two a CU) and five or more K parts for the waves to share:
// k_gemm_rows, the rows in workgroups of one tile up to a workgroup a CU, of two past that.  Else k_gemm_tile.
// Prefill in us with k_gemm_rows to twice the tiles and at any number of parts, and so: 41 rows 1,783 and
// 1,710, 80 rows 2,730 and 2,165, 200 rows 3,160 and 2,740 (0.6B shape), 24 rows 2,820 and 2,330, 41 rows
// 4,230 and 2,980 (1.7B shape); with it only from 16 parts on, 24 rows 1,705 and 1,642 (0.6B).
template <int EPI, bool NORM>
hipError_t tile_shape(const GemmArgs &a, hipStream_t s) {
  const int cols = (a.N + 15) / 16;
  const int64_t tiles = ((int64_t)a.M + 15) / 16;
  if (tiles > 1 && (a.k_parts < 5 || tiles * cols > 512)) return tile_parts<EPI, NORM>(a, s);
  return tiles == 1 || tiles * cols <= 256 ? rows_launch<EPI, NORM, 1>(a, s) : rows_launch<EPI, NORM, 2>(a, s);
}

template <int EPI>
hipError_t tile_norm(const GemmArgs &a, hipStream_t s) {
  return a.gamma ? tile_shape<EPI, true>(a, s) : tile_shape<EPI, false>(a, s);
}

}  // namespace

int gemm_k_parts(int epi, int M, int N, int K) {
  const bool sw = epi == EPI_SWIGLU;
  auto blocks_of = [&](int cols, int rows) { return (int64_t)((N + cols - 1) / cols) * ((M + rows - 1) / rows); };
  int64_t blocks;
  if (M >= 128 && (!sw || N % 64 == 0)) blocks = blocks_of(sw ? 64 : (N % 128 && N % 96 == 0 ? 96 : 128), 128);
  else blocks = blocks_of(sw ? 128 : 256, M <= 16 ? 16 : 32);
  if (blocks >= 128) return 1;
  int p = std::min({(int)((256 + blocks - 1) / blocks), K / 128, kGemmMaxParts});
  while (p > 1 && (int64_t)p * M * N * (sw ? 2 : 1) > (int64_t)4 << 20) --p;
  return std::max(p, 1);
}

hipError_t launch_gemm(int epi, const GemmArgs &args, hipStream_t s) {
  GemmArgs a = args;
  if (a.k_parts == 0) a.k_parts = 1;
  if (a.M <= 0 || a.N <= 0 || a.K <= 0 || a.K % 32 || a.ldx % 4 || !a.w_packed || !a.X || !a.W || !a.Y || a.split2 ||
      a.k_parts < 1 || a.k_parts > std::min(a.K / 32, kGemmMaxParts) || reinterpret_cast<uintptr_t>(a.X) % 16 ||
      reinterpret_cast<uintptr_t>(a.W) % 16 || reinterpret_cast<uintptr_t>(a.gamma) % 16)
    return hipErrorInvalidValue;
  const bool res = epi == EPI_RESIDUAL || epi == EPI_AFFINE_RES || epi == EPI_RES_SNAKE;
  const bool bias = epi == EPI_BIAS || epi == EPI_BIAS_GELU || epi == EPI_BIAS_SILU || epi == EPI_RES_SNAKE;
  if ((res && !a.res) || (bias && !a.bias)) return hipErrorInvalidValue;
  switch (epi) {
    case EPI_STORE: return tile_norm<EPI_STORE>(a, s);
    case EPI_RESIDUAL: return tile_norm<EPI_RESIDUAL>(a, s);
    case EPI_SWIGLU: return tile_norm<EPI_SWIGLU>(a, s);
    case EPI_BIAS: return tile_norm<EPI_BIAS>(a, s);
    case EPI_AFFINE_RES: return a.gamma ? hipErrorInvalidValue : tile_shape<EPI_AFFINE_RES, false>(a, s);
    case EPI_BIAS_GELU: return a.gamma ? hipErrorInvalidValue : tile_shape<EPI_BIAS_GELU, false>(a, s);
    case EPI_BIAS_SILU: return a.gamma ? hipErrorInvalidValue : tile_shape<EPI_BIAS_SILU, false>(a, s);
    case EPI_RES_SNAKE:
      return a.gamma || !a.snake_a || !a.snake_b ? hipErrorInvalidValue : tile_shape<EPI_RES_SNAKE, false>(a, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace q3t
