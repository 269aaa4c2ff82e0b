// Matrix-core GEMM for many rows (prompt prefill, text projection, codec linears and table builds):
// Y[M][N] = f(X[M][K] . W[N][K]^T), bf16 weights in packed order (GemmArgs::w_packed), fp32
// activations as three exact bf16 terms, fp32 accumulation; optional RMSNorm of the rows.
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

// GemmArgs::split2.  Two adds onto zero commute: the result does not depend on which half lands first.
// The first half brings the residual and zeroes it for the GEMM that next accumulates into that buffer.
// Four sums v of columns n .. n + 3 of row m go to t, this wave's LDS image of its ROWS x COLS outputs;
// split_add then adds that image row by row, COLS consecutive columns at a time: an add is worked on
// outside of the XCD, by whole lines.
__device__ __forceinline__ void split_put(const GemmArgs &a, const float *v, const float *r, float *t, int m, int n,
                                          int half, int vec) {
  f32x4_t o{v[0], v[1], v[2], v[3]};
  if (half == 0) {
    o = f32x4_t{r[0] + v[0], r[1] + v[1], r[2] + v[2], r[3] + v[3]};
    if (m < a.M) {
      float *z = a.res_zero + (size_t)m * a.ldr + n;
      if (vec) {
        if (n < a.N) *reinterpret_cast<f32x4_t *>(z) = f32x4_t{0.f, 0.f, 0.f, 0.f};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < a.N) z[e] = 0.f;
      }
    }
  }
  *reinterpret_cast<f32x4_t *>(t) = o;
}

template <int ROWS, int COLS, int LD>
__device__ __forceinline__ void split_add(const GemmArgs &a, const float *t, int m0, int n0, int lane) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  const int r = lane / COLS, c = lane % COLS;
#pragma unroll
  for (int i = 0; i < ROWS; i += 64 / COLS)
    if (m0 + i + r < a.M && n0 + c < a.N)
      unsafeAtomicAdd(a.Y + (size_t)(m0 + i + r) * a.ldy + n0 + c, t[(i + r) * LD + c]);
}

// Block tile 32 rows x 128 packed weight rows (SwiGLU: 64 gate rows and the matching up rows), four
// waves side by side, per K group.  What bounds it: per CU, loading X and the weights (64 bytes a
// clock) and splitting X (7 vector operations an element) take as long as the matrix cores do with
// what is loaded (three MFMAs a product), so all three have to run at once, and a block's own chain
// of k steps must never wait.  Hence:
//   * Everything is loaded well ahead of use: the weights, straight from global memory in
//     matrix-core order (1 KiB contiguous per 16 columns and step, read by one wave only), in a ring
//     of four k steps; X two 64-wide chunks ahead in registers.  The loop is straight-line code with
//     uniform addresses: a branch in it made the compiler copy the rings and wait for them.
//   * X is split into its three terms once per block, into LDS planes of [step][row][4 slots of
//     16 bytes], slots xor-ed with (row / 2) % 4 (any 8 rows of a slot in distinct bank columns),
//     double buffered: one barrier per 64 k.
//   * 32 rows rather than 64: 106-127 registers, four waves a SIMD from different blocks, so that one
//     block's splitting runs under another's matrix-core work, and finer shares of the CUs.  521 rows,
//     1024 -> 4096: 32 us (64 x 128 blocks) -> 25 us; 137 rows, 2048 -> 2 x 6144: 58 -> 35 us.
//   * KG = 2: where blocks are few, two such groups of waves in a block take half of K each and add
//     up through LDS.
//   * RMSNorm needs no launch of its own: every block passes over its rows whole, so the staging
//     threads sum the squares, the matrix cores take x * gain, and the epilogue scales the sums
//     by 1 / rms (one scalar per row).
//   * The weight tile is the A operand: a lane ends with four consecutive columns of one row, so
//     loads and stores of the epilogue are 16 bytes wide.
//   * TAIL: K is not a whole number of pairs of chunks per group; what is missing is staged as zeros.
template <int EPI, bool NORM, int KG, bool TAIL, bool SPLIT>
__global__ __launch_bounds__(256 * KG, 2) void k_gemm_tile(GemmArgs a, int vec) {
  static_assert(!SPLIT || EPI == EPI_RESIDUAL, "the K halves meet in a residual sum");
  constexpr bool SW = EPI == EPI_SWIGLU;
  constexpr int BM = 32, BW = 128;
  constexpr int RT = 2, CT = 2, OT = SW ? 1 : 2;      // row, weight and output tiles per wave
  constexpr int PLANE = 2 * BM * 4, BUF = 3 * PLANE;  // 16-byte units of a term, of a staging buffer
  extern __shared__ bf16x8_t lds[];                   // [KG][2][BUF], then row sums [KG][64]
  const int tid = threadIdx.x & 255, lane = tid & 63, li = lane & 15, kb = lane >> 4;
  const int gwave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform for the compiler too
  const int grp = KG > 1 ? gwave >> 2 : 0, wave = gwave & 3;
  bf16x8_t *xs = lds + grp * 2 * BUF;
  float *rsum = reinterpret_cast<float *>(lds + KG * 2 * BUF);

  // Few column blocks: each XCD (workgroup id % 8) takes a contiguous range of row-major block
  // tiles, so that its L2 reads only its own X rows, once for all column blocks.
  int mb = blockIdx.y, nb = blockIdx.x;
  if (gridDim.x <= 8) {
    const int total = gridDim.x * gridDim.y, L = blockIdx.y * gridDim.x + blockIdx.x;
    const int xcd = L % 8, local = L / 8, C = (total + 7) / 8, r = total % 8;
    const int t = (r == 0 || xcd < r) ? xcd * C + local : r * C + (xcd - r) * (C - 1) + local;
    mb = t / gridDim.x;
    nb = t % gridDim.x;
  }
  const int m0 = mb * BM;
  const int n0 = nb * (SW ? BW / 2 : BW) + wave * OT * 16;  // this wave's first output column
  // k steps [s0, s1) of 32 for this group (SPLIT: of the workgroup's half), worked on in pairs of
  // 64-wide chunks (four steps); what a pair holds past s1 is staged as zeros
  const int steps = a.K / 32, h0 = SPLIT ? steps * (int)blockIdx.z / 2 : 0;
  const int hn = (SPLIT ? steps * ((int)blockIdx.z + 1) / 2 : steps) - h0;
  const int s0 = h0 + hn * grp / KG, s1 = h0 + hn * (grp + 1) / KG;
  const int pairs = ((hn + KG - 1) / KG + 3) / 4;  // of the longest group: every wave meets every barrier

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
  float ss = 0.f;
  auto xstore = [&](int st0, auto set, bool live) {  // to the buffer of the same number
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
      float q = ss;
#pragma unroll
      for (int e = 0; e < 8; ++e) q = __builtin_fmaf(v[e], v[e], q);
      ss = live ? q : ss;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= gr[SET][e >> 2][e & 3];
    }
    bf16x8_t hi, mid, lo;
    split_bf16x8_nc(v, hi, mid, lo);
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

  // Sums over a pair (12 matrix-core additions) are added to the running total: short chains, so the
  // rounding error over a long K stays that of a blocked sum.
  f32x4_t tot[RT][CT], acc[RT][CT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int u = 0; u < CT; ++u) tot[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  constexpr std::integral_constant<int, 0> I0{};
  constexpr std::integral_constant<int, 1> I1{};
  constexpr std::integral_constant<int, 2> I2{};
  constexpr std::integral_constant<int, 3> I3{};
  const bf16x8_t *fsrc = xs + li * 4 + (kb ^ ((li >> 1) & 3));
  // step p of the chunk in buffer SET, weights in ring slot 2 SET + p
  auto mma = [&](auto set, auto step) {
    constexpr int SET = decltype(set)::value, PS = decltype(step)::value;
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
  };

  xload(s0, I0);
  wload(s0, I0);
  wload(s0 + 1, I1);
  xload(s0 + 2, I1);
  wload(s0 + 2, I2);
  wload(s0 + 3, I3);
  xstore(s0, I0, true);
  __syncthreads();
  // Straight-line pairs: no branch, so that the loads of the rings stay in flight across iterations.
  // Entering a pair: chunk st in buffer 0, chunk st + 2 in register set 1, weights of st .. st + 3.
  for (int i = 0, st = s0; i < pairs; ++i, st += 4) {
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int u = 0; u < CT; ++u) acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    xload(st + 4, I0);
    __builtin_amdgcn_sched_barrier(0);
    mma(I0, I0);
    wload(st + 4, I0);
    mma(I0, I1);
    wload(st + 5, I1);
    __builtin_amdgcn_sched_barrier(0);
    xstore(st + 2, I1, true);
    __syncthreads();
    xload(st + 6, I1);
    __builtin_amdgcn_sched_barrier(0);
    mma(I1, I0);
    wload(st + 6, I2);
    mma(I1, I1);
    wload(st + 7, I3);
    __builtin_amdgcn_sched_barrier(0);
    xstore(st + 4, I0, i + 1 < pairs);
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int u = 0; u < CT; ++u) tot[t][u] += acc[t][u];
    __syncthreads();
  }

  // The row's sum of squares over its staging threads: partial sums at rsum[part][row]
  constexpr int NP = 2 * KG;
  if constexpr (NORM) {
    ss += __shfl_xor(ss, 1, 64);
    ss += __shfl_xor(ss, 2, 64);
    if (slot == 0) rsum[(2 * grp + sp) * BM + srow] = ss;
  }
  if constexpr (KG > 1) {  // the other groups' sums, through their own staging buffers, in group order
    f32x4_t *m = reinterpret_cast<f32x4_t *>(lds) + tid;
    if (grp > 0) {
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int u = 0; u < CT; ++u) m[grp * 2 * BUF + (t * CT + u) * 256] = tot[t][u];
    }
    __syncthreads();
    if (grp > 0) return;
#pragma unroll
    for (int k = 1; k < KG; ++k)
#pragma unroll
      for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int u = 0; u < CT; ++u) tot[t][u] += m[k * 2 * BUF + (t * CT + u) * 256];
  } else if constexpr (NORM) {
    __syncthreads();
  }
  float inv[RT];
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    inv[t] = 1.f;
    if constexpr (NORM) {
      float s = rsum[16 * t + li];
#pragma unroll
      for (int i = 1; i < NP; ++i) s += rsum[i * BM + 16 * t + li];
      inv[t] = 1.0f / sqrtf(s / (float)a.K + a.eps);
    }
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
  constexpr int LDI = 36;  // SPLIT: this wave's 32 x 32 outputs, in the staging space of group 0
  float *image = reinterpret_cast<float *>(lds) + wave * BM * LDI;
#pragma unroll
  for (int t = 0; t < RT; ++t) {
    const int m = m0 + 16 * t + li;
#pragma unroll
    for (int u = 0; u < OT; ++u) {
      const int n = n0 + 16 * u + 4 * kb;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = tot[t][u][e];
        if constexpr (NORM) v[e] *= inv[t];
        if constexpr (SW) {
          float up = tot[t][u + OT][e];
          if constexpr (NORM) up *= inv[t];
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
      if constexpr (SPLIT) {
        split_put(a, v, r, image + (16 * t + li) * LDI + 16 * u + 4 * kb, m, n, blockIdx.z, vec);
        continue;
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
  if constexpr (SPLIT) split_add<BM, 32, LDI>(a, image, m0, n0, lane);
}

// Up to 64 rows (MT tiles of 16): a workgroup per 16-column tile (SwiGLU: a gate tile and its up
// tile) and, with GemmArgs::split2, K half.  Eight waves take contiguous shares of K; each issues the
// loads of PS steps together, weights and X straight from global memory in matrix-core order, and the
// waves' sums meet in LDS in wave order.  With so few rows a launch lasts as long as one workgroup:
// one memory round trip, plus what its CU can load (64 bytes a clock, rows x K x 4 of X above all) and
// split.  So the columns are spread as thin as the matrix cores take them, over every CU, nothing is
// waited for between a wave's loads, and no second launch adds up partial sums.
// Same arithmetic as k_gemm_tile: the matrix cores take x * gain, the sums are scaled by 1 / rms.
template <int EPI, bool NORM, int MT, bool SPLIT>
__global__ __launch_bounds__(512, 2) void k_gemm_rows(GemmArgs a, int vec) {
  static_assert(!SPLIT || EPI == EPI_RESIDUAL, "the K halves meet in a residual sum");
  constexpr bool SW = EPI == EPI_SWIGLU;
  constexpr int T = SW ? 2 : 1, W = 8, PS = MT == 1 ? 8 : (MT == 4 && SW && NORM ? 3 : 4);
  constexpr bool RES = EPI == EPI_RESIDUAL || EPI == EPI_AFFINE_RES || EPI == EPI_RES_SNAKE;
  constexpr bool BIAS = EPI == EPI_BIAS || EPI == EPI_AFFINE_RES || EPI == EPI_BIAS_GELU ||
                        EPI == EPI_BIAS_SILU || EPI == EPI_RES_SNAKE;
  __shared__ f32x4_t part[W][MT * T][64];
  __shared__ float ssq[W][MT * 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, kb = lane >> 4;
  const int ntile = (a.N + 15) / 16, steps = a.K / 32;
  const int h0 = SPLIT ? (int)((int64_t)steps * blockIdx.y / 2) : 0;
  const int h1 = SPLIT ? (int)((int64_t)steps * (blockIdx.y + 1) / 2) : steps;
  const int s0 = h0 + (h1 - h0) * wave / W, s1 = h0 + (h1 - h0) * (wave + 1) / W;

  const int r0 = 16 * MT * blockIdx.z;  // first row

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

  const float *xp[MT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xp[t] = a.X + (size_t)min(r0 + 16 * t + li, a.M - 1) * a.ldx + 8 * kb;
  const uint16_t *wp[T];
#pragma unroll
  for (int u = 0; u < T; ++u) wp[u] = a.W + (size_t)(blockIdx.x + u * ntile) * steps * 512 + lane * 8;

  // The high terms' sum apart from the two small ones': a third of the roundings at full magnitude
  f32x4_t acc[MT][T], low[MT][T];
#pragma unroll
  for (int t = 0; t < MT; ++t)
#pragma unroll
    for (int u = 0; u < T; ++u) acc[t][u] = low[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float ss[MT] = {};
  for (int p0 = s0; p0 < s1; p0 += PS) {
    f32x4_t x[PS][MT][2], g[NORM ? PS : 1][2];
    bf16x8_t w[PS][T];
#pragma unroll
    for (int i = 0; i < PS; ++i) {
      const int st = min(p0 + i, s1 - 1);
#pragma unroll
      for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h) x[i][t][h] = *reinterpret_cast<const f32x4_t *>(xp[t] + 32 * st + 4 * h);
      if constexpr (NORM) {
#pragma unroll
        for (int h = 0; h < 2; ++h) g[i][h] = *reinterpret_cast<const f32x4_t *>(a.gamma + 32 * st + 8 * kb + 4 * h);
      }
#pragma unroll
      for (int u = 0; u < T; ++u) w[i][u] = *reinterpret_cast<const bf16x8_t *>(wp[u] + (size_t)st * 512);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < PS; ++i) {
      if (p0 + i >= s1) break;
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = x[i][t][e >> 2][e & 3];
        if constexpr (NORM) {
#pragma unroll
          for (int e = 0; e < 8; ++e) ss[t] = __builtin_fmaf(v[e], v[e], ss[t]);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] *= g[i][e >> 2][e & 3];
        }
        bf16x8_t hi, mid, lo;
        split_bf16x8_nc(v, hi, mid, lo);
#pragma unroll
        for (int u = 0; u < T; ++u) {
          low[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][u], lo, low[t][u], 0, 0, 0);
          low[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][u], mid, low[t][u], 0, 0, 0);
          acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[i][u], hi, acc[t][u], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < MT; ++t) {
#pragma unroll
    for (int u = 0; u < T; ++u) part[wave][t * T + u][lane] = acc[t][u] + low[t][u];
    if constexpr (NORM) {
      float q = ss[t];
      q += __shfl_xor(q, 16, 64);
      q += __shfl_xor(q, 32, 64);
      if (kb == 0) ssq[wave][16 * t + li] = q;
    }
  }
  __syncthreads();
  if (tid >= 64 * MT) return;
  float v[4], up[4];
  {
    f32x4_t s[T];
#pragma unroll
    for (int u = 0; u < T; ++u) {
      s[u] = part[0][ot * T + u][lane];
#pragma unroll
      for (int k = 1; k < W; ++k) s[u] += part[k][ot * T + u][lane];
    }
    float inv = 1.f;
    if constexpr (NORM) {
      float q = 0.f;
#pragma unroll
      for (int k = 0; k < W; ++k) q += ssq[k][16 * ot + li];
      inv = 1.0f / sqrtf(q / (float)a.K + a.eps);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = NORM ? s[0][e] * inv : s[0][e];
      up[e] = NORM ? s[T - 1][e] * inv : s[T - 1][e];
    }
  }
  if constexpr (SPLIT) {
    float r[4], *image = reinterpret_cast<float *>(part[0][ot]);  // 16 x 16; this wave has read its sums
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = rv[e];
    split_put(a, v, r, image + li * 16 + 4 * kb, om, on, blockIdx.y, vec);
    split_add<16, 16, 16>(a, image, r0 + 16 * ot, blockIdx.x * 16, lane);
    return;
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
  const dim3 grid((a.N + 15) / 16, a.split2 ? 2 : 1, (a.M + 16 * MT - 1) / (16 * MT));
  if constexpr (EPI == EPI_RESIDUAL && !NORM) {
    if (a.split2) {
      hipLaunchKernelGGL((k_gemm_rows<EPI, NORM, MT, true>), grid, dim3(512), 0, s, a, gemm_vec(a));
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((k_gemm_rows<EPI, NORM, MT, false>), grid, dim3(512), 0, s, a, gemm_vec(a));
  return hipGetLastError();
}

template <int EPI, bool NORM, int KG, bool SPLIT>
hipError_t tile_launch_split(const GemmArgs &a, hipStream_t s) {
  const int out = EPI == EPI_SWIGLU ? 64 : 128;
  const dim3 grid((a.N + out - 1) / out, (a.M + 31) / 32, SPLIT ? 2 : 1);
  const size_t lds = (size_t)KG * 2 * 3 * 2 * 32 * 64 + (NORM ? (size_t)KG * 2 * 32 * 4 : 0);
  if (!SPLIT && a.K % (128 * KG))
    hipLaunchKernelGGL((k_gemm_tile<EPI, NORM, KG, !SPLIT, SPLIT>), grid, dim3(256 * KG), lds, s, a, gemm_vec(a));
  else
    hipLaunchKernelGGL((k_gemm_tile<EPI, NORM, KG, false, SPLIT>), grid, dim3(256 * KG), lds, s, a, gemm_vec(a));
  return hipGetLastError();
}

template <int EPI, bool NORM, int KG>
hipError_t tile_launch(const GemmArgs &a, hipStream_t s) {
  if constexpr (EPI == EPI_RESIDUAL && !NORM) {
    if (a.split2) return tile_launch_split<EPI, NORM, KG, true>(a, s);
  }
  return tile_launch_split<EPI, NORM, KG, false>(a, s);
}

// Up to 64 rows: k_gemm_rows (whose X traffic per 16 columns is all rows: at 137 rows x 2048 it took
// twice k_gemm_tile's time), the rows in as many parts as bring the workgroups to one per CU at most (O
// and down at 41 rows, 128 workgroups of three tiles: prefill 1.58 -> 1.46 ms with 256 of two and one;
// with 384 of one tile each 1.65, a CU then waits for two).  More: k_gemm_tile, with two K groups a block
// where there are fewer blocks than CUs (137 rows, O and down of the 1.7B shape: prefill 4.63 -> 4.12 ms;
// with 544 blocks one group is 3% faster; four groups measured as two).
template <int EPI, bool NORM>
hipError_t tile_shape(const GemmArgs &a, hipStream_t s) {
  if (a.M <= 64) {
    const int cols = (a.N + 15) / 16 * (a.split2 ? 2 : 1), tiles = (a.M + 15) / 16;
    const int z = std::min(tiles, std::max(1, 256 / cols));
    switch ((tiles + z - 1) / z) {
      case 1: return rows_launch<EPI, NORM, 1>(a, s);
      case 2: return rows_launch<EPI, NORM, 2>(a, s);
      case 3: return rows_launch<EPI, NORM, 3>(a, s);
      default: return rows_launch<EPI, NORM, 4>(a, s);
    }
  }
  const int n = EPI == EPI_SWIGLU ? 2 * a.N : a.N, blocks = (a.M + 31) / 32 * ((n + 127) / 128) * (a.split2 ? 2 : 1);
  return blocks >= 256 || a.K < 128 ? tile_launch<EPI, NORM, 1>(a, s) : tile_launch<EPI, NORM, 2>(a, s);
}

template <int EPI>
hipError_t tile_norm(const GemmArgs &a, hipStream_t s) {
  return a.gamma ? tile_shape<EPI, true>(a, s) : tile_shape<EPI, false>(a, s);
}

}  // namespace

hipError_t launch_gemm(int epi, const GemmArgs &a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0 || a.K <= 0 || a.K % 32 || a.ldx % 4 || !a.w_packed || !a.X || !a.W || !a.Y ||
      reinterpret_cast<uintptr_t>(a.X) % 16 || reinterpret_cast<uintptr_t>(a.W) % 16 ||
      reinterpret_cast<uintptr_t>(a.gamma) % 16)
    return hipErrorInvalidValue;
  const bool res = epi == EPI_RESIDUAL || epi == EPI_AFFINE_RES || epi == EPI_RES_SNAKE;
  const bool bias = epi == EPI_BIAS || epi == EPI_BIAS_GELU || epi == EPI_BIAS_SILU || epi == EPI_RES_SNAKE;
  if ((res && !a.res) || (bias && !a.bias)) return hipErrorInvalidValue;
  if (a.split2 && (epi != EPI_RESIDUAL || a.gamma || a.M > gemm_split_rows(a.N) || !a.res_zero || a.K < 64 ||
                   (a.M > 64 && a.K % 512)))
    return hipErrorInvalidValue;
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
