// Causal convolutions of the codec decoder on the matrix cores, with the Snake activations
// around them folded in: Y[t][n] = f(bias[n] + sum_{j, c} S(X)[t - (TAPS - 1 - j) d][c] W[n][j][c])
// over time-major fp32 rows (rows before time 0 are zeros), S the identity or the input's Snake
// and f the identity or the output's Snake.
//
// What bounds it: the matrix cores.  An fp32 activation enters as three exact bf16 terms
// (q3t_bf16x3.h), so a product costs three v_mfma_f32_16x16x32_bf16.  The block's X rows of 32
// channels (BM + halo rows) are loaded, activated and split once, into LDS, and serve all TAPS
// taps of the block's BW columns from there: the vector work per element is 1 / TAPS of what a
// GEMM over gathered rows spends (which loads and splits each row once per tap), and no padded or
// activated copy of X goes through memory.
//
//   * LDS holds the three terms as planes of [row][32 channels], 64 bytes a row, the four 16-byte
//     slots of a row xor-ed with (row / 2) % 4: any 8 consecutive rows of one slot fall in 8
//     distinct 16-byte columns of the 128-byte bank row, at every tap's row offset.
//   * Two buffers: the next 32 channels are in flight (registers) while the taps of this one run,
//     then activated, split and stored: one barrier per TAPS k steps.
//   * Weights come straight from global memory in matrix-core order (codec_conv_pack: 1 KiB
//     contiguous per 16 columns and step, a step's taps consecutive), one step ahead.  The two
//     waves of a column half read the same lines.
//   * Four waves as 2 x 2: BM / 2 rows by BW / 2 columns each.  The weight tile is the A operand,
//     so a lane ends with four consecutive columns of one row: 16-byte bias loads and stores.
//   * BW = 192, but 96 for the units of 96 channels and the transposed convolution of N = 288: all N are
//     exact multiples.
//   * BM = 64 (45 KB of LDS at dilation 9: up to three blocks a CU).  128-row blocks measured the
//     same on long inputs and leave CUs idle on short ones; residual units, which nothing splits,
//     take BM = 32 when short.  A launch of few blocks splits the
//     channel steps over grid z into split_ws, added in order by k_codec_conv_reduce.
#include "q3t_codec.h"

#include <algorithm>

#include "q3t_bf16x3.h"

namespace q3t {
namespace {

constexpr int kConvMaxDilation = 9;
constexpr int kConvRows = 64;  // BM

// UNIT: BW = N, and the block continues with the residual unit's second half (CodecConvArgs::w2).
template <int TAPS, int BM, int BW, bool SIN, bool SOUT, bool UNIT = false, bool SRES = false>
__global__ __launch_bounds__(256, 2) void k_codec_conv(CodecConvArgs a) {
  constexpr int RT = BM / 32, CT = BW / 32;  // 16-row and 16-column tiles per wave
  constexpr int MAXD = TAPS > 2 ? kConvMaxDilation : 1;
  constexpr int NP = ((BM + (TAPS - 1) * MAXD) * 4 + 255) / 256;  // 8-channel units per thread
  extern __shared__ bf16x8_t xs[];                                // [2][3][rows][4]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, kb = lane >> 4, wr = wave >> 1, wc = wave & 1;
  const int halo = (TAPS - 1) * a.d, rows = BM + halo, units = rows * 4;
  int mb, nb;
  block_tile(UNIT ? 1 : a.N / BW, mb, nb);
  const int m0 = mb * BM;
  const int nch = a.C / 32, nsplit = gridDim.z, z = blockIdx.z;
  const int c0 = (int)((int64_t)nch * z / nsplit), c1 = (int)((int64_t)nch * (z + 1) / nsplit);

  // X units of this thread: row (tid + 256 p) / 4 of the block's rows, channels 8 (tid % 4) .. + 7
  const int slot = tid & 3;
  const float *xp[NP];
  bool xin[NP];
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    const int g = m0 - halo + ((tid + 256 * p) >> 2);
    xin[p] = g >= 0;
    xp[p] = a.X + (size_t)min(max(g, 0), a.T - 1) * a.C + 8 * slot;
  }
  float4 xr[NP][2];
  float4 ta[SIN ? 2 : 1], tb[SIN ? 2 : 1];
  auto xload = [&](int c) {
#pragma unroll
    for (int p = 0; p < NP; ++p)
#pragma unroll
      for (int h = 0; h < 2; ++h) xr[p][h] = *reinterpret_cast<const float4 *>(xp[p] + 32 * c + 4 * h);
    if constexpr (SIN) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        ta[h] = *reinterpret_cast<const float4 *>(a.sa + 32 * c + 8 * slot + 4 * h);
        tb[h] = *reinterpret_cast<const float4 *>(a.sb + 32 * c + 8 * slot + 4 * h);
      }
    }
  };
  auto xstore = [&](int p, int buf) {
    const int idx = tid + 256 * p;
    if (256 * (p + 1) > (BM + TAPS - 1) * 4 && idx >= units) return;
    float v[8] = {xr[p][0].x, xr[p][0].y, xr[p][0].z, xr[p][0].w, xr[p][1].x, xr[p][1].y, xr[p][1].z, xr[p][1].w};
    if constexpr (SIN) {
      const float ea[8] = {ta[0].x, ta[0].y, ta[0].z, ta[0].w, ta[1].x, ta[1].y, ta[1].z, ta[1].w};
      const float ib[8] = {tb[0].x, tb[0].y, tb[0].z, tb[0].w, tb[1].x, tb[1].y, tb[1].z, tb[1].w};
      snake_n<8>(v, ea, ib);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = xin[p] ? v[e] : 0.f;
    bf16x8_t hi, mid, lo;
    split_bf16x8_nc(v, hi, mid, lo);
    const int row = idx >> 2;
    bf16x8_t *dst = xs + (size_t)buf * 3 * units + row * 4 + (slot ^ ((row >> 1) & 3));
    dst[0] = lo;
    dst[units] = mid;
    dst[2 * units] = hi;
  };

  // Weight fragments of k step st = chunk * TAPS + tap of column tile u
  const int steps = nch * TAPS;
  const uint16_t *wbase = a.W + ((size_t)(nb * (BW / 16) + wc * CT) * steps) * 512 + lane * 8;
  const size_t wtile = (size_t)steps * 512;
  bf16x8_t w[CT], wn[CT];
  auto wload = [&](int st, bf16x8_t *dst) {
#pragma unroll
    for (int u = 0; u < CT; ++u) dst[u] = *reinterpret_cast<const bf16x8_t *>(wbase + u * wtile + (size_t)st * 512);
  };

  f32x4_t acc[RT][CT];
#pragma unroll
  for (int t = 0; t < RT; ++t)
#pragma unroll
    for (int u = 0; u < CT; ++u) acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  xload(c0);
  wload(c0 * TAPS, w);
#pragma unroll
  for (int p = 0; p < NP; ++p) xstore(p, 0);
  __syncthreads();
  int buf = 0;
  const int last = c1 * TAPS - 1;
  for (int c = c0; c < c1; ++c) {
    const bool more = c + 1 < c1;
    if (more) xload(c + 1);
#pragma unroll
    for (int tap = 0; tap < TAPS; ++tap) {
      wload(min(c * TAPS + tap + 1, last), wn);
      __builtin_amdgcn_sched_barrier(0);
      const int r = wr * (BM / 2) + li + tap * a.d;
      const bf16x8_t *src = xs + (size_t)buf * 3 * units + r * 4 + (kb ^ ((r >> 1) & 3));
#pragma unroll
      for (int q = 0; q < 3; ++q) {  // lo, mid, hi: every accumulator adds them in that order
        bf16x8_t x[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) x[t] = src[q * units + 64 * t];
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
          for (int u = 0; u < CT; ++u)
            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], x[t], acc[t][u], 0, 0, 0);
      }
#pragma unroll
      for (int u = 0; u < CT; ++u) w[u] = wn[u];
    }
    if (more) {
#pragma unroll
      for (int p = 0; p < NP; ++p) xstore(p, buf ^ 1);
    }
    __syncthreads();
    buf ^= 1;
  }

  if constexpr (UNIT) {
    // Second half: the Snaked rows go to LDS as planes of [channel chunk][row][4 slots] (the
    // staging buffers are free after the loop's last barrier), then through the 1x1 convolution.
    constexpr int PL = BW / 32 * BM * 4;  // 16-byte units of a plane
    float4 rv[RT][CT];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
      for (int u = 0; u < CT; ++u) {
        const int m = min(m0 + wr * (BM / 2) + 16 * t + li, a.T - 1), n = (wc * CT + u) * 16 + 4 * kb;
        rv[t][u] = *reinterpret_cast<const float4 *>(a.X + (size_t)m * BW + n);
      }
#pragma unroll
    for (int u = 0; u < CT; ++u) {
      const int n = (wc * CT + u) * 16 + 4 * kb;
      const float4 b4 = *reinterpret_cast<const float4 *>(a.bias + n);
      const float4 ea4 = *reinterpret_cast<const float4 *>(a.oa + n), ib4 = *reinterpret_cast<const float4 *>(a.ob + n);
      const float ea[4] = {ea4.x, ea4.y, ea4.z, ea4.w}, ib[4] = {ib4.x, ib4.y, ib4.z, ib4.w};
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        float v[4] = {acc[t][u][0] + b4.x, acc[t][u][1] + b4.y, acc[t][u][2] + b4.z, acc[t][u][3] + b4.w};
        snake_n<4>(v, ea, ib);
        bf16x4_t hi, mid, lo;
        split_bf16_nc<4>(v, hi, mid, lo);
        const int r = wr * (BM / 2) + 16 * t + li;
        bf16x4_t *dst = reinterpret_cast<bf16x4_t *>(xs + ((n >> 5) * BM + r) * 4 + (((n >> 3) & 3) ^ ((r >> 1) & 3))) +
                        ((n >> 2) & 1);
        dst[0] = lo;
        dst[2 * PL] = mid;
        dst[4 * PL] = hi;
        acc[t][u] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    constexpr int KS = BW / 32;
    const uint16_t *w2 = a.w2 + (size_t)wc * CT * KS * 512 + lane * 8;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < KS; ++k) {
#pragma unroll
      for (int u = 0; u < CT; ++u) w[u] = *reinterpret_cast<const bf16x8_t *>(w2 + (size_t)(u * KS + k) * 512);
      const int r = wr * (BM / 2) + li;
      const bf16x8_t *src = xs + (k * BM + r) * 4 + (kb ^ ((r >> 1) & 3));
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        bf16x8_t x[RT];
#pragma unroll
        for (int t = 0; t < RT; ++t) x[t] = src[q * PL + 64 * t];
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
          for (int u = 0; u < CT; ++u)
            acc[t][u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[u], x[t], acc[t][u], 0, 0, 0);
      }
    }
#pragma unroll
    for (int u = 0; u < CT; ++u) {
      const int n = (wc * CT + u) * 16 + 4 * kb;
      const float4 b4 = *reinterpret_cast<const float4 *>(a.b2 + n);
      float4 ea4 = b4, ib4 = b4;
      if constexpr (SRES) {
        ea4 = *reinterpret_cast<const float4 *>(a.ra + n);
        ib4 = *reinterpret_cast<const float4 *>(a.rb + n);
      }
#pragma unroll
      for (int t = 0; t < RT; ++t) {
        const int m = m0 + wr * (BM / 2) + 16 * t + li;
        float v[4] = {rv[t][u].x + (acc[t][u][0] + b4.x), rv[t][u].y + (acc[t][u][1] + b4.y),
                      rv[t][u].z + (acc[t][u][2] + b4.z), rv[t][u].w + (acc[t][u][3] + b4.w)};
        if constexpr (SRES) {
          const float ea[4] = {ea4.x, ea4.y, ea4.z, ea4.w}, ib[4] = {ib4.x, ib4.y, ib4.z, ib4.w};
          snake_n<4>(v, ea, ib);
        }
        if (m < a.T) *reinterpret_cast<float4 *>(a.Y + (size_t)m * BW + n) = make_float4(v[0], v[1], v[2], v[3]);
      }
    }
    return;
  }

  // Lane (li, kb) holds columns 4 kb .. 4 kb + 3 of row li of each tile.
#pragma unroll
  for (int u = 0; u < CT; ++u) {
    const int n = nb * BW + (wc * CT + u) * 16 + 4 * kb;
    float4 b4 = make_float4(0.f, 0.f, 0.f, 0.f), ea4 = b4, ib4 = b4;
    if (nsplit == 1) {
      b4 = *reinterpret_cast<const float4 *>(a.bias + n);
      if constexpr (SOUT) {
        ea4 = *reinterpret_cast<const float4 *>(a.oa + n);
        ib4 = *reinterpret_cast<const float4 *>(a.ob + n);
      }
    }
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      const int m = m0 + wr * (BM / 2) + 16 * t + li;
      float v[4] = {acc[t][u][0] + b4.x, acc[t][u][1] + b4.y, acc[t][u][2] + b4.z, acc[t][u][3] + b4.w};
      float *out = a.Y;
      size_t at = (size_t)m * a.N + n;
      if (nsplit > 1) {  // raw sums: [split][T][N]
        out = a.split_ws;
        at += (size_t)z * a.T * a.N;
      } else if constexpr (SOUT) {
        const float ea[4] = {ea4.x, ea4.y, ea4.z, ea4.w}, ib[4] = {ib4.x, ib4.y, ib4.z, ib4.w};
        snake_n<4>(v, ea, ib);
      }
      if (m < a.T) *reinterpret_cast<float4 *>(out + at) = make_float4(v[0], v[1], v[2], v[3]);
    }
  }
}

// The channel splits' sums added in split order, then bias and the output's Snake.
template <bool SOUT>
__global__ __launch_bounds__(256) void k_codec_conv_reduce(CodecConvArgs a, int nsplit) {
  const uint32_t n4 = (uint32_t)a.N / 4, i = blockIdx.x * 256 + threadIdx.x;
  const size_t all = (size_t)a.T * n4;
  if (i >= all) return;
  const uint32_t n = i % n4;
  const float4 *ws = reinterpret_cast<const float4 *>(a.split_ws);
  float4 s = ws[i];
  for (int z = 1; z < nsplit; ++z) {
    const float4 p = ws[z * all + i];
    s.x += p.x; s.y += p.y; s.z += p.z; s.w += p.w;
  }
  const float4 b = reinterpret_cast<const float4 *>(a.bias)[n];
  float v[4] = {s.x + b.x, s.y + b.y, s.z + b.z, s.w + b.w};
  if constexpr (SOUT) {
    const float4 ea4 = reinterpret_cast<const float4 *>(a.oa)[n], ib4 = reinterpret_cast<const float4 *>(a.ob)[n];
    const float ea[4] = {ea4.x, ea4.y, ea4.z, ea4.w}, ib[4] = {ib4.x, ib4.y, ib4.z, ib4.w};
    snake_n<4>(v, ea, ib);
  }
  reinterpret_cast<float4 *>(a.Y)[i] = make_float4(v[0], v[1], v[2], v[3]);
}

template <int TAPS, int BM, int BW, bool SIN, bool SOUT>
void conv_launch(const CodecConvArgs &a, dim3 grid, hipStream_t s) {
  const size_t lds = (size_t)2 * 3 * (BM + (TAPS - 1) * a.d) * 64;
  hipLaunchKernelGGL((k_codec_conv<TAPS, BM, BW, SIN, SOUT>), grid, dim3(256), lds, s, a);
}

template <int TAPS, bool SIN, bool SOUT>
hipError_t conv_shape(const CodecConvArgs &a, hipStream_t s) {
  const int bw = a.N % 192 == 0 ? 192 : 96;
  if (TAPS > 2 && bw == 96) return hipErrorInvalidValue;
  dim3 grid(a.N / bw * ((a.T + kConvRows - 1) / kConvRows));
  // channel splits: towards 256 workgroups, at least two chunks each, within the workspace
  const int blocks = (int)grid.x, nch = a.C / 32;
  int sp = 1;
  if (a.split_ws && blocks < 192) {
    sp = std::max(1, std::min((256 + blocks - 1) / blocks, nch / 2));
    while (sp > 1 && (int64_t)sp * a.T * a.N > a.split_cap) --sp;
  }
  grid.z = sp;
  if constexpr (TAPS == 2) {
    if (bw == 192) conv_launch<TAPS, kConvRows, 192, SIN, SOUT>(a, grid, s);
    else conv_launch<TAPS, kConvRows, 96, SIN, SOUT>(a, grid, s);
  } else {
    conv_launch<TAPS, kConvRows, 192, SIN, SOUT>(a, grid, s);
  }
  if (sp > 1) {
    const size_t n = (size_t)a.T * a.N / 4;
    hipLaunchKernelGGL((k_codec_conv_reduce<SOUT>), dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a, sp);
  }
  return hipGetLastError();
}

// A whole residual unit of C = N channels (C = 96 or 192: one block holds every column).
template <int BM, int BW>
hipError_t unit_launch(const CodecConvArgs &a, hipStream_t s) {
  const size_t stage = (size_t)2 * 3 * (BM + 6 * a.d) * 64, mid = (size_t)3 * BM * BW * 2;
  const dim3 grid((a.T + BM - 1) / BM);
  if (a.ra)
    hipLaunchKernelGGL((k_codec_conv<7, BM, BW, true, true, true, true>), grid, dim3(256), std::max(stage, mid), s, a);
  else
    hipLaunchKernelGGL((k_codec_conv<7, BM, BW, true, true, true, false>), grid, dim3(256), std::max(stage, mid), s, a);
  return hipGetLastError();
}

}  // namespace

std::vector<uint16_t> codec_conv_pack(const std::vector<uint16_t> &w, int N, int C, int taps,
                                      size_t (*at)(int n, int c, int j, int N, int C, int taps)) {
  std::vector<uint16_t> r((size_t)N * C * taps);
  size_t o = 0;
  for (int nt = 0; nt < N / 16; ++nt)
    for (int ch = 0; ch < C / 32; ++ch)
      for (int j = 0; j < taps; ++j)
        for (int lane = 0; lane < 64; ++lane)
          for (int e = 0; e < 8; ++e) r[o++] = w[at(16 * nt + lane % 16, 32 * ch + 8 * (lane / 16) + e, j, N, C, taps)];
  return r;
}

bool codec_unit_ok(int C) { return C == 96 || C == 192; }

hipError_t launch_codec_conv(int taps, const CodecConvArgs &a, hipStream_t s) {
  auto aligned = [](const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (a.T <= 0 || a.C <= 0 || a.C % 32 || a.N <= 0 || a.N % 96 || a.d < 1 || a.d > (taps > 2 ? kConvMaxDilation : 1) ||
      !a.X || !a.W || !a.Y || !a.bias || a.Y == a.X || (!a.sa != !a.sb) || (!a.oa != !a.ob) || !aligned(a.X) ||
      !aligned(a.W) || !aligned(a.Y) || !aligned(a.bias) || !aligned(a.sa) || !aligned(a.sb) || !aligned(a.oa) ||
      !aligned(a.ob) || !aligned(a.split_ws) || (size_t)a.T * a.N / 4 >= UINT32_MAX)
    return hipErrorInvalidValue;
  if (a.w2) {
    if (taps != 7 || !a.sa || !a.oa || a.C != a.N || !codec_unit_ok(a.C) || !a.b2 || (!a.ra != !a.rb) ||
        !aligned(a.w2) || !aligned(a.b2) || !aligned(a.ra) || !aligned(a.rb))
      return hipErrorInvalidValue;
    // Fewer blocks than CUs: half the rows a block.  Decode of 6 frames 749 -> 710 us (60 blocks of 192
    // channels, 180 of 96); of 31 (310 and 930 blocks) with half the rows 1139 -> 1180, each row block
    // reading all the unit's weights.
    if ((a.T + kConvRows - 1) / kConvRows < 256)
      return a.C == 96 ? unit_launch<kConvRows / 2, 96>(a, s) : unit_launch<kConvRows / 2, 192>(a, s);
    return a.C == 96 ? unit_launch<kConvRows, 96>(a, s) : unit_launch<kConvRows, 192>(a, s);
  }
  if (taps == 7 && a.oa) return a.sa ? conv_shape<7, true, true>(a, s) : conv_shape<7, false, true>(a, s);
  if (taps == 2 && !a.sa && !a.oa) return conv_shape<2, false, false>(a, s);
  return hipErrorInvalidValue;
}

}  // namespace q3t
