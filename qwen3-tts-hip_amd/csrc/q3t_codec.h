// Codec decoder (speech tokenizer decoder): codec frames [F][16] -> F * 1920 samples at 24 kHz,
// the reference's HipCodecInitial (src/audio/codec_hip.rs) on the gfx950 matrix cores.
#pragma once

#include <string>
#include <vector>

#include "q3t_device.h"

namespace q3t {

constexpr int kCodecSamplesPerFrame = 1920;  // 2 x 2 (upsampling) x 8 x 5 x 4 x 3 (decoder blocks)
constexpr int kCodecMaxAttnRows = 8192;      // frames one pre-transformer attention covers

struct Codec;

// Loads <model_dir>/speech_tokenizer/model.safetensors (codec_hip.rs:214-336); returns null
// when the file does not exist.  Adds the device bytes it holds to *device_bytes.
Codec *codec_load(const std::string &model_dir, int64_t *device_bytes);
void codec_free(Codec *c);
// Decodes `frames` frames of device codes (frame-major, `groups` per frame) into frames * 1920
// samples (device pointer) on stream s, synchronously.  The workspace grows to the largest
// frame count seen.
void codec_decode(Codec &c, const int32_t *codes, int frames, int groups, float *samples, hipStream_t s);
// Device staging buffers owned by the codec (grown on demand): n codes, n samples.
int32_t *codec_codes_buffer(Codec &c, size_t n);
float *codec_samples_buffer(Codec &c, size_t n);

// Kernels (q3t_codec.hip).
hipError_t launch_codec_rvq(const int32_t *codes, int frames, int groups, const float *first, const float *rest,
                            int V, int D, float *E, hipStream_t s);
// The Snake tables of a checkpoint's alpha / beta, in place: alpha := exp(alpha), beta := 1 /
// (exp(beta) + 1e-9) (snake_beta_f32, kernels.rs).
hipError_t launch_codec_snake_prep(float *alpha, float *beta, int C, hipStream_t s);

// A causal convolution of `taps` taps (7, or 2 at d = 1: the transposed convolutions, whose
// stride phases are columns) over time-major rows, with the Snakes around it (q3t_codec_conv.hip).
// Kinds: 7 taps with an output Snake and with or without an input one; 2 taps with neither.
struct CodecConvArgs {
  const float *X;         // [T][C]; rows before 0 count as zeros
  int32_t T, C, d;        // C a multiple of 32; d = dilation, at most 9
  const float *sa, *sb;   // input Snake tables [C], or null
  const uint16_t *W;      // codec_conv_pack layout
  const float *bias;      // [N]
  const float *oa, *ob;   // output Snake tables [N], or null
  float *Y;               // [T][N], not X
  int32_t N;              // a multiple of 96 (7 taps without w2: of 192)
  float *split_ws;        // channel splits of short inputs: [split][T][N] raw sums, or null
  int64_t split_cap;      // floats in split_ws
  // A whole residual unit (7 taps, both Snakes, C = N, codec_unit_ok): the Snaked output goes on
  // through a 1x1 convolution in the same launch, Y = S(X + (b2 + w2 . out)), S the Snake of
  // ra / rb or, with null tables, the identity.
  const uint16_t *w2;     // [N][C] packed (launch_pack_weights); null: no second half
  const float *b2, *ra, *rb;
};
bool codec_unit_ok(int C);
hipError_t launch_codec_conv(int taps, const CodecConvArgs &a, hipStream_t s);
// Weights in matrix-core order, [N / 16][C / 32][taps][64 lanes][8]: lane i + 16 k of (tile, chunk,
// tap) holds column 16 tile + i, channels 32 chunk + 8 k .. + 7.  at(n, c, j, N, C, taps) is the
// source index of column n, channel c, tap j.
std::vector<uint16_t> codec_conv_pack(const std::vector<uint16_t> &w, int N, int C, int taps,
                                      size_t (*at)(int n, int c, int j, int N, int C, int taps));
// Depthwise convolution (C = 1024, K = 7; w [C][K]) and LayerNorm of its rows.
hipError_t launch_codec_dwconv_norm(const float *x, const float *w, const float *wb, const float *g, const float *b,
                                    int T, int C, int K, float eps, float *out, hipStream_t s);
// Causal attention with RoPE over raw qkv rows (64 dims a head; table [T][32] (cos, sin)).
hipError_t launch_codec_attention(const float *qkv, int T, int ld, int heads, const float2 *table, float scale,
                                  float *out, int ldo, hipStream_t s);
// Last convolution (C = 96, K = 7; rows x[t] of time t) and clamp.
hipError_t launch_codec_final(const float *x, const float *w, const float *b, int T, int C, int K, float *out,
                              hipStream_t s);

}  // namespace q3t
