// Launchers of the audio encoder's gfx950 kernels (encoder_kernels.hip).
// Signals are float32 and channel-major ([channels][positions]); every GEMM
// of the encoder runs through LaunchConv (codec.hpp).
#ifndef OMNIVOICE_AMD_ENCODER_HPP_
#define OMNIVOICE_AMD_ENCODER_HPP_

#include <hip/hip_runtime.h>

#include <cstdint>

namespace ovg {

// The polyphase resampler applied to device samples, written into a buffer
// with `pad` zeros on each side: y[pad + j] = sum_k bank[j % to][k]
// x[(j / to) from - width + k] over the taps inside the signal (summed in
// double), j < out_length; y has out_length + 2 pad elements.
struct ResampleParams {
  const float* x;     // [length]
  const float* bank;  // [to][taps]
  float* y;
  int length, from, to, width, taps, out_length, pad;
};
void LaunchResample(const ResampleParams& p, hipStream_t stream);

// y [cols][rows] = x [rows][cols] transposed.
void LaunchTranspose(const float* x, float* y, int rows, int cols, hipStream_t stream);

// GroupNorm with one group per channel (statistics over the row), affine,
// then GELU, in place: x [channels][length].
void LaunchGroupNormGelu(float* x, const float* w, const float* b, int channels, int length,
                         float eps, hipStream_t stream);

// LayerNorm over the channels of every position: y[c][t] = (x[c][t] -
// mean_t) / sqrt(var_t + eps) w[c] + b[c] (y may be x). sum_mode 1 sets,
// 2 adds y into `sum` (double, the running sum of encoder states).
struct ColumnNormParams {
  const float* x;
  float* y;
  const float* w;
  const float* b;
  double* sum;
  int channels, positions, sum_mode;
  float eps;
};
void LaunchColumnNorm(const ColumnNormParams& p, hipStream_t stream);

// Softmax attention of `heads` heads over `steps` positions: out[d][t] =
// sum_s v[d][s] softmax_s(scale sum_e k[e][s] q[e][t]), every operand
// [heads][head_dim][steps]; `packed` is a workspace of
// PackedHeadsElements(...) elements.
struct HeadAttentionParams {
  const float* q;
  const float* k;
  const float* v;
  float* out;
  std::uint16_t* packed;
  int heads, head_dim, steps;
  float scale;
};
std::size_t PackedHeadsElements(int heads, int head_dim, int steps);
void LaunchHeadAttention(const HeadAttentionParams& p, hipStream_t stream);

// y[c][f] = sum[c][f stride] scale for c < channels, f < frames; sum rows
// `positions` long.
void LaunchPickFrames(const double* sum, int channels, int positions, int stride, int frames,
                      double scale, float* y, hipStream_t stream);

// The residual vector quantizer: for every frame f and stage in turn, the
// projected residual v = bias + project^T r, the entry e of the largest
// -((|v|^2 - 2 v.e) + |e|^2) (the nearest; the lowest index on ties,
// distances in double), codes[stage][f] = e and r -= table[e]; r starts as
// x[:, f].
struct RvqStage {
  const float* project;  // [hidden][dim]
  const float* bias;     // [dim]
  const float* embed;    // [dim][entries]
  const double* norms;   // [entries], |e|^2
  const float* table;    // [entries][hidden]
};
struct RvqEncodeParams {
  const float* x;         // [hidden][frames]
  const RvqStage* stage;  // [stages], device memory
  float* residual;        // workspace of RvqResidualElements(...)
  std::int32_t* codes;    // [stages][frames]
  int stages, dim, entries, hidden, frames;
};
// Elements of `residual`: none where it stays in a work-group's LDS.
std::size_t RvqResidualElements(int dim, int hidden, int frames);
void LaunchRvqEncode(const RvqEncodeParams& p, hipStream_t stream);

}  // namespace ovg

#endif  // OMNIVOICE_AMD_ENCODER_HPP_
