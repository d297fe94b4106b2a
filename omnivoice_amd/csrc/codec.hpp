// Launchers of the audio decoder's gfx950 kernels (codec_kernels.hip).
// Signals are float32, channel-major: [channels][samples].
#ifndef OMNIVOICE_AMD_CODEC_HPP_
#define OMNIVOICE_AMD_CODEC_HPP_

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace ovg {

constexpr int kConvMaxTaps = 7;
constexpr int kConvMaxPhases = 8;
// Largest spread between a convolution's first and last tap (kernel 7 at
// dilation 9 spans 54 samples).
constexpr int kConvMaxSpan = 64;

// Largest residual unit that runs as one launch.
constexpr int kConvFusedChannels = 128;

// Activations a convolution's epilogue applies.
enum ConvAct : int {
  kActNone = 0,
  kActGelu = 1,   // 0.5 v (1 + erf(v / sqrt 2)), pre-activation only
  kActSnake = 2,  // v + sin^2(alpha v) / (alpha + 1e-9), output activation only
  kActElu = 3,    // v > 0 ? v : exp(v) - 1, input or output activation
};

// Float32 weights as the bf16 triples the kernel multiplies (split.hpp), in
// units of eight input channels of one output channel; rows (output channels)
// are padded to whole 32-row blocks, input channels to whole groups of ConvPad.
constexpr int ConvPad(int taps) { return taps == 1 ? 128 : 32; }
struct alignas(16) ConvUnit {
  std::uint32_t pairs[4];
};
constexpr int ConvRows(int cout) { return (cout + 31) / 32 * 32; }
std::size_t ConvWeightUnits(int lead, int taps, int cin, int cout);
// w [lead][taps][cin][cout] to ConvWeightUnits units.
void LaunchPackConvWeights(const float* w, int lead, int taps, int cin, int cout, ConvUnit* out,
                           hipStream_t stream);

// One float32 convolution as an implicit GEMM on the matrix cores:
//   v[o][t] = pre(bias[o] + sum_{k, i} w[phase][k][i][o] *
//                 act_in(x[i][m + first[phase] + k dilation]))
//   y[o][t] = v (+ residual[o][t]), y_act[o][t] = out_act(y[o][t]),  t = m phases + phase
// for output positions m < positions, with x = 0 outside [0, len_in), and
// act_in the Snake activation of the channel's alpha (the identity when
// alpha_in is null), then in_act. A Conv1d is one phase with first = -pad; a
// ConvTranspose1d of stride s is s phases of two taps each (see the codec
// engine). With view_kernel, x has `channels` channels and K index i stands
// for x[i / view_kernel][m view_stride + first + i % view_kernel] (a strided
// or long convolution of one tap, cin = channels x view_kernel). With w2 the
// launch is a residual unit of up to kConvFusedChannels channels: v passes
// through the Snake of alpha_mid and the one-tap convolution w2, bias2 before
// the residual (x is then neither y nor y_act). Either
// output may be null; bias may be null (zero); residual may be y (phases have none).
// `batches` independent convolutions of the same shape run in one launch, the
// pointers of batch b advanced by b times their batch strides, the weights by
// one lead (a grouped convolution).
struct ConvParams {
  const float* x;         // [cin][len_in]
  const float* alpha_in;  // [cin] or null
  const ConvUnit* w;      // lead = batches x phases
  const float* bias;      // [cout] or null
  const ConvUnit* w2;     // [cout][cout], or null
  const float* bias2;     // [cout], with w2
  const float* alpha_mid; // [cout], with w2
  const float* residual;  // [cout][len_out] or null
  float* y;               // [cout][len_out] or null
  float* y_act;           // [cout][len_out] or null
  const float* alpha_out; // [cout], with a Snake output activation
  int cin, len_in, cout, len_out;
  int taps, dilation, phases, positions;
  int view_kernel, view_stride, channels;  // view_kernel 0: none
  int in_act;      // kActNone or kActElu
  int pre_act;     // kActNone or kActGelu
  int out_act;     // for y_act: kActSnake (default when 0) or kActElu
  int batches;     // 0 or 1: one convolution
  std::int64_t x_batch, b_batch, y_batch;  // element strides per batch
  int first[kConvMaxPhases];
  // Optional split-K workspace (float32 elements): when the output tiles
  // alone leave CUs idle, the launcher may split the input channels over
  // several work-groups, which store partial sums here; a second kernel
  // adds them in a fixed order and applies the epilogue. Null: never split.
  float* partial;
  std::int64_t partial_capacity;
  // Set by the launcher.
  int splits, split_chunks, w_rows;
};
void LaunchConv(const ConvParams& p, hipStream_t stream);

// The decoder's last layer, one output channel: y[t] = bias + sum_{k, i}
// w[k][i] x[i][t + k - pad], pad = (taps - 1) / 2.
struct OutputConvParams {
  const float* x;      // [cin][length]
  const float* w;      // [taps][cin]
  const float* bias;   // [1]
  float* y;            // [length]
  int cin, length, taps;
};
void LaunchOutputConv(const OutputConvParams& p, hipStream_t stream);

// RVQ decode folded with fc2: y[o][f] = bias[o] + sum_c
// table[c][codes[c][f]][o], i.e. the latent input of the decoder, channel
// major.
struct RvqParams {
  const float* table;  // [codebooks][entries][latent]
  const float* bias;   // [latent]
  const std::int32_t* codes;  // [codebooks][frames]
  float* y;            // [latent][frames]
  int codebooks, entries, latent, frames;
};
void LaunchRvq(const RvqParams& p, hipStream_t stream);

}  // namespace ovg

#endif  // OMNIVOICE_AMD_CODEC_HPP_
