// The audio decoder's kernels on gfx950 (replacing the reference's
// hipblasSgemm calls and element-wise kernels of the DAC decoder:
// codec_state.hpp:232-300, kernels/codec_kernels.hip:11-84).
//
// Every convolution is one implicit GEMM: output channels x output positions,
// summed over input channels x taps, each float32 product as six products of
// bf16 parts (split.hpp). Bias, activations and the residual addition are
// applied in the epilogue, straight from the accumulators. The sums are
// nearer to the exact ones than the float32 matrix cores' (the decoder's
// audio 1.2-2.3e-6 from 64 bits where those gave 1.9-4.6e-6).
#include "codec.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "split.hpp"

namespace ovg {
namespace {

constexpr int kThreads = 256;
constexpr int kOutTile = kThreads;  // samples per work-group of the output conv

// kernels/codec_kernels.hip:20-22 of the reference: v + sin^2(a v) / (a + 1e-9),
// with 1 / (a + 1e-9) given. x = a v less its nearest multiple of pi (pi in
// two parts; the first difference is exact, both terms being multiples of
// one unit and the difference below 2^24 of them), then the Taylor series of
// the sine up to r^13, whose remainder at pi / 2 is 2^-30 of the sine: about
// 18 operations where sinf has 40 and a branch. The term is at most 1 / |x|
// of v, so past |x| = 2^25, where the multiple is no longer the nearest one,
// any value in 0..1 rounds to the same sum.
__device__ __forceinline__ float Snake(float v, float a, float inverse) {
  const float x = a * v;
  const float n = rintf(x * 0.31830988618379067F);
  float r = fmaf(n, -3.1415927410125732F, x);
  r = fmaf(n, 8.7422776573475858e-8F, r);
  const float u = r * r;
  float s = 1.0F / 6227020800.0F;
  s = fmaf(s, u, -1.0F / 39916800.0F);
  s = fmaf(s, u, 1.0F / 362880.0F);
  s = fmaf(s, u, -1.0F / 5040.0F);
  s = fmaf(s, u, 1.0F / 120.0F);
  s = fmaf(s, u, -1.0F / 6.0F);
  s = fmaf(r * u, s, r);
  s = s * s;
  return v + inverse * (s > 1.0F ? 1.0F : s);
}
__device__ __forceinline__ float SnakeInverse(float a) { return 1.0F / (a + 1e-9F); }
__device__ __forceinline__ float Gelu(float v) {
  return 0.5F * v * (1.0F + erff(v * 0.70710678118654752F));
}
__device__ __forceinline__ float Elu(float v) { return v > 0.0F ? v : expm1f(v); }

// The epilogue of one output: bias, pre-activation, residual accumulation,
// the stores. What it reads is given, loaded before the sum is known.
struct Extras {
  float bias, residual, alpha;
};
__device__ __forceinline__ Extras LoadExtras(const ConvParams& p, const float* bias,
                                             const float* residual, const float* y_act, int co,
                                             size_t at) {
  return {bias != nullptr ? bias[co] : 0.0F, residual != nullptr ? residual[at] : 0.0F,
          y_act != nullptr && p.out_act == kActSnake ? p.alpha_out[co] : 0.0F};
}
__device__ __forceinline__ void Finish(const ConvParams& p, const Extras& x, float* y,
                                       float* y_act, size_t at, float v) {
  v += x.bias;
  if (p.pre_act == kActGelu)
    v = Gelu(v);
  v += x.residual;
  if (y != nullptr)
    y[at] = v;
  if (y_act != nullptr)
    y_act[at] = p.out_act == kActElu ? Elu(v) : Snake(v, x.alpha, SnakeInverse(x.alpha));
}

// Weight (tap k, input j, output co) of a lead of packed weights: its parts'
// sum, exactly.
__device__ __forceinline__ float PackedWeight(const ConvUnit* w, int rows, int taps, int cin,
                                              int lead, int k, int j, int co) {
  const int log2 = taps == 1 ? 7 : 5;  // of ConvPad(taps)
  static_assert(ConvPad(1) == 128 && ConvPad(7) == 32, "padding");
  const int chunks = ((cin - 1) >> log2) + 1, steps = 1 << (log2 - 4);  // of 16, per chunk
  const int step =
      ((lead * chunks + (j >> log2)) * taps + k) * steps + ((j >> 4) & (steps - 1));
  const auto* at = reinterpret_cast<const std::uint16_t*>(
                       w + (static_cast<size_t>(step) * 6 + (j >> 3 & 1)) * rows + co) + (j & 7);
  float part[3];
#pragma unroll
  for (int s = 0; s < 3; ++s)
    part[s] = __builtin_bit_cast(
        float, static_cast<unsigned>(at[static_cast<size_t>(16 * s) * rows]) << 16);
  return __builtin_isfinite(part[0]) ? part[0] + (part[1] + part[2]) : part[0];
}

// One convolution sum (before its bias) from the operands themselves, in
// double. For sums whose split products are infinite or NaN: an operand is,
// or is a finite input too large for its first part (split.hpp), or the sum
// overflows. Such sums are rare, or many where a NaN has spread: one among
// the inputs is looked for first (an encode of 10 s with one in it: 98 ms
// without, now 18; 4.5 of finite samples).
__device__ __forceinline__ float WideSum(const ConvParams& p, int batch, int phase, int co, int m) {
  const float* x = p.x + batch * p.x_batch;
  const bool view = p.view_kernel != 0;
  const int channels = view ? p.channels : p.cin, taps = view ? p.view_kernel : p.taps;
  const int t0 = m * (view ? p.view_stride : 1) + p.first[phase], dilation = view ? 1 : p.dilation;
#pragma unroll 1
  for (int k = 0; k < taps; ++k) {
    const int t = t0 + k * dilation;
    if (t < 0 || t >= p.len_in)
      continue;
#pragma unroll 1
    for (int c0 = 0; c0 < channels; c0 += 8) {
      float zero = 0.0F;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float v = x[static_cast<size_t>(min(c0 + i, channels - 1)) * p.len_in + t];
        zero += v != v ? v : 0.0F;
      }
      if (zero != zero)
        return zero;
    }
  }
  double sum = 0.0;
#pragma unroll 1
  for (int k = 0; k < taps; ++k) {
    const int t = t0 + k * dilation;
    const bool inside = t >= 0 && t < p.len_in;
#pragma unroll 1
    for (int c = 0; c < channels && sum == sum; ++c) {
      float v = 0.0F;
      if (inside) {
        v = x[static_cast<size_t>(c) * p.len_in + t];
        if (p.alpha_in != nullptr)
          v = Snake(v, p.alpha_in[c], SnakeInverse(p.alpha_in[c]));
        if (p.in_act == kActElu)
          v = Elu(v);
      }
      sum += static_cast<double>(v) *
             PackedWeight(p.w, p.w_rows, p.taps, p.cin, p.phases > 1 ? phase : batch,
                          view ? 0 : k, view ? c * taps + k : c, co);
    }
  }
  return static_cast<float>(sum);
}

// The same of a residual unit's second convolution.
__device__ __forceinline__ float WideUnitSum(const ConvParams& p, int co, int m) {
  double sum = 0.0;
#pragma unroll 1
  for (int j = 0; j < p.cout && sum == sum; ++j) {
    const float v = Snake(WideSum(p, 0, 0, j, m) + p.bias[j], p.alpha_mid[j],
                          SnakeInverse(p.alpha_mid[j]));
    sum += static_cast<double>(v) * PackedWeight(p.w2, p.w_rows, 1, p.cout, 0, 0, j, co);
  }
  return static_cast<float>(sum);
}

// Four floats at any 4-byte address.
typedef float Unaligned4 __attribute__((ext_vector_type(4), aligned(4)));

// The six products of a step's one or two 32 x 32 blocks, part by part of the
// operand b, whose parts are read again for the next step (next(part)) as
// soon as they are done with. A product waits some 90 cycles for the one
// before it on the same accumulator but only 32 for the pipe, so two blocks
// (or, for a single one, two low accumulators) are multiplied in turn; the
// scheduling barriers keep the order, which the compiler would otherwise turn
// back into one chain after the other. other(k) is vector work to put behind
// product k.
template <int N, typename Next, typename Other>
__device__ __forceinline__ void Products(const uintx4* a, const uintx4 (*b)[3], floatx16* main,
                                         floatx16* low, Next&& next, Other&& other) {
  auto multiply = [&](int k, int i, int j, floatx16* sum) {
#pragma unroll
    for (int t = 0; t < N; ++t)
      sum[t] = MfmaBf16(a[i], b[t][j], sum[t]);
    other(k);
    __builtin_amdgcn_sched_barrier(0);
  };
  floatx16* second = N == 1 ? low + 1 : low;
  multiply(0, 0, 2, low);
  next(2);
  multiply(1, 0, 1, second);
  multiply(2, 1, 1, low);
  next(1);
  multiply(3, 0, 0, main);
  multiply(4, 1, 0, second);
  multiply(5, 2, 0, low);
  next(0);
}

// Work-group `id` of `count` to a tile such that each XCD (id % 8) has a run
// of consecutive tiles.
__device__ __forceinline__ int XcdTile(int id, int count) {
  const int xcd = id % kXcds, per = count / kXcds, more = count % kXcds;
  return xcd * per + min(xcd, more) + id / kXcds;
}

// Input channels per chunk of a tile (a divisor of the weights' padding): two
// work-groups' windows fit a CU's LDS.
constexpr int TileChunk(int taps, int columns) {
  return taps > 1 || columns > 64 ? 32 : columns == 64 ? 64 : 128;
}

// One float32 convolution as an implicit GEMM over bf16 triples (split.hpp):
// rows are output channels, columns output positions, the sum runs over
// chunks of 32 to 128 input channels x taps in steps of 16 channels. A wave
// owns 32 rows x NT blocks of 32 columns, WM x WN waves a work-group.
//
// The weights come split and in step order from memory (PackConvWeights):
// each wave reads its own rows' 16-byte operands straight into registers
// kAhead steps ahead, so they cost no LDS traffic and no barrier; with all
// waves on the same columns (WN = 1) nothing is read twice. The chunk's input
// window (the tile's positions plus the taps' spread) is fetched as float32
// while the previous chunk is multiplied, split once per work-group on its
// way to LDS as [part][8 channels][position] 16-byte units, and every tap
// reads the window at its own shift. One barrier per chunk: two LDS buffers,
// or one where there is one chunk.
//
// A residual unit's k1 convolution follows in the same work-group where one
// tile holds every channel (FUSED): the k7 results, biased and through their
// Snake, are split back into LDS as the second product's operand and never
// see memory. A transposed convolution (kUp) gives each wave one phase of the
// same 32 channels, so that the work-group's outputs are whole runs.
//
// VIEW reads the input through a strided window: K index j is tap j %
// view_kernel of channel j / view_kernel (an im2col that is never stored).
//
// Bound by the matrix cores (their pipes 58-69 % busy at the 1.9 GHz this
// work draws) at 128 channels and more; at 32 and 64 (27 and 41 %) by them,
// the activations' vector work and memory alike. At a 60 s signal: the k7
// convolutions of 256 and 512 channels 195 TFLOP/s of float32 products (87 on
// the float32 matrix cores), a residual unit of 128 / 64 / 32 channels 403 /
// 268 / 280 us where its two launches took 492 / 329 / 397, the transposed
// convolutions 202 us a launch where one phase per work-group, its outputs
// scattered, took 295.
// Splitting a chunk between its predecessor's products instead of before its
// own: one-tap layers of 768 to 3072 channels at 500 positions 22.3 -> 20.6
// and 28.8 -> 25.0 us, the transposed convolutions 230 -> 204 us a launch.
enum ConvKind : int { kPlain, kView, kFused, kUp };

template <int WM, int WN, int NT, int TAPS, int BUFS, ConvKind KIND>
__global__ __launch_bounds__(64 * WM * WN, 2) void ConvKernel(ConvParams p) {
  constexpr bool VIEW = KIND == kView, FUSED = KIND == kFused, UP = KIND == kUp;
  static_assert(!VIEW || TAPS == 1, "a view has its taps in K");
  static_assert(!UP || (TAPS == 2 && WN == 1), "a wave per phase");
  constexpr int kT = 64 * WM * WN;
  constexpr int S = UP ? WM : 1;  // output positions per position of the tile
  constexpr int BM = UP ? 32 : 32 * WM, BN = 32 * WN * NT;
  constexpr int kChunk = TileChunk(TAPS, BN);
  constexpr int kMaxWidth = BN + (TAPS == 1 ? 0 : UP ? 2 : TAPS == 2 ? 1 : kConvMaxSpan);
  constexpr int kSlots = (kChunk / 8 * kMaxWidth + kT - 1) / kT;
  constexpr int kMaxUnits = kSlots * kT;  // whole turns of the threads
  constexpr int kSubs = kChunk / 16;
  constexpr int kSteps = kSubs * TAPS;  // of 16 channels, per chunk
  // Steps the weights are loaded ahead: a narrow tile's short steps and large
  // weights need more.
  constexpr int kAhead = TAPS == 7 ? 2 : BN == 32 && TAPS == 1 ? 8 : UP || WM == 4 ? 4 : 2;
  static_assert(kSteps % kAhead == 0, "weight registers");
  // The tile's results pass through LDS on their way out, kOutRows rows of
  // channels at a time.
  constexpr int kRowFloats = BN * S + 4;
  constexpr int kLds0 = BUFS * 3 * kMaxUnits;
  constexpr int kOutRows = UP ? 16 : kLds0 * 4 / kRowFloats >= BM || BN == 32 ? BM
                                 : kLds0 * 4 / kRowFloats >= 64   ? 64
                                                                  : 32;
  constexpr int kLds1 = (kOutRows * kRowFloats + 3) / 4;
  constexpr int kLds = kLds0 > kLds1 ? kLds0 : kLds1;
  static_assert(!FUSED || 3 * BM / 8 * BN <= kLds, "the second operand's LDS");
  __shared__ uintx4 xs[kLds];

  // Work-group to tile: consecutive tiles, the positions of a row block, stay
  // on one XCD, whose cache then holds few of the weights. (The row blocks of
  // a position tile first, or that only where the input is the larger operand:
  // within 2 % at every layer but the linear ones of 768 channels, where rows
  // first are slower, 27.8 -> 33.2 us to 3072 channels at 500 positions.)
  const int tiles_n = (p.positions + BN - 1) / BN, tiles_m = (p.cout + BM - 1) / BM;
  int tile = XcdTile(blockIdx.x, gridDim.x);
  const int tile_n = tile % tiles_n;
  tile /= tiles_n;
  const int tile_m = tile % tiles_m;
  tile /= tiles_m;
  const int split = tile % p.splits;
  const int batch = tile / p.splits;
  const int chunks = (p.cin + kChunk - 1) / kChunk;
  const int c_begin = split * p.split_chunks;
  const int c_end = min(chunks, c_begin + p.split_chunks);
  const float* x = p.x + batch * p.x_batch;
  const int m0 = tile_n * BN;
  const int co0 = tile_m * BM;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int phase = UP ? wave : 0;
  const int rest = UP ? wave : batch;               // the weights' lead
  const int row = UP ? 0 : (wave / WN) * 32;        // first output channel of the wave
  const int col = (wave % WN) * 32 * NT;            // first position of the wave
  const int half = lane >> 5;                       // K half of the lane's operands
  const int l32 = lane & 31;
  const int dilation = TAPS == 1 ? 0 : p.dilation;
  const int width = TAPS <= 2 ? kMaxWidth : BN + (TAPS - 1) * dilation;
  const int units = kChunk / 8 * width;
  // The window's first column is the first phase's, the least of them.
  const int lo = p.first[0];
  const int shift = UP ? p.first[phase] - lo : 0;

  // Unit u = tid + q kT of a chunk's window: channels 8 (u / width) .. + 7
  // at window column u % width.
  int at[kSlots], group[kSlots];  // first input position, 8-channel group
  // Windows fetched ahead of the one multiplied: a one-tap chunk is over
  // before its successor's loads have come back.
  constexpr int kDepth = TAPS == 1 && NT <= 2 && BUFS == 2 ? 2 : 1;
  unsigned inside[kDepth][kSlots];  // bit i: channel i of the unit is a value
#pragma unroll
  for (int q = 0; q < kSlots; ++q) {
    const int u = min(tid + q * kT, units - 1);
    group[q] = u / width;
    const int m = m0 + u % width;
    if (VIEW) {
      at[q] = min(m, p.positions - 1) * p.view_stride + lo;  // columns past the last: not stored
    } else {
      const int t = m + lo;
#pragma unroll
      for (int d = 0; d < kDepth; ++d)
        inside[d][q] = t >= 0 && t < p.len_in ? 0xFFU : 0U;
      at[q] = min(max(t, 0), p.len_in - 1);
    }
  }
  float window[kDepth][kSlots][8];
  // Every wave issues the same number of loads on every path (clamped ones
  // where there is nothing to load): the compiler then waits for the weights
  // by counting past the window's loads instead of for all of them.
  auto fetch = [&](int chunk, int d) __attribute__((always_inline)) {
    auto& xr = window[d];
    if (VIEW) {
#pragma unroll
      for (int q = 0; q < kSlots; ++q) {
        const int j = chunk * kChunk + 8 * group[q];
        int c = j / p.view_kernel, k = j % p.view_kernel;
        unsigned mask = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int t = at[q] + k;
          if (t >= 0 && t < p.len_in && j + i < p.cin)
            mask |= 1U << i;
          const int cc = min(c, p.channels - 1);
          xr[q][i] = x[static_cast<size_t>(cc) * p.len_in + min(max(t, 0), p.len_in - 1)];
          if (++k == p.view_kernel) {
            k = 0;
            ++c;
          }
        }
        inside[d][q] = mask;
      }
    } else if ((chunk + 1) * kChunk <= p.cin) {
#pragma unroll
      for (int q = 0; q < kSlots; ++q) {
        const float* from =
            x + at[q] + static_cast<size_t>(chunk * kChunk + 8 * group[q]) * p.len_in;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          xr[q][i] = from[static_cast<size_t>(i) * p.len_in];
      }
    } else {
#pragma unroll
      for (int q = 0; q < kSlots; ++q) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          xr[q][i] = x[at[q] + static_cast<size_t>(min(chunk * kChunk + 8 * group[q] + i,
                                                       p.cin - 1)) * p.len_in];
      }
    }
  };
  // Window d to LDS in 4 kSlots slices of two values: mask, split, and with
  // a unit's last pair the unit's stores (past the window's units too, where
  // nothing reads).
  auto activate = [&](int chunk, int d) __attribute__((always_inline)) {
    if (p.alpha_in == nullptr && p.in_act == kActNone)
      return;
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
      const int j = chunk * kChunk + 8 * group[q];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int c = VIEW ? min((j + i) / p.view_kernel, p.channels - 1) : min(j + i, p.cin - 1);
        const float alpha = p.alpha_in != nullptr ? p.alpha_in[c] : 0.0F;
        float& v = window[d][q][i];
        if (p.alpha_in != nullptr)
          v = Snake(v, alpha, SnakeInverse(alpha));
        if (p.in_act == kActElu)
          v = Elu(v);
      }
    }
  };
  uintx4 part[3];
  unsigned mask = 0;
  auto slice = [&](int k, int chunk, int buf, int d) __attribute__((always_inline)) {
    const int q = k / 4, h = k % 4;
    if (TAPS == 7 && q == kSlots - 1 && wave * 64 + q * kT >= units)
      return;
    if (h == 0) {
      mask = inside[d][q];
      const int j = chunk * kChunk + 8 * group[q];
      if (!VIEW)
        mask &= 0xFFU >> min(max(j + 8 - p.cin, 0), 8);
    }
    floatx2 rest{(mask >> 2 * h & 1U) != 0U ? window[d][q][2 * h] : 0.0F,
                 (mask >> 2 * h & 2U) != 0U ? window[d][q][2 * h + 1] : 0.0F};
    part[0][h] = RoundPair(rest);
    rest = Rest(rest, part[0][h]);
    part[1][h] = RoundPair(rest);
    rest = Rest(rest, part[1][h]);
    part[2][h] = RoundPair(rest);
    if (h == 3) {
#pragma unroll
      for (int s = 0; s < 3; ++s)
        xs[(buf * 3 + s) * kMaxUnits + tid + q * kT] = part[s];
    }
  };

  // The weights of the wave's 32 rows, one step after the other.
  const size_t step_units = 6 * static_cast<size_t>(p.w_rows);
  const uintx4* w = reinterpret_cast<const uintx4*>(p.w) +
                    (static_cast<size_t>(rest) * ((p.cin + ConvPad(TAPS) - 1) / ConvPad(TAPS)) *
                         (ConvPad(TAPS) / 16 * TAPS) +
                     c_begin * kSteps) * step_units +
                    static_cast<size_t>(half) * p.w_rows + min(co0 + row + l32, p.w_rows - 1);
  auto load = [&](uintx4* a) {
#pragma unroll
    for (int s = 0; s < 3; ++s)
      a[s] = w[static_cast<size_t>(2 * s) * p.w_rows];
    w += step_units;
  };

  constexpr int kTurn = NT > 1 ? 2 : 1;  // blocks multiplied in turn
  floatx16 main[NT] = {}, low[NT > 1 ? NT : 2] = {};
  uintx4 a[kAhead][3], b[kTurn][3];
#pragma unroll
  for (int d = 0; d < kDepth; ++d)
    fetch(min(c_begin + d, c_end - 1), d);
#pragma unroll
  for (int i = 0; i < kAhead; ++i)
    load(a[i]);
  activate(c_begin, 0);
#pragma unroll
  for (int k = 0; k < 4 * kSlots; ++k)
    slice(k, c_begin, 0, 0);
  if (BUFS > 1)
    fetch(min(c_begin + kDepth, c_end - 1), 0);
  __syncthreads();
  // Multiplies a chunk; with `more`, splits the next one into the other
  // buffer between the products, whose pipe it leaves free (before them it
  // took as long as a one-tap chunk's products), and fetches another.
  auto multiply = [&](int chunk, int buf, bool more) __attribute__((always_inline)) {
    const int d = kDepth == 2 ? 1 - buf : 0;
    if (more)
      activate(chunk + 1, d);
    const uintx4* base = xs + buf * 3 * kMaxUnits + half * width + col + l32 + shift;
    // Part s of blocks i kTurn .. of a chunk: column block % NT of step / NT.
    auto read = [&](int i, int s) {
#pragma unroll
      for (int j = 0; j < kTurn; ++j) {
        const int step = (i * kTurn + j) / NT;
        b[j][s] = base[s * kMaxUnits + step % kSubs * 2 * width + step / kSubs * dilation +
                       32 * ((i * kTurn + j) % NT)];
      }
    };
    read(0, 2);
    read(0, 1);
    read(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    constexpr int kTurns = kSteps * NT / kTurn;
    // The slices go behind the last two thirds of the products, when the
    // window has arrived.
    constexpr int kSlices = 4 * kSlots, kFrom = kTurns * 2, kOver = kTurns * 6 - kFrom;
#pragma unroll
    for (int i = 0; i < kTurns; ++i) {
      const int t = i * kTurn % NT, step = i * kTurn / NT;
      Products<kTurn>(
          a[step % kAhead], b, main + t, low + t,
          [&](int s) {
            if (i + 1 < kTurns)
              read(i + 1, s);
          },
          [&](int k) {
            const int g = i * 6 + k - kFrom;
            if (!more || g < 0)
              return;
#pragma unroll
            for (int n = g * kSlices / kOver; n < (g + 1) * kSlices / kOver; ++n)
              slice(n, chunk + 1, 1 - buf, d);
          });
      if (t + kTurn == NT && (more || step + kAhead < kSteps))
        load(a[step % kAhead]);
    }
    if (more) {
      fetch(min(chunk + 1 + kDepth, c_end - 1), d);
      __syncthreads();
    }
  };
  if (BUFS == 1) {
    multiply(c_begin, 0, false);
  } else {
    int chunk = c_begin;
    for (; chunk + 2 < c_end; chunk += 2) {
      multiply(chunk, 0, true);
      multiply(chunk + 1, 1, true);
    }
    if (chunk + 1 < c_end) {
      multiply(chunk, 0, true);
      multiply(chunk + 1, 1, false);
    } else {
      multiply(chunk, 0, false);
    }
  }
  if (NT == 1)
    low[0] += low[1];

  // Element r of the accumulators: output channel row + 8 (r / 4) + 4 half +
  // r % 4, position col + 32 t + l32.
  const float* bias = p.bias != nullptr ? p.bias + batch * p.b_batch : nullptr;
  if (!FUSED && p.splits > 1) {
    // partial[batch or phase][split][co][m]
    float* part = p.partial + (static_cast<size_t>(rest) * p.splits + split) * p.cout * p.positions;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int m = m0 + col + 32 * t + l32;
#pragma unroll
      for (int r = 0; r < 16; ++r)
        main[t][r] += low[t][r];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int co = co0 + row + 8 * (r >> 2) + 4 * half + (r & 3);
        if (m < p.positions && co < p.cout)
          part[static_cast<size_t>(co) * p.positions + m] = main[t][r];
      }
    }
    return;
  }

  if (FUSED) {
    // The second convolution: 8 channels of a position are the 4 + 4 of a
    // lane pair.
    const uintx4* w2 = reinterpret_cast<const uintx4*>(p.w2) +
                       static_cast<size_t>(half) * p.w_rows + min(row + l32, p.w_rows - 1);
    auto load2 = [&](int step, uintx4* v) {
#pragma unroll
      for (int s = 0; s < 3; ++s)
        v[s] = w2[(static_cast<size_t>(step) * 6 + 2 * s) * p.w_rows];
    };
    load2(0, a[0]);
    __syncthreads();
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float bias4[4], alpha4[4], inverse4[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int co = min(row + 8 * g + 4 * half + r, p.cout - 1);
        bias4[r] = bias[co];
        alpha4[r] = p.alpha_mid[co];
        inverse4[r] = SnakeInverse(alpha4[r]);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          v[r] = Snake((main[t][4 * g + r] + low[t][4 * g + r]) + bias4[r], alpha4[r],
                       inverse4[r]);
          v[r] = row + 8 * g + 4 * half + r < p.cout ? v[r] : 0.0F;
        }
        floatx2 rest0{v[0], v[1]}, rest1{v[2], v[3]};
        auto* to = reinterpret_cast<uintx2*>(xs + (row / 8 + g) * BN + col + 32 * t + l32) + half;
#pragma unroll
        for (int s = 0; s < 3; ++s) {
          const uintx2 pairs{RoundPair(rest0), RoundPair(rest1)};
          to[s * 2 * (BM / 8 * BN)] = pairs;
          rest0 = Rest(rest0, pairs[0]);
          rest1 = Rest(rest1, pairs[1]);
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t)
      main[t] = low[t] = floatx16{};
    const uintx4* base = xs + half * BN + col + l32;
    static_assert(!FUSED || NT == kTurn, "a step is one turn of blocks");
    if (NT == 1)
      low[1] = floatx16{};
    auto read = [&](int step, int s) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        b[t][s] = base[s * (BM / 8 * BN) + 2 * step * BN + 32 * t];
    };
    read(0, 2);
    read(0, 1);
    read(0, 0);
#pragma unroll
    for (int step = 0; step < BM / 16; ++step) {
      if (step + 1 < BM / 16)
        load2(step + 1, a[(step + 1) & 1]);
      Products<kTurn>(
          a[step & 1], b, main, low,
          [&](int s) {
            if (step + 1 < BM / 16)
              read(step + 1, s);
          },
          [](int) {});
    }
    if (NT == 1)
      low[0] += low[1];
    bias = p.bias2;
  }

  // Out through LDS, as rows of positions, then in a loop over 16-byte runs:
  // the residual loads and the stores are wide, and the code that every
  // work-group runs once, and has to fetch, is short (straight from the
  // accumulators it was most of the kernel). Four runs at a time, the next
  // four's loads issued before these four's stores, which may alias them as
  // far as the compiler knows.
  float* y = p.y != nullptr ? p.y + batch * p.y_batch : nullptr;
  float* y_act = p.y_act != nullptr ? p.y_act + batch * p.y_batch : nullptr;
  const float* residual =
      !UP && p.residual != nullptr ? p.residual + batch * p.y_batch : nullptr;
  constexpr int kRuns = BN * S / 4;      // per row
  constexpr int kStride = kT / kRuns;    // rows between a thread's runs
  constexpr int kPer = kOutRows / kStride / 4;
  static_assert(kT % kRuns == 0 && kOutRows % (4 * kStride) == 0, "runs");
  const int length = p.positions * S;
  const int at0 = m0 * S + tid % kRuns * 4;  // the thread's first output position
  const int n = min(length - at0, 4);
  struct Runs {
    float bias[4], alpha[4];
    floatx4 residual[4];
  };
  auto gather = [&](int first) __attribute__((always_inline)) {
    Runs v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int co = min(co0 + first + i * kStride, p.cout - 1);
      v.bias[i] = bias != nullptr ? bias[co] : 0.0F;
      v.alpha[i] = y_act != nullptr && p.out_act == kActSnake ? p.alpha_out[co] : 0.0F;
      v.residual[i] = floatx4{0.0F, 0.0F, 0.0F, 0.0F};
      if (residual != nullptr && n > 0) {
        const float* from = residual + static_cast<size_t>(co) * p.len_out + at0;
        if (n == 4)
          v.residual[i] = *reinterpret_cast<const Unaligned4*>(from);
        else
          for (int e = 0; e < n; ++e)
            v.residual[i][e] = from[e];
      }
    }
    return v;
  };
  float* out = reinterpret_cast<float*>(xs);
#pragma unroll
  for (int r0 = 0; r0 < BM; r0 += kOutRows) {
    const int mine = r0 + tid / kRuns;
    Runs next = gather(mine);
    __syncthreads();
    if (UP) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 8; ++r)
          out[(8 * (r >> 2) + 4 * half + (r & 3)) * kRowFloats + (32 * t + l32) * S + phase] =
              main[t][r0 / 2 + r] + low[t][r0 / 2 + r];
    } else if (row >= r0 && row < r0 + kOutRows) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          out[(row - r0 + 8 * (r >> 2) + 4 * half + (r & 3)) * kRowFloats + col + 32 * t + l32] =
              main[t][r] + low[t][r];
    }
    __syncthreads();
    bool wide = false;
    // Four runs, and whether all of them are finite.
    auto run = [&](int q, int i) __attribute__((always_inline)) {
      return *reinterpret_cast<const floatx4*>(
          out + (mine - r0 + (4 * q + i) * kStride) * kRowFloats + tid % kRuns * 4);
    };
    auto check = [](floatx4 v, floatx4* zero) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        (*zero)[e] = fmaf(v[e], 0.0F, (*zero)[e]);
    };
    auto finite = [](floatx4 zero) __attribute__((always_inline)) {
      return (zero[0] + zero[1]) + (zero[2] + zero[3]) == 0.0F;
    };
#pragma unroll 1
    for (int q = 0; q < kPer; ++q) {
      const Runs cur = next;
      if (q + 1 < kPer)
        next = gather(mine + 4 * (q + 1) * kStride);
      // Four runs are left out where one is not finite, since y may be the
      // residual; phases have none, and none to leave out.
      floatx4 sums[4], zero = {0.0F, 0.0F, 0.0F, 0.0F};
      if (!UP) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          sums[i] = run(q, i);
          check(sums[i], &zero);
        }
        if (__builtin_expect(!finite(zero), 0)) {
          wide = true;
          continue;
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int local = mine + (4 * q + i) * kStride;
        if (co0 + local >= p.cout || n <= 0)
          continue;
        floatx4 v = UP ? run(q, i) : sums[i];
        if (UP)
          check(v, &zero);
        const size_t to = static_cast<size_t>(co0 + local) * p.len_out + at0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] += cur.bias[i];
          if (p.pre_act == kActGelu)
            v[e] = Gelu(v[e]);
          v[e] += cur.residual[i][e];
        }
        if (y != nullptr) {
          if (n == 4)
            *reinterpret_cast<Unaligned4*>(y + to) = v;
          else
            for (int e = 0; e < n; ++e)
              y[to + e] = v[e];
        }
        if (y_act != nullptr) {
          const float inverse = SnakeInverse(cur.alpha[i]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[e] = p.out_act == kActElu ? Elu(v[e]) : Snake(v[e], cur.alpha[i], inverse);
          if (n == 4)
            *reinterpret_cast<Unaligned4*>(y_act + to) = v;
          else
            for (int e = 0; e < n; ++e)
              y_act[to + e] = v[e];
        }
      }
      if (UP)
        wide |= !finite(zero);
    }
    // The sums that are not finite are formed again, and their fours finished.
    if (__builtin_expect(wide, 0)) {
      const ConvParams& wp = ParamsAgain<ConvParams>();
#pragma unroll 1
      for (int q = 0; q < kPer; ++q) {
        floatx4 zero = {0.0F, 0.0F, 0.0F, 0.0F};
#pragma unroll
        for (int i = 0; i < 4; ++i)
          check(run(q, i), &zero);
        if (finite(zero))
          continue;
#pragma unroll 1
        for (int k = 0; k < 16; ++k) {
          const int local = mine + (4 * q + k / 4) * kStride, t = at0 + k % 4;
          const int co = co0 + local;
          if (co >= wp.cout || k % 4 >= n)
            continue;
          float v = out[(local - r0) * kRowFloats + tid % kRuns * 4 + k % 4];
          if (!__builtin_isfinite(v))
            v = FUSED ? WideUnitSum(wp, co, t) : WideSum(wp, batch, UP ? t % S : 0, co, t / S);
          const size_t at = static_cast<size_t>(co) * wp.len_out + t;
          Finish(wp, LoadExtras(wp, bias, residual, y_act, co, at), y, y_act, at, v);
        }
      }
    }
  }
}

// Splits float32 weights [lead][taps][cin][cout] into the operands the
// kernel reads, [lead][chunk][tap][step][part 3][half 2][w_rows] units of
// eight channels, zero past cin and cout.
__global__ __launch_bounds__(kThreads) void PackConvWeightsKernel(const float* w, int lead, int taps,
                                                                  int cin, int cout, int rows,
                                                                  uintx4* out) {
  const int groups = ConvPad(taps) / 8;
  const int chunks = (cin + ConvPad(taps) - 1) / ConvPad(taps);
  const size_t total = static_cast<size_t>(lead) * chunks * taps * groups * rows;
  for (size_t e = static_cast<size_t>(blockIdx.x) * kThreads + threadIdx.x; e < total;
       e += static_cast<size_t>(gridDim.x) * kThreads) {
    const int o = static_cast<int>(e % rows);
    size_t at = e / rows;
    const int g = static_cast<int>(at % groups);  // step x half
    at /= groups;
    const int tap = static_cast<int>(at % taps);
    const int chunk = static_cast<int>(at / taps % chunks);
    const size_t ld = at / taps / chunks;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int c = chunk * ConvPad(taps) + 8 * g + i;
      v[i] = c < cin && o < cout ? w[((ld * taps + tap) * cin + c) * cout + o] : 0.0F;
    }
    uintx4 part[3];
    Split8<true>(v, part);
    uintx4* to = out + (at * (groups / 2) + (g >> 1)) * 6 * rows + (g & 1) * static_cast<size_t>(rows) + o;
#pragma unroll
    for (int s = 0; s < 3; ++s)
      to[static_cast<size_t>(2 * s) * rows] = part[s];
  }
}

// Sums the split-K partials of every output in split order, then the
// convolution's epilogue.
__global__ __launch_bounds__(kThreads) void SplitReduceKernel(ConvParams p) {
  const size_t per = static_cast<size_t>(p.cout) * p.positions;
  const size_t total = per * p.batches * p.phases;
  for (size_t e = static_cast<size_t>(blockIdx.x) * kThreads + threadIdx.x; e < total;
       e += static_cast<size_t>(gridDim.x) * kThreads) {
    const int rest = static_cast<int>(e / per);
    const size_t within = e % per;
    const int co = static_cast<int>(within / p.positions);
    const int m = static_cast<int>(within % p.positions);
    const int phase = rest % p.phases, batch = rest / p.phases;
    const float* bias = p.bias != nullptr ? p.bias + batch * p.b_batch : nullptr;
    float* y = p.y != nullptr ? p.y + batch * p.y_batch : nullptr;
    float* y_act = p.y_act != nullptr ? p.y_act + batch * p.y_batch : nullptr;
    const float* residual = p.residual != nullptr ? p.residual + batch * p.y_batch : nullptr;
    const size_t at = static_cast<size_t>(co) * p.len_out + static_cast<size_t>(m) * p.phases + phase;
    const Extras extras = LoadExtras(p, bias, residual, y_act, co, at);
    const float* part = p.partial + static_cast<size_t>(rest) * p.splits * per + within;
    float v = 0.0F;
#pragma unroll 8
    for (int s = 0; s < p.splits; ++s)
      v += part[static_cast<size_t>(s) * per];
    if (__builtin_expect(!__builtin_isfinite(v), 0))
      v = WideSum(ParamsAgain<ConvParams>(), batch, phase, co, m);
    Finish(p, extras, y, y_act, at, v);
  }
}

// Four outputs a thread from a register window of 4 + taps - 1 samples per
// channel, read in 16-byte runs whose overlaps stay in the caches; the waves
// of a work-group take a quarter of the channels each, eight in flight, and
// meet in LDS. Bound by memory at long signals (with a work-group's window in
// LDS and one read per product 60 s of 32 channels, 184 MB, took 131 us), by
// one round trip to it at short ones.
template <int TAPS>
__global__ __launch_bounds__(kThreads) void OutputConvKernel(OutputConvParams p) {
  constexpr int kPad = (TAPS - 1) / 2, kRuns = (4 + TAPS - 1 + 3) / 4;
  constexpr int kWaves = kThreads / 64;
  __shared__ floatx4 sums[kWaves][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int t0 = blockIdx.x * kOutTile + lane * 4;
  const int per = (p.cin + kWaves - 1) / kWaves;
  const int c_end = min(p.cin, (wave + 1) * per);
  const bool inside = t0 >= kPad && t0 - kPad + 4 * kRuns <= p.length;
  floatx4 sum = {0.0F, 0.0F, 0.0F, 0.0F};
#pragma unroll 8
  for (int c = wave * per; c < c_end; ++c) {
    const float* row = p.x + static_cast<size_t>(c) * p.length;
    float v[4 * kRuns];
    if (inside) {
#pragma unroll
      for (int r = 0; r < kRuns; ++r)
        *reinterpret_cast<floatx4*>(v + 4 * r) =
            *reinterpret_cast<const Unaligned4*>(row + t0 - kPad + 4 * r);
    } else {
#pragma unroll
      for (int i = 0; i < 4 * kRuns; ++i) {
        const int t = t0 - kPad + i;
        const float sample = row[min(max(t, 0), p.length - 1)];
        v[i] = t >= 0 && t < p.length ? sample : 0.0F;
      }
    }
#pragma unroll
    for (int k = 0; k < TAPS; ++k)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        sum[e] += p.w[k * p.cin + c] * v[e + k];
  }
  sums[wave][lane] = sum;
  __syncthreads();
  const int t = blockIdx.x * kOutTile + threadIdx.x;
  if (t < p.length) {
    float v = 0.0F;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      v += sums[w][threadIdx.x / 4][threadIdx.x % 4];
    p.y[t] = v + p.bias[0];
  }
}

__global__ __launch_bounds__(kThreads) void RvqKernel(RvqParams p) {
  const int f = blockIdx.x;
  for (int o = threadIdx.x; o < p.latent; o += kThreads) {
    float v = 0.0F;
    for (int c = 0; c < p.codebooks; ++c) {
      // Codes were range-checked by the host; the clamp keeps a bad device
      // input inside the table.
      const int code = min(max(p.codes[static_cast<size_t>(c) * p.frames + f], 0),
                           p.entries - 1);
      v += p.table[(static_cast<size_t>(c) * p.entries + code) * p.latent + o];
    }
    p.y[static_cast<size_t>(o) * p.frames + f] = v + p.bias[o];
  }
}

template <int WM, int WN, int NT, int TAPS, int BUFS, ConvKind KIND>
void DispatchTile(const ConvParams& p, hipStream_t stream) {
  constexpr int BM = KIND == kUp ? 32 : 32 * WM, BN = 32 * WN * NT;
  const int64_t grid = static_cast<int64_t>((p.positions + BN - 1) / BN) *
                       ((p.cout + BM - 1) / BM) * p.batches * p.splits;
  Require(grid < (int64_t{1} << 31), "conv: too many tiles");
  Dispatch(ConvKernel<WM, WN, NT, TAPS, BUFS, KIND>, dim3(static_cast<unsigned>(grid)),
           dim3(64 * WM * WN), 0, stream, true, p.splits == 1, p);
}

// Splits the input channels of a convolution of `tiles` work-groups until
// about `target` run, at least two chunks and at most `most` splits, if there
// is a workspace.
void ChooseSplits(ConvParams* p, int64_t tiles, int chunk, int64_t target, int most) {
  const int chunks = (p->cin + chunk - 1) / chunk;
  p->splits = 1;
  p->split_chunks = chunks;
  if (p->partial == nullptr)
    return;
  int64_t want = std::min<int64_t>(target / tiles, std::min(most, chunks / 2));
  const int64_t outputs = static_cast<int64_t>(p->cout) * p->positions * p->phases * p->batches;
  want = std::min<int64_t>(want, p->partial_capacity / std::max<int64_t>(outputs, 1));
  want = std::min<int64_t>(want, 65535 / (static_cast<int64_t>(p->phases) * p->batches));
  if (want >= 2) {
    p->split_chunks = static_cast<int>((chunks + want - 1) / want);
    p->splits = (chunks + p->split_chunks - 1) / p->split_chunks;
  }
}

void Reduce(const ConvParams& p, hipStream_t stream) {
  if (p.splits == 1)
    return;
  const size_t total = static_cast<size_t>(p.cout) * p.positions * p.phases * p.batches;
  const int blocks = static_cast<int>(std::min<size_t>((total + kThreads - 1) / kThreads, 16384));
  Dispatch(SplitReduceKernel, dim3(blocks), dim3(kThreads), 0, stream, false, true, p);
}

int64_t Tiles(const ConvParams& p, int bm, int bn) {
  return static_cast<int64_t>((p.positions + bn - 1) / bn) * ((p.cout + bm - 1) / bm) * p.batches;
}

// The tile and the splits. All output channels of a narrow layer: 32 x 256
// when the input is one chunk, so that two work-groups' windows fit a CU's
// LDS, else 32 x 128; 64 x 128; about 512 work-groups.
//
// Wider layers take 128 x 64, or 128 x 32 where that keeps the CUs as busy.
// One tap: up to three narrow tiles a CU cost as much as one wide one, or less
// than two (768 -> 3072 channels: 216 wide tiles 25.6 us and 25.4 narrow, 264
// 36.8 and 35.2, 384 39.7 and 38.6, 408 40.3 and 45.6; 3072 -> 768: 360 128
// and 126, 390 131 and 154; 512 x 3 taps of a view: 200 59.7 and 53.4, 328
// 89.3 and 82.5, 392 92.7 and 101). Seven taps, with splits: wide ones once
// they and their splits number the CUs; without: one narrow tile a CU (512
// channels: 128 wide tiles 64.8 us and 55.4 narrow, 200 70.6 and 78.2), two
// where the sum is short (32 channels: 200 11.6 and 10.8, 256 12.2 and 11.9,
// 300 15.4 and 15.6, 512 17.4 and 19.8).
//
// A split costs a pass of partial sums, so it only has to give each CU one
// work-group, unless the sums are so long (over 512 channels x 7 taps) that
// three balance better. Measured at one tap: 768 -> 3072 channels x 500 20.6
// us at 384 tiles of 128 x 32, 29-30 split in two; 768 -> 768 at 150
// positions 15.0 at 30 tiles, 11.9 and 10.7 split in two and three. At seven
// taps: 512 channels x 2000 positions 63.6 at 128 tiles of 128 x 64, 43.4,
// 44.9, 48.0 split in two, four, six; x 200 positions 16.4 (16 tiles, eight
// splits) and 13.8 (28 tiles of 128 x 32, eight); 1024 x 750 65.7 at two
// splits of 96 tiles, 57.8 at five, 54.3 at eight. 128 x 128 tiles were
// slower at every size (512 x 12000, seven taps: 191 to 160).
template <int TAPS, ConvKind KIND>
void DispatchTaps(const ConvParams& params, hipStream_t stream) {
  ConvParams p = params;
  if (p.cout <= 64) {
    const bool one = p.cin <= 32;
    const int rows = p.cout <= 32 ? 32 : 64, columns = rows == 32 && one ? 256 : 128;
    const int64_t tiles = Tiles(p, rows, columns);
    ChooseSplits(&p, tiles, TileChunk(TAPS, columns), tiles < 256 ? 512 + tiles - 1 : 1, 65535);
    if (rows == 32 && one)
      DispatchTile<1, 4, 2, TAPS, 1, KIND>(p, stream);
    else if (rows == 32)
      DispatchTile<1, 4, 1, TAPS, 2, KIND>(p, stream);
    else
      DispatchTile<2, 2, 2, TAPS, 2, KIND>(p, stream);
  } else {
    const int64_t tiles = Tiles(p, 128, 64);
    const int most = TAPS == 7 ? 8 : 65535;
    const int splits = p.partial == nullptr ? 1 : std::min(most, (p.cin + 31) / 32 / 2);
    const bool wide = TAPS == 1    ? Tiles(p, 128, 32) > 3 * kCus
                      : splits > 1 ? tiles * splits >= kCus
                                   : Tiles(p, 128, 32) > (p.cin <= 64 ? 2 : 1) * kCus;
    ChooseSplits(&p, wide ? tiles : Tiles(p, 128, 32), TileChunk(TAPS, wide ? 64 : 32),
                 TAPS == 7 && p.cin > 512 ? 768 : 256, most);
    if (wide)
      DispatchTile<4, 1, 2, TAPS, 2, KIND>(p, stream);
    else
      DispatchTile<4, 1, 1, TAPS, 2, KIND>(p, stream);
  }
  Reduce(p, stream);
}

// A residual unit of up to 128 channels in one launch. Half the columns where
// the wider tile leaves CUs idle: 24000 samples of 32 channels 18.5 -> 13.3 us,
// 8000 of 64 22.3 -> 16.8, 4000 of 128 29.9 -> 23.3; at 60 s the wider tile is
// 15-25 % faster, but for the one chunk of 32 channels, where the narrow one
// leaves LDS for more work-groups (301 -> 282 us).
void DispatchFused(const ConvParams& params, hipStream_t stream) {
  ConvParams p = params;
  ChooseSplits(&p, 1, 32, 1, 1);
  const auto few = [&](int columns) { return Tiles(p, 128, columns) < 256; };
  if (p.cout <= 32)
    DispatchTile<1, 4, 1, 7, 1, kFused>(p, stream);
  else if (p.cout <= 64 && few(128))
    DispatchTile<2, 2, 1, 7, 2, kFused>(p, stream);
  else if (p.cout <= 64)
    DispatchTile<2, 2, 2, 7, 2, kFused>(p, stream);
  else if (few(64))
    DispatchTile<4, 1, 1, 7, 2, kFused>(p, stream);
  else
    DispatchTile<4, 1, 2, 7, 2, kFused>(p, stream);
}

// A transposed convolution: a wave per phase.
void DispatchUp(const ConvParams& params, hipStream_t stream) {
  ConvParams p = params;
  const int64_t tiles = Tiles(p, 32, 64);
  ChooseSplits(&p, tiles, 32, tiles < 256 ? 512 + tiles - 1 : 1, 65535);
  switch (p.phases) {
    case 2: DispatchTile<2, 1, 2, 2, 2, kUp>(p, stream); break;
    case 3: DispatchTile<3, 1, 2, 2, 2, kUp>(p, stream); break;
    case 4: DispatchTile<4, 1, 2, 2, 2, kUp>(p, stream); break;
    case 5: DispatchTile<5, 1, 2, 2, 2, kUp>(p, stream); break;
    case 6: DispatchTile<6, 1, 2, 2, 2, kUp>(p, stream); break;
    case 7: DispatchTile<7, 1, 2, 2, 2, kUp>(p, stream); break;
    default: DispatchTile<8, 1, 2, 2, 2, kUp>(p, stream); break;
  }
  Reduce(p, stream);
}

}  // namespace

std::size_t ConvWeightUnits(int lead, int taps, int cin, int cout) {
  return static_cast<std::size_t>(lead) * taps * ((cin + ConvPad(taps) - 1) / ConvPad(taps)) *
         (ConvPad(taps) / 8 * 3) * ConvRows(cout);
}

void LaunchPackConvWeights(const float* w, int lead, int taps, int cin, int cout, ConvUnit* out,
                           hipStream_t stream) {
  Require(w && out, "conv weights: null pointer");
  Require(lead >= 1 && taps >= 1 && cin >= 1 && cout >= 1, "conv weights: empty shape");
  const std::size_t total = ConvWeightUnits(lead, taps, cin, cout) / 3;
  Dispatch(PackConvWeightsKernel,
           dim3(static_cast<unsigned>(std::min<std::size_t>((total + kThreads - 1) / kThreads, 16384))),
           dim3(kThreads), 0, stream, true, true, w, lead, taps, cin, cout, ConvRows(cout),
           reinterpret_cast<uintx4*>(out));
}

void LaunchConv(const ConvParams& params, hipStream_t stream) {
  ConvParams p = params;
  if (p.batches == 0)
    p.batches = 1;
  if (p.out_act == kActNone)
    p.out_act = kActSnake;
  p.w_rows = ConvRows(p.cout);
  Require(p.x && p.w, "conv: null pointer");
  Require(p.y != nullptr || p.y_act != nullptr, "conv: no output");
  Require(p.y_act == nullptr || p.out_act != kActSnake || p.alpha_out != nullptr,
          "conv: activated output needs alpha");
  Require(p.pre_act == kActNone || p.pre_act == kActGelu, "conv: bad pre-activation");
  Require(p.in_act == kActNone || p.in_act == kActElu, "conv: bad input activation");
  Require(p.out_act == kActSnake || p.out_act == kActElu, "conv: bad output activation");
  Require(p.batches >= 1 && static_cast<int64_t>(p.batches) * p.phases <= 65535,
          "conv: 1 to 65535 batches x phases");
  Require(p.batches == 1 || (p.x_batch >= 0 && p.b_batch >= 0 && p.y_batch >= 0),
          "conv: negative batch stride");
  Require(p.cin >= 1 && p.cout >= 1 && p.len_in >= 1 && p.positions >= 1,
          "conv: empty shape");
  Require(p.taps == 1 || p.taps == 2 || p.taps == 7, "conv: 1, 2 or 7 taps");
  Require(p.phases >= 1 && p.phases <= kConvMaxPhases, "conv: 1 to 8 phases");
  Require(p.phases == 1 || (p.taps == 2 && p.batches == 1 && p.residual == nullptr),
          "conv: phases have two taps and no residual");
  for (int i = 1; i < p.phases; ++i)
    Require(p.first[i] - p.first[0] == 0 || p.first[i] - p.first[0] == 1,
            "conv: the phases' windows differ by one position at most");
  Require(static_cast<int64_t>(p.positions) * p.phases <= p.len_out,
          "conv: output positions past the output length");
  Require(p.taps == 1 || (p.dilation >= 1 &&
                          (p.taps - 1) * static_cast<int64_t>(p.dilation) <=
                              (p.taps == 2 ? 1 : kConvMaxSpan)),
          "conv: taps spread too far for their count");
  if (p.view_kernel != 0) {
    Require(p.taps == 1 && p.phases == 1, "conv: a view has one tap and phase");
    Require(p.view_kernel >= 1 && p.view_stride >= 1 && p.channels >= 1 &&
                static_cast<int64_t>(p.channels) * p.view_kernel == p.cin &&
                (p.positions - int64_t{1}) * p.view_stride + p.view_kernel <
                    (std::int64_t{1} << 31),
            "conv: bad view");
    DispatchTaps<1, kView>(p, stream);
  } else if (p.w2 != nullptr) {
    Require(p.taps == 7 && p.batches == 1 && p.cin == p.cout && p.cout <= kConvFusedChannels &&
                p.bias != nullptr && p.bias2 != nullptr && p.alpha_mid != nullptr &&
                p.pre_act == kActNone && p.x != p.y && p.x != p.y_act,
            "conv: bad residual unit");
    DispatchFused(p, stream);
  } else if (p.phases > 1) {
    DispatchUp(p, stream);
  } else if (p.taps == 1) {
    DispatchTaps<1, kPlain>(p, stream);
  } else if (p.taps == 2) {
    DispatchTaps<2, kPlain>(p, stream);
  } else {
    DispatchTaps<7, kPlain>(p, stream);
  }
}

void LaunchOutputConv(const OutputConvParams& p, hipStream_t stream) {
  Require(p.x && p.w && p.bias && p.y, "output conv: null pointer");
  Require(p.cin >= 1 && p.length >= 1, "output conv: empty shape");
  Require(p.taps >= 1 && p.taps <= kConvMaxTaps && p.taps % 2 == 1,
          "output conv: 1, 3, 5 or 7 taps");
  const dim3 grid(static_cast<unsigned>((p.length + int64_t{kOutTile} - 1) / kOutTile));
  auto launch = [&](auto* kernel) {
    Dispatch(kernel, grid, dim3(kThreads), 0, stream, true, true, p);
  };
  switch (p.taps) {
    case 1: launch(OutputConvKernel<1>); break;
    case 3: launch(OutputConvKernel<3>); break;
    case 5: launch(OutputConvKernel<5>); break;
    default: launch(OutputConvKernel<7>); break;
  }
}

void LaunchRvq(const RvqParams& p, hipStream_t stream) {
  Require(p.table && p.bias && p.codes && p.y, "rvq: null pointer");
  Require(p.codebooks >= 1 && p.entries >= 1 && p.latent >= 1 && p.frames >= 1,
          "rvq: empty shape");
  Dispatch(RvqKernel, dim3(p.frames), dim3(kThreads), 0, stream, true, true, p);
}

}  // namespace ovg
