// The audio decoder's kernels on gfx950 (replacing the reference's
// hipblasSgemm calls and element-wise kernels of the DAC decoder:
// codec_state.hpp:232-300, kernels/codec_kernels.hip:11-84).
//
// Every convolution is one implicit GEMM: output channels x output positions,
// summed over input channels x taps, each float32 product as six products of
// bf16 parts (split.hpp). Bias, activations and the residual addition are
// applied in the epilogue, straight from the accumulators. The sums are
// nearer to the exact ones than the float32 matrix cores' (the decoder's
// audio 1.2-2.1e-6 from 64 bits where those gave 1.9-4.6e-6).
#include "codec.hpp"
#include "common.hpp"
#include "kernels.hpp"
#include "split.hpp"

namespace ovg {
namespace {

constexpr int kThreads = 256;
constexpr int kOutTile = 256;  // samples per work-group of the output conv
constexpr int kOutChunk = 32;  // input channels per chunk of the output conv

// kernels/codec_kernels.hip:20-22 of the reference: v + sin^2(a v) / (a + 1e-9),
// with 1 / (a + 1e-9) given. x = a v less its nearest multiple of pi (pi in
// three parts; the first difference is exact, both terms being multiples of
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
  r = fmaf(n, 3.4302490902798e-15F, r);
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
// the stores.
__device__ __forceinline__ void Finish(const ConvParams& p, const float* bias,
                                       const float* residual, float* y, float* y_act, int co,
                                       size_t at, float v) {
  if (bias != nullptr)
    v += bias[co];
  if (p.pre_act == kActGelu)
    v = Gelu(v);
  if (residual != nullptr)
    v += residual[at];
  if (y != nullptr)
    y[at] = v;
  if (y_act != nullptr)
    y_act[at] = p.out_act == kActElu ? Elu(v) : Snake(v, p.alpha_out[co], SnakeInverse(p.alpha_out[co]));
}

// Work-group `id` of `count` to a tile such that each XCD (id % 8) has a run
// of consecutive tiles.
__device__ __forceinline__ int XcdTile(int id, int count) {
  const int xcd = id % kXcds, per = count / kXcds, more = count % kXcds;
  return xcd * per + min(xcd, more) + id / kXcds;
}

// Input channels per chunk of a tile (a divisor of the weights' padding): two
// work-groups' windows fit a CU's LDS.
constexpr int TileChunk(int taps, int columns) { return taps == 1 && columns <= 64 ? 64 : 32; }

// One float32 convolution as an implicit GEMM over bf16 triples (split.hpp):
// rows are output channels, columns output positions, the sum runs over
// chunks of 32 or 64 input channels x taps in steps of 16 channels. A wave owns 32
// rows x NT blocks of 32 columns, WM x WN waves a work-group.
//
// The weights come split and in step order from memory (PackConvWeights):
// each wave reads its own rows' 16-byte operands straight into registers
// some 1500 cycles of products ahead, so they cost no LDS traffic and no barrier; with all waves on
// one row block of columns (WN = 1) nothing is read twice. The chunk's input
// window (the tile's positions plus the taps' spread) is fetched as float32
// while the previous chunk is multiplied, split once per work-group on its
// way to LDS as [part][8 channels][position] 16-byte units, and every tap
// reads the window at its own shift. One barrier per chunk: two LDS buffers,
// or one where there is one chunk.
//
// VIEW reads the input through a strided window: K index j is tap j % view_kernel of channel j /
// view_kernel (an im2col that is never stored).
template <int WM, int WN, int NT, int TAPS, int BUFS, bool VIEW>
__global__ __launch_bounds__(kThreads, 2) void ConvKernel(ConvParams p) {
  static_assert(WM * WN * 64 == kThreads, "four waves");
  static_assert(!VIEW || TAPS == 1, "a view has its taps in K");
  constexpr int BM = 32 * WM, BN = 32 * WN * NT;
  constexpr int kMaxWidth = BN + (TAPS == 1 ? 0 : TAPS == 2 ? 1 : kConvMaxSpan);
  constexpr int kChunk = TileChunk(TAPS, BN);
  constexpr int kMaxUnits = kChunk / 8 * kMaxWidth;
  constexpr int kSlots = (kMaxUnits + kThreads - 1) / kThreads;
  constexpr int kSubs = kChunk / 16;
  constexpr int kSteps = kSubs * TAPS;  // of 16 channels, per chunk
  // Steps the weights are loaded ahead: a narrow tile's short steps and large
  // weights need more.
  constexpr int kAhead = WM < 4 || NT == 4 ? 2 : TAPS == 7 ? 7 : 4;
  static_assert(kSteps % kAhead == 0, "weight registers");
  __shared__ uintx4 xs[BUFS][3][kMaxUnits];

  // Work-group to tile: consecutive tiles stay on one XCD, the
  // positions of a row block where the weights are the larger operand, the
  // row blocks of a position tile where the input is, so that the XCDs'
  // caches do not all hold the larger one.
  const int tiles_n = (p.positions + BN - 1) / BN, tiles_m = (p.cout + BM - 1) / BM;
  int tile = XcdTile(blockIdx.x, gridDim.x), tile_n, tile_m;
  if (p.rows_first) {
    tile_m = tile % tiles_m;
    tile /= tiles_m;
    tile_n = tile % tiles_n;
    tile /= tiles_n;
  } else {
    tile_n = tile % tiles_n;
    tile /= tiles_n;
    tile_m = tile % tiles_m;
    tile /= tiles_m;
  }
  const int split = tile % p.splits;
  const int rest = tile / p.splits;  // batch x phases + phase
  const int phase = rest % p.phases;
  const int batch = rest / p.phases;
  const int chunks = (p.cin + kChunk - 1) / kChunk;
  const int c_begin = split * p.split_chunks;
  const int c_end = min(chunks, c_begin + p.split_chunks);
  const float* x = p.x + batch * p.x_batch;
  const int m0 = tile_n * BN;
  const int co0 = tile_m * BM;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int row = (wave / WN) * 32;       // first output channel of the wave
  const int col = (wave % WN) * 32 * NT;  // first position of the wave
  const int half = lane >> 5;             // K half of the lane's operands
  const int l32 = lane & 31;
  const int dilation = TAPS == 1 ? 0 : p.dilation;
  const int width = TAPS <= 2 ? kMaxWidth : BN + (TAPS - 1) * dilation;
  const int units = kChunk / 8 * width;

  // Unit u = tid + 256 q of a chunk's window: channels 8 (u / width) .. + 7
  // at window column u % width.
  int at[kSlots], group[kSlots];  // first input position, 8-channel group
  unsigned inside[kSlots];        // bit i: channel i of the unit is a value
#pragma unroll
  for (int q = 0; q < kSlots; ++q) {
    const int u = min(tid + q * kThreads, units - 1);
    group[q] = u / width;
    const int m = m0 + u % width;
    if (VIEW) {
      at[q] = m * p.view_stride + p.first[phase];
    } else {
      const int t = m + p.first[phase];
      inside[q] = t >= 0 && t < p.len_in ? 0xFFU : 0U;
      at[q] = min(max(t, 0), p.len_in - 1);
    }
  }
  float xr[kSlots][8];
  auto fetch = [&](int chunk) {
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
      if (wave * 64 + q * kThreads >= units)
        break;
      const int j = chunk * kChunk + 8 * group[q];
      if (VIEW) {
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
        inside[q] = mask;
      } else {
        const float* from = x + at[q];
        if (j + 8 <= p.cin) {
          from += static_cast<size_t>(j) * p.len_in;
#pragma unroll
          for (int i = 0; i < 8; ++i)
            xr[q][i] = from[static_cast<size_t>(i) * p.len_in];
        } else {
#pragma unroll
          for (int i = 0; i < 8; ++i)
            xr[q][i] = from[static_cast<size_t>(min(j + i, p.cin - 1)) * p.len_in];
        }
      }
    }
  };
  auto stash = [&](int chunk, int buf) {
#pragma unroll
    for (int q = 0; q < kSlots; ++q) {
      const int u = tid + q * kThreads;
      if (wave * 64 + q * kThreads >= units)
        break;
      const int j = chunk * kChunk + 8 * group[q];
      if (p.alpha_in != nullptr) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          xr[q][i] = Snake(xr[q][i], p.alpha_in[min(j + i, p.cin - 1)],
                           SnakeInverse(p.alpha_in[min(j + i, p.cin - 1)]));
      }
      if (p.in_act == kActElu) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          xr[q][i] = Elu(xr[q][i]);
      }
      unsigned mask = inside[q];
      if (!VIEW && j + 8 > p.cin)
        mask &= (1U << max(p.cin - j, 0)) - 1U;
#pragma unroll
      for (int i = 0; i < 8; ++i)
        xr[q][i] = (mask >> i & 1U) != 0U ? xr[q][i] : 0.0F;
      uintx4 part[3];
      Split8(xr[q], part);
      if (u < units) {
#pragma unroll
        for (int s = 0; s < 3; ++s)
          xs[buf][s][u] = part[s];
      }
    }
  };

  // The weights of the wave's 32 rows, one step after the other.
  const int steps = (c_end - c_begin) * kSteps;
  const size_t step_units = 6 * static_cast<size_t>(p.w_rows);
  const uintx4* w = reinterpret_cast<const uintx4*>(p.w) +
                    (static_cast<size_t>(rest) * ((p.cin + ConvPad(TAPS) - 1) / ConvPad(TAPS)) *
                         (ConvPad(TAPS) / 16 * TAPS) +
                     c_begin * kSteps) * step_units +
                    static_cast<size_t>(half) * p.w_rows + min(co0 + row + l32, p.w_rows - 1);
  int ahead = 0;  // the next step to load, held at the last one
  auto load = [&](uintx4* a) {
#pragma unroll
    for (int s = 0; s < 3; ++s)
      a[s] = w[static_cast<size_t>(2 * s) * p.w_rows];
    if (++ahead < steps)
      w += step_units;
  };

  floatx16 main[NT] = {}, low[NT] = {};
  uintx4 a[kAhead][3], b[2][3];
  fetch(c_begin);
#pragma unroll
  for (int i = 0; i < kAhead; ++i)
    load(a[i]);
  for (int chunk = c_begin; chunk < c_end; ++chunk) {
    const int buf = BUFS == 1 ? 0 : (chunk - c_begin) & 1;
    stash(chunk, buf);
    __syncthreads();
    if (BUFS > 1 && chunk + 1 < c_end)
      fetch(chunk + 1);
    const uintx4* base = &xs[buf][0][half * width + col + l32];
    // Block i of a chunk: column block i % NT of step i / NT.
    auto read = [&](int i, uintx4* v) {
      const int step = i / NT;
      const uintx4* from =
          base + step % kSubs * 2 * width + step / kSubs * dilation + 32 * (i % NT);
#pragma unroll
      for (int s = 0; s < 3; ++s)
        v[s] = from[s * kMaxUnits];
    };
    read(0, b[0]);
#pragma unroll
    for (int i = 0; i < kSteps * NT; ++i) {
      const int t = i % NT, step = i / NT;
      if (i + 1 < kSteps * NT)
        read(i + 1, b[(i + 1) & 1]);
      // Keeps the next block's reads ahead of this block's products.
      __builtin_amdgcn_sched_barrier(0);
      const uintx4* aa = a[step % kAhead];
      const uintx4* bb = b[i & 1];
      low[t] = MfmaBf16(aa[0], bb[2], low[t]);
      main[t] = MfmaBf16(aa[0], bb[0], main[t]);
      low[t] = MfmaBf16(aa[2], bb[0], low[t]);
      low[t] = MfmaBf16(aa[1], bb[1], low[t]);
      low[t] = MfmaBf16(aa[0], bb[1], low[t]);
      low[t] = MfmaBf16(aa[1], bb[0], low[t]);
      __builtin_amdgcn_sched_barrier(0);
      if (t == NT - 1)
        load(a[step % kAhead]);
    }
  }

  // Element r of the accumulators: output channel row + 8 (r / 4) +
  // 4 half + r % 4, position col + 32 t + l32.
  const float* bias = p.bias != nullptr ? p.bias + batch * p.b_batch : nullptr;
  float* y = p.y != nullptr ? p.y + batch * p.y_batch : nullptr;
  float* y_act = p.y_act != nullptr ? p.y_act + batch * p.y_batch : nullptr;
  const float* prior_of = p.residual != nullptr ? p.residual + batch * p.y_batch : nullptr;
  const int co1 = co0 + row + 4 * half;
  const int first = m0 + col + l32;
  if (p.splits > 1) {
    // partial[rest][split][co][m]
    float* part = p.partial + (static_cast<size_t>(rest) * p.splits + split) * p.cout * p.positions;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int m = first + 32 * t;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int co = co1 + 8 * (r >> 2) + (r & 3);
        if (m < p.positions && co < p.cout)
          part[static_cast<size_t>(co) * p.positions + m] = Join(main[t][r], low[t][r]);
      }
    }
    return;
  }
  // Four channels at a time. Every load of a group (bias, the residual, the
  // Snake alphas) is issued before the previous group's stores: the stores may
  // alias them as far as the compiler knows, so loads left between them would
  // each wait out a memory round trip.
  struct Group {
    float bias[4], alpha[4], residual[NT][4];
  };
  auto gather = [&](int g) {
    Group v;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int co = min(co1 + 8 * g + r, p.cout - 1);
      v.bias[r] = bias != nullptr ? bias[co] : 0.0F;
      v.alpha[r] = y_act != nullptr && p.out_act == kActSnake ? p.alpha_out[co] : 0.0F;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        v.residual[t][r] =
            prior_of != nullptr
                ? prior_of[static_cast<size_t>(co) * p.len_out +
                           static_cast<size_t>(min(first + 32 * t, p.positions - 1)) * p.out_stride +
                           phase]
                : 0.0F;
    }
    return v;
  };
  Group next = gather(0);
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const Group cur = next;
    if (g < 3)
      next = gather(g + 1);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int co = co1 + 8 * g + r;
      const float inverse = SnakeInverse(cur.alpha[r]);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int m = first + 32 * t;
        if (m < p.positions && co < p.cout) {
          const size_t to = static_cast<size_t>(co) * p.len_out +
                            static_cast<size_t>(m) * p.out_stride + phase;
          float v = Join(main[t][4 * g + r], low[t][4 * g + r]) + cur.bias[r];
          if (p.pre_act == kActGelu)
            v = Gelu(v);
          v += cur.residual[t][r];
          if (y != nullptr)
            y[to] = v;
          if (y_act != nullptr)
            y_act[to] = p.out_act == kActElu ? Elu(v) : Snake(v, cur.alpha[r], inverse);
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
    Split8(v, part);
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
    const float* part = p.partial + static_cast<size_t>(rest) * p.splits * per + within;
    float v = 0.0F;
    for (int s = 0; s < p.splits; ++s)
      v += part[static_cast<size_t>(s) * per];
    const int phase = rest % p.phases, batch = rest / p.phases;
    const float* bias = p.bias != nullptr ? p.bias + batch * p.b_batch : nullptr;
    float* y = p.y != nullptr ? p.y + batch * p.y_batch : nullptr;
    float* y_act = p.y_act != nullptr ? p.y_act + batch * p.y_batch : nullptr;
    const float* residual = p.residual != nullptr ? p.residual + batch * p.y_batch : nullptr;
    const size_t t = static_cast<size_t>(m) * p.out_stride + phase;
    Finish(p, bias, residual, y, y_act, co, static_cast<size_t>(co) * p.len_out + t, v);
  }
}

__global__ __launch_bounds__(kThreads) void OutputConvKernel(OutputConvParams p) {
  __shared__ float xs[kOutChunk][kOutTile + kConvMaxTaps - 1];
  const int tid = threadIdx.x;
  const int t0 = blockIdx.x * kOutTile;
  const int pad = (p.taps - 1) / 2;
  const int width = kOutTile + p.taps - 1;
  float acc = 0.0F;
  for (int c0 = 0; c0 < p.cin; c0 += kOutChunk) {
    for (int j = tid; j < width; j += kThreads) {
      const int t = t0 - pad + j;
      const bool inside = t >= 0 && t < p.length;
      const int tc = min(max(t, 0), p.length - 1);
      float v[kOutChunk];
#pragma unroll
      for (int c = 0; c < kOutChunk; ++c)
        v[c] = p.x[static_cast<size_t>(min(c0 + c, p.cin - 1)) * p.length + tc];
#pragma unroll
      for (int c = 0; c < kOutChunk; ++c)
        xs[c][j] = inside && c0 + c < p.cin
                       ? (p.alpha != nullptr ? Snake(v[c], p.alpha[min(c0 + c, p.cin - 1)],
                                                     SnakeInverse(p.alpha[min(c0 + c, p.cin - 1)]))
                                             : v[c])
                       : 0.0F;
    }
    __syncthreads();
    const int channels = min(kOutChunk, p.cin - c0);
    for (int c = 0; c < channels; ++c)
      for (int k = 0; k < p.taps; ++k)
        acc += p.w[k * p.cin + c0 + c] * xs[c][tid + k];
    __syncthreads();
  }
  const int t = t0 + tid;
  if (t < p.length)
    p.y[t] = acc + p.bias[0];
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

template <int WM, int WN, int NT, int TAPS, int BUFS, bool VIEW>
void DispatchTile(const ConvParams& p, hipStream_t stream) {
  constexpr int BM = 32 * WM, BN = 32 * WN * NT;
  const int64_t grid = static_cast<int64_t>((p.positions + BN - 1) / BN) *
                       ((p.cout + BM - 1) / BM) * p.phases * p.batches * p.splits;
  Require(grid < (int64_t{1} << 31), "conv: too many tiles");
  Dispatch(ConvKernel<WM, WN, NT, TAPS, BUFS, VIEW>, dim3(static_cast<unsigned>(grid)),
           dim3(kThreads), 0, stream, true, p.splits == 1, p);
}

// The tile: all output channels of a narrow layer (32 x 256 when the input is
// one chunk, so that two work-groups' windows fit a CU's LDS, else 32 x 128;
// 64 x 128), else 128 x 128 where that gives every CU a work-group, else
// 128 x 64.
//
// With a split-K workspace, a convolution whose tiles number under 256
// instead splits its input channels until about 512 work-groups run, and a
// reduction kernel finishes it.
template <int TAPS, bool VIEW>
void DispatchTaps(const ConvParams& params, hipStream_t stream) {
  ConvParams p = params;
  const auto groups = [&](int bm, int bn) {
    return static_cast<int64_t>((p.positions + bn - 1) / bn) * ((p.cout + bm - 1) / bm) *
           p.phases * p.batches;
  };
  const int64_t inputs = static_cast<int64_t>(VIEW ? p.channels : p.cin) * p.len_in * p.batches;
  p.rows_first = 2 * inputs > int64_t{3} * p.taps * p.cin * p.cout * p.phases * p.batches;
  const bool wide = p.cout > 64 && groups(128, 128) >= 256;
  const bool one = p.cin <= 32;
  const int columns = p.cout <= 32 ? (one ? 256 : 128) : p.cout <= 64 || wide ? 128 : 64;
  const int64_t tiles = groups(p.cout <= 32 ? 32 : p.cout <= 64 ? 64 : 128, columns);
  const int chunk = TileChunk(TAPS, columns), chunks = (p.cin + chunk - 1) / chunk;
  p.splits = 1;
  p.split_chunks = chunks;
  if (p.partial != nullptr && tiles < 256 && chunks >= 4) {
    int64_t want = std::min<int64_t>((512 + tiles - 1) / tiles, chunks / 2);
    const int64_t outputs = static_cast<int64_t>(p.cout) * p.positions * p.phases * p.batches;
    want = std::min<int64_t>(want, p.partial_capacity / std::max<int64_t>(outputs, 1));
    want = std::min<int64_t>(want, 65535 / (static_cast<int64_t>(p.phases) * p.batches));
    if (want >= 2) {
      p.split_chunks = static_cast<int>((chunks + want - 1) / want);
      p.splits = (chunks + p.split_chunks - 1) / p.split_chunks;
    }
  }
  if (p.cout <= 32 && one)
    DispatchTile<1, 4, 2, TAPS, 1, VIEW>(p, stream);
  else if (p.cout <= 32)
    DispatchTile<1, 4, 1, TAPS, 2, VIEW>(p, stream);
  else if (p.cout <= 64)
    DispatchTile<2, 2, 2, TAPS, 2, VIEW>(p, stream);
  else if (wide)
    DispatchTile<4, 1, 4, TAPS, 2, VIEW>(p, stream);
  else
    DispatchTile<4, 1, 2, TAPS, 2, VIEW>(p, stream);
  if (p.splits > 1) {
    const size_t total = static_cast<size_t>(p.cout) * p.positions * p.phases * p.batches;
    const int blocks = static_cast<int>(std::min<size_t>((total + kThreads - 1) / kThreads, 16384));
    Dispatch(SplitReduceKernel, dim3(blocks), dim3(kThreads), 0, stream, false, true, p);
  }
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
  Require(p.out_stride >= p.phases, "conv: phases overlap in the output");
  Require(static_cast<int64_t>(p.positions - 1) * p.out_stride + p.phases - 1 < p.len_out,
          "conv: output positions past the output length");
  Require(p.taps == 1 || (p.dilation >= 1 &&
                          (p.taps - 1) * static_cast<int64_t>(p.dilation) <=
                              (p.taps == 2 ? 1 : kConvMaxSpan)),
          "conv: taps spread too far for their count");
  if (p.view_kernel != 0) {
    Require(p.taps == 1 && p.phases == 1, "conv: a view has one tap and phase");
    Require(p.view_kernel >= 1 && p.view_stride >= 1 && p.channels >= 1 &&
                static_cast<int64_t>(p.channels) * p.view_kernel == p.cin &&
                (p.positions + int64_t{256}) * p.view_stride + p.view_kernel <
                    (std::int64_t{1} << 31),
            "conv: bad view");
    DispatchTaps<1, true>(p, stream);
  } else if (p.taps == 1) {
    DispatchTaps<1, false>(p, stream);
  } else if (p.taps == 2) {
    DispatchTaps<2, false>(p, stream);
  } else {
    DispatchTaps<7, false>(p, stream);
  }
}

void LaunchOutputConv(const OutputConvParams& p, hipStream_t stream) {
  Require(p.x && p.w && p.bias && p.y, "output conv: null pointer");
  Require(p.cin >= 1 && p.length >= 1, "output conv: empty shape");
  Require(p.taps >= 1 && p.taps <= kConvMaxTaps && p.taps % 2 == 1,
          "output conv: 1, 3, 5 or 7 taps");
  Dispatch(OutputConvKernel, dim3((p.length + kOutTile - 1) / kOutTile), dim3(kThreads), 0,
           stream, true, true, p);
}

void LaunchRvq(const RvqParams& p, hipStream_t stream) {
  Require(p.table && p.bias && p.codes && p.y, "rvq: null pointer");
  Require(p.codebooks >= 1 && p.entries >= 1 && p.latent >= 1 && p.frames >= 1,
          "rvq: empty shape");
  Dispatch(RvqKernel, dim3(p.frames), dim3(kThreads), 0, stream, true, true, p);
}

}  // namespace ovg
