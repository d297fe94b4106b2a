// The audio encoder's element-wise, normalisation and selection kernels on
// gfx950 (the reference's kernels/encoder_kernels.hip counterparts: the
// resampler that audio.cpp:265-322 runs on the host, GroupNorm + GELU,
// LayerNorm, attention, the frame pick and the residual vector quantizer).
// Every GEMM-shaped layer of the encoder but attention runs through the
// convolution kernel; these kernels move each element once or twice and are
// bound by HBM or, at the encoder's small sizes, by launch.
//
// The column kernel (LayerNorm over channels) reads a channel-major matrix
// along its slow dimension: a work-group owns 8 adjacent columns, each
// column 32 lanes that hold every 32nd row in registers, so each element is
// read once, all of a thread's loads are in flight together, and the partial
// sums meet in LDS.
#include <algorithm>
#include <cfloat>
#include <type_traits>

#include "codec.hpp"
#include "common.hpp"
#include "encoder.hpp"
#include "kernels.hpp"
#include "split.hpp"

namespace ovg {
namespace {

constexpr int kThreads = 256;

__device__ __forceinline__ float Gelu(float v) {
  return 0.5F * v * (1.0F + erff(v * 0.70710678118654752F));
}

__global__ __launch_bounds__(kThreads) void ResampleKernel(ResampleParams p) {
  const int total = p.out_length + 2 * p.pad;
  for (int i = blockIdx.x * kThreads + threadIdx.x; i < total; i += gridDim.x * kThreads) {
    const int j = i - p.pad;
    float out = 0.0F;
    if (j >= 0 && j < p.out_length) {
      const int phase = j % p.to;
      const int origin = (j / p.to) * p.from - p.width;
      const float* w = p.bank + static_cast<size_t>(phase) * p.taps;
      const int lo = max(0, -origin), hi = min(p.taps, p.length - origin);
      double sum = 0.0;
      for (int k = lo; k < hi; ++k)
        sum += static_cast<double>(w[k]) * p.x[origin + k];
      out = static_cast<float>(sum);
    }
    p.y[i] = out;
  }
}

// 32 x 32 tiles through LDS, both sides in whole 128-byte runs.
__global__ __launch_bounds__(kThreads) void TransposeKernel(const float* x, float* y, int rows,
                                                            int cols) {
  __shared__ float tile[32][33];
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int i = threadIdx.x % 32;
  for (int j = threadIdx.x / 32; j < 32; j += kThreads / 32)
    if (r0 + j < rows && c0 + i < cols)
      tile[j][i] = x[static_cast<size_t>(r0 + j) * cols + c0 + i];
  __syncthreads();
  for (int j = threadIdx.x / 32; j < 32; j += kThreads / 32)
    if (c0 + j < cols && r0 + i < rows)
      y[static_cast<size_t>(c0 + j) * rows + r0 + i] = tile[i][j];
}

// Sum of one double per thread over the work-group (every thread gets it).
__device__ double BlockSum(double v, double* scratch) {
  for (int o = 32; o > 0; o >>= 1)
    v += __shfl_xor(v, o);
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0)
    scratch[wave] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < kThreads / 64; ++i)
    s += scratch[i];
  return s;
}

__global__ __launch_bounds__(kThreads) void GroupNormGeluKernel(float* x, const float* w,
                                                                const float* b, int length,
                                                                float eps) {
  __shared__ double scratch[kThreads / 64];
  float* row = x + static_cast<size_t>(blockIdx.x) * length;
  // One pass for the sum and the sum of squares (double), unrolled so that
  // eight loads are in flight per thread.
  double s = 0.0, q = 0.0;
#pragma unroll 8
  for (int t = threadIdx.x; t < length; t += kThreads) {
    const double v = row[t];
    s += v;
    q += v * v;
  }
  const double mean = BlockSum(s, scratch) / length;
  const double var = fmax(BlockSum(q, scratch) / length - mean * mean, 0.0);
  const double inv = 1.0 / sqrt(var + eps);
  const double wc = w[blockIdx.x], bc = b[blockIdx.x];
#pragma unroll 8
  for (int t = threadIdx.x; t < length; t += kThreads)
    row[t] = Gelu(static_cast<float>((row[t] - mean) * inv * wc + bc));
}

// The column kernel: a work-group of kCols adjacent columns x kLanes lanes;
// lane l of a column holds rows l, l + kLanes, ... (up to kPer of them) in
// registers, so every element is read once with all its loads in flight.
constexpr int kCols = 8;
constexpr int kLanes = kThreads / kCols;

// Sum over the lanes of a column: those of a wave by shuffles, then the
// waves' sums through LDS. With every lane reading all 32 partial sums from
// LDS, and the store loop's loads behind the sums, a LayerNorm of 768 channels
// took 7.2, 9.3 and 13.3 us at 150, 500 and 1045 positions; now 6.4, 8.4, 12.3.
__device__ double LaneSum(double v, double (*scratch)[kCols]) {
  for (int o = kCols; o < 64; o *= 2)
    v += __shfl_xor(v, o);
  const int col = threadIdx.x % kCols;
  __syncthreads();
  if ((threadIdx.x & 63) < kCols)
    scratch[threadIdx.x >> 6][col] = v;
  __syncthreads();
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < kThreads / 64; ++i)
    s += scratch[i][col];
  return s;
}

template <int kPer>
__global__ __launch_bounds__(kThreads) void ColumnNormKernel(ColumnNormParams p) {
  __shared__ double scratch[kThreads / 64][kCols];
  const int t = blockIdx.x * kCols + threadIdx.x % kCols;
  const int lane = threadIdx.x / kCols;
  const int tc = min(t, p.positions - 1);
  float v[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = min(lane + i * kLanes, p.channels - 1);
    v[i] = p.x[static_cast<size_t>(c) * p.positions + tc];
  }
  // The store loop's loads too, all in flight with the column's.
  float w[kPer], b[kPer];
  double prior[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = min(lane + i * kLanes, p.channels - 1);
    w[i] = p.w[c];
    b[i] = p.b[c];
    prior[i] = p.sum_mode == 2 ? p.sum[static_cast<size_t>(c) * p.positions + tc] : 0.0;
  }
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    if (lane + i * kLanes < p.channels)
      s += v[i];
  const double mean = LaneSum(s, scratch) / p.channels;
  double q = 0.0;
#pragma unroll
  for (int i = 0; i < kPer; ++i)
    if (lane + i * kLanes < p.channels) {
      const double d = v[i] - mean;
      q += d * d;
    }
  const double inv = 1.0 / sqrt(LaneSum(q, scratch) / p.channels + p.eps);
  if (t >= p.positions)
    return;
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int c = lane + i * kLanes;
    if (c < p.channels) {
      const size_t at = static_cast<size_t>(c) * p.positions + t;
      const float o = static_cast<float>((v[i] - mean) * inv * w[i] + b[i]);
      p.y[at] = o;
      if (p.sum_mode != 0)
        p.sum[at] = prior[i] + o;
    }
  }
}

// HuBERT's attention: the projections into matrix-core operands, then one
// kernel over the heads, instead of scores, softmax, transpose and context
// launches that move the [heads][steps][steps] scores through memory. Bound
// by each wave's chain of dependent products and its softmax, hence eight
// waves (two per SIMD) over the keys of only 32 queries. Both launches, 12
// heads of 64 dims: 14.8, 20.7 and 47.1 us at 150, 500 and 1045 steps, against
// 37.6, 52.9 and 156 us for the four launches (four waves: 15.8, 22.2, 59.2;
// operands gathered and split by every work-group from the channel-major
// projections: 24.9, 46.2, 119).
//
// Operand order, per head and tile of 32 positions (zeros past the head's
// dims and past the last position), three parts (split.hpp) of 64 lanes x 16
// bytes each:
//   q, k  [16 dims s][part]: lane l is position l % 32, dims 16 s + 8 (l / 32)
//         .. + 7
//   v     [32 dims n][16 keys j][part]: lane l is dim 32 n + l % 32, keys 16 j
//         + 8 (i / 4) + 4 (l / 32) + i % 4 for i < 8, the order in which the
//         scores' accumulators hold the keys
constexpr int kAttentionTile = 32;   // queries per work-group, keys per tile
constexpr int kAttentionDims = 64;   // output dims per work-group
constexpr int kAttentionThreads = 512;
// 16-byte vectors of one tile of q or k and of v.
__host__ __device__ constexpr int QkVectors(int head_dim) { return (head_dim + 15) / 16 * 192; }
__host__ __device__ constexpr int ValueVectors(int head_dim) {
  return (head_dim + 31) / 32 * 384;
}

__global__ __launch_bounds__(kThreads) void PackHeadsKernel(HeadAttentionParams p) {
  const int T = p.steps, hd = p.head_dim;
  const int tile = blockIdx.x, head = blockIdx.y, which = blockIdx.z;
  const int tiles = gridDim.x;
  const int t0 = tile * kAttentionTile;
  const float* from = (which == 0 ? p.q : which == 1 ? p.k : p.v) +
                      static_cast<size_t>(head) * hd * T;
  uintx4* to = reinterpret_cast<uintx4*>(p.packed);
  const size_t at = static_cast<size_t>(head) * tiles + tile;
  const size_t heads_tiles = static_cast<size_t>(p.heads) * tiles;
  if (which < 2)
    to += (heads_tiles * which + at) * QkVectors(hd);
  else
    to += heads_tiles * 2 * QkVectors(hd) + at * ValueVectors(hd);
  const int items = (which < 2 ? QkVectors(hd) : ValueVectors(hd)) / 3;
  for (int e = threadIdx.x; e < items; e += kThreads) {
    const int lane = e & 63, half = lane >> 5, l32 = lane & 31;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      int d, t;
      if (which < 2) {
        d = (e >> 6) * 16 + 8 * half + i;
        t = t0 + l32;
      } else {
        d = (e >> 7) * 32 + l32;
        t = t0 + ((e >> 6) & 1) * 16 + 8 * (i >> 2) + 4 * half + (i & 3);
      }
      v[i] = from[static_cast<size_t>(min(d, hd - 1)) * T + min(t, T - 1)];
      if (d >= hd || t >= T)
        v[i] = 0.0F;
    }
    uintx4 part[3];
    Split8<true>(v, part);
#pragma unroll
    for (int k = 0; k < 3; ++k)
      to[((e >> 6) * 3 + k) * 64 + lane] = part[k];
  }
}

// One output in double, for sums that are not finite: the sum of values next
// to the largest overflows where their mean does not. Ends at the first NaN.
__device__ __forceinline__ float WideContext(const HeadAttentionParams& p, int head, int d, int t) {
  const size_t T = p.steps, at = static_cast<size_t>(head) * p.head_dim * T;
  const auto score = [&](int s) {
    double sum = 0.0;
#pragma unroll 1
    for (int e = 0; e < p.head_dim; ++e)
      sum += static_cast<double>(p.q[at + e * T + t]) * p.k[at + e * T + s];
    return sum * p.scale;
  };
  double peak = -DBL_MAX, sum = 0.0, out = 0.0;
#pragma unroll 1
  for (int s = 0; s < p.steps; ++s) {
    const double v = score(s), top = v > peak || v != v ? v : peak;
    const double keep = exp(peak - top), share = exp(v - top);
    sum = sum * keep + share;
    out = out * keep + share * p.v[at + d * T + s];
    peak = top;
    if (out != out)
      break;
  }
  return static_cast<float>(out / sum);
}

// A work-group owns one head's 32 queries (and 64 of the head's dims; wider
// heads take more work-groups); its eight waves take every eighth tile of
// 32 keys. Scores are formed transposed (S^T = K^T Q, each lane one query
// column) and never leave registers: they become the operand of O = V P^T
// there. The softmax runs online per wave (a running maximum, the sum in
// double, the output rescaled when the maximum grows), and the waves'
// states meet in LDS at the end. The queries are in LDS (kQueriesInLds: up to
// 256 dims), a tile's keys and values come straight into registers, the next
// keys during the softmax.
template <bool kQueriesInLds>
__global__ __launch_bounds__(kAttentionThreads) void HeadAttentionKernel(HeadAttentionParams p) {
  constexpr int kWaves = kAttentionThreads / 64;
  // The queries, then (once every wave is past them) the waves' outputs.
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ float peaks[kWaves][kAttentionTile];
  __shared__ double sums[kWaves][kAttentionTile];
  auto merged = reinterpret_cast<float(*)[kAttentionDims][kAttentionTile]>(lds);
  const int T = p.steps, hd = p.head_dim;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int half = lane >> 5, l32 = lane & 31;
  const int tiles = gridDim.x, head = blockIdx.y;
  const int q0 = blockIdx.x * kAttentionTile;
  const int slab = blockIdx.z * kAttentionDims;  // first output dim
  const int rounds = (hd + 15) / 16;             // 16 dims each
  const int blocks = (hd + 31) / 32;             // 32 output dims each
  const size_t heads_tiles = static_cast<size_t>(p.heads) * tiles;
  const uintx4* packed = reinterpret_cast<const uintx4*>(p.packed);
  const size_t first = static_cast<size_t>(head) * tiles;
  const uintx4* queries = packed + (first + blockIdx.x) * QkVectors(hd);
  const uintx4* keys = packed + (heads_tiles + first) * QkVectors(hd) + lane;
  const uintx4* values = packed + heads_tiles * 2 * QkVectors(hd) + first * ValueVectors(hd) + lane;
  uintx4* const staged = reinterpret_cast<uintx4*>(lds);
  if constexpr (kQueriesInLds) {
    for (int e = threadIdx.x; e < rounds * 192; e += kAttentionThreads)
      staged[e] = queries[e];
    __syncthreads();
  }
  const int n_last = blocks - 1;

  uintx4 kf[4][3];
  auto load_keys = [&](int tile, int s0) {
    const uintx4* from = keys + static_cast<size_t>(min(tile, tiles - 1)) * QkVectors(hd);
#pragma unroll
    for (int s = 0; s < 4; ++s)
#pragma unroll
      for (int k = 0; k < 3; ++k)
        kf[s][k] = from[(min(s0 + s, rounds - 1) * 3 + k) * 64];
  };
  floatx16 main[2] = {}, corr[2] = {};
  float peak = -FLT_MAX;
  double sum = 0.0;
  load_keys(wave, 0);
  for (int tile = wave; tile < tiles; tile += kWaves) {
    const int k0 = tile * kAttentionTile;
    // Values of this tile, in flight during the scores and the softmax.
    uintx4 vf[2][2][3];
#pragma unroll
    for (int n = 0; n < 2; ++n) {
      const uintx4* from = values + static_cast<size_t>(tile) * ValueVectors(hd) +
                           min(slab / 32 + n, n_last) * 384;
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int k = 0; k < 3; ++k)
          vf[n][j][k] = from[(j * 3 + k) * 64];
    }
    floatx16 sm = {}, sc = {};
    for (int s0 = 0; s0 < rounds; s0 += 4) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (s0 + s >= rounds)
          break;
        uintx4 qf[3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
          qf[k] = kQueriesInLds ? staged[((s0 + s) * 3 + k) * 64 + lane]
                                : queries[((s0 + s) * 3 + k) * 64 + lane];
        sc = MfmaBf16(kf[s][2], qf[0], sc);
        sm = MfmaBf16(kf[s][0], qf[0], sm);
        sc = MfmaBf16(kf[s][0], qf[2], sc);
        sc = MfmaBf16(kf[s][1], qf[1], sc);
        sc = MfmaBf16(kf[s][1], qf[0], sc);
        sc = MfmaBf16(kf[s][0], qf[1], sc);
      }
      // The next round of dims, or the next tile's first one.
      if (s0 + 4 < rounds)
        load_keys(tile, s0 + 4);
      else
        load_keys(tile + kWaves, 0);
    }
    float s[16], top = peak;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = Join(sm[r], sc[r]);
      if (k0 + 8 * (r >> 2) + 4 * half + (r & 3) < T)
        top = fmaxf(top, s[r]);
    }
    top = fmaxf(top, __shfl_xor(top, 32));
    const float keep = expf((peak - top) * p.scale);
    peak = top;
    double part = 0.0;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s[r] = k0 + 8 * (r >> 2) + 4 * half + (r & 3) < T ? expf((s[r] - top) * p.scale) : 0.0F;
      part += s[r];
    }
    sum = sum * keep + (part + __shfl_xor(part, 32));
#pragma unroll
    for (int n = 0; n < 2; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        main[n][r] *= keep;
        corr[n][r] *= keep;
      }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      uintx4 pf[3];
      Split8<false>(s + 8 * j, pf);
#pragma unroll
      for (int n = 0; n < 2; ++n) {
        corr[n] = MfmaBf16(vf[n][j][2], pf[0], corr[n]);
        main[n] = MfmaBf16(vf[n][j][0], pf[0], main[n]);
        corr[n] = MfmaBf16(vf[n][j][0], pf[2], corr[n]);
        corr[n] = MfmaBf16(vf[n][j][1], pf[1], corr[n]);
        corr[n] = MfmaBf16(vf[n][j][1], pf[0], corr[n]);
        corr[n] = MfmaBf16(vf[n][j][0], pf[1], corr[n]);
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int n = 0; n < 2; ++n)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      merged[wave][32 * n + 8 * (r >> 2) + 4 * half + (r & 3)][l32] = Join(main[n][r], corr[n][r]);
  if (half == 0) {
    peaks[wave][l32] = peak;
    sums[wave][l32] = sum;
  }
  __syncthreads();
  const int q = threadIdx.x % kAttentionTile;
  float top = peaks[0][q];
#pragma unroll
  for (int w = 1; w < kWaves; ++w)
    top = fmaxf(top, peaks[w][q]);
  float keep[kWaves];
  double total = 0.0;
#pragma unroll
  for (int w = 0; w < kWaves; ++w) {
    keep[w] = expf((peaks[w][q] - top) * p.scale);
    total += sums[w][q] * keep[w];
  }
  const float inv = static_cast<float>(1.0 / total);
  for (int d = threadIdx.x / kAttentionTile; d < kAttentionDims;
       d += kAttentionThreads / kAttentionTile) {
    float o = 0.0F;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
      o += merged[w][d][q] * keep[w];
    o *= inv;
    if (q0 + q < T && slab + d < hd) {
      if (__builtin_expect(!__builtin_isfinite(o), 0))
        o = WideContext(ParamsAgain<HeadAttentionParams>(), head, slab + d, q0 + q);
      p.out[(static_cast<size_t>(head) * hd + slab + d) * T + q0 + q] = o;
    }
  }
}

__global__ __launch_bounds__(kThreads) void PickFramesKernel(const double* sum, int channels,
                                                             int positions, int stride,
                                                             int frames, double scale,
                                                             float* y) {
  const int total = channels * frames;
  for (int e = blockIdx.x * kThreads + threadIdx.x; e < total; e += gridDim.x * kThreads) {
    const int c = e / frames, f = e % frames;
    y[e] = static_cast<float>(sum[static_cast<size_t>(c) * positions +
                                  static_cast<size_t>(f) * stride] * scale);
  }
}

// The residual vector quantizer, every stage of FRAMES frames in one
// work-group: a frame's stages depend on each other, frames do not. Per stage
// the projection (float32 sums over an eighth of the input per wave, the
// eight added in order), the distances to every entry (double, dims in
// order), the nearest entry (the lowest index on ties) and the subtraction of
// its decoded row from the residual, which stays in LDS (in `residual` where
// it does not fit, kInLds false).
//
// A stage reads the projection and the codebook once per work-group (512 KB
// at 1024 x 64 x 1024, 4 us of the CU's 64 B/clk load path) in a chain of
// load batches, barriers and the search's reduction, whose latency bounds the
// kernel at about 14 us per stage. All eight stages: 113 us at 75 and 250
// frames against 262 and 277 us for a projection and a search launch each;
// 163 us at 523 frames (400 us), where more frames than CUs go two to a
// work-group. Batches of 64 and 32 loads (350 us: the unrolled code no longer
// fits the instruction cache) and 16-byte loads (122 us, 291 us at 523
// frames) were slower.
constexpr int kRvqThreads = 512;
constexpr int kRvqWaves = kRvqThreads / 64;
constexpr int kRvqMaxDim = 1024;
constexpr std::uint32_t kRvqLdsLimit = 144 * 1024;
constexpr std::uint64_t RvqLdsBytes(int frames, int dim, std::int64_t hidden) {
  return static_cast<std::uint64_t>(frames) *
         (dim * (8 + 4 * kRvqWaves) + 4 * static_cast<std::uint64_t>(hidden));
}

template <int FRAMES, bool kInLds>
__global__ __launch_bounds__(kRvqThreads) void RvqEncodeKernel(RvqEncodeParams p) {
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ double best_d[FRAMES][kRvqWaves];
  __shared__ int best_e[FRAMES][kRvqWaves];
  const int D = p.dim, E = p.entries, H = p.hidden;
  double* const v = reinterpret_cast<double*>(lds);                  // [FRAMES][D]
  float* const part = reinterpret_cast<float*>(v + FRAMES * D);      // [waves][FRAMES][D]
  float* const lds_r = part + kRvqWaves * FRAMES * D;                // [FRAMES][H]
  const int f0 = blockIdx.x * FRAMES;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  auto residual = [&](int f, int h) -> float& {
    if constexpr (kInLds)
      return lds_r[f * H + h];
    else
      return p.residual[static_cast<size_t>(min(f0 + f, p.frames - 1)) * H + h];
  };
#pragma unroll
  for (int f = 0; f < FRAMES; ++f)
    for (int h = tid; h < H; h += kRvqThreads)
      residual(f, h) = p.x[static_cast<size_t>(h) * p.frames + min(f0 + f, p.frames - 1)];
  const int per = (H + kRvqWaves - 1) / kRvqWaves;
  const int h_begin = min(wave * per, H), h_end = min(h_begin + per, H);
  for (int q = 0; q < p.stages; ++q) {
    const RvqStage st = p.stage[q];
    __syncthreads();
    for (int d0 = 0; d0 < D; d0 += 64) {
      const int d = min(d0 + lane, D - 1);
      float acc[FRAMES] = {};
#pragma unroll 16
      for (int h = h_begin; h < h_end; ++h) {
        const float w = st.project[static_cast<size_t>(h) * D + d];
#pragma unroll
        for (int f = 0; f < FRAMES; ++f)
          acc[f] = fmaf(w, residual(f, h), acc[f]);
      }
      if (d0 + lane < D)
#pragma unroll
        for (int f = 0; f < FRAMES; ++f)
          part[(wave * FRAMES + f) * D + d] = acc[f];
    }
    __syncthreads();
    for (int i = tid; i < FRAMES * D; i += kRvqThreads) {
      float sum = 0.0F;
#pragma unroll
      for (int w = 0; w < kRvqWaves; ++w)
        sum += part[w * FRAMES * D + i];
      v[i] = sum + st.bias[i % D];
    }
    __syncthreads();
    double best[FRAMES];
    int arg[FRAMES];
#pragma unroll
    for (int f = 0; f < FRAMES; ++f) {
      best[f] = -DBL_MAX;
      arg[f] = 0;
    }
    // Entries tid and tid + 512 of every 1024, their loads interleaved.
    for (int e0 = tid; e0 < E; e0 += 2 * kRvqThreads) {
      const int e1 = e0 + kRvqThreads;
      const float* c0 = st.embed + e0;
      const float* c1 = st.embed + min(e1, E - 1);
      double pp[FRAMES] = {}, dot0[FRAMES] = {}, dot1[FRAMES] = {};
#pragma unroll 8
      for (int d = 0; d < D; ++d) {
        const double w0 = c0[static_cast<size_t>(d) * E], w1 = c1[static_cast<size_t>(d) * E];
#pragma unroll
        for (int f = 0; f < FRAMES; ++f) {
          const double x = v[f * D + d];
          pp[f] += x * x;
          dot0[f] += x * w0;
          dot1[f] += x * w1;
        }
      }
      // Entries ascend per thread: ties keep the lower.
#pragma unroll
      for (int f = 0; f < FRAMES; ++f) {
        const double dist0 = -((pp[f] - 2.0 * dot0[f]) + st.norms[e0]);
        if (dist0 > best[f]) {
          best[f] = dist0;
          arg[f] = e0;
        }
        const double dist1 = -((pp[f] - 2.0 * dot1[f]) + st.norms[min(e1, E - 1)]);
        if (e1 < E && dist1 > best[f]) {
          best[f] = dist1;
          arg[f] = e1;
        }
      }
    }
#pragma unroll
    for (int f = 0; f < FRAMES; ++f) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) {
        const double od = __shfl_xor(best[f], o);
        const int oe = __shfl_xor(arg[f], o);
        if (od > best[f] || (od == best[f] && oe < arg[f])) {
          best[f] = od;
          arg[f] = oe;
        }
      }
      if (lane == 0) {
        best_d[f][wave] = best[f];
        best_e[f][wave] = arg[f];
      }
    }
    __syncthreads();
#pragma unroll
    for (int f = 0; f < FRAMES; ++f) {
      double top = best_d[f][0];
      int code = best_e[f][0];
#pragma unroll
      for (int w = 1; w < kRvqWaves; ++w)
        if (best_d[f][w] > top || (best_d[f][w] == top && best_e[f][w] < code)) {
          top = best_d[f][w];
          code = best_e[f][w];
        }
      if (tid == 0 && f0 + f < p.frames)
        p.codes[static_cast<size_t>(q) * p.frames + f0 + f] = code;
      if (kInLds || f0 + f < p.frames)
        for (int h = tid; h < H; h += kRvqThreads)
          residual(f, h) -= st.table[static_cast<size_t>(code) * H + h];
    }
  }
}

// The column kernel holds up to 32 rows per lane: 1024 channels.
constexpr int kMaxNormChannels = 32 * kLanes;

template <typename K>
void ColumnDispatch(int rows, K&& launch) {
  if (rows <= 8 * kLanes)
    launch(std::integral_constant<int, 8>());
  else if (rows <= 16 * kLanes)
    launch(std::integral_constant<int, 16>());
  else if (rows <= 24 * kLanes)
    launch(std::integral_constant<int, 24>());
  else
    launch(std::integral_constant<int, 32>());
}

int Blocks(size_t work) {
  return static_cast<int>(std::min<size_t>((work + kThreads - 1) / kThreads, 256 * 64));
}

}  // namespace

void LaunchTranspose(const float* x, float* y, int rows, int cols, hipStream_t stream) {
  Require(x && y, "transpose: null pointer");
  Require(rows >= 1 && cols >= 1 && rows <= 32 * 65535, "transpose: bad shape");
  Dispatch(TransposeKernel, dim3((cols + 31) / 32, (rows + 31) / 32), dim3(kThreads), 0, stream,
           true, true, x, y, rows, cols);
}

void LaunchResample(const ResampleParams& p, hipStream_t stream) {
  Require(p.x && p.bank && p.y, "resample: null pointer");
  Require(p.length >= 1 && p.from >= 1 && p.to >= 1 && p.taps >= 1 && p.width >= 0 &&
              p.out_length >= 1 && p.pad >= 0,
          "resample: bad shape");
  Dispatch(ResampleKernel, dim3(Blocks(static_cast<size_t>(p.out_length) + 2 * p.pad)),
           dim3(kThreads), 0, stream, true, true, p);
}

void LaunchGroupNormGelu(float* x, const float* w, const float* b, int channels, int length,
                         float eps, hipStream_t stream) {
  Require(x && w && b, "group norm: null pointer");
  Require(channels >= 1 && length >= 1, "group norm: empty shape");
  Dispatch(GroupNormGeluKernel, dim3(channels), dim3(kThreads), 0, stream, true, true, x, w, b,
           length, eps);
}

void LaunchColumnNorm(const ColumnNormParams& p, hipStream_t stream) {
  Require(p.x && p.y && p.w && p.b, "layer norm: null pointer");
  Require(p.sum_mode == 0 || p.sum != nullptr, "layer norm: no sum buffer");
  Require(p.channels >= 1 && p.channels <= kMaxNormChannels && p.positions >= 1,
          "layer norm: 1 to 1024 channels");
  ColumnDispatch(p.channels, [&](auto per) {
    Dispatch(ColumnNormKernel<decltype(per)::value>, dim3((p.positions + kCols - 1) / kCols),
             dim3(kThreads), 0, stream, true, true, p);
  });
}

std::size_t PackedHeadsElements(int heads, int head_dim, int steps) {
  const std::size_t tiles = (static_cast<std::size_t>(steps) + kAttentionTile - 1) / kAttentionTile;
  return heads * tiles * (2 * QkVectors(head_dim) + ValueVectors(head_dim)) * 8;
}

void LaunchHeadAttention(const HeadAttentionParams& p, hipStream_t stream) {
  Require(p.q && p.k && p.v && p.packed && p.out, "attention: null pointer");
  const int slabs = (p.head_dim + kAttentionDims - 1) / kAttentionDims;
  Require(p.heads >= 1 && p.heads <= 65535 && p.head_dim >= 1 && slabs <= 65535 &&
              p.steps >= 1,
          "attention: bad shape");
  const unsigned tiles = (p.steps + kAttentionTile - 1) / kAttentionTile;
  Dispatch(PackHeadsKernel, dim3(tiles, p.heads, 3), dim3(kThreads), 0, stream, true, false, p);
  const dim3 grid(tiles, p.heads, slabs);
  const std::uint32_t merge = kAttentionThreads / 64 * kAttentionDims * kAttentionTile * 4;
  const std::uint32_t queries = QkVectors(p.head_dim) * 16;
  if (p.head_dim <= 256)
    Dispatch(HeadAttentionKernel<true>, grid, dim3(kAttentionThreads), std::max(merge, queries),
             stream, false, true, p);
  else
    Dispatch(HeadAttentionKernel<false>, grid, dim3(kAttentionThreads), merge, stream, false,
             true, p);
}

void LaunchPickFrames(const double* sum, int channels, int positions, int stride, int frames,
                      double scale, float* y, hipStream_t stream) {
  Require(sum && y, "pick frames: null pointer");
  Require(channels >= 1 && frames >= 1 && stride >= 1 &&
              static_cast<int64_t>(frames - 1) * stride < positions,
          "pick frames: frames past the states");
  Dispatch(PickFramesKernel, dim3(Blocks(static_cast<size_t>(channels) * frames)),
           dim3(kThreads), 0, stream, true, true, sum, channels, positions, stride, frames,
           scale, y);
}

std::size_t RvqResidualElements(int dim, int hidden, int frames) {
  return RvqLdsBytes(1, dim, hidden) <= kRvqLdsLimit ? 0
                                                     : static_cast<std::size_t>(hidden) * frames;
}

void LaunchRvqEncode(const RvqEncodeParams& p, hipStream_t stream) {
  Require(p.x && p.stage && p.codes, "quantizer: null pointer");
  Require(p.dim >= 1 && p.dim <= kRvqMaxDim && p.entries >= 1 && p.hidden >= 1 &&
              p.frames >= 1 && p.stages >= 1,
          "quantizer: bad shape");
  Require(p.residual != nullptr || RvqResidualElements(p.dim, p.hidden, p.frames) == 0,
          "quantizer: no workspace");
  auto launch = [&](auto kernel, int frames, std::uint64_t bytes) {
    Dispatch(kernel, dim3((p.frames + frames - 1) / frames), dim3(kRvqThreads),
             static_cast<std::uint32_t>(bytes), stream, true, true, p);
  };
  // Two frames per work-group once one each would take more than one round of
  // the CUs.
  if (p.frames > kCus && RvqLdsBytes(2, p.dim, p.hidden) <= kRvqLdsLimit)
    launch(RvqEncodeKernel<2, true>, 2, RvqLdsBytes(2, p.dim, p.hidden));
  else if (RvqLdsBytes(1, p.dim, p.hidden) <= kRvqLdsLimit)
    launch(RvqEncodeKernel<1, true>, 1, RvqLdsBytes(1, p.dim, p.hidden));
  else
    launch(RvqEncodeKernel<1, false>, 1, RvqLdsBytes(1, p.dim, 0));
}

}  // namespace ovg
