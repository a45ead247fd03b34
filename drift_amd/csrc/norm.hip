// Row-wise norms for gfx950: RMSNorm (with the residual add), LayerNorm,
// AdaLN (LayerNorm then per-sample modulation, one pass) and modulate.
//
// Layout: row-major [rows, cols]. A row belongs to one wave (or to a group of
// four waves when it is long and rows are few), each lane holding K 16-byte
// chunks of it in registers, so the row crosses HBM once each way. Chunk k of
// lane l is chunk (k * W + wave) * 64 + l of the row: every load and store
// instruction of a wave covers 1 KiB of contiguous memory.
//
// Arithmetic is the runner's CPU reference's (ops/CpuNormalisation.scala:53-71,
// :128-151, ops/CpuElementwise.scala:33-38): sums, factor and every output in
// double, rounded once to float (then to bf16). CDNA4 runs double at the same
// vector rate as unpacked float, so this costs no more than float math and
// the results match the reference to the last bit but for sums taken in
// another order.
#include "common.hpp"

#include <algorithm>
#include <atomic>
#include <climits>

namespace drift {
namespace {

// The sum over a row's group of W waves (W = 1 or 4), the same in every lane.
template <int W>
__device__ __forceinline__ double row_sum(double v, double* partial) {
  v = group_sum<64>(v);
  if constexpr (W > 1) {
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) partial[wave] = v;
    __syncthreads();
    v = partial[0];
#pragma unroll
    for (int w = 1; w < W; ++w) v += partial[w];
    __syncthreads();  // partial is reused by the next sum
  }
  return v;
}

// Four or eight consecutive F32 weights, as the chunk of type T they pair with.
template <int N>
__device__ __forceinline__ void load_f32(const float* p, float (&v)[N]) {
#pragma unroll
  for (int j = 0; j < N; j += 4) {
    const float4 q = *reinterpret_cast<const float4*>(p + j);
    v[j] = q.x;
    v[j + 1] = q.y;
    v[j + 2] = q.z;
    v[j + 3] = q.w;
  }
}

// ------------------------------------------------------------------ RMSNorm

// A chunk's squares, summed in order in double. A row's sum of squares is
// taken as: per lane, its chunks' sums in increasing chunk order, then over
// the wave, then over the row's waves in order; with four waves a row, wave s
// holding the lane's chunks 64 * (4m + s) + lane. rms_norm_rows and
// rms_norm_wide keep that order, so a row norms the same in either.
template <int N>
__device__ __forceinline__ double chunk_squares(const float (&v)[N]) {
  double p = 0.0;
#pragma unroll
  for (int j = 0; j < N; ++j) p = fma((double)v[j], (double)v[j], p);  // the square is exact
  return p;
}

// 1 / sqrt(squares / cols + eps), the same in every kernel here (one form for
// any eps: with a second, shorter one chosen by eps > 0, bf16 [2000, 1024] took
// 7.8 us behind reads in place of 7.4).
__device__ __forceinline__ double row_factor(double squares, int cols, float eps) {
  const double mean = squares / (double)cols + (double)eps;
  return inverse_sqrt(mean);
}

// The variance from a row's moments about one of its values. Rounding may take
// it below zero; a NaN (of a row with an infinity or a NaN in it) stays one, as
// two passes give and the reference writes.
__device__ __forceinline__ double moment_variance(double s2, double m1, double inverse_cols) {
  const double v = fma(s2, inverse_cols, -(m1 * m1));
  return v < 0.0 ? 0.0 : v;
}

// With q.xq, out is quantized too as it is written (quantize_chunk; cols a
// multiple of 32, so a row holds whole blocks).
template <typename T, int K, int W>
__global__ void __launch_bounds__(256) rms_norm_rows(T* x, const T* y, const float* weight, T* out, int64_t rows,
                                                     int cols, float eps, float offset, int weight_rows,
                                                     Quantized q) {
  constexpr int N = Chunk<T>::N;
  constexpr int kRowsPerBlock = 4 / W;
  __shared__ double partial[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = wave % W;
  const int chunks = cols / N;
  for (int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + wave / W; row < rows;
       row += (int64_t)gridDim.x * kRowsPerBlock) {
    T* xr = x + row * cols;
    const float* w = weight + (row % weight_rows) * cols;
    // Short rows (decode) are latency-bound: their weights are loaded with x,
    // before the sum, so the two loads' latencies overlap.
    constexpr bool kEarlyWeights = K * N <= 16;
    float early[kEarlyWeights ? K : 1][N];
    if constexpr (kEarlyWeights) {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int c = (k * W + sub) * kWave + lane;
        if (c < chunks) load_f32<N>(w + c * N, early[k]);
      }
    }
    float v[K][N];
    double squares = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k * W + sub) * kWave + lane;
      if (c < chunks) {
        Chunk<T>::load(xr + c * N, v[k]);
        if (y) {
          float u[N];
          Chunk<T>::load(y + row * cols + c * N, u);
#pragma unroll
          for (int j = 0; j < N; ++j) v[k][j] += u[j];  // the F32 sum, as add() rounds it
        }
        squares += chunk_squares(v[k]);
      }
    }
    squares = row_sum<W>(squares, partial);
    const double factor = row_factor(squares, cols, eps);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k * W + sub) * kWave + lane;
      if (c < chunks) {
        if (y) Chunk<T>::store(xr + c * N, v[k]);  // the residual stream, before out (which may be x)
        float wv[N], o[N];
        if constexpr (kEarlyWeights) {
#pragma unroll
          for (int j = 0; j < N; ++j) wv[j] = early[k][j];
        } else {
          load_f32<N>(w + c * N, wv);
        }
#pragma unroll
        for (int j = 0; j < N; ++j) o[j] = (float)((double)v[k][j] * factor * ((double)wv[j] + (double)offset));
        Chunk<T>::store(out + row * cols + c * N, o);
        if (q.xq) {
          as_written<T>(o);
          quantize_chunk<N>(o, (row * cols + c * N) / 32, q);
        }
      }
    }
  }
}

// Many long rows, no side output and one weight row: a wave per row, in
// one-wave blocks, so a row waits on no barrier; its sum is taken in the
// four-wave group's order (chunk_squares): four sums over the wave, chunk k's
// squares in sum k % 4. Loads are never branched around (chunks past the row
// are clamped to its last and left out).
//
// Once a row a wave (RESIDENT false) the weights are read after the sum, from
// the L1 (at 5120 values they are 20 KiB of it, and more registers hold fewer
// waves); RESIDENT keeps them in registers over the rows a wave takes, with
// the next row's loads in flight. Memory bounds it. Measured, us a launch in
// graph replays, four-wave group / once a row / RESIDENT at a wave a SIMD:
//   bf16 [4093, 4096] 15.8 / 12.6 / 13.5, with the residual 26.4 / 22.6 / 25.3
//   F32 [2000, 2560] 11.8 / 7.6 / 8.3, with the residual 16.7 / 13.6 / 14.2
//   F32 [2500, 5120] 22.9 / 17.9 / 20.1, with the residual 37.2 / 40.8 / 53.6
//   bf16 [6000, 4096] 21.5 / 17.6 / 18.7, with the residual 36.4 / 39.0 / 36.4
//   bf16 [14040, 3072] 39.0 / 33.2 / 31.4 (172 MB), with the residual 64.3 / 61.8 / 59.9
//   bf16 [8000, 5120] 36.1 / 36.6 / 30.3, with the residual 61.1 / 60.9 / 59.3
//   F32 [7800, 3072] 37.4 / 37.5 / 33.5, with the residual 65.2 / 70.8 / 67.8
//   bf16 [1000, 4096] 5.3 / 5.4 / 4.8; F32 [509, 2560] 4.8 / 4.7 / 3.9; bf16 [300, 4096] 3.8 / 4.4 / 3.9,
//   with the residual 5.0 / 6.1 / 6.0
// Alone, two waves a SIMD in the resident grid were 1 to 4% slower on the
// larger of these, three and four up to 15%.
//
// KEEP: the output is stored through the caches, for the rope that reads it
// next. RMSNorm and ropeTable (or rope3d) of queries and keys, bf16 [14040,
// 3072] 122.0 -> 116.2 (125.5 -> 114.4), [12470, 3072] 109.9 -> 104.6; in a
// dense layer, whose next kernels do not read it, 119.6 -> 131.0 for 4,093
// tokens of 4096. Rows past the resident line keep it, where such a layer is
// even: behind a matrix product 7,168 tokens of 4096 223.0 -> 221.5, 8,192 249.1
// -> 250.7, 16,384 480.3 -> 478.8, F32 8,192 of 2560 340.9 -> 344.9 (behind reads
// 343.0 -> 339.2), and the norm by itself bf16 [8192, 4096] 28.6 -> 26.8, F32
// 50.7 -> 46.4, bf16 [16384, 4096] 50.7 -> 46.5.
template <typename T, int K, bool ADD, bool RESIDENT, bool KEEP>
__global__ void __launch_bounds__(kWave) rms_norm_waves(T* x, const T* y, const float* weight, T* out, int64_t rows,
                                                        int cols, float eps, float offset) {
  constexpr int N = Chunk<T>::N;
  using Raw = typename Chunk<T>::Raw;
  const int lane = threadIdx.x;
  const int chunks = cols / N;
  auto load_row = [&](int64_t r, Raw(&into)[K], Raw(&also)[ADD ? K : 1]) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = min(k * kWave + lane, chunks - 1);
      into[k] = Chunk<T>::load_raw(x + r * cols + c * N);
      if constexpr (ADD) also[k] = Chunk<T>::load_raw(y + r * cols + c * N);
    }
  };
  int64_t row = blockIdx.x;
  Raw raw[K], add[ADD ? K : 1];
  load_row(row, raw, add);
  float w[RESIDENT ? K : 1][N];
  if constexpr (RESIDENT) {
#pragma unroll
    for (int k = 0; k < K; ++k) load_f32<N>(weight + min(k * kWave + lane, chunks - 1) * N, w[k]);
  }
  // chunk k's values, with the residual the F32 sum as add() rounds it
  auto values = [&](int k, float(&v)[N]) {
    Chunk<T>::unpack(raw[k], v);
    if constexpr (ADD) {
      float u[N];
      Chunk<T>::unpack(add[k], u);
#pragma unroll
      for (int j = 0; j < N; ++j) v[j] += u[j];
    }
  };
  while (true) {
    const int64_t following = row + gridDim.x;
    Raw next[K], next_add[ADD ? K : 1];
    if constexpr (RESIDENT)
      if (following < rows) load_row(following, next, next_add);
    constexpr int kSums = K < 4 ? K : 4;
    double sums[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < K; ++k) {
      float v[N];
      values(k, v);
      const double squares = chunk_squares(v);
      sums[k % 4] += k * kWave + lane < chunks ? squares : 0.0;
    }
#pragma unroll
    for (int i = 0; i < kSums; ++i) sums[i] = group_sum<64>(sums[i]);
    const double factor = row_factor(((sums[0] + sums[1]) + sums[2]) + sums[3], cols, eps);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = k * kWave + lane;
      if (c < chunks) {
        opaque(raw[k]);
        if constexpr (ADD) opaque(add[k]);
        float v[N], wk[N], o[N];
        values(k, v);
        if constexpr (ADD) Chunk<T>::store(x + row * cols + c * N, v);  // before out (which may be x)
        if constexpr (RESIDENT) {
#pragma unroll
          for (int j = 0; j < N; ++j) wk[j] = w[k][j];
        } else {
          load_f32<N>(weight + c * N, wk);
        }
#pragma unroll
        for (int j = 0; j < N; ++j) o[j] = (float)((double)v[j] * factor * ((double)wk[j] + (double)offset));
        if constexpr (KEEP) Chunk<T>::store_cached(out + row * cols + c * N, o);
        else Chunk<T>::store(out + row * cols + c * N, o);
      }
    }
    if constexpr (!RESIDENT) return;
    if (following >= rows) return;
    row = following;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      raw[k] = next[k];
      if constexpr (ADD) add[k] = next_add[k];
    }
  }
}

// Rows of at most 64 chunks (attention heads): G lanes a row, G the power of
// two at or above its chunks, a wave taking U passes of 64 / G rows, every
// load issued before the first sum and the lane's weights read once for all
// its rows. The sum over G lanes is the wave's with zeros beyond
// (rms_norm_rows), the same to the last bit. Memory bounds it from about 10
// MB. Measured, us a launch in graph replays, rms_norm_rows (a row a wave,
// half its lanes or more idle) / U = 1 / 2 / 4 / 8:
//   F32 [65248, 128] 22.3 / 12.1 / 12.6 / 12.7 / 12.8
//   bf16 [157104, 256] (161 MB) 60.4 / 29.5 / 28.1 / 27.8 / 29.4
//   bf16 [100000, 128] 38.2 / 10.8 / 10.8 / 10.8 / 11.5
//   F32 [70000, 72] 21.8 / 10.8 / 9.4 / 9.7 / 10.2
//   bf16 [4192, 256] 3.5 / 2.5 / - / 3.1 / -; F32 [32, 128] 1.95 / 1.75 / - / 2.2 / -
//
// KEEP: the output is stored through the caches, for the rope that reads it
// next (F32: norms, ropes and the cache write of 2,039 tokens of 32 + 8 heads
// 42.6 -> 40.1, of 5,000 87.4 -> 83.3; BF16 moved 2% either way by shape).
template <typename T, int G, int U, bool KEEP>
__global__ void __launch_bounds__(kWave) rms_norm_groups(const T* x, const float* weight, T* out, int64_t rows,
                                                         int cols, float eps, float offset) {
  constexpr int N = Chunk<T>::N;
  constexpr int kRows = kWave / G;
  const int lane = threadIdx.x;
  const bool inside = lane % G < cols / N;
  const int c = min(lane % G, cols / N - 1) * N;
  const int64_t first = (int64_t)blockIdx.x * (kRows * U) + lane / G;
  typename Chunk<T>::Raw raw[U];
#pragma unroll
  for (int u = 0; u < U; ++u) raw[u] = Chunk<T>::load_raw(x + min(first + u * kRows, rows - 1) * cols + c);
  float w[N];
  load_f32<N>(weight + c, w);
#pragma unroll
  for (int u = 0; u < U; ++u) {
    float v[N], o[N];
    Chunk<T>::unpack(raw[u], v);
    double squares = chunk_squares(v);
    if (!inside) squares = 0.0;
    const double factor = row_factor(group_sum<G>(squares), cols, eps);
    const int64_t row = first + u * kRows;
#pragma unroll
    for (int j = 0; j < N; ++j) o[j] = (float)((double)v[j] * factor * ((double)w[j] + (double)offset));
    if (inside && row < rows) {
      if constexpr (KEEP) Chunk<T>::store_cached(out + row * cols + c, o);
      else Chunk<T>::store(out + row * cols + c, o);
    }
  }
}

// Few rows (a decode step's tokens): a row's chunks spread over W = 8 or 16
// waves (512 or 1024 threads), so each lane's serial work is 2 or 4 times
// shorter than in the four-wave group. The chunks' sums of squares go through
// LDS to the first four waves, which add them in the four-wave group's order
// (chunk_squares), so the result is the same to the last bit.
template <typename T, int K, int W>
__global__ void __launch_bounds__(64 * W) rms_norm_wide(T* x, const T* y, const float* weight, T* out, int64_t rows,
                                                       int cols, float eps, float offset, int weight_rows,
                                                       Quantized q) {
  static_assert(W == 8 || W == 16, "the wide group is 8 or 16 waves");
  constexpr int N = Chunk<T>::N;
  constexpr int kSlots = K * W;  // 64-chunk slots a row can have
  __shared__ double sums[kSlots][kWave];
  __shared__ double partial[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int chunks = cols / N;
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    T* xr = x + row * cols;
    const float* w = weight + (row % weight_rows) * cols;
    float wv[K][N];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k * W + wave) * kWave + lane;
      if (c < chunks) load_f32<N>(w + c * N, wv[k]);
    }
    float v[K][N];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int slot = k * W + wave, c = slot * kWave + lane;
      if (c < chunks) {
        Chunk<T>::load(xr + c * N, v[k]);
        if (y) {
          float u[N];
          Chunk<T>::load(y + row * cols + c * N, u);
#pragma unroll
          for (int j = 0; j < N; ++j) v[k][j] += u[j];
        }
        sums[slot][lane] = chunk_squares(v[k]);
      }
    }
    __syncthreads();
    if (wave < 4) {
      double squares = 0.0;
#pragma unroll
      for (int m = 0; m < kSlots / 4; ++m) {
        const int slot = 4 * m + wave;
        if (slot * kWave + lane < chunks) squares += sums[slot][lane];
      }
      squares = group_sum<64>(squares);
      if (lane == 0) partial[wave] = squares;
    }
    __syncthreads();
    const double total = ((partial[0] + partial[1]) + partial[2]) + partial[3];
    const double factor = row_factor(total, cols, eps);
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k * W + wave) * kWave + lane;
      if (c < chunks) {
        if (y) Chunk<T>::store(xr + c * N, v[k]);
        float o[N];
#pragma unroll
        for (int j = 0; j < N; ++j) o[j] = (float)((double)v[k][j] * factor * ((double)wv[k][j] + (double)offset));
        Chunk<T>::store(out + row * cols + c * N, o);
        if (q.xq) {
          as_written<T>(o);
          quantize_chunk<N>(o, (row * cols + c * N) / 32, q);
        }
      }
    }
    __syncthreads();  // sums and partial are reused by the next row
  }
}

// Any width and alignment: a block of 256 per row, reading the row twice.
template <typename T>
__global__ void __launch_bounds__(256) rms_norm_rows_scalar(T* x, const T* y, const float* weight, T* out,
                                                            int64_t rows, int cols, float eps, float offset,
                                                            int weight_rows) {
  __shared__ double partial[4];
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    T* xr = x + row * cols;
    const T* yr = y ? y + row * cols : nullptr;
    double squares = 0.0;
    for (int c = threadIdx.x; c < cols; c += 256) {
      float v = load_one(xr + c);
      if (yr) v += load_one(yr + c);
      squares += (double)v * (double)v;
    }
    squares = row_sum<4>(squares, partial);
    const double factor = row_factor(squares, cols, eps);
    const float* w = weight + (row % weight_rows) * cols;
    for (int c = threadIdx.x; c < cols; c += 256) {
      float v = load_one(xr + c);
      if (yr) {
        v += load_one(yr + c);
        store_one(xr + c, v);
      }
      store_one(out + row * cols + c, (float)((double)v * factor * ((double)w[c] + (double)offset)));
    }
  }
}

// Narrow rows (at most 32 values, a pixel's channels, often millions of
// rows): a thread per row, as the reference's rms_norm_narrow_f32
// (kernels/norm.hip:414-426). The sum runs over the row in order, as the
// CPU's left fold does, so the result is the CPU's to the last bit.
constexpr int kNarrowCols = 32;

template <typename T>
__global__ void __launch_bounds__(256) rms_norm_narrow(T* x, const T* y, const float* weight, T* out, int64_t rows,
                                                       int cols, float eps, float offset, int weight_rows) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; row < rows; row += stride) {
    T* xr = x + row * cols;
    const T* yr = y ? y + row * cols : nullptr;
    float v[kNarrowCols];
    double squares = 0.0;
#pragma unroll
    for (int c = 0; c < kNarrowCols; ++c) {
      if (c < cols) {
        v[c] = load_one(xr + c);
        if (yr) v[c] += load_one(yr + c);
        squares += (double)v[c] * (double)v[c];
      }
    }
    const double factor = row_factor(squares, cols, eps);
    const float* w = weight + (row % weight_rows) * cols;
#pragma unroll
    for (int c = 0; c < kNarrowCols; ++c) {
      if (c < cols) {
        if (yr) store_one(xr + c, v[c]);
        store_one(out + row * cols + c, (float)((double)v[c] * factor * ((double)w[c] + (double)offset)));
      }
    }
  }
}

// ------------------------------------------------------------------ LayerNorm / AdaLN

// MODULATE false: out = normal * (weight or 1) + (bias or 0).
// MODULATE true: n = float(normal + 0) (layerNorm's F32 result, no affine),
// out = n * (1 + scale[s, c]) + shift[s, c], s the row's sample.
template <typename T, int K, int W, bool MODULATE>
__global__ void __launch_bounds__(256) layer_norm_rows(const T* x, const float* weight, const float* bias, T* out,
                                                       int64_t rows, int cols, int64_t rows_per_sample, float eps) {
  constexpr int N = Chunk<T>::N;
  constexpr int kRowsPerBlock = 4 / W;
  __shared__ double partial[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int sub = wave % W;
  const int chunks = cols / N;
  for (int64_t row = (int64_t)blockIdx.x * kRowsPerBlock + wave / W; row < rows;
       row += (int64_t)gridDim.x * kRowsPerBlock) {
    float v[K][N];
    double sum = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k * W + sub) * kWave + lane;
      if (c < chunks) {
        Chunk<T>::load(x + row * cols + c * N, v[k]);
#pragma unroll
        for (int j = 0; j < N; ++j) sum += (double)v[k][j];
      }
    }
    const double mean = row_sum<W>(sum, partial) / (double)cols;
    double squares = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k * W + sub) * kWave + lane;
      if (c < chunks) {
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const double d = (double)v[k][j] - mean;
          squares = fma(d, d, squares);
        }
      }
    }
    const double factor = row_factor(row_sum<W>(squares, partial), cols, eps);
    const float* s0 = weight;  // MODULATE: the sample's scale row
    const float* s1 = bias;    // MODULATE: the sample's shift row
    if constexpr (MODULATE) {
      const int64_t sample = row / rows_per_sample;
      s0 = weight + sample * cols;
      s1 = bias + sample * cols;
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = (k * W + sub) * kWave + lane;
      if (c < chunks) {
        float o[N];
        if constexpr (MODULATE) {
          float sc[N], sh[N];
          load_f32<N>(s0 + c * N, sc);
          load_f32<N>(s1 + c * N, sh);
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const float n = (float)fma((double)v[k][j] - mean, factor, 0.0);
            o[j] = (float)fma((double)n, 1.0 + (double)sc[j], (double)sh[j]);
          }
        } else {
          float wv[N], bv[N];
          if (s0) load_f32<N>(s0 + c * N, wv);
          if (s1) load_f32<N>(s1 + c * N, bv);
#pragma unroll
          for (int j = 0; j < N; ++j) {
            const double normal = ((double)v[k][j] - mean) * factor;
            o[j] = (float)(normal * (s0 ? (double)wv[j] : 1.0) + (s1 ? (double)bv[j] : 0.0));
          }
        }
        Chunk<T>::store(out + row * cols + c * N, o);
      }
    }
  }
}

// LayerNorm of many rows of four waves' chunks: a wave a row in one-wave
// blocks, so a row waits on no barrier (the four-wave group has four). Its
// sums are taken in the four-wave group's order, chunk k's in sum k % 4. The
// weights and biases are read after the sums: read first, their registers (as
// doubles) held half as many waves. Measured, us a launch in graph replays,
// four-wave group / weights first / this: [4087, 1152] (38 MB) 12.6 / 8.9 /
// 8.4, [4830, 1280] 14.9 / 12.7 / 9.8, [9000, 1024] 19.1 / 18.1 / 15.5. The
// group stays up to 2^19 chunks, and up to 1,792 rows of at most 6 chunks a
// lane and 2,048 of longer ones: at two rows a SIMD a row's own chain counts,
// which replays of one buffer hide. With events around the launch, its input
// left by earlier work in the MALL / just written / in HBM, group against this:
// [1700, 1536] 10.2 against 10.5, even, 14% slower, [1800, 1536] 12.4 against
// 10.6, 5% and 4% faster; [1100, 3072] 11.0 / 10.5 / 11.0 against 14.0 / 14.5 /
// 17.6, [1700, 3072] 15.0 / 13.8 / 15.4 against 14.8 / 15.8 / 19.0, [2000, 2560]
// 15.2 / 14.1 / 15.1 against 14.3 / 14.1 / 17.3, [2300, 2560] 17.6 / 15.3 / 16.8
// against 15.0 / 14.6 / 18.1, [3000, 3072] 22.4 / 19.0 / 22.2 against 18.9 / 18.2
// / 21.9.
//
// MODULATE (as layer_norm_rows): AdaLN rows of 4,097 to 5,120 values, past
// adaln_launch's, a sample's rows by blockIdx.y, in 256-thread blocks. Us a
// launch, events around it, its input in HBM behind a matrix product / just
// written, four-wave group against one-wave blocks and these: bf16 [16380,
// 5120] 105.3 / 88.2, 80.9 / 67.4, 80.7 / 66.2; bf16 [4000, 5120] 30.7 / 26.0,
// 23.1 / 23.0, 22.2 / 22.0; F32 [16380, 5120] 183.8 / 155.9, 130.8 / 129.1,
// 131.1 / 130.5; F32 [1700, 5120] 24.7 / 20.5, 18.8 / 18.8, 18.8 / 18.5. At
// 1,500 rows bf16 15.3 / 14.0 in the group, 14.4 / 14.1 here, and with the
// input in HBM behind reads 15.7 and 17.0 (F32 21.3 and 24.7): up to 1,536
// rows (one and a half a SIMD) keep the group.
template <bool MODULATE>
constexpr int kNormBlock = MODULATE ? 256 : kWave;

template <typename T, int K, bool MODULATE>
__global__ void __launch_bounds__(kNormBlock<MODULATE>) layer_norm_waves(const T* x, const float* weight,
                                                                       const float* bias, T* out, int64_t rows,
                                                                       int cols, int64_t rows_per_sample, float eps) {
  constexpr int N = Chunk<T>::N;
  const int lane = threadIdx.x & 63;
  const int chunks = cols / N;
  int64_t row = (int64_t)blockIdx.x * (kNormBlock<MODULATE> / kWave) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if constexpr (MODULATE) {
    if (row >= rows_per_sample) return;
    row += (int64_t)blockIdx.y * rows_per_sample;
    if (row >= rows) return;
    weight += (int64_t)blockIdx.y * cols;
    bias += (int64_t)blockIdx.y * cols;
  }
  typename Chunk<T>::Raw raw[K];
#pragma unroll
  for (int k = 0; k < K; ++k) raw[k] = Chunk<T>::load_raw(x + row * cols + min(k * kWave + lane, chunks - 1) * N);
  constexpr int kSums = K < 4 ? K : 4;
  double sums[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int k = 0; k < K; ++k) {
    float v[N];
    Chunk<T>::unpack(raw[k], v);
    if (k * kWave + lane < chunks) {
#pragma unroll
      for (int j = 0; j < N; ++j) sums[k % 4] += (double)v[j];
    }
  }
#pragma unroll
  for (int i = 0; i < kSums; ++i) sums[i] = group_sum<64>(sums[i]);
  const double mean = (((sums[0] + sums[1]) + sums[2]) + sums[3]) / (double)cols;
#pragma unroll
  for (int i = 0; i < 4; ++i) sums[i] = 0.0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    opaque(raw[k]);
    float v[N];
    Chunk<T>::unpack(raw[k], v);
    if (k * kWave + lane < chunks) {
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const double d = (double)v[j] - mean;
        sums[k % 4] = fma(d, d, sums[k % 4]);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < kSums; ++i) sums[i] = group_sum<64>(sums[i]);
  const double factor = row_factor(((sums[0] + sums[1]) + sums[2]) + sums[3], cols, eps);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = k * kWave + lane;
    if (c < chunks) {
      opaque(raw[k]);
      float v[N], w[N], b[N], o[N];
      Chunk<T>::unpack(raw[k], v);
      if (MODULATE || weight) load_f32<N>(weight + c * N, w);
      if (MODULATE || bias) load_f32<N>(bias + c * N, b);
#pragma unroll
      for (int j = 0; j < N; ++j) {
        if constexpr (MODULATE) {
          const float n = (float)fma((double)v[j] - mean, factor, 0.0);
          o[j] = (float)fma((double)n, 1.0 + (double)w[j], (double)b[j]);
        } else {
          const double normal = ((double)v[j] - mean) * factor;
          o[j] = (float)(normal * (weight ? (double)w[j] : 1.0) + (bias ? (double)b[j] : 0.0));
        }
      }
      Chunk<T>::store(out + row * cols + c * N, o);
    }
  }
}

template <typename T, bool MODULATE>
__global__ void __launch_bounds__(256) layer_norm_rows_scalar(const T* x, const float* weight, const float* bias,
                                                              T* out, int64_t rows, int cols,
                                                              int64_t rows_per_sample, float eps) {
  __shared__ double partial[4];
  for (int64_t row = blockIdx.x; row < rows; row += gridDim.x) {
    const T* xr = x + row * cols;
    double sum = 0.0;
    for (int c = threadIdx.x; c < cols; c += 256) sum += (double)load_one(xr + c);
    const double mean = row_sum<4>(sum, partial) / (double)cols;
    double squares = 0.0;
    for (int c = threadIdx.x; c < cols; c += 256) {
      const double d = (double)load_one(xr + c) - mean;
      squares = fma(d, d, squares);
    }
    const double factor = row_factor(row_sum<4>(squares, partial), cols, eps);
    const float* s0 = weight;
    const float* s1 = bias;
    if constexpr (MODULATE) {
      const int64_t sample = row / rows_per_sample;
      s0 = weight + sample * cols;
      s1 = bias + sample * cols;
    }
    for (int c = threadIdx.x; c < cols; c += 256) {
      const double d = (double)load_one(xr + c) - mean;
      float o;
      if constexpr (MODULATE) {
        const float n = (float)fma(d, factor, 0.0);
        o = (float)fma((double)n, 1.0 + (double)s0[c], (double)s1[c]);
      } else {
        o = (float)(d * factor * (s0 ? (double)s0[c] : 1.0) + (s1 ? (double)s1[c] : 0.0));
      }
      store_one(out + row * cols + c, o);
    }
  }
}

// F32 AdaLN, one wave per row, four rows of one sample per block (grid.y =
// sample), the grid covering the rows in one pass. Each lane reads its
// chunks' scale and shift from the sample's rows (cached: every row of the
// sample reads them). One-wave blocks spread a sample of few rows over every
// XCD, each of which fetches its table: us a launch behind a matrix product,
// one-wave blocks / these: [2000, 3072] of 256 samples 18.5 / 14.0, [4000,
// 1536] of 1,000 17.9 / 13.4, [7000, 3840] of 1,000 64.0 / 48.0, of one 46.0 /
// 44.9; [1500, 3840] of one 14.4 / 14.5.
//
// The mean and variance come from one pass over the row about its first
// value x0 (sums of d = x - x0 and d^2): the same as the reference's two
// passes to the last bits, since |mean - x0| is a few standard deviations at
// most. The arithmetic is the reference's, in double: n = float((x - mean) *
// factor) is layerNorm's F32 result, out = n * (1 + scale) + shift rounded
// once, as modulate.
constexpr int kAdalnMaxCols = 4096;

template <int K, bool FULL>
__global__ void __launch_bounds__(256) adaln_waves(const float* x, const float* scale, const float* shift, float* out,
                                                   int64_t rows, int cols, int64_t rows_per_sample, float eps) {
  constexpr int N = 4;
  using Raw = uint4;
  const int chunks = FULL ? K * kWave : cols / N;
  const int64_t sample = blockIdx.y;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t row = sample * rows_per_sample + (int64_t)blockIdx.x * 4 + wave;
  if (row >= min(rows, (sample + 1) * rows_per_sample)) return;
  Raw raw[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = k * kWave + lane;
    if (FULL || c < chunks) raw[k] = Chunk<float>::load_raw(x + row * cols + c * N);
  }
  float first_value[N];
  Chunk<float>::unpack(raw[0], first_value);
  const double x0 = (double)__shfl(first_value[0], 0);
  double s1 = 0.0, s2 = 0.0;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if (FULL || k * kWave + lane < chunks) {
      float v[N];
      Chunk<float>::unpack(raw[k], v);
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const double d = (double)v[j] - x0;
        s1 += d;
        s2 = fma(d, d, s2);
      }
    }
  }
  s1 = group_sum<64>(s1);
  s2 = group_sum<64>(s2);
  const double inverse_cols = 1.0 / (double)cols;
  const double m1 = s1 * inverse_cols;  // mean - x0
  const double mean = x0 + m1;
  const double variance = moment_variance(s2, m1, inverse_cols);
  const double factor = eps > 0.0f ? inverse_sqrt<true>(variance + (double)eps) : inverse_sqrt(variance + (double)eps);
  const double offset = -mean * factor;
  const float* sc = scale + sample * cols;
  const float* sh = shift + sample * cols;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = k * kWave + lane;
    if (FULL || c < chunks) {
      opaque(raw[k]);
      float v[N], o[N], a[N], b[N];
      Chunk<float>::unpack(raw[k], v);
      load_f32<N>(sc + c * N, a);
      load_f32<N>(sh + c * N, b);
#pragma unroll
      for (int j = 0; j < N; ++j) {
        const float n = (float)fma((double)v[j], factor, offset);
        o[j] = (float)fma((double)n, 1.0 + (double)a[j], (double)b[j]);
      }
      Chunk<float>::store(out + row * cols + c * N, o);
    }
  }
}

// F32 AdaLN of few rows (up to one a wave) or many (seven or more a wave), at
// a wave a SIMD: the lane's scale and shift in registers across the rows it
// takes, the next row's loads in flight (adaln_resident's plan, the tables
// kept as float: as doubles they would not fit). Measured against adaln_waves
// in 256-thread blocks, us a launch in graph replays: [300, 3072] 5.0 -> 4.1,
// [7800, 3072] (192 MB) 36.9 -> 34.9, [16000, 3072] of two samples 70.8 ->
// 69.5, [8190, 1536] 19.2 -> 18.1; but [1500, 3840] 11.2 against 9.5. In many
// samples it is slower alone ([8192, 3072] of 64, behind a matrix product 41.8
// against 45.2, just written 34.9 against 42.3), but a block's convert, AdaLN,
// gatedAdd, AdaLN, GELU-tanh of those rows is faster with it, 201.9 -> 183.6
// (of one sample 177.9 -> 171.5).
template <int K, bool FULL>
__global__ void __launch_bounds__(kWave) adaln_resident_f32(const float* x, const float* scale, const float* shift,
                                                      float* out, int64_t rows, int cols, int64_t rows_per_sample,
                                                      float eps, int64_t waves_per_sample) {
  constexpr int N = 4;
  using Raw = uint4;
  const int chunks = FULL ? K * kWave : cols / N;
  const int64_t sample = blockIdx.y;
  const int lane = threadIdx.x;
  const int64_t w = blockIdx.x;
  const int64_t end = min(rows, (sample + 1) * rows_per_sample);
  int64_t row = sample * rows_per_sample + w;
  if (row >= end) return;
  auto load_row = [&](int64_t r, Raw(&into)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = FULL ? k * kWave + lane : min(k * kWave + lane, chunks - 1);
      into[k] = stream_load(x + r * cols + c * N);
    }
  };
  Raw raw[K];
  load_row(row, raw);
  float a[K][N], b[K][N];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = FULL ? k * kWave + lane : min(k * kWave + lane, chunks - 1);
    load_f32<N>(scale + sample * cols + c * N, a[k]);
    load_f32<N>(shift + sample * cols + c * N, b[k]);
  }
  const double inverse_cols = 1.0 / (double)cols;
  for (; row < end; row += waves_per_sample) {
    Raw next[K];
    if (row + waves_per_sample < end) load_row(row + waves_per_sample, next);
    const double x0 = (double)__shfl(__uint_as_float(raw[0].x), 0);
    double s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (FULL || k * kWave + lane < chunks) {
        float v[N];
        Chunk<float>::unpack(raw[k], v);
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const double d = (double)v[j] - x0;
          s1 += d;
          s2 = fma(d, d, s2);
        }
      }
    }
    s1 = group_sum<64>(s1);
    s2 = group_sum<64>(s2);
    const double m1 = s1 * inverse_cols;
    const double mean = x0 + m1;
    const double variance = moment_variance(s2, m1, inverse_cols);
    const double var_eps = variance + (double)eps;
    const double factor = eps > 0.0f ? inverse_sqrt<true>(var_eps) : inverse_sqrt(var_eps);
    const double offset = -mean * factor;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = k * kWave + lane;
      if (FULL || c < chunks) {
        opaque(raw[k]);
        float v[N], o[N];
        Chunk<float>::unpack(raw[k], v);
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const float n = (float)fma((double)v[j], factor, offset);
          o[j] = (float)fma((double)n, 1.0 + (double)a[k][j], (double)b[k][j]);
        }
        Chunk<float>::store(out + row * cols + c * N, o);
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) raw[k] = next[k];
  }
}

// BF16 AdaLN with each lane's (1 + scale, shift) held in registers across the
// rows it takes: re-reading them per row would move four times the row's own
// bytes through the L1. Wave w of a sample takes rows w, w + W, w + 2W, ... of
// it (W waves per sample, all resident at once), with the next row's loads in
// flight while it computes the current one.
//
// The arithmetic is adaln_waves', in double. It has to be: where the output
// nearly cancels (n * (1 + scale) ~ -shift) a float ulp of n or of 1 + scale
// is many bf16 ulps of the result. d = x - x0 is exact in float for bf16
// values within a factor 2^15 of each other, and d^2 exact in double.
template <int K, bool FULL>
__global__ void __launch_bounds__(256) adaln_resident(const uint16_t* x, const float* scale, const float* shift,
                                                      uint16_t* out, int64_t rows, int cols, int64_t rows_per_sample,
                                                      float eps, int64_t waves_per_sample) {
  constexpr int N = 8;
  using Raw = uint4;
  const int chunks = FULL ? K * kWave : cols / N;
  const int64_t sample = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int64_t w = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t end = min(rows, (sample + 1) * rows_per_sample);
  int64_t row = sample * rows_per_sample + w;
  if (w >= waves_per_sample || row >= end) return;
  auto load_row = [&](int64_t r, Raw(&into)[K]) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = k * kWave + lane;
      if (FULL || c < chunks) into[k] = Chunk<uint16_t>::load_raw(x + r * cols + c * N);
    }
  };
  Raw raw[K];
  load_row(row, raw);
  double a[K][N];
  float b[K][N];
  const float* sc = scale + sample * cols;
  const float* sh = shift + sample * cols;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int c = k * kWave + lane;
    if (FULL || c < chunks) {
      float f[N];
      load_f32<N>(sc + c * N, f);
      load_f32<N>(sh + c * N, b[k]);
#pragma unroll
      for (int j = 0; j < N; ++j) a[k][j] = 1.0 + (double)f[j];
    }
  }
  const double inverse_cols = 1.0 / (double)cols;
  for (; row < end; row += waves_per_sample) {
    Raw next[K];
    if (row + waves_per_sample < end) load_row(row + waves_per_sample, next);
    float first_value[N];
    Chunk<uint16_t>::unpack(raw[0], first_value);
    const float x0 = __shfl(first_value[0], 0);
    double s1 = 0.0, s2 = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      if (FULL || k * kWave + lane < chunks) {
        float v[N];
        Chunk<uint16_t>::unpack(raw[k], v);
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const double d = (double)(v[j] - x0);
          s1 += d;
          s2 = fma(d, d, s2);
        }
      }
    }
    s1 = group_sum<64>(s1);
    s2 = group_sum<64>(s2);
    // the row's statistics are a chain the wave waits on, alone on its
    // SIMD: the width's reciprocal (made once) for the two divisions, and
    // 1/sqrt by the hardware's reciprocal root refined, not a root and a
    // division (each within a double ulp or two)
    const double m1 = s1 * inverse_cols;  // mean - x0
    const double mean = (double)x0 + m1;
    const double variance = moment_variance(s2, m1, inverse_cols);
    const double var_eps = variance + (double)eps;
    const double factor = eps > 0.0f ? inverse_sqrt<true>(var_eps) : inverse_sqrt(var_eps);
    const double offset = -mean * factor;
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const int c = k * kWave + lane;
      if (FULL || c < chunks) {
        opaque(raw[k]);
        float v[N], o[N];
        Chunk<uint16_t>::unpack(raw[k], v);
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const float n = (float)fma((double)v[j], factor, offset);
          o[j] = (float)fma((double)n, a[k][j], (double)b[k][j]);
        }
        Chunk<uint16_t>::store(out + row * cols + c * N, o);
      }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) raw[k] = next[k];
  }
}

// ------------------------------------------------------------------ modulate

template <typename T>
__global__ void __launch_bounds__(256) modulate_elements(const T* x, const float* scale, const float* shift, T* out,
                                                         int64_t n, int cols) {
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int c = (int)(i % cols);
    store_one(out + i, (float)fma((double)load_one(x + i), 1.0 + (double)scale[c], (double)shift[c]));
  }
}

template <typename T>
__global__ void __launch_bounds__(256) modulate_chunks(const T* x, const float* scale, const float* shift, T* out,
                                                       int64_t chunks, int cols) {
  constexpr int N = Chunk<T>::N;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < chunks; i += stride) {
    const int c = (int)((i * N) % cols);
    float v[N], sc[N], sh[N], o[N];
    Chunk<T>::load(x + i * N, v);
    load_f32<N>(scale + c, sc);
    load_f32<N>(shift + c, sh);
#pragma unroll
    for (int j = 0; j < N; ++j) o[j] = (float)fma((double)v[j], 1.0 + (double)sc[j], (double)sh[j]);
    Chunk<T>::store(out + i * N, o);
  }
}

// ------------------------------------------------------------------ launch layer

// MI355X's 256 CUs of 4, which the lines between the splits were measured on
// (adaln_resident's grid follows its registers and asks the device).
constexpr int64_t kSimds = 1024;

// How a row is split: W waves per row, K chunks per lane; K = 0 means the
// scalar path.
struct RowPlan {
  int waves = 1;
  int per_lane = 0;
};

template <typename T>
RowPlan plan_rows(int64_t rows, int cols, bool vector_ok) {
  constexpr int N = Chunk<T>::N;
  RowPlan plan;
  if (!vector_ok || cols % N != 0) return plan;
  const int chunks = cols / N;
  // long rows: a 4-wave group per row shortens each lane's chain. The order
  // of a row's sums depends on its width only, never on how many rows come
  // with it (rms_norm_wide, rms_norm_groups, rms_norm_waves and
  // layer_norm_waves keep this split's order), so a row is the same to the
  // last bit whether it is normed alone, as a decode step's token, or in a
  // batch
  plan.waves = chunks >= 4 * kWave ? 4 : 1;
  (void)rows;
  const int per_lane = (int)ceil_div(chunks, kWave * plan.waves);
  static const int kSteps[] = {1, 2, 3, 4, 6, 8, 12, 16};
  for (int k : kSteps)
    if (per_lane <= k) {
      plan.per_lane = k;
      break;
    }
  return plan;
}

#define DRIFT_ROW_CASES(MACRO) \
  MACRO(1)                     \
  MACRO(2)                     \
  MACRO(3)                     \
  MACRO(4)                     \
  MACRO(6)                     \
  MACRO(8)                     \
  MACRO(12)                    \
  MACRO(16)

// Rows for rms_norm_wide: a few (at most one a CU) long rows, spread over 8
// waves (one or two chunks a lane) or 16 (one to four). 0: the four-wave
// group (or one wave) of plan_rows.
constexpr int64_t kWideRows = 256;

template <typename T>
int wide_waves(int64_t rows, int cols, const RowPlan& plan) {
  const int chunks = cols / Chunk<T>::N;
  if (plan.waves != 4 || rows > kWideRows || rows < 1) return 0;
  if (chunks >= 16 * kWave && chunks <= 4 * 16 * kWave) return 16;
  if (chunks >= 8 * kWave && chunks < 16 * kWave) return 8;
  return 0;
}

// rms_norm_waves for rows of four waves' chunks, where it measured faster than
// the four-wave group (its comment's figures). Alone from 384 to 1024 rows
// (BF16 of at most 8 chunks a lane: [600, 6144] 5.5 us in the group, 5.9 so),
// RESIDENT, a row a wave (1024 waves: one a SIMD). Above, from 1281 rows on, or
// from 1537 if a row is long (BF16 of more than 8 chunks a lane, F32 alone of
// 11 or 12), or at once (F32 alone of more): RESIDENT from 7 rows a wave. With
// the residual the same lines, to 4096 rows of at most 12 chunks a lane, and
// BF16 rows of at most 10 past the resident line ([9000, 6144] 77.9 in the
// group, 80.2 so). Returns false for the others.
//
// Just past a row a SIMD the second row's chain counts, which replays of one
// buffer hide. With events around the launch, its input left by earlier work
// in the MALL / just written / in HBM, group against waves: bf16 [1100, 4096]
// 10.2 / 8.9 / 10.1 against 9.9 / 9.3 / 11.7, [1350, 4096] 11.1 against 10.3, 3%
// slower, 12%; [1100, 5120] 10.8 / 10.0 / 10.5 against 11.7 / 11.2 / 13.8,
// [1536, 5120] 12.5 against 12.4, 5% slower, 31%, [1700, 5120] 14.3 / 12.6 / 14.6
// against 12.4 / 11.9 / 15.3; with the residual [1200, 4096] 12.6 against 12.3,
// 10% slower, 25%, [1450, 4096] 14.3 against 12.9, 4%, 16%; F32 [1100, 2560]
// 11.1 / 9.4 / 10.7 against 10.7 / 10.3 / 12.7, [1350, 2560] 11.8 against 10.8,
// 6%, 14%, [1281, 3072] 11.7 against 11.9, 12%, 25%, [1100, 4096] 15.2 / 13.0 /
// 15.4 against 13.4 / 13.0 / 17.9, with the residual [1350, 2560] 14.7 against
// 13.5, 2% faster, 17% slower. A layer's calls with F32 [1300, 4096] take 87.8
// us in the group, 86.0 so, [1500, 2560] 69.4 and 67.4.
template <typename T>
bool rms_waves_launch(T* x, const T* y, const float* weight, T* out, int64_t rows, int cols, float eps, float offset,
                      hipStream_t s) {
  const int per_lane = (int)ceil_div(cols / Chunk<T>::N, kWave);
  const bool resident = rows <= kSimds || rows >= 7 * kSimds;
  if (rows < 384 || rows > kOneWaveBlocks || per_lane > (sizeof(T) == 4 ? 20 : 16)) return false;
  if (sizeof(T) == 2 && per_lane > 8 && rows <= kSimds) return false;
  const bool longer = sizeof(T) == 2 ? per_lane > 8 : !y && per_lane > 10;
  const int64_t from = sizeof(T) == 4 && per_lane > 12 ? kSimds : longer ? 3 * kSimds / 2 : 5 * kSimds / 4;
  if (rows <= from && (y || !resident)) return false;
  if (y && per_lane > 12) return false;
  if (y && rows > 4 * kSimds && !(sizeof(T) == 2 && resident && per_lane <= 10)) return false;
  // waves of the resident grid: two a SIMD for BF16 alone, whose output a rope
  // reads next (with ropeTable over [14040, 24, 128] queries and keys 122.7 us
  // against 130.3 at one a SIMD; F32 and the residual 1% faster at one)
  const int64_t waves = sizeof(T) == 2 && !y ? 2 * kSimds : kSimds;
  const dim3 grid((unsigned)(resident ? std::min(rows, waves) : rows)), block(kWave);
  const bool keep = !y && rows >= 7 * kSimds && rows * cols * (int64_t)sizeof(T) <= kKeptBytes;
#define DRIFT_RMS_WAVES(K, ADD)                                                                                     \
  if (per_lane <= K) {                                                                                              \
    if constexpr (sizeof(T) == 2 || !ADD) { /* F32 with the residual is never resident */                           \
      if (keep) {                                                                                                   \
        hipLaunchKernelGGL((rms_norm_waves<T, K, ADD, true, !ADD>), grid, block, 0, s, x, y, weight, out, rows,     \
                           cols, eps, offset);                                                                      \
        return true;                                                                                                \
      }                                                                                                             \
      if (resident) {                                                                                               \
        hipLaunchKernelGGL((rms_norm_waves<T, K, ADD, true, false>), grid, block, 0, s, x, y, weight, out, rows,    \
                           cols, eps, offset);                                                                      \
        return true;                                                                                                \
      }                                                                                                             \
    }                                                                                                               \
    hipLaunchKernelGGL((rms_norm_waves<T, K, ADD, false, false>), grid, block, 0, s, x, y, weight, out, rows, cols, \
                       eps, offset);                                                                                \
    return true;                                                                                                    \
  }
  if (y) {
    DRIFT_RMS_WAVES(4, true)
    DRIFT_RMS_WAVES(6, true)
    DRIFT_RMS_WAVES(8, true)
    DRIFT_RMS_WAVES(10, true)
    DRIFT_RMS_WAVES(12, true)
  } else {
    DRIFT_RMS_WAVES(4, false)
    DRIFT_RMS_WAVES(6, false)
    DRIFT_RMS_WAVES(8, false)
    DRIFT_RMS_WAVES(10, false)
    DRIFT_RMS_WAVES(12, false)
    DRIFT_RMS_WAVES(16, false)
    if constexpr (sizeof(T) == 4) DRIFT_RMS_WAVES(20, false)
  }
#undef DRIFT_RMS_WAVES
  return false;
}

// rms_norm_groups: two passes a wave past 16 waves a CU, else one.
template <typename T, int G>
void rms_groups_launch(const T* x, const float* weight, T* out, int64_t rows, int cols, float eps, float offset,
                       hipStream_t s) {
  constexpr int kRows = kWave / G;
  const int64_t waves = ceil_div(rows, kRows);
  const bool keep = sizeof(T) == 4 && rows * cols * (int64_t)sizeof(T) <= kKeptBytes;
  const bool one = waves <= 4 * kSimds;
  const dim3 grid((unsigned)(one ? waves : ceil_div(waves, 2))), block(kWave);
  if (one && keep)
    hipLaunchKernelGGL((rms_norm_groups<T, G, 1, sizeof(T) == 4>), grid, block, 0, s, x, weight, out, rows, cols, eps,
                       offset);
  else if (one)
    hipLaunchKernelGGL((rms_norm_groups<T, G, 1, false>), grid, block, 0, s, x, weight, out, rows, cols, eps, offset);
  else if (keep)
    hipLaunchKernelGGL((rms_norm_groups<T, G, 2, sizeof(T) == 4>), grid, block, 0, s, x, weight, out, rows, cols, eps,
                       offset);
  else
    hipLaunchKernelGGL((rms_norm_groups<T, G, 2, false>), grid, block, 0, s, x, weight, out, rows, cols, eps, offset);
}

template <typename T>
int rms_norm(const char* entry, T* x, const T* y, const float* weight, T* out, int64_t rows, int32_t cols, float eps,
             float offset, int32_t weight_rows, Quantized q, void* stream) {
  clear_error();
  if (rows < 0) return refuse("%s: %lld rows", entry, (long long)rows);
  if (cols <= 0) return refuse("%s: rows of %d values", entry, cols);
  if (weight_rows <= 0) return refuse("%s: %d weight rows", entry, weight_rows);
  if (q.xq && cols % 32 != 0) return refuse("%s: rows of %d values are not whole blocks of 32 to quantize", entry, cols);
  if (const int bad = check_quantized(entry, q, rows * cols)) return bad;
  if (rows == 0) return 0;
  if (!x || !weight || !out) return refuse("%s: null x, weight or out", entry);
  const hipStream_t s = (hipStream_t)stream;
  const bool vector_ok = aligned16(x) && aligned16(out) && aligned16(weight) && (!y || aligned16(y));
  const RowPlan plan = plan_rows<T>(rows, cols, vector_ok);
  // the side output is written by the norm when its chunks can store the
  // codes, else by a quantize_x launch over out right after
  const bool fused = q.xq && plan.per_lane > 0 && codes_storable(q.xq, Chunk<T>::N);
  const Quantized in_kernel = fused ? q : Quantized{nullptr, nullptr, nullptr};
  if (cols <= kNarrowCols && !q.xq) {
    hipLaunchKernelGGL(rms_norm_narrow<T>, dim3(grid_for(rows, 256)), dim3(256), 0, s, x, y, weight, out, rows,
                       (int)cols, eps, offset, (int)weight_rows);
  } else if (plan.per_lane == 0) {
    hipLaunchKernelGGL(rms_norm_rows_scalar<T>, dim3(grid_for(rows, 1)), dim3(256), 0, s, x, y, weight, out, rows,
                       (int)cols, eps, offset, (int)weight_rows);
  } else if (weight_rows == 1 && !y && !q.xq && cols / Chunk<T>::N <= kWave && rows <= kOneWaveBlocks) {
    const int chunks = cols / Chunk<T>::N;
    if (chunks <= 8)
      rms_groups_launch<T, 8>(x, weight, out, rows, cols, eps, offset, s);
    else if (chunks <= 16)
      rms_groups_launch<T, 16>(x, weight, out, rows, cols, eps, offset, s);
    else if (chunks <= 32)
      rms_groups_launch<T, 32>(x, weight, out, rows, cols, eps, offset, s);
    else
      rms_groups_launch<T, 64>(x, weight, out, rows, cols, eps, offset, s);
  } else if (weight_rows == 1 && !q.xq && plan.waves == 4 &&
             rms_waves_launch(x, y, weight, out, rows, cols, eps, offset, s)) {
    return launched(entry);
  } else if (const int wide = wide_waves<T>(rows, cols, plan)) {
    const int per_lane = (int)ceil_div(cols / Chunk<T>::N, kWave * wide);
    const dim3 grid((unsigned)rows), block(kWave * wide);
    if (wide == 8 && per_lane == 1)
      hipLaunchKernelGGL((rms_norm_wide<T, 1, 8>), grid, block, 0, s, x, y, weight, out, rows, cols, eps, offset,
                         weight_rows, in_kernel);
    else if (wide == 8)
      hipLaunchKernelGGL((rms_norm_wide<T, 2, 8>), grid, block, 0, s, x, y, weight, out, rows, cols, eps, offset,
                         weight_rows, in_kernel);
    else if (per_lane == 1)
      hipLaunchKernelGGL((rms_norm_wide<T, 1, 16>), grid, block, 0, s, x, y, weight, out, rows, cols, eps, offset,
                         weight_rows, in_kernel);
    else if (per_lane == 2)
      hipLaunchKernelGGL((rms_norm_wide<T, 2, 16>), grid, block, 0, s, x, y, weight, out, rows, cols, eps, offset,
                         weight_rows, in_kernel);
    else if (per_lane == 3)
      hipLaunchKernelGGL((rms_norm_wide<T, 3, 16>), grid, block, 0, s, x, y, weight, out, rows, cols, eps, offset,
                         weight_rows, in_kernel);
    else
      hipLaunchKernelGGL((rms_norm_wide<T, 4, 16>), grid, block, 0, s, x, y, weight, out, rows, cols, eps, offset,
                         weight_rows, in_kernel);
  } else {
    const unsigned grid = grid_for(rows, 4 / plan.waves);
#define DRIFT_RMS_CASE(K)                                                                                     \
  case K:                                                                                                     \
    if (plan.waves == 1)                                                                                      \
      hipLaunchKernelGGL((rms_norm_rows<T, K, 1>), dim3(grid), dim3(256), 0, s, x, y, weight, out, rows,     \
                         cols, eps, offset, weight_rows, in_kernel);                                          \
    else                                                                                                      \
      hipLaunchKernelGGL((rms_norm_rows<T, K, 4>), dim3(grid), dim3(256), 0, s, x, y, weight, out, rows,     \
                         cols, eps, offset, weight_rows, in_kernel);                                          \
    break;
    switch (plan.per_lane) { DRIFT_ROW_CASES(DRIFT_RMS_CASE) }
#undef DRIFT_RMS_CASE
  }
  if (q.xq && !fused) {
    if (const int status = launched(entry)) return status;
    launch_quantize(out, q, rows * cols / 32, s);
  }
  return launched(entry);
}

// Waves of `kernel` (256-thread blocks) the device holds at once.
template <typename Kernel>
int64_t resident_waves(Kernel kernel) {
  int device = 0, cus = 0, blocks = 0;
  if (hipGetDevice(&device) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&blocks, kernel, 256, 0) != hipSuccess)
    return 0;
  return (int64_t)cus * blocks * 4;
}

template <int K, bool FULL>
void adaln_resident_launch(const uint16_t* x, const float* scale, const float* shift, uint16_t* out, int64_t rows,
                           int cols, int64_t rows_per_sample, int64_t samples, float eps, hipStream_t s) {
  // every wave resident at once, rows shared out as evenly as they go; the
  // residency is the current device's, found once per device
  constexpr int kDevices = 64;
  static std::atomic<int64_t> budget[kDevices] = {};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kDevices) device = 0;
  int64_t waves = budget[device].load(std::memory_order_relaxed);
  if (waves == 0) {
    waves = std::max<int64_t>(resident_waves(adaln_resident<K, FULL>), 4);
    budget[device].store(waves, std::memory_order_relaxed);
  }
  int64_t per_sample = std::max<int64_t>(1, std::min(rows_per_sample, waves / samples));
  per_sample = ceil_div(rows_per_sample, ceil_div(rows_per_sample, per_sample));
  const dim3 grid((unsigned)ceil_div(per_sample, 4), (unsigned)samples);
  hipLaunchKernelGGL((adaln_resident<K, FULL>), grid, dim3(256), 0, s, x, scale, shift, out, rows, cols,
                     rows_per_sample, eps, per_sample);
}

// AdaLN of rows of whole 16-byte chunks, at most 4096 values: BF16 through
// adaln_resident, F32 through adaln_resident_f32 or adaln_waves (their
// comments' figures), which take a row's sums alike. Returns -1 when the shape
// does not qualify.
template <typename T>
int adaln_launch(const T* x, const float* scale, const float* shift, T* out, int64_t rows, int cols,
                 int64_t rows_per_sample, float eps, hipStream_t s) {
  constexpr int N = Chunk<T>::N;
  const int64_t samples = ceil_div(rows, rows_per_sample);
  if (cols % N != 0 || cols > kAdalnMaxCols || samples > 65535 || rows_per_sample > kOneWaveBlocks) return -1;
  const int chunks = cols / N;
  const int per_lane = (int)ceil_div(chunks, kWave);
  if constexpr (sizeof(T) == 2) {
#define DRIFT_ADALN_CASE(K)                                                                                   \
  if (per_lane <= K) {                                                                                        \
    if (chunks == K * kWave)                                                                                  \
      adaln_resident_launch<K, true>(x, scale, shift, out, rows, cols, rows_per_sample, samples, eps, s);     \
    else                                                                                                      \
      adaln_resident_launch<K, false>(x, scale, shift, out, rows, cols, rows_per_sample, samples, eps, s);    \
    return 0;                                                                                                 \
  }
    DRIFT_ADALN_CASE(1)
    DRIFT_ADALN_CASE(2)
    DRIFT_ADALN_CASE(3)
    DRIFT_ADALN_CASE(4)
    DRIFT_ADALN_CASE(6)
    DRIFT_ADALN_CASE(8)
#undef DRIFT_ADALN_CASE
  } else {
    if (per_lane <= 12 && (rows <= kSimds || rows >= 7 * kSimds)) {
      // rows shared out as evenly as they go
      int64_t waves = std::max<int64_t>(1, std::min(rows_per_sample, kSimds / samples));
      waves = ceil_div(rows_per_sample, ceil_div(rows_per_sample, waves));
      const dim3 grid((unsigned)waves, (unsigned)samples), block(kWave);
#define DRIFT_ADALN_CASE(K)                                                                                      \
  if (per_lane <= K) {                                                                                           \
    if (chunks == K * kWave)                                                                                     \
      hipLaunchKernelGGL((adaln_resident_f32<K, true>), grid, block, 0, s, x, scale, shift, out, rows, cols,     \
                         rows_per_sample, eps, waves);                                                           \
    else                                                                                                         \
      hipLaunchKernelGGL((adaln_resident_f32<K, false>), grid, block, 0, s, x, scale, shift, out, rows, cols,    \
                         rows_per_sample, eps, waves);                                                           \
    return 0;                                                                                                    \
  }
      DRIFT_ADALN_CASE(3)
      DRIFT_ADALN_CASE(6)
      DRIFT_ADALN_CASE(8)
      DRIFT_ADALN_CASE(12)
#undef DRIFT_ADALN_CASE
    }
    const dim3 grid((unsigned)ceil_div(rows_per_sample, 4), (unsigned)samples);
#define DRIFT_ADALN_CASE(K)                                                                               \
  if (per_lane <= K) {                                                                                    \
    if (chunks == K * kWave)                                                                              \
      hipLaunchKernelGGL((adaln_waves<K, true>), grid, dim3(256), 0, s, x, scale, shift, out, rows, cols,  \
                         rows_per_sample, eps);                                                           \
    else                                                                                                  \
      hipLaunchKernelGGL((adaln_waves<K, false>), grid, dim3(256), 0, s, x, scale, shift, out, rows, cols, \
                         rows_per_sample, eps);                                                           \
    return 0;                                                                                             \
  }
    DRIFT_ADALN_CASE(1)
    DRIFT_ADALN_CASE(2)
    DRIFT_ADALN_CASE(3)
    DRIFT_ADALN_CASE(4)
    DRIFT_ADALN_CASE(6)
    DRIFT_ADALN_CASE(8)
    DRIFT_ADALN_CASE(12)
    DRIFT_ADALN_CASE(16)
#undef DRIFT_ADALN_CASE
  }
  return -1;
}

template <typename T, bool MODULATE>
int layer_norm(const char* entry, const T* x, const float* weight, const float* bias, T* out, int64_t rows,
               int32_t cols, int64_t rows_per_sample, float eps, void* stream) {
  clear_error();
  if (rows < 0) return refuse("%s: %lld rows", entry, (long long)rows);
  if (cols <= 0) return refuse("%s: rows of %d values", entry, cols);
  if (MODULATE && rows_per_sample <= 0) return refuse("%s: %lld rows per sample", entry, (long long)rows_per_sample);
  if (rows == 0) return 0;
  if (!x || !out) return refuse("%s: null x or out", entry);
  if (MODULATE && (!weight || !bias)) return refuse("%s: null scale or shift", entry);
  // a sample of more rows than there are is one of them all: the grids are
  // made of a sample's rows ([2000, 3840] F32, 2^20 rows a sample: 222 us of
  // empty blocks, 14 so)
  rows_per_sample = std::min(rows_per_sample, rows);
  const hipStream_t s = (hipStream_t)stream;
  const bool vector_ok =
      aligned16(x) && aligned16(out) && (!weight || aligned16(weight)) && (!bias || aligned16(bias));
  if (MODULATE && vector_ok && adaln_launch<T>(x, weight, bias, out, rows, cols, rows_per_sample, eps, s) == 0)
    return launched(entry);
  const RowPlan plan = plan_rows<T>(rows, cols, vector_ok);
  if (plan.per_lane == 0) {
    hipLaunchKernelGGL((layer_norm_rows_scalar<T, MODULATE>), dim3(grid_for(rows, 1)), dim3(256), 0, s, x, weight,
                       bias, out, rows, (int)cols, rows_per_sample, eps);
    return launched(entry);
  }
  const int per_lane = (int)ceil_div(cols / Chunk<T>::N, kWave);
  if constexpr (MODULATE) {
    const int64_t samples = ceil_div(rows, rows_per_sample);
    if (plan.waves == 4 && cols <= 5120 && rows > 3 * kSimds / 2 && samples <= 65535 &&
        rows_per_sample <= kOneWaveBlocks) {
      const dim3 grid((unsigned)ceil_div(rows_per_sample, 4), (unsigned)samples);
      hipLaunchKernelGGL((layer_norm_waves<T, 5120 / Chunk<T>::N / kWave, true>), grid, dim3(kNormBlock<true>), 0, s, x,
                         weight, bias, out, rows, cols, rows_per_sample, eps);
      return launched(entry);
    }
  } else {
    if (plan.waves == 4 && rows > (per_lane <= 6 ? 7 * kSimds / 4 : 2 * kSimds) &&
        rows * (cols / 4) >= (1 << 19) && rows <= kOneWaveBlocks &&
        per_lane <= 20) {
      const dim3 one((unsigned)rows), block(kWave);
#define DRIFT_LN_WAVES(K)                                                                                     \
  if (per_lane <= K) {                                                                                        \
    hipLaunchKernelGGL((layer_norm_waves<T, K, false>), one, block, 0, s, x, weight, bias, out, rows, cols,    \
                       rows_per_sample, eps);                                                                 \
    return launched(entry);                                                                                   \
  }
      DRIFT_LN_WAVES(4)
      DRIFT_LN_WAVES(5)
      DRIFT_LN_WAVES(6)
      DRIFT_LN_WAVES(8)
      DRIFT_LN_WAVES(10)
      DRIFT_LN_WAVES(12)
      DRIFT_LN_WAVES(16)
      DRIFT_LN_WAVES(20)
#undef DRIFT_LN_WAVES
    }
  }
  const unsigned grid = grid_for(rows, 4 / plan.waves);
#define DRIFT_LN_CASE(K)                                                                                     \
  case K:                                                                                                    \
    if (plan.waves == 1)                                                                                     \
      hipLaunchKernelGGL((layer_norm_rows<T, K, 1, MODULATE>), dim3(grid), dim3(256), 0, s, x, weight, bias, \
                         out, rows, cols, rows_per_sample, eps);                                             \
    else                                                                                                     \
      hipLaunchKernelGGL((layer_norm_rows<T, K, 4, MODULATE>), dim3(grid), dim3(256), 0, s, x, weight, bias, \
                         out, rows, cols, rows_per_sample, eps);                                             \
    break;
  switch (plan.per_lane) { DRIFT_ROW_CASES(DRIFT_LN_CASE) }
#undef DRIFT_LN_CASE
  return launched(entry);
}

}  // namespace
}  // namespace drift

using namespace drift;

extern "C" int drift_rms_norm_f32(float* x, const float* y, const float* weight, float* out, int64_t rows,
                                  int32_t cols, float eps, float offset, int32_t weight_rows, int8_t* xq, float* xd,
                                  float* xs, void* stream) {
  return rms_norm<float>("drift_rms_norm_f32", x, y, weight, out, rows, cols, eps, offset, weight_rows,
                         Quantized{xq, xd, xs}, stream);
}

extern "C" int drift_rms_norm_bf16(uint16_t* x, const uint16_t* y, const float* weight, uint16_t* out,
                                   int64_t rows, int32_t cols, float eps, float offset, int32_t weight_rows,
                                   int8_t* xq, float* xd, float* xs, void* stream) {
  return rms_norm<uint16_t>("drift_rms_norm_bf16", x, y, weight, out, rows, cols, eps, offset, weight_rows,
                            Quantized{xq, xd, xs}, stream);
}

extern "C" int drift_layer_norm_f32(const float* x, const float* weight, const float* bias, float* out,
                                    int64_t rows, int32_t cols, float eps, void* stream) {
  return layer_norm<float, false>("drift_layer_norm_f32", x, weight, bias, out, rows, cols, 1, eps, stream);
}

extern "C" int drift_layer_norm_modulate_f32(const float* x, const float* scale, const float* shift, float* out,
                                             int64_t rows, int32_t cols, int64_t rows_per_sample, float eps,
                                             void* stream) {
  return layer_norm<float, true>("drift_layer_norm_modulate_f32", x, scale, shift, out, rows, cols,
                                 rows_per_sample, eps, stream);
}

extern "C" int drift_layer_norm_modulate_bf16(const uint16_t* x, const float* scale, const float* shift,
                                              uint16_t* out, int64_t rows, int32_t cols, int64_t rows_per_sample,
                                              float eps, void* stream) {
  return layer_norm<uint16_t, true>("drift_layer_norm_modulate_bf16", x, scale, shift, out, rows, cols,
                                    rows_per_sample, eps, stream);
}

extern "C" int drift_modulate_f32(const float* x, const float* scale, const float* shift, float* out, int64_t rows,
                                  int32_t cols, void* stream) {
  const char* entry = "drift_modulate_f32";
  clear_error();
  if (rows < 0) return refuse("%s: %lld rows", entry, (long long)rows);
  if (cols <= 0) return refuse("%s: rows of %d values", entry, cols);
  if (rows == 0) return 0;
  if (!x || !scale || !shift || !out) return refuse("%s: null x, scale, shift or out", entry);
  const hipStream_t s = (hipStream_t)stream;
  const int64_t n = rows * cols;
  if (cols % 4 == 0 && aligned16(x) && aligned16(out) && aligned16(scale) && aligned16(shift)) {
    const int64_t chunks = n / 4;
    hipLaunchKernelGGL(modulate_chunks<float>, dim3(grid_for(chunks, 256)), dim3(256), 0, s, x, scale, shift, out,
                       chunks, (int)cols);
  } else {
    hipLaunchKernelGGL(modulate_elements<float>, dim3(grid_for(n, 256)), dim3(256), 0, s, x, scale, shift, out, n,
                       (int)cols);
  }
  return launched(entry);
}
