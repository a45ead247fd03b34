// Rotary embeddings for gfx950: rope by positions (NeoX, interleaved, mRoPE
// sections, per-axis), rope from cos/sin tables, Wan's 3-D rope with its
// angles made in the kernel, and per-head query/key RMSNorm fused with rope.
//
// Layout: x, out [tokens, heads, head_dim], row-major. A wave (or, for the
// awkward shapes, a block) first makes its tokens' cos/sin for every pair
// (shared by the heads it takes: the reference recomputes them per value),
// then turns the heads' pairs. Where a head is whole 16-byte chunks, each lane
// reads a pair's two chunks (NeoX: a chunk and its partner half a rotary
// away; interleaved: pairs sit inside a chunk), turns them in registers and
// writes them back, so out may be x.
//
// Arithmetic is the CPU reference's (ops/CpuAttention.scala:53-146):
// inverse frequency = 1f / float(pow(theta, 2i/rotary)) (host-side, double
// pow, as the CPU), angle = float(position) * inverse in float, cos and sin
// of it in double, the turn a*c - b*s, a*s + b*c in double, rounded once.
// Wan's tables (models/Wan.scala:324-361) are cos and sin of a double angle
// rounded to float; rope_3d makes exactly those values.
#include "rope.hpp"

#include <algorithm>
#include <climits>
#include <initializer_list>

namespace drift {
namespace {

// ------------------------------------------------------------------ rope

// Chunked turn of a head: lane items are chunk pairs. NeoX: chunk i (< half/N)
// with chunk i + half/N; interleaved: one chunk, its N/2 pairs inside. Tail
// chunks (from rotary on) are copied.
template <typename T>
__device__ __forceinline__ void turn_chunks(const T* xh, T* oh, int item, int rotary, int layout, const double2* cs) {
  constexpr int N = Chunk<T>::N;
  const int half = rotary / 2;
  if (layout == DRIFT_ROPE_NEOX) {
    const int rotating = half / N;  // chunk pairs
    if (item < rotating) {
      float a[N], b[N];
      Chunk<T>::load(xh + item * N, a);
      Chunk<T>::load(xh + half + item * N, b);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const double2 q = cs[item * N + i];
        turn(a[i], b[i], q.x, q.y, a[i], b[i]);
      }
      Chunk<T>::store(oh + item * N, a);
      Chunk<T>::store(oh + half + item * N, b);
    } else {
      const int d = rotary + (item - rotating) * N;
      float v[N];
      Chunk<T>::load(xh + d, v);
      Chunk<T>::store(oh + d, v);
    }
  } else {
    const int d = item * N;
    float v[N];
    Chunk<T>::load(xh + d, v);
    if (d < rotary) {
#pragma unroll
      for (int i = 0; i < N; i += 2) {
        const double2 q = cs[d / 2 + i / 2];
        turn(v[i], v[i + 1], q.x, q.y, v[i], v[i + 1]);
      }
    }
    Chunk<T>::store(oh + d, v);
  }
}

// Any width and alignment: a block a token, a value or pair at a time. A
// thread's next head and slot follow from its last ones, with no division
// (in 64 bits, for any number of heads, it took bf16 [4087, 16, 72] from 14.4
// to 16.1 us behind a matrix product).
template <typename T>
__global__ void __launch_bounds__(256) rope_kernel(const T* x, const int32_t* positions, T* out, RopeArgs p) {
  __shared__ double2 cs[kMaxPairs];
  const int slots = (p.dim + 1) / 2;
  const int first_h = threadIdx.x / slots, first_j = threadIdx.x % slots;
  const int step_h = blockDim.x / slots, step_j = blockDim.x % slots;
  for (int64_t t = blockIdx.x; t < p.tokens; t += gridDim.x) {
    token_angles(p, positions, t, cs);
    __syncthreads();
    const T* xt = x + t * p.heads * p.dim;
    T* ot = out + t * p.heads * p.dim;
    uint32_t h = first_h;
    int j = first_j;
    while (true) {
      if (j >= slots) {
        j -= slots;
        ++h;
      }
      if (h >= (uint32_t)p.heads) break;
      const T* xh = xt + (int64_t)h * p.dim;
      turn_slot<T>(j, p.dim, p.rotary, p.layout, cs, [&](int d) { return (double)load_one(xh + d); },
                   ot + (int64_t)h * p.dim);
      h += step_h;
      j += step_j;
    }
    __syncthreads();  // cs is remade for the next token
  }
}

// Heads and rotating parts of whole 16-byte chunks, in one-wave blocks with no
// barrier. An item is turn_chunks' (NeoX: a chunk and its partner;
// interleaved: a chunk), a head has `rotating` of them and then its tail's
// chunks (none in place: they stay as they are). A wave takes K * 64 items of
// one token (`runs` waves a token) or, where a token has fewer, of `per_wave`
// tokens. It issues its loads, makes its tokens' cos and sin while they land
// (a pair a lane, into its LDS), and turns its items from there.
//
// Memory bounds the large launches. Measured, us a launch in graph replays, a
// 256-thread block a token with two barriers and the library's sincos / this:
// F32 in place [2039, 32, 128] (67 MB) 12.8 / 12.5, [2039, 8, 128] 5.8 / 4.3;
// bf16 [6546, 24, 256] with 64 values turning, in place 43.5 / 10.9 (its tail
// copied onto itself before), out of place (161 MB) 44.0 / 31.7, [6546, 4,
// 256] in place 17.1 / 3.6; bf16 interleaved [4096, 32, 128] 15.8 / 12.1; F32
// over two axes [4087, 16, 72] 10.4 / 9.9; one token of 32 heads 2.2 / 1.9.
// K = 1, 2, 4 there: [2039, 32, 128] 12.1, 11.9, 12.5; out of place [6546, 24,
// 256] 30.6, 32.5, 31.7; [4087, 16, 72] 9.7, 13.1 (its second wave nearly
// empty), 9.8; [262, 16, 256] in place 2.4, 2.9, 3.9.
//
// Pair m of an item j sits in LDS at m * rotating + j, so that lanes on
// consecutive items read consecutive entries.
// Row i / slots comes from a product with slots_inverse = ceil(2^32 / slots)
// (exact where i * slots < 2^32: the launcher's bound on a token; 0 where
// slots is 1). TOKENS: a wave's items are of several tokens.
//
// STREAM: the loads are non-temporal, for chunks rewritten where they were
// read, whole lines at a time (plain loads there: F32 [2039, 32, 128] 12.5 ->
// 15.1, bf16 interleaved [4096, 32, 128] 11.9 -> 14.5). Elsewhere plain loads
// are faster: bf16 [6546, 24, 256] with 64 turning 31.9 -> 28.7, in place
// (halves of a line) 10.9 -> 9.4, F32 [4087, 16, 72] 9.9 -> 8.0, [4830, 12,
// 64] 6.6 -> 5.4, [2039, 32, 128] out of place 12.5 -> 11.9.
template <typename T, bool NEOX, int K, bool TOKENS, bool STREAM>
__global__ void __launch_bounds__(kWave) rope_waves(const T* x, const int32_t* positions, T* out, RopeArgs p, int slots,
                                                    uint32_t slots_inverse, uint32_t runs, int per_wave) {
  constexpr int N = Chunk<T>::N;
  constexpr int P = NEOX ? N : N / 2;  // pairs of an item
  using Raw = typename Chunk<T>::Raw;
  constexpr int kPairsPerLane = kMaxPairs / kWave;
  __shared__ double2 cs[kMaxPairs];
  const int lane = threadIdx.x;
  const int half = p.rotary / 2, rotating = half / P;
  const int items = p.heads * slots;  // a token's
  const uint32_t group = blockIdx.x / runs, run = blockIdx.x - group * runs;
  const int64_t t0 = TOKENS ? (int64_t)group * per_wave : (int64_t)group;
  const int tokens = TOKENS ? (int)min((int64_t)per_wave, p.tokens - t0) : 1;
  // the small operands load first (a pair's position and frequency), and are
  // used only once the items' loads are issued
  const int pairs = tokens * half;
  int32_t position[kPairsPerLane];
  float inverse[kPairsPerLane];
#pragma unroll
  for (int u = 0; u < kPairsPerLane; ++u) {
    if (u * kWave < pairs) {
      const int i = min(u * kWave + lane, pairs - 1);
      const int tt = TOKENS ? i / half : 0, j = i - tt * half;
      position[u] = positions[(int64_t)rope_section(j, p) * p.tokens + t0 + tt];
      inverse[u] = p.inverse[j];
    }
  }
  const T* xt = x + t0 * p.heads * p.dim;
  T* ot = out + t0 * p.heads * p.dim;
  const int last = tokens * items - 1;
  Raw r0[K], r1[NEOX ? K : 1];
  int at[K], slot[K];
  bool turns[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int i = min((int)(run * K + k) * kWave + lane, last);
    const int row = slots_inverse ? (int)__umulhi((uint32_t)i, slots_inverse) : i;  // (token, head) of the wave's
    const int j = i - row * slots;
    turns[k] = j < rotating;
    at[k] = row * p.dim + (NEOX && !turns[k] ? p.rotary + (j - rotating) * N : j * N);
    slot[k] = (TOKENS ? row / p.heads * half : 0) + j;
    auto load = [](const T* from) {
      if constexpr (STREAM) return Chunk<T>::load_raw(from);
      else return *reinterpret_cast<const Raw*>(from);
    };
    r0[k] = load(xt + at[k]);
    if constexpr (NEOX) r1[k] = load(xt + at[k] + (turns[k] ? half : 0));
  }
#pragma unroll
  for (int u = 0; u < kPairsPerLane; ++u) {
    const int i = u * kWave + lane;
    if (i < pairs) {
      const int tt = TOKENS ? i / half : 0, j = i - tt * half;
      asm volatile("" : "+v"(position[u]));  // converted here, not (waiting) before the items' loads
      cs[tt * half + j % P * rotating + j / P] = cos_sin((float)position[u] * inverse[u]);
    }
  }
  wave_sync();
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if ((int)(run * K + k) * kWave + lane > last) return;
    float a[N], b[N];
    Chunk<T>::unpack(r0[k], a);
    if constexpr (NEOX) Chunk<T>::unpack(r1[k], b);
    if (turns[k]) {
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const double2 q = cs[slot[k] + i * rotating];
        if constexpr (NEOX)
          turn_fused(a[i], b[i], q.x, q.y, a[i], b[i]);
        else
          turn_fused(a[2 * i], a[2 * i + 1], q.x, q.y, a[2 * i], a[2 * i + 1]);
      }
    }
    Chunk<T>::store(ot + at[k], a);
    if constexpr (NEOX)
      if (turns[k]) Chunk<T>::store(ot + at[k] + half, b);
  }
}

// ------------------------------------------------------------------ rope from tables

template <typename T>
__global__ void __launch_bounds__(256) rope_table_kernel(const T* x, const float* cosines, const float* sines, T* out,
                                                         int tokens, int heads, int dim, int pairs, int per_head,
                                                         int halves) {
  const int slots = (dim + 1) / 2;
  const int64_t items = (int64_t)tokens * heads * slots;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < items; i += stride) {
    const int j = (int)(i % slots);
    const int64_t head_row = i / slots;  // token * heads + head
    const int64_t row = per_head ? head_row : head_row / heads;
    const T* xh = x + head_row * dim;
    T* oh = out + head_row * dim;
    if (j < pairs) {
      const int d0 = halves ? j : 2 * j;
      const int d1 = halves ? j + pairs : 2 * j + 1;
      const double c = (double)cosines[row * pairs + j], s = (double)sines[row * pairs + j];
      const double a = (double)load_one(xh + d0), b = (double)load_one(xh + d1);
      float f, g;
      turn(a, b, c, s, f, g);
      store_one(oh + d0, f);
      store_one(oh + d1, g);
    } else {
      const int e = 2 * pairs + 2 * (j - pairs);
      const float v0 = load_one(xh + e);
      const float v1 = e + 1 < dim ? load_one(xh + e + 1) : 0.0f;
      store_one(oh + e, v0);
      if (e + 1 < dim) store_one(oh + e + 1, v1);
    }
  }
}

// Heads and rotating parts of whole 16-byte chunks: one-wave blocks, a wave
// per run of K * 64 items of a token, an item a chunk (interleaved: its pairs
// sit inside it) or a chunk and its partner (halves), as turn_chunks' items.
// The loads are all issued before any turn and never branched around. The
// products a*c of floats are exact in double, so the one fma is the
// reference's a*c - b*s rounded once.
//
// Memory sets its pace: in place over [14040, 24, 128] bf16 with a table row a
// token (172 MB, written just before by a norm) it takes 24.5 us, 7 TB/s; the
// kernel above, two values a thread, took 68. An RMSNorm and this for
// queries and keys there took 146.1, 136.7, 138.2 and 153.1 us with K = 1, 2,
// 3 and 4; over 72 tokens (432 waves at K = 1) 10.4, 12.0, 13.6 and 14.6.
template <typename T, int K, bool HALVES, bool PER_HEAD>
__global__ void __launch_bounds__(kWave) rope_table_chunks(const T* x, const float* cosines, const float* sines,
                                                           T* out, uint32_t runs, int heads, int dim, int pairs) {
  constexpr int N = Chunk<T>::N;
  constexpr int P = HALVES ? N : N / 2;  // pairs of an item
  using Raw = typename Chunk<T>::Raw;
  const uint32_t token = blockIdx.x / runs, run = blockIdx.x - token * runs;
  const int rotating = HALVES ? pairs / N : 2 * pairs / N;  // a head's items that turn
  const int slots = HALVES ? rotating + (dim - 2 * pairs) / N : dim / N;
  const int items = heads * slots;
  const T* xt = x + (int64_t)token * heads * dim;
  T* ot = out + (int64_t)token * heads * dim;
  Raw r0[K], r1[HALVES ? K : 1];
  float c[K][P], s[K][P];
  int at[K];
  bool turns[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int item = min((int)(run * K + k) * kWave + (int)threadIdx.x, items - 1);
    const int h = item / slots, j = item - h * slots;
    turns[k] = j < rotating;
    at[k] = h * dim + (HALVES && !turns[k] ? 2 * pairs + (j - rotating) * N : j * N);
    r0[k] = Chunk<T>::load_raw(xt + at[k]);
    if constexpr (HALVES) r1[k] = Chunk<T>::load_raw(xt + at[k] + (turns[k] ? pairs : 0));
    const int64_t row = PER_HEAD ? (int64_t)token * heads + h : (int64_t)token;
    const int64_t q = row * pairs + (turns[k] ? j * P : 0);
    if (pairs > 0) {
#pragma unroll
      for (int i = 0; i < P; i += P >= 4 ? 4 : 2) {
        if constexpr (P >= 4) {
          const float4 a = *reinterpret_cast<const float4*>(cosines + q + i);
          const float4 b = *reinterpret_cast<const float4*>(sines + q + i);
          c[k][i] = a.x, c[k][i + 1] = a.y, c[k][i + 2] = a.z, c[k][i + 3] = a.w;
          s[k][i] = b.x, s[k][i + 1] = b.y, s[k][i + 2] = b.z, s[k][i + 3] = b.w;
        } else {
          const float2 a = *reinterpret_cast<const float2*>(cosines + q + i);
          const float2 b = *reinterpret_cast<const float2*>(sines + q + i);
          c[k][i] = a.x, c[k][i + 1] = a.y;
          s[k][i] = b.x, s[k][i + 1] = b.y;
        }
      }
    }
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    if ((int)(run * K + k) * kWave + (int)threadIdx.x >= items) return;
    float a[N], b[N];
    Chunk<T>::unpack(r0[k], a);
    if constexpr (HALVES) Chunk<T>::unpack(r1[k], b);
    if (turns[k]) {
#pragma unroll
      for (int i = 0; i < P; ++i) {
        if constexpr (HALVES)
          turn_fused(a[i], b[i], c[k][i], s[k][i], a[i], b[i]);
        else
          turn_fused(a[2 * i], a[2 * i + 1], c[k][i], s[k][i], a[2 * i], a[2 * i + 1]);
      }
    }
    Chunk<T>::store(ot + at[k], a);
    if constexpr (HALVES)
      if (turns[k]) Chunk<T>::store(ot + at[k] + pairs, b);
  }
}

// ------------------------------------------------------------------ Wan 3-D rope

struct Rope3dArgs {
  double denominator[kMaxPairs];  // theta^(2 index / (2 pairs_axis)) per pair
  int64_t tokens, token_offset, grid;
  int32_t heads, dim, rows, cols, pairs0, pairs1;
};

template <typename T, bool CHUNKED>
__global__ void __launch_bounds__(256) rope_3d_kernel(const T* x, T* out, Rope3dArgs p) {
  __shared__ double2 cs[kMaxPairs];
  constexpr int N = Chunk<T>::N;
  const int half = p.dim / 2;
  const int slots = CHUNKED ? p.dim / N : half;
  for (int64_t t = blockIdx.x; t < p.tokens; t += gridDim.x) {
    const int64_t g = (p.token_offset + t) % p.grid;
    for (int j = threadIdx.x; j < half; j += blockDim.x) {
      const int64_t position = j < p.pairs0 ? g / ((int64_t)p.rows * p.cols)
                                            : (j < p.pairs0 + p.pairs1 ? g / p.cols % p.rows : g % p.cols);
      const double angle = (double)position / p.denominator[j];
      double sn, cn;
      sincos(angle, &sn, &cn);
      cs[j] = make_double2((double)(float)cn, (double)(float)sn);  // the F32 tables' values
    }
    __syncthreads();
    const T* xt = x + t * p.heads * p.dim;
    T* ot = out + t * p.heads * p.dim;
    for (int i = threadIdx.x; i < p.heads * slots; i += blockDim.x) {
      const int h = i / slots, j = i % slots;
      const T* xh = xt + (int64_t)h * p.dim;
      T* oh = ot + (int64_t)h * p.dim;
      if constexpr (CHUNKED)
        turn_chunks<T>(xh, oh, j, p.dim, DRIFT_ROPE_INTERLEAVED, cs);
      else
        turn_slot<T>(j, p.dim, p.dim, DRIFT_ROPE_INTERLEAVED, cs, [&](int d) { return (double)load_one(xh + d); },
                     oh);
    }
    __syncthreads();
  }
}

// One wave per token, the grid covering the tokens in one pass. A wave issues
// its token's loads first; while they land, each lane makes one pair's angle
// (Wan's angle depends on one axis position: frame, row or column) and its
// cos and sin, exactly as the host tables hold them (cos and sin of the
// double angle, rounded to float), into the wave's LDS slice. Then each lane
// turns its chunks' pairs. With a, b bf16 or F32 and c, s floats, a*c and b*s
// are exact in double, so fma(a, c, -b*s) is the reference's a*c - b*s
// rounded once.
constexpr int kRope3dWaves = 8;

template <typename T, int K, bool FIXED>
__global__ void __launch_bounds__(kRope3dWaves * 64) rope_3d_waves(const T* x, T* out, Rope3dArgs p) {
  constexpr int N = Chunk<T>::N;
  using Raw = typename Chunk<T>::Raw;
  __shared__ float2 cs_all[kRope3dWaves][kMaxPairs];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t t = (int64_t)blockIdx.x * kRope3dWaves + wave;
  if (t >= p.tokens) return;  // no block-wide barrier follows
  const int per_token = p.heads * p.dim / N;  // chunks of a token, at most K * 64
  const int per_head = p.dim / N;
  const T* xt = x + t * p.heads * p.dim;
  // loads are never branched around (a branch makes each wait for the one
  // before): chunk indices past the token are clamped and their values unused
  Raw raw[K];
#pragma unroll
  for (int k = 0; k < K; ++k) raw[k] = Chunk<T>::load_raw(xt + min(k * kWave + lane, per_token - 1) * N);
  const int64_t g = (p.token_offset + t) % p.grid;
  const int plane = p.rows * p.cols;
  const int frame = (int)(g / plane), rem = (int)(g % plane);
  const int row = rem / p.cols, col = rem % p.cols;
  const int half = p.dim / 2;
  float2* cs = cs_all[wave];
  for (int m = lane; m < half; m += kWave) {
    const int position = m < p.pairs0 ? frame : (m < p.pairs0 + p.pairs1 ? row : col);
    double sn, cn;
    sincos((double)position / p.denominator[m], &sn, &cn);
    cs[m] = make_float2((float)cn, (float)sn);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // the lane's pairs' cos and sin, when they are the same in every chunk
  double fc[N / 2], fs[N / 2];
  if constexpr (FIXED) {
    const int m0 = (lane % per_head) * N / 2;
#pragma unroll
    for (int i = 0; i < N / 2; ++i) {
      const float2 q = cs[m0 + i];
      fc[i] = q.x;
      fs[i] = q.y;
    }
  }
  T* ot = out + t * p.heads * p.dim;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int q = k * kWave + lane;
    if (q < per_token) {
      float v[N];
      Chunk<T>::unpack(raw[k], v);
      const int m0 = (q % per_head) * N / 2;
#pragma unroll
      for (int i = 0; i < N / 2; ++i) {
        double c, sn;
        if constexpr (FIXED) {
          c = fc[i];
          sn = fs[i];
        } else {
          const float2 e = cs[m0 + i];
          c = e.x;
          sn = e.y;
        }
        const double a = v[2 * i], b = v[2 * i + 1];
        v[2 * i] = (float)fma(a, c, -(b * sn));
        v[2 * i + 1] = (float)fma(a, sn, b * c);
      }
      Chunk<T>::store(ot + q * N, v);
    }
  }
}

// ------------------------------------------------------------------ launch layer

template <typename T>
int rope(const char* entry, const T* x, const int32_t* positions, T* out, int32_t tokens, int32_t heads,
         int32_t dim, int32_t rotary, float theta, int32_t layout, int32_t sections, int32_t s0, int32_t s1,
         int32_t s2, int32_t s3, void* stream) {
  clear_error();
  const int32_t s[4] = {s0, s1, s2, s3};
  if (const int bad = check_rope(entry, tokens, heads, dim, rotary, layout, sections, s)) return bad;
  if ((int64_t)tokens * heads == 0) return 0;
  if (!x || !positions || !out) return refuse("%s: null x, positions or out", entry);
  RopeArgs p;
  fill_rope(p, tokens, heads, dim, rotary, theta, layout, sections, s);
  constexpr int N = Chunk<T>::N;
  const bool neox = layout == DRIFT_ROPE_NEOX;
  const bool chunked = aligned16(x) && aligned16(out) && dim % N == 0 && rotary % (neox ? 2 * N : N) == 0 &&
                       (int64_t)heads * dim <= INT32_MAX;
  const hipStream_t st = (hipStream_t)stream;
  const int rotating = neox ? rotary / 2 / N : rotary / N;
  const int slots = x == out ? rotating : rotating + (dim - rotary) / N;
  if (chunked && slots == 0) return 0;  // in place with nothing to turn
  const int64_t items = (int64_t)heads * std::max(slots, 1);
  // items a lane: one in launches of up to 8 waves a CU of one; else the count
  // of 4, 3 or 2 whose waves hold a token's items with the fewest idle lanes
  int per_lane = 1;
  if (tokens * items > 2048 * kWave) {
    per_lane = 4;
    for (int k : {3, 2})
      if (ceil_div(items, k * kWave) * k < ceil_div(items, per_lane * kWave) * per_lane &&
          items > per_lane * kWave / 2)
        per_lane = k;
  }
  const int64_t runs = ceil_div(items, per_lane * kWave);
  // whole tokens of a wave: as many as its items and its LDS's pairs hold
  const int64_t fit = std::min<int64_t>(per_lane * kWave / items, rotary > 0 ? kMaxPairs / (rotary / 2) : kMaxPairs);
  const int64_t per_wave = std::max<int64_t>(1, std::min<int64_t>(fit, tokens));
  const int64_t blocks = ceil_div(tokens, per_wave) * runs;
  if (chunked && blocks <= kOneWaveBlocks && items * slots < (int64_t)1 << 32) {
    const dim3 grid((unsigned)blocks), block(kWave);
    const uint32_t slots_inverse = slots == 1 ? 0 : (uint32_t)ceil_div((int64_t)1 << 32, slots);
    const bool stream = x == out && (!neox || rotary / 2 * sizeof(T) % 128 == 0);
#define DRIFT_ROPE_LAUNCH(NEOX, K, TOKENS)                                                                         \
  if (stream)                                                                                                      \
    hipLaunchKernelGGL((rope_waves<T, NEOX, K, TOKENS, true>), grid, block, 0, st, x, positions, out, p, slots,    \
                       slots_inverse, (uint32_t)runs, (int)per_wave);                                              \
  else                                                                                                             \
    hipLaunchKernelGGL((rope_waves<T, NEOX, K, TOKENS, false>), grid, block, 0, st, x, positions, out, p, slots,   \
                       slots_inverse, (uint32_t)runs, (int)per_wave)
#define DRIFT_ROPE_CASE(K)                  \
  case K:                                   \
    if (neox && per_wave > 1) {             \
      DRIFT_ROPE_LAUNCH(true, K, true);     \
    } else if (neox) {                      \
      DRIFT_ROPE_LAUNCH(true, K, false);    \
    } else if (per_wave > 1) {              \
      DRIFT_ROPE_LAUNCH(false, K, true);    \
    } else {                                \
      DRIFT_ROPE_LAUNCH(false, K, false);   \
    }                                       \
    break;
    switch (per_lane) {
      DRIFT_ROPE_CASE(1)
      DRIFT_ROPE_CASE(2)
      DRIFT_ROPE_CASE(3)
      DRIFT_ROPE_CASE(4)
    }
#undef DRIFT_ROPE_CASE
#undef DRIFT_ROPE_LAUNCH
  } else {
    hipLaunchKernelGGL(rope_kernel<T>, dim3(grid_for(tokens, 1, 1 << 16)), dim3(256), 0, st, x, positions, out, p);
  }
  return launched(entry);
}

template <typename T>
int rope_table(const char* entry, const T* x, const float* cosines, const float* sines, T* out, int32_t tokens,
               int32_t heads, int32_t dim, int32_t pairs, int32_t per_head, int32_t halves, void* stream) {
  clear_error();
  if (tokens < 0 || heads < 0 || dim <= 0) return refuse("%s: %d tokens of %d heads of %d", entry, tokens, heads, dim);
  if (pairs < 0 || 2 * pairs > dim) return refuse("%s: %d pairs in heads of %d", entry, pairs, dim);
  if ((int64_t)tokens * heads == 0) return 0;
  if (!x || !cosines || !sines || !out) return refuse("%s: null x, cosines, sines or out", entry);
  constexpr int N = Chunk<T>::N;
  const hipStream_t st = (hipStream_t)stream;
  const bool chunked = aligned16(x) && aligned16(out) && aligned16(cosines) && aligned16(sines) && dim % N == 0 &&
                       (halves ? pairs % N == 0 : 2 * pairs % N == 0) && (int64_t)heads * dim <= INT32_MAX;
  const int64_t items = heads * (halves ? (dim - pairs) / N : dim / N);
  // a lane's items: one where they are chunk pairs, and in launches of at most
  // 16 waves a CU of one; else two (rope_table_chunks' comment)
  const int per_lane = halves || tokens * ceil_div(items, kWave) <= 4096 ? 1 : 2;
  const int64_t runs = ceil_div(items, per_lane * kWave);
  if (chunked && tokens * runs <= kOneWaveBlocks) {
    const dim3 grid((unsigned)(tokens * runs)), block(kWave);
#define DRIFT_TABLE_LAUNCH(K, HALVES, PER_HEAD)                                                               \
  hipLaunchKernelGGL((rope_table_chunks<T, K, HALVES, PER_HEAD>), grid, block, 0, st, x, cosines, sines, out, \
                     (uint32_t)runs, heads, dim, pairs)
    if (halves && per_head)
      DRIFT_TABLE_LAUNCH(1, true, true);
    else if (halves)
      DRIFT_TABLE_LAUNCH(1, true, false);
    else if (per_head && per_lane == 2)
      DRIFT_TABLE_LAUNCH(2, false, true);
    else if (per_head)
      DRIFT_TABLE_LAUNCH(1, false, true);
    else if (per_lane == 2)
      DRIFT_TABLE_LAUNCH(2, false, false);
    else
      DRIFT_TABLE_LAUNCH(1, false, false);
#undef DRIFT_TABLE_LAUNCH
    return launched(entry);
  }
  const int64_t threads = (int64_t)tokens * heads * ((dim + 1) / 2);
  hipLaunchKernelGGL(rope_table_kernel<T>, dim3(grid_for(threads, 256, 1 << 16)), dim3(256), 0, st, x, cosines, sines,
                     out, tokens, heads, dim, pairs, per_head ? 1 : 0, halves ? 1 : 0);
  return launched(entry);
}

template <typename T>
int rope_3d(const char* entry, const T* x, T* out, int64_t tokens, int32_t heads, int32_t dim, int32_t frames,
            int32_t rows, int32_t cols, int64_t token_offset, double theta, void* stream) {
  clear_error();
  if (tokens < 0 || heads < 0) return refuse("%s: %lld tokens of %d heads", entry, (long long)tokens, heads);
  if (dim <= 0 || dim % 2 != 0 || dim > 2 * kMaxPairs) return refuse("%s: heads of %d values", entry, dim);
  if (frames <= 0 || rows <= 0 || cols <= 0 || (int64_t)frames * rows * cols > INT32_MAX)
    return refuse("%s: a %d x %d x %d grid", entry, frames, rows, cols);
  if (token_offset < 0) return refuse("%s: token offset %lld", entry, (long long)token_offset);
  if (tokens * heads == 0) return 0;
  if (!x || !out) return refuse("%s: null x or out", entry);
  // WanConfig.ropePairs (models/Wan.scala:35-41)
  const int side = 2 * (dim / 6);
  const int axes[3] = {(dim - 2 * side) / 2, side / 2, side / 2};
  if (axes[0] <= 0 || axes[1] <= 0) return refuse("%s: heads of %d values are too narrow for 3 axes", entry, dim);
  Rope3dArgs p;
  p.tokens = tokens;
  p.token_offset = token_offset;
  p.grid = (int64_t)frames * rows * cols;
  p.heads = heads;
  p.dim = dim;
  p.rows = rows;
  p.cols = cols;
  p.pairs0 = axes[0];
  p.pairs1 = axes[1];
  for (int pair = 0; pair < kMaxPairs; ++pair) {
    if (pair >= dim / 2) {
      p.denominator[pair] = 1.0;
      continue;
    }
    const int axis = pair < axes[0] ? 0 : (pair < axes[0] + axes[1] ? 1 : 2);
    const int index = pair - (axis > 0 ? axes[0] : 0) - (axis > 1 ? axes[1] : 0);
    p.denominator[pair] = std::pow(theta, 2.0 * index / (double)(2 * axes[axis]));
  }
  constexpr int N = Chunk<T>::N;
  const bool chunked = aligned16(x) && aligned16(out) && dim % N == 0;
  const hipStream_t st = (hipStream_t)stream;
  const int per_lane = (int)ceil_div((int64_t)heads * dim / N, kWave);
  const int64_t blocks = ceil_div(tokens, kRope3dWaves);
  if (chunked && blocks <= kOneShotBlocks) {
    const bool fixed = (64 % (dim / N)) == 0;
#define DRIFT_ROPE3D_CASE(K)                                                                                  \
  if (per_lane <= K) {                                                                                        \
    if (fixed)                                                                                                \
      hipLaunchKernelGGL((rope_3d_waves<T, K, true>), dim3((unsigned)blocks), dim3(64 * kRope3dWaves), 0, st, \
                         x, out, p);                                                                          \
    else                                                                                                      \
      hipLaunchKernelGGL((rope_3d_waves<T, K, false>), dim3((unsigned)blocks), dim3(64 * kRope3dWaves), 0,    \
                         st, x, out, p);                                                                      \
    return launched(entry);                                                                                   \
  }
    DRIFT_ROPE3D_CASE(1)
    DRIFT_ROPE3D_CASE(2)
    DRIFT_ROPE3D_CASE(4)
    DRIFT_ROPE3D_CASE(6)
    DRIFT_ROPE3D_CASE(8)
    DRIFT_ROPE3D_CASE(12)
    DRIFT_ROPE3D_CASE(16)
#undef DRIFT_ROPE3D_CASE
  }
  const dim3 grid(grid_for(tokens, 1, 1 << 16));
  if (chunked)
    hipLaunchKernelGGL((rope_3d_kernel<T, true>), grid, dim3(256), 0, st, x, out, p);
  else
    hipLaunchKernelGGL((rope_3d_kernel<T, false>), grid, dim3(256), 0, st, x, out, p);
  return launched(entry);
}

}  // namespace
}  // namespace drift

using namespace drift;

extern "C" int drift_rope_f32(const float* x, const int32_t* positions, float* out, int32_t tokens, int32_t heads,
                              int32_t head_dim, int32_t rotary, float theta, int32_t layout, int32_t sections,
                              int32_t s0, int32_t s1, int32_t s2, int32_t s3, void* stream) {
  return rope<float>("drift_rope_f32", x, positions, out, tokens, heads, head_dim, rotary, theta, layout, sections,
                     s0, s1, s2, s3, stream);
}

extern "C" int drift_rope_bf16(const uint16_t* x, const int32_t* positions, uint16_t* out, int32_t tokens,
                               int32_t heads, int32_t head_dim, int32_t rotary, float theta, int32_t layout,
                               int32_t sections, int32_t s0, int32_t s1, int32_t s2, int32_t s3, void* stream) {
  return rope<uint16_t>("drift_rope_bf16", x, positions, out, tokens, heads, head_dim, rotary, theta, layout,
                        sections, s0, s1, s2, s3, stream);
}

extern "C" int drift_rope_table_f32(const float* x, const float* cosines, const float* sines, float* out,
                                    int32_t tokens, int32_t heads, int32_t head_dim, int32_t pairs, int32_t per_head,
                                    int32_t halves, void* stream) {
  return rope_table<float>("drift_rope_table_f32", x, cosines, sines, out, tokens, heads, head_dim, pairs, per_head,
                           halves, stream);
}

extern "C" int drift_rope_table_bf16(const uint16_t* x, const float* cosines, const float* sines, uint16_t* out,
                                     int32_t tokens, int32_t heads, int32_t head_dim, int32_t pairs,
                                     int32_t per_head, int32_t halves, void* stream) {
  return rope_table<uint16_t>("drift_rope_table_bf16", x, cosines, sines, out, tokens, heads, head_dim, pairs,
                              per_head, halves, stream);
}

extern "C" int drift_rope_3d_f32(const float* x, float* out, int64_t tokens, int32_t heads, int32_t head_dim,
                                 int32_t frames, int32_t grid_rows, int32_t grid_cols, int64_t token_offset,
                                 double theta, void* stream) {
  return rope_3d<float>("drift_rope_3d_f32", x, out, tokens, heads, head_dim, frames, grid_rows, grid_cols,
                        token_offset, theta, stream);
}

extern "C" int drift_rope_3d_bf16(const uint16_t* x, uint16_t* out, int64_t tokens, int32_t heads,
                                  int32_t head_dim, int32_t frames, int32_t grid_rows, int32_t grid_cols,
                                  int64_t token_offset, double theta, void* stream) {
  return rope_3d<uint16_t>("drift_rope_3d_bf16", x, out, tokens, heads, head_dim, frames, grid_rows, grid_cols,
                           token_offset, theta, stream);
}
