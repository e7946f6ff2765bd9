// Row kernels of decoders whose residual stream is kept in fp32 and whose sublayer
// outputs are normalised before they are added to it:
//
//  * residual_norm_kernel: pending sublayer output -> its norm -> residual add -> average
//    with the results of earlier layers -> the next sublayer's norm, one launch per step
//    between two sublayers (the embedding lookup rides in the first).
//  * rows_linear_kernel: the matrix-vector products of a decode step, with that step
//    as an optional prologue, and a gated unit, a second scaled term, or the residual sum
//    and the average over depth as epilogue.
//  * gated_unit_kernel: the gated unit alone, for prompts.
#include <algorithm>

#include "elem.h"

namespace {

constexpr int kRowThreads = 256;

// One row of the step described at socket_residual_norm by a workgroup of kRowThreads
// lanes.  `buf`: LDS, `dim` floats; a lane reads back only what it wrote itself.  V = 4
// (dim a multiple of 4) or 1.  emit(i, v): V normalised elements at column i.
template <class DT, int V, bool DEPTH, class Emit>
__device__ __forceinline__ void residual_row(const socket_residual& a, int64_t row, float* buf, float (*red)[4],
                                             bool store_x, Emit emit) {
  const int dim = a.dim;
  const int64_t base = row * dim;
  float rs_y = 1.f;
  if (a.a) {
    float ss = 0.f;
    for (int i = threadIdx.x * V; i < dim; i += kRowThreads * V) {
      float y[V];
      if (a.pending_f32) load_vec<DType_f32, V>(a.a, base + i, y);
      else load_vec<DT, V>(a.a, base + i, y);
#pragma unroll
      for (int e = 0; e < V; ++e) y[e] *= a.scale_a;
      if (a.b) {
        float z[V];
        if (a.pending_f32) load_vec<DType_f32, V>(a.b, base + i, z);
        else load_vec<DT, V>(a.b, base + i, z);
#pragma unroll
        for (int e = 0; e < V; ++e) y[e] = fmaf(a.scale_b, z[e], y[e]);
      }
#pragma unroll
      for (int e = 0; e < V; ++e) ss = fmaf(y[e], y[e], ss);
      store_vec<DType_f32, V>(buf, i, y);
    }
    if (a.post_w) rs_y = rsqrt_f32(block_sum(ss, red[0]) / (float)dim + a.eps);
  }
  int64_t src = a.x_stride ? row * a.x_stride : base;
  if (!a.x) {
    int64_t id = a.ids64 ? ((const int64_t*)a.ids)[row] : (int64_t)((const int32_t*)a.ids)[row];
    id = id < 0 ? 0 : (id >= a.vocab ? a.vocab - 1 : id);
    src = id * dim;
  }
  float ss = 0.f;
  for (int i = threadIdx.x * V; i < dim; i += kRowThreads * V) {
    float x[V];
    if (a.x) load_vec<DType_f32, V>(a.x, src + i, x);
    else {
      load_vec<DT, V>(a.embed, src + i, x);
#pragma unroll
      for (int e = 0; e < V; ++e) x[e] *= a.embed_scale;
    }
    if (a.a) {
      float y[V];
      load_vec<DType_f32, V>(buf, i, y);
      if (a.post_w) {
        float w[V];
        load_vec<DType_f32, V>(a.post_w, i, w);
#pragma unroll
        for (int e = 0; e < V; ++e) y[e] = y[e] * rs_y * w[e];
      }
#pragma unroll
      for (int e = 0; e < V; ++e) x[e] += y[e];
    }
    if constexpr (DEPTH) {
      const socket_depth_mix& d = a.depth;
      store_vec<DType_f32, V>(d.result, base + i, x);
      const float own = d.w[d.n];
#pragma unroll
      for (int e = 0; e < V; ++e) x[e] *= own;
#pragma unroll 4
      for (int j = 0; j < d.n; ++j) {
        float p[V];
        load_vec<DType_f32, V>(d.past, j * d.past_stride + base + i, p);
#pragma unroll
        for (int e = 0; e < V; ++e) x[e] = fmaf(d.w[j], p[e], x[e]);
      }
    }
#pragma unroll
    for (int e = 0; e < V; ++e) ss = fmaf(x[e], x[e], ss);
    store_vec<DType_f32, V>(buf, i, x);
    if (store_x && a.x_out) store_vec<DType_f32, V>(a.x_out, base + i, x);
  }
  const float rs = rsqrt_f32(block_sum(ss, red[1]) / (float)dim + a.eps);
  for (int i = threadIdx.x * V; i < dim; i += kRowThreads * V) {
    float x[V], w[V];
    load_vec<DType_f32, V>(buf, i, x);
    load_vec<DType_f32, V>(a.pre_w, i, w);
#pragma unroll
    for (int e = 0; e < V; ++e) x[e] = x[e] * rs * w[e];
    emit(i, x);
  }
}

template <class DT, int V, bool DEPTH>
__global__ __launch_bounds__(kRowThreads) void residual_norm_kernel(socket_residual a) {
  extern __shared__ __attribute__((aligned(16))) float row_buf[];
  __shared__ float red[2][4];
  const int64_t row = blockIdx.x;
  residual_row<DT, V, DEPTH>(a, row, row_buf, red, true, [&](int i, const float* v) {
    if (a.h_out) store_vec<DT, V>(a.h_out, row * a.dim + i, v);
  });
}

__device__ __forceinline__ float clamped_glu(float g, float u, float limit) {
  g = fminf(g, limit);
  u = fminf(fmaxf(u, -limit), limit);
  return g * sigmoid_f32(1.702f * g) * (u + 1.f);
}

__device__ __forceinline__ float gated_unit(int kind, float g, float u, float limit) {
  return kind == 1 ? clamped_glu(g, u, limit) : g * sigmoid_f32(g) * u;
}

template <class DT, int V>
__global__ __launch_bounds__(256) void gated_unit_kernel(const void* __restrict__ gu, void* __restrict__ out,
                                                         int64_t rows, int ff, int kind, float limit) {
  const int64_t per_row = ff / V;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t >= rows * per_row) return;
  const int64_t r = t / per_row, j = (t % per_row) * V;
  float g[V], u[V];
  load_vec<DT, V>(gu, r * 2 * ff + j, g);
  load_vec<DT, V>(gu, r * 2 * ff + ff + j, u);
#pragma unroll
  for (int e = 0; e < V; ++e) g[e] = gated_unit(kind, g[e], u[e], limit);
  store_vec<DT, V>(out, r * ff + j, g);
}

constexpr int kVec = 8;                    // weights per lane and load
constexpr int kDepth = 4;                  // loads of a chunk of a row
constexpr int kShortDepth = 2;             // the same of rows that are one short chunk, whose inputs the lanes keep
constexpr int kChunkElems = 64 * kVec * kDepth, kShortElems = 64 * kVec * kShortDepth;
constexpr int kWgPerCu = 4;                // workgroups per CU of a persistent launch
constexpr int kInputVecs = 8;              // 16-byte vectors of a lane that wait in registers on their way to LDS

__host__ __device__ __forceinline__ int chunks_of(int K, int elems = kChunkElems) { return (K + elems - 1) / elems; }

typedef uint32_t rl_u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

// Where the input rows come from.
enum RowsInput {
  kFromMemory,      // x1 (and x2), requested with the weights that they meet: rows that do not fit into LDS
  kFromLds,         // x1 (and x2), brought into LDS
  kNormRows,        // residual_row's, one row after the other, behind the first weights: half of a wave's slots
  kNormRowsLong,    // the same behind all of its slots, where a wave has more chunks than that
  kNormEarly2,      // residual_row's for one row of up to 2 float4 vectors a lane, its operands requested ahead of the weights
  kNormEarly4,      // the same, up to 4
};

// Chunks of a wave in flight: 16 KB of weights, or two chunks and the inputs' beside them.
constexpr int most_slots(RowsInput in, int two) { return in == kFromMemory || two == 1 ? 2 : 4; }

// A row of weights as a buffer: loads past its end give zeros and ask the memory for nothing, so that whether there is a
// row at all is no branch (behind one, the compiler's wait for a chunk would be a wait for everything in flight).
__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_buffer(const uint16_t* w, int64_t n, int K, bool there) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w + (there ? n * K : 0)), 0, there ? K * 2 : 0, 0x00027000);
}

constexpr int kStreaming = 2;              // cache policy of a buffer load: nt

// Chunk kc of a row, DEPTH vectors a lane; `last`: of which those behind it are zeros without a load.
template <int POLICY = kStreaming, int DEPTH>
__device__ __forceinline__ void fetch_chunk(rl_u32x4 (&v)[DEPTH], __amdgpu_buffer_rsrc_t row, int kc, int lane, int last = DEPTH - 1) {
  const int at = kc * (DEPTH * 1024) + lane * 16;
#pragma unroll
  for (int u = 0; u < DEPTH; ++u)
    if (u > last) v[u] = rl_u32x4{0, 0, 0, 0};
    else v[u] = __builtin_bit_cast(rl_u32x4, __builtin_amdgcn_raw_buffer_load_b128(row, at + u * 1024, 0, POLICY));
}

// acc + the two products of bf16 pairs (an element of a vector has to be a value of its own here: a bit cast of the element
// itself takes the vector's first).  Products are exact in 32 bits; how the three are rounded is the instruction's own.  Error of
// whole rows against float64 beside a chain of two multiply-adds, 300 draws each: N(0, 1) 7.48e-8 / 7.43e-8 at 2048 elements, 1.19e-7 /
// 1.16e-7 at 14336, positive 4.23e-8 / 4.24e-8 (+- 0.1 %), heavy-tailed 2.45e-7 / 2.00e-7.  Subnormal operands and results are kept;
// products past 2^128 are infinities, which of opposite signs in one pair give a NaN where the chain gives the infinity.
__device__ __forceinline__ float dot2(uint32_t w, uint32_t x, float acc) {
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w), __builtin_bit_cast(bf16x2, x), acc, false);
}

// A chunk of a row with the M input rows in LDS.  Lanes past the rows' end have zero weights; ZEROS: and find zeros in place of the
// input, else take them, for what they would read might be an infinity (and several rows end with their last vector that holds
// any of it: 4 rows of 12296, 3392 results with the residual, 29.1 us as it was, 30.1 with all four vectors, 28.8 now).
template <int M, bool ZEROS>
__device__ __forceinline__ void mul_chunk(float (&acc)[M], const rl_u32x4 (&v)[kDepth], const uint16_t* x, int64_t xs, int K,
                                          int kc, int lane) {
  auto mul = [&](auto whole) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kDepth; ++u) {
      const int k = kc * kChunkElems + (u * 64 + lane) * kVec;
      if (!decltype(whole)::value && u > 0 && kc * kChunkElems + u * 64 * kVec >= K) break;      // (uniform: nothing left)
#pragma unroll
      for (int m = 0; m < M; ++m) {
        constexpr bool kWhole = decltype(whole)::value;
        const rl_u32x4 xv = *reinterpret_cast<const rl_u32x4*>(x + m * xs + (kWhole ? k : min(k, K - kVec)));
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[m] = dot2(v[u][i], kWhole || k < K ? xv[i] : 0u, acc[m]);
      }
    }
  };
  if (ZEROS || (kc + 1) * kChunkElems <= K) mul(std::true_type{});
  else mul(std::false_type{});
}

// The same with the input's chunk in registers, zeros where there is none.
template <int M, int DEPTH>
__device__ __forceinline__ void mul_chunk(float (&acc)[M], const rl_u32x4 (&v)[DEPTH], const rl_u32x4 (&x)[M][DEPTH], int last = DEPTH - 1) {
#pragma unroll
  for (int u = 0; u < DEPTH; ++u)
#pragma unroll
    for (int m = 0; m < M && u <= last; ++m)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[m] = dot2(v[u][i], x[m][u][i], acc[m]);
}

// Zeros behind a row of K elements in LDS, up to the end of its last chunk.
__device__ __forceinline__ void zeros_behind(uint16_t* row, int K) {
  const int at = K + (int)threadIdx.x * kVec;
  if (at < chunks_of(K) * kChunkElems) *reinterpret_cast<rl_u32x4*>(row + at) = rl_u32x4{0, 0, 0, 0};
}

// M input rows of K elements on their way to LDS: N vectors of every lane's wait in registers (zeros past the rows' end, by
// the same means as the weights'), what is left goes there at once.
template <int M, int N>
__device__ __forceinline__ void request_input(rl_u32x4 (&v)[N], uint16_t* lds, const uint16_t* x, int K) {
  const __amdgpu_buffer_rsrc_t rows = row_buffer(x, 0, M * K, true);
#pragma unroll
  for (int i = 0; i < N; ++i) {
    if (i * kRowThreads * kVec >= M * K) break;     // (uniform)
    v[i] = __builtin_bit_cast(rl_u32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, (i * kRowThreads + (int)threadIdx.x) * 16, 0, 0));
  }
#pragma unroll 1
  for (int at = N * kRowThreads; at < M * K / kVec; at += N * kRowThreads) {
    rl_u32x4 r[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
      r[i] = __builtin_bit_cast(rl_u32x4, __builtin_amdgcn_raw_buffer_load_b128(rows, (at + i * kRowThreads + (int)threadIdx.x) * 16, 0, 0));
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (at + i * kRowThreads + (int)threadIdx.x < M * K / kVec)
        reinterpret_cast<rl_u32x4*>(lds)[at + i * kRowThreads + threadIdx.x] = r[i];
  }
}
template <int M, int N>
__device__ __forceinline__ void place_input(const rl_u32x4 (&v)[N], uint16_t* lds, int K) {
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (i * kRowThreads + (int)threadIdx.x < M * K / kVec) reinterpret_cast<rl_u32x4*>(lds)[i * kRowThreads + threadIdx.x] = v[i];
}

// residual_row for a row of at most kRowThreads * 4 * NV elements without a second pending term, in two parts: the
// operands' requests, and the rest, which finds them on their way.  The same sums in the same order.
template <int NV>
struct EarlyNorm {
  float4 x[NV], w[NV], y[NV], pw[NV];

  static __host__ bool serves(const socket_residual& a) { return a.dim % 4 == 0 && a.dim <= kRowThreads * 4 * NV && !a.b; }

  __device__ __forceinline__ void request(const socket_residual& a) {
    const bool pending = a.a != nullptr, post = pending && a.post_w;
    int64_t src = 0;
    if (!a.x) {
      const int64_t id = a.ids64 ? ((const int64_t*)a.ids)[0] : (int64_t)((const int32_t*)a.ids)[0];
      src = (id < 0 ? 0 : (id >= a.vocab ? a.vocab - 1 : id)) * a.dim;
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = (v * kRowThreads + (int)threadIdx.x) * 4;
      if (i >= a.dim) break;
      if (a.x) x[v] = *reinterpret_cast<const float4*>(a.x + i);
      else load_vec<DType_bf16, 4>(a.embed, src + i, &x[v].x);
      if (pending) {
        if (a.pending_f32) y[v] = *reinterpret_cast<const float4*>((const float*)a.a + i);
        else load_vec<DType_bf16, 4>(a.a, i, &y[v].x);
      }
      if (post) pw[v] = *reinterpret_cast<const float4*>(a.post_w + i);
      w[v] = *reinterpret_cast<const float4*>(a.pre_w + i);
    }
  }

  template <class Emit>
  __device__ __forceinline__ void finish(const socket_residual& a, float (*red)[4], bool store_x, Emit emit) {
    float rs_y = 1.f;
    if (a.a) {
      float ss = 0.f;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        if ((v * kRowThreads + (int)threadIdx.x) * 4 >= a.dim) break;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float& t = (&y[v].x)[e];
          t *= a.scale_a;
          ss = fmaf(t, t, ss);
        }
      }
      if (a.post_w) rs_y = rsqrt_f32(block_sum(ss, red[0]) / (float)a.dim + a.eps);
    }
    float ss = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = (v * kRowThreads + (int)threadIdx.x) * 4;
      if (i >= a.dim) break;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float& t = (&x[v].x)[e];
        if (!a.x) t *= a.embed_scale;
        if (a.a) {
          float u = (&y[v].x)[e];
          if (a.post_w) u = u * rs_y * (&pw[v].x)[e];
          t += u;
        }
        ss = fmaf(t, t, ss);
      }
      if (store_x && a.x_out) *reinterpret_cast<float4*>(a.x_out + i) = x[v];
    }
    const float rs = rsqrt_f32(block_sum(ss, red[1]) / (float)a.dim + a.eps);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int i = (v * kRowThreads + (int)threadIdx.x) * 4;
      if (i >= a.dim) break;
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = (&x[v].x)[e] * rs * (&w[v].x)[e];
      emit(i, o);
    }
  }
};

// One wave per output feature; wave g of the launch takes features g, g + waves, ...
// TWO: 0 one product, 1 the gated unit (w1 and w2 share the input row), 2 a second scaled product (x2 . w2).  RES: the
// residual sum and the average over depth in the epilogue; a wave takes one feature, whose earlier results its lanes gather
// (one each) before the weights arrive.
//
// Bound by the stream of weights, and a launch is so short (5 to 20 us) that what counts is how soon all of it is asked
// for.  The input's operands are requested first, behind them up to 16 KB of weights a wave (its next SLOTS chunks, each
// register refilled right after its use); loads return in order, so an input requested behind the weights would arrive
// behind them.  `row_buffer` keeps every wait a wait for one chunk.  The products are the pairwise dot instruction's: with
// a conversion of each operand in front of a multiply-add the vector ALUs took 4 of the 14 us of the first line.
// us a launch, weights that no cache holds, before (weights first, two chunks in flight, inputs without a norm read from
// memory behind them) / now, beside a launch that only reads as many bytes:
//   norm, gated 2 x 8192 x 2048       14.25 / 12.3 (10.8)     one row; 2 rows 19.9 / 16.0; 4 rows 26.4 / 20.8
//   norm, 32000 x 2048                23.4 / 22.0 (20.2)      norm, 3392 x 2048   5.8 / 5.1
//   sum and average, 2048 x 8192       8.45 / 7.75 (6.2)      2048 x 2048         3.46 / 3.27 (2.8)
//   norm, gated 2 x 14336 x 4096      40.7 / 38.3             4096 x 14336       21.9 / 19.9
// Inputs that LDS does not hold ride with the weights (read from memory as before / as they are used, between requests for weights / now):
//   4 rows: 1000 x 20480   17.0 / 25.0 / 12.6     5120 x 20480   62.6 / 78.5 / 55.8     1000 x 98304   75 / 208 / 58
//           two terms of 14336: 1000 rows of each 22.0 / 34.5 / 18.9, 14336 231 / 224 / 221;  3 rows, 1000: 19.9 / 29.2 / 17.0
// SHORT: rows of at most kShortElems, whose inputs every lane takes into registers before the first product (from memory by
// itself, IN == kFromMemory, or what a norm left in LDS), so that a row's work is two loads and two vectors' products, not four.
// us a launch, loads past a row's end skipped by branches (as it was) / chunks of four vectors / now:
//   one row   3392 x 256 2.64 / 3.04 / 2.52    32000 x 256 7.4 / 8.5 / 6.0    32000 x 1000 14.3 / 11.9 / 11.6    residual, 3392 x 256 2.67 / 3.01 / 2.67
//   4 rows    3392 x 256 3.38 / 3.95 / 3.10    32000 x 256 12.3 / 18.5 / 10.4   32000 x 1000 20.9 / 20.8 / 14.7   norm, gated 2 x 32000 x 256 27 / 37 / 21
// From 1032 elements on the chunks of four are ahead of what was: 4 rows of 1032, 3392 results 4.99 / 4.57, 1000 4.28 / 3.41.
template <int M, RowsInput IN, int TWO, bool RES, int SLOTS, bool SHORT>
__global__ __launch_bounds__(kRowThreads) void rows_linear_kernel(socket_rows_linear a, socket_residual nrm) {
  extern __shared__ __attribute__((aligned(16))) float rl_lds[];
  __shared__ float red[2][4];
  constexpr bool EARLY = IN == kNormEarly2 || IN == kNormEarly4;
  constexpr bool ZEROS = M == 1 && (EARLY || IN == kFromLds), MEM = IN == kFromMemory && !SHORT;
  constexpr int kLoads = SHORT ? kShortDepth : kDepth, kElems = SHORT ? kShortElems : kChunkElems;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = gridDim.x * (kRowThreads / 64);
  int n = blockIdx.x * (kRowThreads / 64) + wave;   // (wave-uniform)
  const uint16_t* w1 = (const uint16_t*)a.w1;
  const uint16_t* w2 = (const uint16_t*)a.w2;
  const uint16_t* x1 = (const uint16_t*)a.x1;
  const uint16_t* x2 = TWO == 2 ? (const uint16_t*)a.x2 : x1;
  const int K1 = a.K1, K2 = TWO == 2 ? a.K2 : K1;
  constexpr bool NORM_ROWS = IN == kNormRows || IN == kNormRowsLong;
  const int nk1 = chunks_of(K1, kElems), nk = TWO == 2 ? nk1 + chunks_of(K2, kElems) : nk1;
  const int rows1 = ZEROS ? nk1 * kChunkElems : M * K1;     // elements of LDS in front of the second input's

  // (which vectors of a short row hold any of it: a branch, which costs nothing where a wave has one row, but for the residual's
  // single row, 2.67 us without and 2.75 with it for 3392 x 256)
  const int last1 = SHORT && SLOTS == 1 && !(RES && M == 1) ? (K1 - 1) / (64 * kVec) : kLoads - 1;

  // ---- the input's requests ----
  uint16_t* xs = reinterpret_cast<uint16_t*>(rl_lds) + (NORM_ROWS ? 2 * K1 : 0);    // (behind residual_row's floats)
  constexpr int kIn = TWO == 2 ? kInputVecs / 2 : kInputVecs;      // vectors a lane requests of either input
  rl_u32x4 in1[IN == kFromLds ? kIn : 1], in2[IN == kFromLds && TWO == 2 ? kIn : 1];
  EarlyNorm<IN == kNormEarly4 ? 4 : 2> early;
  rl_u32x4 held1[SHORT ? M : 1][kLoads], held2[SHORT ? M : 1][kLoads];
  if constexpr (EARLY) early.request(nrm);
  if constexpr (SHORT && IN == kFromMemory) {
#pragma unroll
    for (int m = 0; m < M; ++m) {
      fetch_chunk<0>(held1[m], row_buffer(x1, m, K1, true), 0, lane, last1);
      if constexpr (TWO == 2) fetch_chunk<0>(held2[m], row_buffer(x2, m, K2, true), 0, lane);
    }
  }
  if constexpr (IN == kFromLds) {
    request_input<M, kIn>(in1, xs, x1, K1);
    if constexpr (TWO == 2) request_input<M, kIn>(in2, xs + rows1, x2, K2);
  }
  // RES: the stream, the share of the result in the average, and this lane's earlier result with its share
  float before[M], past[M], own = 1.f, share = 0.f;
  if constexpr (RES) {
    const socket_depth_mix& d = a.depth;
    const bool averaged = d.w && n < a.N && lane < d.n;
    if (d.w) own = d.w[d.n];
    if (averaged) share = d.w[lane];
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int64_t at = (int64_t)m * a.N + min(n, a.N - 1);
      before[m] = a.res[at];
      past[m] = averaged ? d.past[lane * d.past_stride + at] : 0.f;
    }
  }

  // ---- the first weights' ----
  rl_u32x4 wv[SLOTS][kLoads], gv[TWO == 1 ? SLOTS : 1][kLoads], xv[MEM ? SLOTS : 1][M][kLoads];
  uint16_t bias1[SLOTS], bias2[TWO == 1 ? SLOTS : 1];
  const __amdgpu_buffer_rsrc_t b1 = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.b1), 0, a.b1 ? a.N * 2 : 0, 0x00027000);
  const __amdgpu_buffer_rsrc_t b2 = __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(a.b2), 0, a.b2 ? a.N * 2 : 0, 0x00027000);
  int fn = n, fkc = 0;                     // the next chunk to request
  auto fetch = [&](auto slot) __attribute__((always_inline)) {
    constexpr int i = decltype(slot)::value;
    const bool there = fn < a.N;
    const bool second = TWO == 2 && fkc >= nk1;
    const int K = second ? K2 : K1, at = second ? fkc - nk1 : fkc;
    if constexpr (MEM)
#pragma unroll
      for (int m = 0; m < M; ++m) fetch_chunk<0>(xv[i][m], row_buffer(second ? x2 : x1, m, K, there), at, lane);
    fetch_chunk(wv[i], row_buffer(second ? w2 : w1, fn, K, there), at, lane, last1);
    bias1[i] = __builtin_amdgcn_raw_buffer_load_b16(b1, there ? fn * 2 : 0, 0, 0);
    if constexpr (TWO == 1) {
      fetch_chunk(gv[i], row_buffer(w2, fn, K1, there), fkc, lane, last1);
      bias2[i] = __builtin_amdgcn_raw_buffer_load_b16(b2, there ? fn * 2 : 0, 0, 0);
    }
    const bool row_ends = ++fkc == nk;
    fn = row_ends ? fn + waves : fn;
    fkc = row_ends ? 0 : fkc;
  };
  // (Rows normed one after the other have trips to memory for each, which all of a wave's weights, requested first, would keep
  // waiting to the last.  2 and 4 rows, us with all slots / half of them first: 14336 x 2048 15.7 / 14.7 and 20.3 / 18.9, gated
  // 2 x 3392 x 4096 17.6 / 16.2 and 34.2 / 32.3; past as many chunks the stream counts, 32000 x 2048 24.4 / 25.0 and 30.2 / 29.8.)
  constexpr int kFirst = IN == kNormRows && !SHORT && SLOTS > 1 ? SLOTS / 2 : SLOTS;
  static_for<kFirst>(fetch);

  // ---- the input ----
  if constexpr (EARLY) {
    early.finish(nrm, red, blockIdx.x == 0, [&](int i, const float* v) { store_vec<DType_bf16, 4>(xs, i, v); });
    zeros_behind(xs, K1);
    __syncthreads();
  } else if constexpr (NORM_ROWS) {
    for (int m = 0; m < M; ++m) {
      residual_row<DType_bf16, 4, false>(nrm, m, rl_lds, red, blockIdx.x == 0,
                                  [&](int i, const float* v) { store_vec<DType_bf16, 4>(xs, (int64_t)m * K1 + i, v); });
      __syncthreads();
    }
    static_for<SLOTS - kFirst>([&](auto slot) __attribute__((always_inline)) { fetch(std::integral_constant<int, decltype(slot)::value + kFirst>{}); });
  } else if constexpr (IN == kFromLds) {
    place_input<M, kIn>(in1, xs, K1);
    if constexpr (TWO == 2) place_input<M, kIn>(in2, xs + rows1, K2);
    if constexpr (ZEROS) zeros_behind(xs, K1);
    if constexpr (ZEROS && TWO == 2) zeros_behind(xs + rows1, K2);
    __syncthreads();
  }
  if constexpr (IN != kFromMemory) {
    x1 = xs;
    x2 = IN == kFromLds ? xs + rows1 : xs;
  }
  if constexpr (SHORT && IN != kFromMemory) {
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
      for (int u = 0; u < kLoads; ++u) {
        const int k = (u * 64 + lane) * kVec;
        held1[m][u] = *reinterpret_cast<const rl_u32x4*>(xs + m * K1 + (k < K1 ? k : 0));
        if (k >= K1) held1[m][u] = rl_u32x4{0, 0, 0, 0};
      }
  }

  float mixed[M];
  if constexpr (RES) {
    const socket_depth_mix& d = a.depth;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      mixed[m] = share * past[m];
      if (d.w && n < a.N)
#pragma unroll 1
        for (int j = lane + 64; j < d.n; j += 64) mixed[m] = fmaf(d.w[j], d.past[j * d.past_stride + (int64_t)m * a.N + n], mixed[m]);
    }
  }

  // ---- the products ----
  float acc[M], acc2[M];
#pragma unroll
  for (int m = 0; m < M; ++m) acc[m] = acc2[m] = 0.f;
  int kc = 0;
  auto step = [&](auto slot, auto refill) __attribute__((always_inline)) {
    constexpr int i = decltype(slot)::value;
    const bool row_ends = kc + 1 == nk;
    if constexpr (SHORT) {
      if (TWO == 2 && kc >= nk1) mul_chunk<M>(acc2, wv[i], held2);
      else mul_chunk<M>(acc, wv[i], held1, last1);
      if constexpr (TWO == 1) mul_chunk<M>(acc2, gv[i], held1, last1);
    } else if constexpr (MEM) {
      if (TWO == 2 && kc >= nk1) mul_chunk<M>(acc2, wv[i], xv[i]);
      else mul_chunk<M>(acc, wv[i], xv[i]);
      if constexpr (TWO == 1) mul_chunk<M>(acc2, gv[i], xv[i]);
    } else if (n < a.N) {
      if (TWO == 2 && kc >= nk1) mul_chunk<M, ZEROS>(acc2, wv[i], x2, K2, K2, kc - nk1, lane);
      else mul_chunk<M, ZEROS>(acc, wv[i], x1, K1, K1, kc, lane);
      if constexpr (TWO == 1) mul_chunk<M, ZEROS>(acc2, gv[i], x1, K1, K1, kc, lane);
    }
    float c1 = bf16_bits_to_f32(bias1[i]), c2 = TWO == 1 ? bf16_bits_to_f32(bias2[TWO == 1 ? i : 0]) : 0.f;
    if constexpr (decltype(refill)::value) {
      // (all of the slot has been read by here, or its refill would take other registers and have to be copied, which
      // waits for it)
      asm volatile("" : "+v"(c1), "+v"(c2));
      __builtin_amdgcn_sched_barrier(0);
      fetch(slot);
    }
    if (row_ends && n < a.N) {
#pragma unroll
      for (int m = 0; m < M; ++m) {
        float o = wave_reduce_to_last<false>(acc[m]);
        if (TWO) {
          const float o2 = wave_reduce_to_last<false>(acc2[m]);
          o = TWO == 1 ? gated_unit(a.kind, o + c1, o2 + c2, a.limit) : fmaf(a.s2, o2, a.s1 * o) + c1;
        } else {
          o = a.s1 * o + c1;
        }
        if constexpr (RES) {
          o += before[m];
          const float earlier = wave_reduce_to_last<false>(mixed[m]);
          if (lane == 63 && a.depth.w) a.depth.result[(int64_t)m * a.N + n] = o;
          o = fmaf(own, o, earlier);
        }
        if (lane == 63) {
          if (a.y_f32) ((float*)a.y)[(int64_t)m * a.N + n] = o;
          else ((uint16_t*)a.y)[(int64_t)m * a.N + n] = f32_to_bf16_bits(o);
        }
        acc[m] = acc2[m] = 0.f;
      }
    }
    n = row_ends ? n + waves : n;
    kc = row_ends ? 0 : kc + 1;
  };
  // (all slots in every turn: to leave in the middle of one would make the waits of the next for everything, too)
  if constexpr (SHORT ? SLOTS > 1 : SLOTS == most_slots(IN, TWO))
    while (fn < a.N) static_for<SLOTS>([&](auto slot) __attribute__((always_inline)) { step(slot, std::true_type{}); });
  static_for<SLOTS>([&](auto slot) __attribute__((always_inline)) { step(slot, std::false_type{}); });
}

template <int M, RowsInput IN, int TWO, bool RES, int SLOTS, bool SHORT = false>
int launch_rows_linear(const socket_rows_linear& a, int n_wg, size_t lds, hipStream_t s) {
  auto kern = rows_linear_kernel<M, IN, TWO, RES, SLOTS, SHORT>;
  if (lds > 48 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                             (int)lds) != hipSuccess)
    return SOCKET_ERR_LAUNCH;
  hipLaunchKernelGGL(kern, dim3((unsigned)n_wg), dim3(kRowThreads), lds, s, a, a.norm ? *a.norm : socket_residual{});
  return SOCKET_OK;
}

// A wave's slots: as many as it has chunks, up to 16 KB of weights (a load that finds no row left brings nothing, but takes
// its turn).
template <int M, RowsInput IN, int TWO, bool RES, bool SHORT = false>
int dispatch_slots(const socket_rows_linear& a, size_t lds, hipStream_t s) {
  constexpr int kWaves = kRowThreads / 64;
  int n_wg = (a.N + kWaves - 1) / kWaves;
  // (few workgroups pay for the input's passage: each keeps its waves streaming from row to row)
  if (!RES && (SHORT || IN != kFromMemory)) n_wg = std::min(n_wg, socket_device_limits().cu_count * kWgPerCu);
  constexpr int kElems = SHORT ? kShortElems : kChunkElems, kMost = SHORT && TWO != 1 ? 4 : most_slots(IN, TWO);
  const int nk = chunks_of(a.K1, kElems) + (TWO == 2 ? chunks_of(a.K2, kElems) : 0);
  const int64_t chunks = (int64_t)((a.N + n_wg * kWaves - 1) / (n_wg * kWaves)) * nk;
  if constexpr (RES && SHORT) return launch_rows_linear<M, IN, TWO, RES, 1, true>(a, n_wg, lds, s);      // (a wave, a row)
  if constexpr (TWO != 2 && (SHORT || IN != kFromMemory || (RES && M < 4))) {
    if (chunks == 1) return launch_rows_linear<M, IN, TWO, RES, 1, SHORT>(a, n_wg, lds, s);
    if (!SHORT && IN != kFromMemory && chunks == 2) return launch_rows_linear<M, IN, TWO, RES, 2>(a, n_wg, lds, s);
  }
  if constexpr (IN == kNormRows && !SHORT)
    if (chunks > kMost) return launch_rows_linear<M, kNormRowsLong, TWO, RES, kMost>(a, n_wg, lds, s);
  return launch_rows_linear<M, IN, TWO, RES, kMost, SHORT>(a, n_wg, lds, s);
}

template <int M, RowsInput IN, int TWO, bool SHORT = false>
int dispatch_res(const socket_rows_linear& a, size_t lds, hipStream_t s) {
  if constexpr (TWO == 0 && (IN == kFromMemory || IN == kFromLds))
    if (a.res) return dispatch_slots<M, IN, TWO, true, SHORT>(a, lds, s);
  return dispatch_slots<M, IN, TWO, false, SHORT>(a, lds, s);
}

template <int M, int TWO>
int dispatch_input(const socket_rows_linear& a, hipStream_t s) {
  const size_t room = (size_t)socket_device_limits().max_lds_per_block - 256;
  auto in_lds = [](int K) { return M == 1 ? ((size_t)K + kChunkElems - 1) / kChunkElems * kChunkElems * 2 : (size_t)M * K * 2; };
  const bool is_short = a.K1 <= kShortElems && (TWO != 2 || a.K2 <= kShortElems);
  if (!a.norm) {
    if (is_short) return dispatch_res<M, kFromMemory, TWO, true>(a, 0, s);
    // A residual's rows of one chunk while each CU has a workgroup at most: the way through LDS is on the chain of what the launch
    // waits for.  2048 elements, us through LDS / from memory: one row, 64 results 2.45 / 2.16, 1000 2.88 / 2.76, two rows 3.17 / 3.07,
    // three 3.41 / 3.36, four 3.60 / 3.68; one row, 3392 results 4.44 / 4.59; without a residual, one row, 1000 results 2.74 / 3.04.
    if (M < 4 && a.res && chunks_of(a.K1) == 1 && a.N <= kRowThreads / 64 * socket_device_limits().cu_count)
      return dispatch_res<M, kFromMemory, TWO>(a, 0, s);
    // (LDS also where it leaves a CU one workgroup: us from memory, a chunk ahead / from LDS, 4 rows of 14336: 1000 results 12.2 / 8.8,
    // 4096 33.5 / 29.9, 14336 111 / 70, the last with the residual 113 / 98; 3 rows 94.9 / 66.3; 2 rows 77.5 / 62.5)
    const size_t lds = in_lds(a.K1) + (TWO == 2 ? in_lds(a.K2) : 0);
    return lds <= room ? dispatch_res<M, kFromLds, TWO>(a, lds, s) : dispatch_res<M, kFromMemory, TWO>(a, 0, s);
  }
  if constexpr (TWO == 2) {
    return SOCKET_ERR_UNSUPPORTED;
  } else {
    const size_t rows = (size_t)a.K1 * (4 + 2 * M);
    if (rows > room) return SOCKET_ERR_UNSUPPORTED;
    if constexpr (M == 1) {
      if (EarlyNorm<2>::serves(*a.norm)) return dispatch_res<M, kNormEarly2, TWO>(a, in_lds(a.K1), s);
      if (EarlyNorm<4>::serves(*a.norm)) return dispatch_res<M, kNormEarly4, TWO>(a, in_lds(a.K1), s);
    }
    if constexpr (M > 1)
      if (is_short) return dispatch_res<M, kNormRows, TWO, true>(a, rows, s);
    return dispatch_res<M, kNormRows, TWO>(a, rows, s);
  }
}

template <int M>
int dispatch_rows_linear(const socket_rows_linear& a, hipStream_t s) {
  if (a.kind != 0) return dispatch_input<M, 1>(a, s);
  return a.x2 ? dispatch_input<M, 2>(a, s) : dispatch_input<M, 0>(a, s);
}

int check_residual(const socket_residual* a) {
  SOCKET_REQUIRE(a && a->pre_w, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(a->x || (a->embed && a->ids), SOCKET_ERR_NULL);
  SOCKET_REQUIRE(a->x || a->vocab > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(a->a || !a->b, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(!a->depth.w || (a->depth.result && a->depth.n >= 0 && (a->depth.past || a->depth.n == 0)), SOCKET_ERR_NULL);
  SOCKET_REQUIRE(a->x_stride >= 0 && (a->x_stride == 0 || a->x_out != a->x), SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(a->dim > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(a->dtype == SOCKET_F32 || a->dtype == SOCKET_BF16, SOCKET_ERR_UNSUPPORTED);
  if (a->dim % 4 == 0) {
    const void* ptrs[] = {a->x, a->embed, a->a, a->b, a->post_w, a->pre_w, a->x_out, a->h_out};
    for (const void* p : ptrs) SOCKET_REQUIRE(p == nullptr || socket_aligned16(p), SOCKET_ERR_ALIGN);
    SOCKET_REQUIRE(a->x_stride % 4 == 0 && (!a->depth.w || (a->depth.past_stride % 4 == 0 && socket_aligned16(a->depth.past) &&
                                                            socket_aligned16(a->depth.result))), SOCKET_ERR_ALIGN);
  }
  return SOCKET_OK;
}

}  // namespace

extern "C" int socket_residual_norm(const socket_residual* args, int64_t rows, void* stream) {
  const int rc = check_residual(args);
  if (rc != SOCKET_OK) return rc;
  SOCKET_REQUIRE(rows > 0 && rows < (1LL << 31), SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(args->dim <= 32768, SOCKET_ERR_UNSUPPORTED);
  const size_t lds = (size_t)args->dim * 4;
  hipStream_t s = (hipStream_t)stream;
#define SOCKET_RN(DT, V)                                                                                            \
  do {                                                                                                              \
    auto kern = args->depth.w ? residual_norm_kernel<DT, V, true> : residual_norm_kernel<DT, V, false>;                                                                        \
    if (lds > 48 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern),                                 \
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess) \
      return SOCKET_ERR_LAUNCH;                                                                                     \
    hipLaunchKernelGGL(kern, dim3((unsigned)rows), dim3(kRowThreads), lds, s, *args);                               \
  } while (0)
  const bool v4 = args->dim % 4 == 0;
  if (args->dtype == SOCKET_F32) {
    if (v4) SOCKET_RN(DType_f32, 4);
    else SOCKET_RN(DType_f32, 1);
  } else {
    if (v4) SOCKET_RN(DType_bf16, 4);
    else SOCKET_RN(DType_bf16, 1);
  }
#undef SOCKET_RN
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

extern "C" int socket_rows_linear_bf16(const socket_rows_linear* args, void* stream) {
  SOCKET_REQUIRE(args && args->w1 && args->y, SOCKET_ERR_NULL);
  const socket_rows_linear& a = *args;
  SOCKET_REQUIRE(a.kind >= 0 && a.kind <= 2, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(a.M >= 1 && a.N >= 1 && a.K1 >= 1, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(a.M <= 4 && a.K1 % 8 == 0, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(socket_aligned16(a.w1) && (!a.w2 || socket_aligned16(a.w2)), SOCKET_ERR_ALIGN);
  SOCKET_REQUIRE(a.kind == 0 || a.w2, SOCKET_ERR_NULL);
  if (a.norm) {
    const int rc = check_residual(a.norm);
    if (rc != SOCKET_OK) return rc;
    SOCKET_REQUIRE(!a.x2 && !a.res && !a.norm->depth.w && a.norm->dtype == SOCKET_BF16, SOCKET_ERR_UNSUPPORTED);
    SOCKET_REQUIRE(a.norm->dim == a.K1 && (a.norm->x_out == nullptr || a.norm->x_out != a.norm->x), SOCKET_ERR_SHAPE);
  } else {
    SOCKET_REQUIRE(a.x1 != nullptr, SOCKET_ERR_NULL);
    SOCKET_REQUIRE(socket_aligned16(a.x1), SOCKET_ERR_ALIGN);
  }
  if (a.res) {
    SOCKET_REQUIRE(a.kind == 0 && !a.x2 && a.y_f32 && (const void*)a.res != a.y, SOCKET_ERR_UNSUPPORTED);
    SOCKET_REQUIRE(!a.depth.w || (a.depth.result && a.depth.n >= 0 && (a.depth.past || a.depth.n == 0)), SOCKET_ERR_NULL);
  }
  if (a.x2) {
    SOCKET_REQUIRE(a.w2 && a.kind == 0, SOCKET_ERR_NULL);
    SOCKET_REQUIRE(a.K2 >= 8 && a.K2 % 8 == 0, SOCKET_ERR_UNSUPPORTED);
    SOCKET_REQUIRE(socket_aligned16(a.x2), SOCKET_ERR_ALIGN);
  }
  hipStream_t s = (hipStream_t)stream;
  int rc;
  switch (a.M) {
    case 1: rc = dispatch_rows_linear<1>(a, s); break;
    case 2: rc = dispatch_rows_linear<2>(a, s); break;
    case 3: rc = dispatch_rows_linear<3>(a, s); break;
    default: rc = dispatch_rows_linear<4>(a, s); break;
  }
  if (rc != SOCKET_OK) return rc;
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

extern "C" int socket_gated_unit(const void* gu, void* out, int dtype, int64_t rows, int ff, int kind, float limit,
                                 void* stream) {
  SOCKET_REQUIRE(gu && out, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(kind == 1 || kind == 2, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(dtype == SOCKET_F32 || dtype == SOCKET_BF16, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(rows > 0 && ff > 0, SOCKET_ERR_SHAPE);
  const bool v8 = ff % 8 == 0 && socket_aligned16(gu) && socket_aligned16(out);
  const int64_t items = rows * (v8 ? ff / 8 : ff);
  SOCKET_REQUIRE((items + 255) / 256 < (1LL << 31), SOCKET_ERR_SHAPE);
  const dim3 grid((unsigned)((items + 255) / 256)), block(256);
  hipStream_t s = (hipStream_t)stream;
#define SOCKET_CG(DT, V) hipLaunchKernelGGL((gated_unit_kernel<DT, V>), grid, block, 0, s, gu, out, rows, ff, kind, limit)
  if (dtype == SOCKET_F32) {
    if (v8) SOCKET_CG(DType_f32, 8);
    else SOCKET_CG(DType_f32, 1);
  } else {
    if (v8) SOCKET_CG(DType_bf16, 8);
    else SOCKET_CG(DType_bf16, 1);
  }
#undef SOCKET_CG
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}
