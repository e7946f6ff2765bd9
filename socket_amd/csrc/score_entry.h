// The entries of a soft-hash table in LDS, their sums, and the operands of the packed cache's scorers (score.hip,
// score_short.hip).
#pragma once
#include <type_traits>

#include "socket_common.h"

namespace {

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2_t;

struct TabF32 {
  typedef float elem;
  static constexpr int kEnum = SOCKET_F32;
};
struct TabBF16 {
  typedef uint16_t elem;
  static constexpr int kEnum = SOCKET_BF16;
};

// One LDS entry (the GP heads' values for one bucket of one table) as raw words,
// so that the gather (load) and the accumulation can be scheduled apart.
template <int BYTES>
struct RawEntry;
template <>
struct RawEntry<2> { uint16_t w; };
template <>
struct RawEntry<4> { uint32_t w; };
template <>
struct RawEntry<8> { uint2 w; };
template <>
struct RawEntry<16> { uint4 w; };
template <>
struct RawEntry<32> { uint4 w[2]; };

template <int BYTES>
__device__ __forceinline__ RawEntry<BYTES> load_entry(const void* lds) {
  return *reinterpret_cast<const RawEntry<BYTES>*>(lds);
}

// bf16 entries are widened and added by the matrix core used as a four-wide
// adder: v_mfma_f32_4x4x4_16B_bf16 computes, in each of its 16 independent 4x4
// blocks (4 lanes each), D[i][j] = C[i][j] + sum_k A[i][k] * B[k][j], where lane
// j of a block supplies column B[:,j] (4 bf16 = one 8-byte LDS entry: the four
// heads' values) and holds column D[:,j] (4 fp32 = that lane's four head sums),
// and lane i supplies row A[i,:].  With A the identity (lane i holds e_i) this is
// acc[h] += entry[h] for h = 0..3 in one instruction, on a pipe that is
// otherwise idle, instead of four VALU operations.  The products are exact; the
// matrix core's accumulate may round differently from the fp32 adder in the last
// place (and flushes denormals), hence the 2e-6 relative bound stated for bf16
// tables; the fp32-table path uses plain adds and reproduces the reference sum
// exactly.
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// Streamed once: loads and stores that should not displace the table slices,
// which every tile of a (b, kv head) pair re-reads, from the L2.
__device__ __forceinline__ uint4 load_stream16(const uint32_t* p) {
  const u32x4_t v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void store_stream16(float* p, float a, float b, float c, float d) {
  float4_t v = {a, b, c, d};
  __builtin_nontemporal_store(v, reinterpret_cast<float4_t*>(p));
}

struct Bf16Select {
  short4_t identity_row;  // e_{lane % 4} as four bf16
};

__device__ __forceinline__ Bf16Select make_bf16_select(uint32_t bf16_one) {
  const int r = threadIdx.x & 3;
  uint2 w = make_uint2(0u, 0u);
  if (r == 0) w.x = bf16_one;
  else if (r == 1) w.x = bf16_one << 16;
  else if (r == 2) w.y = bf16_one;
  else w.y = bf16_one << 16;
  Bf16Select s;
  __builtin_memcpy(&s.identity_row, &w, 8);
  return s;
}

__device__ __forceinline__ void add4_bf16(float* acc, uint2 four, const Bf16Select& sel) {
  short4_t b;
  __builtin_memcpy(&b, &four, 8);
  float4_t c = {acc[0], acc[1], acc[2], acc[3]};
  c = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(sel.identity_row, b, c, 0, 0, 0);
  acc[0] = c[0];
  acc[1] = c[1];
  acc[2] = c[2];
  acc[3] = c[3];
}

// acc[g] += entry[g], fp32 table
template <int GP>
__device__ __forceinline__ void accumulate(float* acc, const RawEntry<GP * 4>& e, const TabF32*,
                                           const Bf16Select&) {
  if constexpr (GP == 1) {
    acc[0] += __uint_as_float(e.w);
  } else if constexpr (GP == 2) {
    acc[0] += __uint_as_float(e.w.x);
    acc[1] += __uint_as_float(e.w.y);
  } else if constexpr (GP == 4) {
    acc[0] += __uint_as_float(e.w.x);
    acc[1] += __uint_as_float(e.w.y);
    acc[2] += __uint_as_float(e.w.z);
    acc[3] += __uint_as_float(e.w.w);
  } else {
#pragma unroll
    for (int v = 0; v < 2; ++v) {
      acc[4 * v + 0] += __uint_as_float(e.w[v].x);
      acc[4 * v + 1] += __uint_as_float(e.w[v].y);
      acc[4 * v + 2] += __uint_as_float(e.w[v].z);
      acc[4 * v + 3] += __uint_as_float(e.w[v].w);
    }
  }
}

// acc[g] += entry[g], bf16 table
template <int GP>
__device__ __forceinline__ void accumulate(float* acc, const RawEntry<GP * 2>& e, const TabBF16*,
                                           const Bf16Select& sel) {
  if constexpr (GP == 1) {
    acc[0] += bf16_bits_to_f32(e.w);
  } else if constexpr (GP == 2) {
    float a4[4] = {acc[0], acc[1], 0.f, 0.f};
    add4_bf16(a4, make_uint2(e.w, 0u), sel);
    acc[0] = a4[0];
    acc[1] = a4[1];
  } else if constexpr (GP == 4) {
    add4_bf16(acc, e.w, sel);
  } else {
    add4_bf16(acc, make_uint2(e.w.x, e.w.y), sel);
    add4_bf16(acc + 4, make_uint2(e.w.z, e.w.w), sel);
  }
}

// LDS past the table buffers in every launch: scratch of the key-range reduction
constexpr size_t kScoreScratchBytes = 1024;


}  // namespace

struct ScoreArgs {
  const void* q_probs;
  const uint32_t* codes;
  const uint16_t* v_norm;
  const int32_t* lens;
  float* scores;
  int B, Hq, Hkv, L, P, R, T;
  int64_t Tcap, score_stride;
  uint32_t* row_range;
  int range_parts;
  hipStream_t stream;
  int grouped;  // table layout: 0 = [B,Hq,L,R], 1 = [B*Hkv*parts, L, R, group width]
  int flags;    // SOCKET_SCORE_*
};

// score_short.hip: calls with few tokens per CU
bool socket_score_short_serves(const ScoreArgs& a, size_t elem_bytes);
int socket_score_short(const ScoreArgs& a, size_t elem_bytes);
