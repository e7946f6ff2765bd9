// K5: query soft hash -- the producer of the scorer's bucket-probability table.
//
//   proj[l,k]  = q . planes[l,k,:]
//   t[k]       = tanh(proj[l,k]) * tanh_scale            (tanh_scale = 1 / sqrt(D))
//   logit[l,r] = inv_temperature * sum_k t[k] * protos_T[k,r]
//   probs[l,:] = softmax_r(logit[l,:])
//
// GPT-FAST/model.py:392-401 (inv_temperature 1) and the HuggingFace twin
// pipeline/train_quest/modeling/modeling_llama.py:618-638 (logits / 0.3), which
// run this as two einsums, a tanh, a division and a softmax, five launches with
// [B,H,L,K] and [B,H,L,R] intermediates rounded to the model dtype.  Here it is
// one launch computing in fp32 from the inputs as stored and rounding once, to
// the output dtype.
//
// Three forms: on the matrix cores (bf16, 128 dims, K = 10, R = 1024), a wave to a
// head (R <= 256), and the general one.  In that, one workgroup per (table l, batch b,
// KV head): the K planes of the table and the G query heads of the group sit in LDS,
// four lanes to a projection,
// then every lane owns runs of four buckets and makes three sweeps over them
// (maximum, sum of exponentials, normalised write), recomputing the K-term
// logits each time rather than holding R/64 of them per head in registers.
#include <type_traits>

#include "socket_common.h"

namespace {

constexpr int kSHThreads = 256;
constexpr int kSHWaves = kSHThreads / SOCKET_WAVE;
constexpr int kSHMaxK = 16;
constexpr int kSHMaxG = 8;
constexpr int kSHMaxD = 256;

template <class DT>
__device__ __forceinline__ float sh_load(const void* p, int64_t i);
template <>
__device__ __forceinline__ float sh_load<DType_f32>(const void* p, int64_t i) {
  return ((const float*)p)[i];
}
template <>
__device__ __forceinline__ float sh_load<DType_bf16>(const void* p, int64_t i) {
  return bf16_bits_to_f32(((const uint16_t*)p)[i]);
}
template <>
__device__ __forceinline__ float sh_load<DType_f16>(const void* p, int64_t i) {
  return f16_bits_to_f32(((const uint16_t*)p)[i]);
}

// Four consecutive elements starting at index i (the address must be aligned to
// the size of the four).
template <class DT>
__device__ __forceinline__ void sh_load4(const void* p, int64_t i, float (&o)[4]);
template <>
__device__ __forceinline__ void sh_load4<DType_f32>(const void* p, int64_t i, float (&o)[4]) {
  const float4 v = *reinterpret_cast<const float4*>((const float*)p + i);
  o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
}
template <>
__device__ __forceinline__ void sh_load4<DType_bf16>(const void* p, int64_t i, float (&o)[4]) {
  const uint2 v = *reinterpret_cast<const uint2*>((const uint16_t*)p + i);
  o[0] = bf16_bits_to_f32(v.x & 0xffffu); o[1] = bf16_bits_to_f32(v.x >> 16);
  o[2] = bf16_bits_to_f32(v.y & 0xffffu); o[3] = bf16_bits_to_f32(v.y >> 16);
}
template <>
__device__ __forceinline__ void sh_load4<DType_f16>(const void* p, int64_t i, float (&o)[4]) {
  const uint2 v = *reinterpret_cast<const uint2*>((const uint16_t*)p + i);
  o[0] = f16_bits_to_f32((uint16_t)(v.x & 0xffffu)); o[1] = f16_bits_to_f32((uint16_t)(v.x >> 16));
  o[2] = f16_bits_to_f32((uint16_t)(v.y & 0xffffu)); o[3] = f16_bits_to_f32((uint16_t)(v.y >> 16));
}

// x rounded to the storage type and widened again (what a stored value reads back as)
template <class DT>
__device__ __forceinline__ float sh_round(float x);
template <>
__device__ __forceinline__ float sh_round<DType_f32>(float x) { return x; }
template <>
__device__ __forceinline__ float sh_round<DType_bf16>(float x) { return bf16_bits_to_f32(f32_to_bf16_bits(x)); }
template <>
__device__ __forceinline__ float sh_round<DType_f16>(float x) { return f16_bits_to_f32(f32_to_f16_bits(x)); }

// Four consecutive elements (already representable in the storage type) to index i.
template <class DT>
__device__ __forceinline__ void sh_store4(void* p, int64_t i, const float (&v)[4]);
template <>
__device__ __forceinline__ void sh_store4<DType_f32>(void* p, int64_t i, const float (&v)[4]) {
  *reinterpret_cast<float4*>((float*)p + i) = make_float4(v[0], v[1], v[2], v[3]);
}
template <>
__device__ __forceinline__ void sh_store4<DType_bf16>(void* p, int64_t i, const float (&v)[4]) {
  *reinterpret_cast<uint2*>((uint16_t*)p + i) =
      make_uint2(f32x2_to_bf16_bits(v[0], v[1]), f32x2_to_bf16_bits(v[2], v[3]));
}
template <>
__device__ __forceinline__ void sh_store4<DType_f16>(void* p, int64_t i, const float (&v)[4]) {
  *reinterpret_cast<uint2*>((uint16_t*)p + i) =
      make_uint2((uint32_t)f32_to_f16_bits(v[0]) | ((uint32_t)f32_to_f16_bits(v[1]) << 16),
                 (uint32_t)f32_to_f16_bits(v[2]) | ((uint32_t)f32_to_f16_bits(v[3]) << 16));
}

// ---------------------------------------------------------------------------
// bf16 queries and planes of 128 dims, K = 10, R = 1024 (whatever the group): both products on the
// matrix cores, sixteen heads of one table to a workgroup.
//
//   proj^T[plane, head] = planes . q^T          v_mfma_f32_16x16x32_bf16, exact products, fp32 sums
//   logit[head, bucket] = t . protos            t in three bf16 terms (hi, mid, lo: all 24 bits), so that
//                                               two products of 16 x 16 x 32 keep what fp32 keeps
// The head is the N index of the first: lane x holds head x % 16, and the planes of lane quarter q are 4 q .. + 3; the terms a
// lane splits off are the operand it has to supply to the second, where the head is the M index: register r of quarter q is head 4 q + r,
// so that the heads of a unit lie in one lane and an entry of the table is stored as it is.  Bucket order inside a product is free:
// a lane's prototypes and its results are runs of kMxRun16 buckets.  A wave has 256 buckets.  Of what all four waves need, each works out a share: a
// quarter of the dims of the rotation and the projections, one plane of four of the tanh.  Logits are made in base-2 units
// (log2 e goes into t) for the hardware's exponential, and nothing is taken off them first where all of a head's are small,
// which they are with +-1 prototypes (tanh / sqrt(D) / temperature: at most 4.3); it is seen from the logits themselves.
// What bounds it are vector instructions, about 600 a wave at 64 logits a lane, and at few heads dependent trips to memory.
// Before (head as the N index of both products: entries put together by lane exchanges; every wave rotated and projected
// everything; maxima exchanged and taken off) and now, the decode prologue with the rest of its roles: one sequence of 32 heads x
// 60 tables 7.7 / 5.4 us, four 13.4 / 9.4, sixteen of 28 x 48 27.2 / 18.1.  (The scalar form below spends ten multiply-adds
// and a library exponential per head and bucket: 10.4, 23 and 56 us.)
//
// W: heads of a unit (the scorer's grouped layout [unit, L, R, W]; 1 for the reference's [B,Hq,L,R], whose
// units are heads).  OutDT: the table's type.  FT: void, or the element type of a rotary table, as above.
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 sh_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float sh_f32x4;
union ShFrag {
  uint4 u;
  sh_bf16x8 v;
};
__device__ __forceinline__ sh_f32x4 sh_mfma(const uint4& a, const uint4& b, sh_f32x4 c) {
  ShFrag x, y;
  x.u = a;
  y.u = b;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x.v, y.v, c, 0, 0, 0);
}

// eight consecutive table entries (cos, sin of four pairs) as floats
template <class FT>
__device__ __forceinline__ void sh_load8(const void* p, int64_t i, float (&o)[8]);
template <>
__device__ __forceinline__ void sh_load8<DType_bf16>(const void* p, int64_t i, float (&o)[8]) {
  unpack16<DType_bf16>(*reinterpret_cast<const uint4*>((const uint16_t*)p + i), o);
}
template <>
__device__ __forceinline__ void sh_load8<DType_f32>(const void* p, int64_t i, float (&o)[8]) {
  const float4 a = *reinterpret_cast<const float4*>((const float*)p + i);
  const float4 c = *reinterpret_cast<const float4*>((const float*)p + i + 4);
  o[0] = a.x, o[1] = a.y, o[2] = a.z, o[3] = a.w, o[4] = c.x, o[5] = c.y, o[6] = c.z, o[7] = c.w;
}

constexpr int kMxHeads = 16, kMxD = 128, kMxK = 10, kMxR = 1024;
constexpr float kMxPlain = 32.f;      // base-2 logits up to which nothing is taken off before the exponential

// Which heads the units are: `parts` units of W heads to a kv head's G (0: a unit is a head of Hq).
// per_seq: units of a sequence; the reciprocals are for mx_div.
struct MxUnits {
  int count, parts, Hq, Hkv, G, per_seq;
  float inv_per_seq, inv_parts;
};

// x / d of x >= 0 and 0 < d with inv = 1 / d in fp32: the rounded quotient is off by at most one while it is below 2^22.
__device__ __forceinline__ int mx_div(int x, int d, float inv) {
  int k = (int)((float)x * inv);
  k -= k * d > x ? 1 : 0;
  return k + ((k + 1) * d <= x ? 1 : 0);
}

// Sum or maximum over the sixteen lanes of a row, in every lane of it.
template <bool MAX>
__device__ __forceinline__ float mx_row(float x) {
#define SOCKET_STEP(ctrl)                                                                                               \
  {                                                                                                                     \
    const float o = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), ctrl, 0xf, 0xf, false));           \
    x = MAX ? fmaxf(x, o) : x + o;                                                                                      \
  }
  SOCKET_STEP(0x128)      // row_ror: 8, 4, 2, 1
  SOCKET_STEP(0x124)
  SOCKET_STEP(0x122)
  SOCKET_STEP(0x121)
#undef SOCKET_STEP
  return x;
}

// What the matrix-core forms share: where a lane's head is, the waves' shares of the projections put together, and the
// softmax and the write of one table.
struct MxHead {
  int b, head;
  bool live;
};
template <int W>
__device__ __forceinline__ MxHead mx_head(const int group, const MxUnits& units, int n) {
  const int first = group * (kMxHeads / W), b0 = first / units.per_seq;         // (uniform)
  const bool in_units = first + n / W < units.count;
  const int at0 = first - b0 * units.per_seq + (in_units ? n / W : 0), over = mx_div(at0, units.per_seq, units.inv_per_seq);
  const int at = at0 - over * units.per_seq;
  MxHead h{b0 + over, at, in_units};
  if (units.parts > 0) {
    const int kvh = mx_div(at, units.parts, units.inv_parts), member = (at - kvh * units.parts) * W + n % W;     // (of the kv head's group)
    h.live = in_units && member < units.G;
    h.head = kvh * units.G + (h.live ? member : 0);
  }
  return h;
}

// part: register r is this wave's share of plane 4 quarter + r of head n.  Returns t of those planes, each wave having worked out
// one register's (planes past the tenth: zero).
__device__ __forceinline__ sh_f32x4 mx_angles(const sh_f32x4& part, float scale, int wave, int lane) {
  __shared__ __attribute__((aligned(16))) sh_f32x4 shares[kSHWaves][SOCKET_WAVE];
  __shared__ __attribute__((aligned(16))) float angles[SOCKET_WAVE][4];
  shares[wave][lane] = part;
  __syncthreads();
  const float* at = (const float*)shares + 4 * lane + wave;
  constexpr int kStep = 4 * SOCKET_WAVE;
  const float proj = (at[0] + at[2 * kStep]) + (at[kStep] + at[3 * kStep]);
  angles[lane][wave] = 4 * (lane >> 4) + wave < kMxK ? tanhf(proj) * scale : 0.f;
  __syncthreads();
  return *reinterpret_cast<const sh_f32x4*>(angles[lane]);
}

// Buckets that follow one another in a lane, the same number for every layout and type of the table, whose sums are then the same:
// block ii of a 64-bucket chunk takes bucket mx_bucket<RUN>(n, ii) of it for column n.  Two 16-bit
// prototypes are fetched at once and 32-bit ones one by one, so that a lane's entries of four heads are 16 bytes in a row and its
// quarter's 256: more at once would leave them further apart.  Decode prologue in bf16, runs of four / two: one sequence of 32 heads x 60
// tables 6.0 / 5.4 us, four 10.7 / 9.4, sixteen of 28 x 48 20.9 / 18.1.  fp32 table of one / eight sequences of 32 heads x 60 by itself,
// runs of two / one: grouped 7.6, 22.3 / 6.6, 19.3 us, plain 7.0, 19.7 / 6.7, 19.4 (before, heads as columns: 8.1, 23.3 and 10.1, 34.2);
// steps over 15617 tokens of two sequences of 64 heads, four layers, runs of four 270 us, two 257, one 252 (before 264).
constexpr int kMxRun16 = 2, kMxRun32 = 1;
template <int RUN>
__device__ __forceinline__ int mx_bucket(int n, int ii) {
  return 16 * RUN * (ii / RUN) + RUN * n + ii % RUN;
}

// N neighbouring elements, aligned to all of them (to 16 bytes where they are more).
template <int N, class OT>
__device__ __forceinline__ void mx_store(OT* to, const float* v) {
  if constexpr (sizeof(OT) == 4) {
    if constexpr (N == 1) *to = v[0];
    else if constexpr (N == 2) *reinterpret_cast<float2*>(to) = make_float2(v[0], v[1]);
    else
#pragma unroll
      for (int i = 0; i < N; i += 4) *reinterpret_cast<float4*>(to + i) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
  } else {
    if constexpr (N == 1) *to = f32_to_bf16_bits(v[0]);
    else if constexpr (N == 2) *reinterpret_cast<uint32_t*>(to) = f32x2_to_bf16_bits(v[0], v[1]);
    else if constexpr (N == 4) *reinterpret_cast<uint2*>(to) = make_uint2(f32x2_to_bf16_bits(v[0], v[1]), f32x2_to_bf16_bits(v[2], v[3]));
    else
#pragma unroll
      for (int i = 0; i < N; i += 8)
        *reinterpret_cast<uint4*>(to + i) = make_uint4(f32x2_to_bf16_bits(v[i], v[i + 1]), f32x2_to_bf16_bits(v[i + 2], v[i + 3]),
                                                       f32x2_to_bf16_bits(v[i + 4], v[i + 5]), f32x2_to_bf16_bits(v[i + 6], v[i + 7]));
  }
}

// logits(c, lg): lg[ii][r] is bucket 256 wave + 64 c + mx_bucket<RUN>(n, ii) of head 4 quarter + r, in base-2 units.
// A wave in which some logit is past kMxPlain takes the largest of its own off, in the heads that have one, and rounded to a
// whole number, so that putting the waves' sums together multiplies by powers of two.  Logits of +-1 prototypes at a
// temperature of 0.02, bf16, us with the maximum over all waves taken off everywhere / worked out again where a logit is large /
// now: one sequence of 32 heads x 60 tables 6.3 / 16.0 / 6.0, four 9.7 / 27.9 / 9.2, sixteen of 28 x 48 19.3 / 66.7 / 17.0 (small logits:
// 4.8, 7.7, 14.2).
template <int W, class OutDT, int RUN, class LOGITS>
__device__ __forceinline__ void mx_table(const LOGITS& logits, bool live, void* __restrict__ out, int l, int group, int n_units, int L,
                                         int wave, int lane) {
  __shared__ __attribute__((aligned(16))) float sums[kSHWaves][kMxHeads], offs[kSHWaves][kMxHeads];
  __shared__ __attribute__((aligned(16))) float alive[kMxHeads];
  __shared__ int wide[kSHWaves];
  const int n = lane & 15, quarter = lane >> 4;
  sh_f32x4 lg[4][4];
  float top = 0.f;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    logits(c, lg[c]);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) top = fmaxf(top, fabsf(lg[c][i][r]));
  }
  const bool far = __builtin_amdgcn_ballot_w64(top > kMxPlain) != 0;
  if (__builtin_expect(far, 0)) {
    sh_f32x4 off;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float mx = -INFINITY, size = 0.f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        mx = fmaxf(mx, lg[i >> 2][i & 3][r]);
        size = fmaxf(size, fabsf(lg[i >> 2][i & 3][r]));
      }
      off[r] = mx_row<true>(size) > kMxPlain ? rintf(mx_row<true>(mx)) : 0.f;      // (0: what the head has when it is with others)
      const float taken = off[r] == -INFINITY ? 0.f : off[r];
#pragma unroll
      for (int i = 0; i < 16; ++i) lg[i >> 2][i & 3][r] -= taken;
    }
    if (n == 0) *reinterpret_cast<sh_f32x4*>(&offs[wave][4 * quarter]) = off;
  }
  sh_f32x4 sum = sh_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 16; ++i) {
#pragma unroll
    for (int r = 0; r < 4; ++r) lg[i >> 2][i & 3][r] = __builtin_amdgcn_exp2f(lg[i >> 2][i & 3][r]);
    sum += lg[i >> 2][i & 3];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) sum[r] = mx_row<false>(sum[r]);
  if (n == 0) *reinterpret_cast<sh_f32x4*>(&sums[wave][4 * quarter]) = sum;
  if (quarter == 0) alive[n] = live ? 1.f : 0.f;
  if (lane == 0) wide[wave] = far ? 1 : 0;
  __syncthreads();
  sh_f32x4 part[kSHWaves], scale = sh_f32x4{1.f, 1.f, 1.f, 1.f};      // the waves' sums; this wave's entries times that
#pragma unroll
  for (int i = 0; i < kSHWaves; ++i) part[i] = *reinterpret_cast<const sh_f32x4*>(&sums[i][4 * quarter]);
  if (__builtin_expect(__builtin_amdgcn_readfirstlane(wide[0] | wide[1] | wide[2] | wide[3]) != 0, 0)) {
    sh_f32x4 off[kSHWaves];
#pragma unroll
    for (int i = 0; i < kSHWaves; ++i)
      off[i] = wide[i] ? *reinterpret_cast<const sh_f32x4*>(&offs[i][4 * quarter]) : sh_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float most = fmaxf(fmaxf(off[0][r], off[1][r]), fmaxf(off[2][r], off[3][r]));
#pragma unroll
      for (int i = 0; i < kSHWaves; ++i) {
        const float f = ldexpf(1.f, (int)fmaxf(off[i][r] - most, -200.f));      // (0 from -150 down, and where all are infinite)
        part[i][r] *= f;
        scale[r] = wave == i ? f : scale[r];
      }
    }
  }
  sum = (part[0] + part[1]) + (part[2] + part[3]);
  const sh_f32x4 real = *reinterpret_cast<const sh_f32x4*>(&alive[4 * quarter]);
  sh_f32x4 inv;
#pragma unroll
  for (int r = 0; r < 4; ++r) inv[r] = real[r] != 0.f ? scale[r] / sum[r] : 0.f;      // (heads that only fill a unit up are zero)
  typedef typename OutDT::storage OT;
#pragma unroll
  for (int g = 0; g < 4; g += W) {      // the lane's units: heads 4 quarter + g .. + W - 1
    const int unit = group * (kMxHeads / W) + (4 * quarter + g) / W;
    if (unit >= n_units) break;
    OT* base = (OT*)out + (((int64_t)unit * L + l) * kMxR + wave * 256) * W;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      float v[4 * W];                   // four buckets of W heads, in runs
#pragma unroll
      for (int i = 0; i < 4 * W; ++i) v[i] = lg[c][i / W][g + i % W] * inv[g + i % W];
#pragma unroll
      for (int ii = 0; ii < 4; ii += RUN) mx_store<RUN * W>(base + (64 * c + mx_bucket<RUN>(n, ii)) * W, v + ii * W);
    }
  }
}

template <class FT, int W, class OutDT>
__device__ __forceinline__ void soft_hash_mx_block(const int l, const int group, const MxUnits& units, const uint16_t* __restrict__ q,
                                                   int64_t q_sb, int64_t q_sh, const uint16_t* __restrict__ planes,
                                                   const uint16_t* __restrict__ protos_T, void* __restrict__ out, int L, float scale,
                                                   const void* __restrict__ freqs, const int64_t* __restrict__ pos, int pos_stride,
                                                   int64_t n_pos, uint16_t* __restrict__ q_out) {
  constexpr bool kRope = !std::is_void<FT>::value;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, quarter = lane >> 4;
  const MxHead at = mx_head<W>(group, units, n);

  // everything is asked for first: the wave's quarter of the queries, angles and planes, prototypes
  const int d0 = 32 * wave + 8 * quarter;
  int64_t p = 0;
  if constexpr (kRope) p = pos[(int64_t)at.b * pos_stride];
  uint4 qf = *reinterpret_cast<const uint4*>(q + at.b * q_sb + at.head * q_sh + d0);
  const uint4 pl = *reinterpret_cast<const uint4*>(planes + ((int64_t)l * kMxK + min(n, kMxK - 1)) * kMxD + d0);
  uint2 pr[4][4];
  // (byte offsets of 32 bits beside a common address)
  const char* at0 = (const char*)protos_T + wave * 512;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const uint32_t off = (uint32_t)min(4 * quarter + r, kMxK - 1) * (kMxR * 2) + 2 * kMxRun16 * n;
#pragma unroll
    for (int c = 0; c < 4; ++c)
      pr[c][r] = make_uint2(*reinterpret_cast<const uint32_t*>(at0 + off + 128 * c), *reinterpret_cast<const uint32_t*>(at0 + off + 128 * c + 64));
  }
  if (quarter >= 2) {         // (no prototype past the tenth: zeros, whatever the tenth is)
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * quarter + r >= kMxK) pr[c][r] = make_uint2(0, 0);
  }
  if constexpr (kRope) {
    const bool turn = p >= 0 && p < n_pos;
    // (angles of row 0 for a position outside the table: a load under a condition is waited for at once)
    float f[8];
    sh_load8<FT>(freqs, (turn ? p : 0) * kMxD + d0, f);
    if (turn) {
      float x[8];
      unpack16<DType_bf16>(qf, x);
      uint32_t w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float re, im;
        rotate_pair(x[2 * j], x[2 * j + 1], f[2 * j], f[2 * j + 1], re, im);
        w[j] = f32x2_to_bf16_bits(re, im);
      }
      qf = make_uint4(w[0], w[1], w[2], w[3]);
    }
    if (l == 0 && at.live) *reinterpret_cast<uint4*>(q_out + ((int64_t)at.b * units.Hq + at.head) * kMxD + d0) = qf;
  }

  const sh_f32x4 t = mx_angles(sh_mfma(pl, qf, sh_f32x4{0.f, 0.f, 0.f, 0.f}), scale, wave, lane);
  float hi[4], mid[4], lo[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    hi[r] = sh_round<DType_bf16>(t[r]);
    mid[r] = sh_round<DType_bf16>(t[r] - hi[r]);
    lo[r] = t[r] - hi[r] - mid[r];
  }
  const uint4 t_high = make_uint4(f32x2_to_bf16_bits(hi[0], hi[1]), f32x2_to_bf16_bits(hi[2], hi[3]),
                                  f32x2_to_bf16_bits(mid[0], mid[1]), f32x2_to_bf16_bits(mid[2], mid[3]));
  const uint4 t_low = make_uint4(f32x2_to_bf16_bits(lo[0], lo[1]), f32x2_to_bf16_bits(lo[2], lo[3]), 0, 0);
  auto logits = [&](int c, sh_f32x4 (&lg)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) {
      const uint32_t sel = (ii & 1) ? 0x07060302u : 0x05040100u;
      auto word = [&](int r) { return ii < 2 ? pr[c][r].x : pr[c][r].y; };
      const uint32_t a0 = __builtin_amdgcn_perm(word(1), word(0), sel), a1 = __builtin_amdgcn_perm(word(3), word(2), sel);
      lg[ii] = sh_mfma(t_low, make_uint4(a0, a1, 0, 0), sh_f32x4{0.f, 0.f, 0.f, 0.f});
      lg[ii] = sh_mfma(t_high, make_uint4(a0, a1, a0, a1), lg[ii]);
    }
  };
  mx_table<W, OutDT, kMxRun16>(logits, at.live, out, l, group, units.count, L, wave, lane);
}

__host__ __device__ __forceinline__ float mx_scale(float tanh_scale, float inv_temperature) {
  return tanh_scale * inv_temperature * 1.4426950408889634f;
}

// The same for fp32 queries, planes and prototypes: v_mfma_f32_16x16x4_f32, which multiplies and adds in fp32 throughout, so
// nothing is split.  Lane x holds column (or row) x % 16 and one k of four; which k that is is free as long as both operands
// agree: for the projections quarter q of wave w takes dims 32 q + 8 w .. + 7, a run, and for the logits step r takes plane 4 q + r,
// which is what the lane's own projections are.
// One sequence of 16 heads, 60 tables, by itself: 6.0 us, 8.9 of the scalar form below; a chain of trips to memory and of matrix
// products, on 60 workgroups.  Against float64 (2-norm, queries and planes N(0, 1)): 1.9e-7, the scalar form 2.5e-7.
// OutDT: the table's type (bf16: the fp32 value rounded once).
template <class FT, int W, class OutDT>
__device__ __forceinline__ void soft_hash_mx32_block(const int l, const int group, const MxUnits& units, const float* __restrict__ q,
                                                     int64_t q_sb, int64_t q_sh, const float* __restrict__ planes,
                                                     const float* __restrict__ protos_T, void* __restrict__ out, int L, float scale,
                                                     const void* __restrict__ freqs, const int64_t* __restrict__ pos, int pos_stride,
                                                     int64_t n_pos, float* __restrict__ q_out) {
  constexpr bool kRope = !std::is_void<FT>::value;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n = lane & 15, quarter = lane >> 4;
  const MxHead at = mx_head<W>(group, units, n);

  const int d0 = 32 * quarter + 8 * wave;
  const float* qrow = q + at.b * q_sb + at.head * q_sh + d0;
  const float* prow = planes + ((int64_t)l * kMxK + min(n, kMxK - 1)) * kMxD + d0;
  int64_t p = 0;
  if constexpr (kRope) p = pos[(int64_t)at.b * pos_stride];
  float x[8], pl[8], pr[4][4][4];
#pragma unroll
  for (int i = 0; i < 8; i += 4) {
    float t[4];
    sh_load4<DType_f32>(qrow, i, t);
#pragma unroll
    for (int e = 0; e < 4; ++e) x[i + e] = t[e];
    sh_load4<DType_f32>(prow, i, t);
#pragma unroll
    for (int e = 0; e < 4; ++e) pl[i + e] = t[e];
  }
#pragma unroll
  for (int c = 0; c < 4; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float* from = protos_T + min(4 * quarter + r, kMxK - 1) * kMxR + wave * 256 + 64 * c;
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) pr[c][r][ii] = from[mx_bucket<kMxRun32>(n, ii)];
    }
  if constexpr (kRope) {
    const bool turn = p >= 0 && p < n_pos;
    // (angles of row 0 for a position outside the table: a load under a condition is waited for at once)
    float f[8];
    sh_load8<FT>(freqs, (turn ? p : 0) * kMxD + d0, f);
    if (turn) {
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        float re, im;
        rotate_pair(x[i], x[i + 1], f[i], f[i + 1], re, im);
        x[i] = re, x[i + 1] = im;
      }
    }
    if (l == 0 && at.live) {
#pragma unroll
      for (int i = 0; i < 8; i += 4) {
        const float t[4] = {x[i], x[i + 1], x[i + 2], x[i + 3]};
        sh_store4<DType_f32>(q_out, ((int64_t)at.b * units.Hq + at.head) * kMxD + d0 + i, t);
      }
    }
  }

  // register r: plane 4 quarter + r of head n (planes past the tenth repeat it and are dropped).  Eight sums of sixteen
  // products over the four waves, added in pairs: one of 128 loses more than the scalar form's.
  sh_f32x4 proj[2] = {sh_f32x4{0.f, 0.f, 0.f, 0.f}, sh_f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
  for (int i = 0; i < 8; ++i) proj[i % 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(pl[i], x[i], proj[i % 2], 0, 0, 0);
  const sh_f32x4 t = mx_angles(proj[0] + proj[1], scale, wave, lane);
  auto logits = [&](int c, sh_f32x4 (&lg)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int ii = 0; ii < 4; ++ii) lg[ii] = sh_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int ii = 0; ii < 4; ++ii)
        // (no prototype past the tenth: zeros, whatever the tenth is)
        lg[ii] = __builtin_amdgcn_mfma_f32_16x16x4f32(t[r], 4 * quarter + r < kMxK ? pr[c][r][ii] : 0.f, lg[ii], 0, 0, 0);
  };
  mx_table<W, OutDT, kMxRun32>(logits, at.live, out, l, group, units.count, L, wave, lane);
}

template <int W, class OutDT>
__global__ __launch_bounds__(kSHThreads) void soft_hash_mx32_kernel(const float* __restrict__ q, int64_t q_sb, int64_t q_sh,
                                                                    const float* __restrict__ planes, const float* __restrict__ protos_T,
                                                                    void* __restrict__ out, MxUnits units, int L, float scale) {
  soft_hash_mx32_block<void, W, OutDT>(blockIdx.x, blockIdx.y, units, q, q_sb, q_sh, planes, protos_T, out, L, scale, nullptr, nullptr, 0, 0,
                                nullptr);
}

template <int W, class OutDT>
__global__ __launch_bounds__(kSHThreads, 4) void soft_hash_mx_kernel(const uint16_t* __restrict__ q, int64_t q_sb, int64_t q_sh,
                                                                  const uint16_t* __restrict__ planes,
                                                                  const uint16_t* __restrict__ protos_T, void* __restrict__ out,
                                                                  MxUnits units, int L, float scale) {
  soft_hash_mx_block<void, W, OutDT>(blockIdx.x, blockIdx.y, units, q, q_sb, q_sh, planes, protos_T, out, L, scale, nullptr, nullptr, 0, 0,
                                  nullptr);
}

// GC: heads per group the registers are sized for (4 or 8).  KC: K when known at
// compile time (then, with a single sweep, a lane's 4 x K prototype entries are
// fetched straight into registers at kernel entry: no LDS copy of the prototypes,
// a small LDS footprint and several workgroups per CU), 0 = runtime K.
// LDS (dynamic): qs [G][D] | ps [K][D+1] | ts [G][K] | red [waves][GC] | protos [K][R] (optional)
//
// FT: void, or the element type of a rotary table: then the queries arrive
// unrotated (the q part of a fused qkv projection), are rotated by the angles of
// position `rope_pos` (when `rope_on`) and rounded to DT as they are staged, and
// the workgroups of table 0 also write them to `q_out` [B,Hq,D] (vector path only).
template <class DT, int GC, int KC, class FT>
__device__ __forceinline__ void soft_hash_block(
    const int l, const int pair, const void* __restrict__ q, int64_t q_sb, int64_t q_sh,
    const void* __restrict__ planes, const void* __restrict__ protos_T, void* __restrict__ out, int out_dtype,
    int Hq, int Hkv, int G, int D, int L, int K, int R, float tanh_scale, float inv_temperature, int parts,
    int width, int protos_in_lds, int vec_ok, const void* __restrict__ freqs, int64_t rope_pos, bool rope_on,
    void* __restrict__ q_out) {
  constexpr bool kRope = !std::is_void<FT>::value;
  extern __shared__ __attribute__((aligned(16))) float lds[];
  float* qs = lds;
  float* ps = qs + G * D;
  float* ts = ps + ((K * (D + 1) + 3) / 4) * 4;   // (16-byte aligned when G * D is a multiple of 4: read as float4)
  float* red = ts + ((G * K + 3) / 4) * 4;
  float* protos_lds = lds + ((G * D + ((K * (D + 1) + 3) / 4) * 4 + ((G * K + 3) / 4) * 4 + kSHWaves * GC + 3) / 4) * 4;
  const int DP = D + 1;
  const int b = pair / Hkv, kvh = pair % Hkv;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  constexpr bool direct = KC > 0;   // prototypes from global memory into registers, once

  float pk[direct ? KC : 1][4];
  if (direct && tid * 4 < R) {
#pragma unroll
    for (int k = 0; k < KC; ++k) sh_load4<DT>(protos_T, (int64_t)k * R + tid * 4, pk[k]);
  }

  if (vec_ok) {
    // Staging with every global load issued before the first LDS store: the whole
    // set-up costs one memory latency.  (A load-convert-store loop exposes one per
    // iteration.)
    constexpr int QV = kSHMaxG * kSHMaxD / 4 / kSHThreads;   // vectors of four per lane
    constexpr int PV = kSHMaxK * kSHMaxD / 4 / kSHThreads;
    constexpr int RV = direct ? 1 : 10;                       // prototype vectors per batch
    float qv[QV][4], pv[PV][4], rv[RV][4];
    const int nr4 = (!direct && protos_in_lds) ? K * R / 4 : 0;
    float fv[kRope ? QV : 1][4];   // (cos, sin) of the two pairs a vector holds
#pragma unroll
    for (int u = 0; u < QV; ++u) {
      const int i = (tid + u * kSHThreads) * 4;
      if (i < G * D) {
        sh_load4<DT>(q, b * q_sb + (int64_t)(kvh * G + i / D) * q_sh + i % D, qv[u]);
        if constexpr (kRope) {
          // (always fetched, from row 0 when the position is outside the table: a load under a
          // condition would make the compiler wait for every load issued so far, one by one)
          sh_load4<FT>(freqs, ((rope_on ? rope_pos : 0) * (D / 2) + (i % D) / 2) * 2, fv[u]);
        }
      }
    }
#pragma unroll
    for (int u = 0; u < PV; ++u) {
      const int i = (tid + u * kSHThreads) * 4;
      if (i < K * D) sh_load4<DT>(planes, (int64_t)l * K * D + i, pv[u]);
    }
    if (!direct) {
#pragma unroll
      for (int u = 0; u < RV; ++u) {
        const int i = tid + u * kSHThreads;
        if (i < nr4) sh_load4<DT>(protos_T, (int64_t)i * 4, rv[u]);
      }
    }
#pragma unroll
    for (int u = 0; u < QV; ++u) {
      const int i = (tid + u * kSHThreads) * 4;
      if (i < G * D) {
        if constexpr (kRope) {
          if (rope_on) {
            float re, im;
            rotate_pair(qv[u][0], qv[u][1], fv[u][0], fv[u][1], re, im);
            qv[u][0] = sh_round<DT>(re), qv[u][1] = sh_round<DT>(im);
            rotate_pair(qv[u][2], qv[u][3], fv[u][2], fv[u][3], re, im);
            qv[u][2] = sh_round<DT>(re), qv[u][3] = sh_round<DT>(im);
          }
          if (l == 0) sh_store4<DT>(q_out, ((int64_t)b * Hq + kvh * G + i / D) * D + i % D, qv[u]);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) qs[i + e] = qv[u][e];
      }
    }
#pragma unroll
    for (int u = 0; u < PV; ++u) {
      const int i = (tid + u * kSHThreads) * 4;
      if (i < K * D) {
#pragma unroll
        for (int e = 0; e < 4; ++e) ps[(i / D) * DP + i % D + e] = pv[u][e];
      }
    }
    if (!direct) {
#pragma unroll
      for (int u = 0; u < RV; ++u) {
        const int i = tid + u * kSHThreads;
        if (i < nr4) *reinterpret_cast<float4*>(protos_lds + (size_t)i * 4) = make_float4(rv[u][0], rv[u][1], rv[u][2], rv[u][3]);
      }
      // (prototype tables beyond one batch: the rest in further batches)
      for (int i0 = RV * kSHThreads; i0 < nr4; i0 += RV * kSHThreads) {
#pragma unroll
        for (int u = 0; u < RV; ++u) {
          const int i = i0 + tid + u * kSHThreads;
          if (i < nr4) sh_load4<DT>(protos_T, (int64_t)i * 4, rv[u]);
        }
#pragma unroll
        for (int u = 0; u < RV; ++u) {
          const int i = i0 + tid + u * kSHThreads;
          if (i < nr4) *reinterpret_cast<float4*>(protos_lds + (size_t)i * 4) = make_float4(rv[u][0], rv[u][1], rv[u][2], rv[u][3]);
        }
      }
    }
  } else {
    for (int i = tid; i < G * D; i += kSHThreads) {
      const int g = i / D, d = i % D;
      qs[i] = sh_load<DT>(q, b * q_sb + (int64_t)(kvh * G + g) * q_sh + d);
    }
    for (int i = tid; i < K * D; i += kSHThreads) ps[(i / D) * DP + i % D] = sh_load<DT>(planes, (int64_t)l * K * D + i);
    if (protos_in_lds)
      for (int i = tid; i < K * R; i += kSHThreads) protos_lds[i] = sh_load<DT>(protos_T, i);
  }
  __syncthreads();
  // projections: four lanes per (head, plane) pair, a quarter of the dimension each
  for (int p0 = 0; p0 < G * K; p0 += kSHThreads / 4) {
    const int p = p0 + tid / 4, part = tid % 4;
    float s = 0.f;
    if (p < G * K) {
      const float* qrow = qs + (p / K) * D;
      const float* prow = ps + (p % K) * DP;
#pragma unroll 8
      for (int d = part; d < D; d += 4) s += qrow[d] * prow[d];
    }
    s = group_sum<4>(s);
    if (p < G * K && part == 0) ts[p] = tanhf(s) * tanh_scale * inv_temperature;   // ts[g][k], p = g*K + k
  }
  __syncthreads();

  // logits of buckets r0..r0+3 for every head of the group
  auto logits4 = [&](int r0, float (&lg)[GC][4]) {
#pragma unroll
    for (int g = 0; g < GC; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) lg[g][i] = 0.f;
    auto add_plane = [&](int k, const float (&pr)[4]) {
#pragma unroll
      for (int g = 0; g < GC; ++g) {
        if (g < G) {
          const float t = ts[g * K + k];
#pragma unroll
          for (int i = 0; i < 4; ++i) lg[g][i] += t * pr[i];
        }
      }
    };
    if constexpr (direct) {
      // the G x K scaled projections as a handful of 16-byte broadcast reads instead
      // of one LDS read per (head, plane) term
      if ((G * D) % 4 == 0) {
        constexpr int NV = (GC * (KC > 0 ? KC : 1) + 3) / 4;
        float tv[NV * 4];
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const float4 t4 = (i * 4 < G * K) ? *reinterpret_cast<const float4*>(ts + i * 4) : make_float4(0.f, 0.f, 0.f, 0.f);
          tv[4 * i] = t4.x, tv[4 * i + 1] = t4.y, tv[4 * i + 2] = t4.z, tv[4 * i + 3] = t4.w;
        }
#pragma unroll
        for (int g = 0; g < GC; ++g) {
          if (g < G) {
#pragma unroll
            for (int k = 0; k < KC; ++k) {
              const float t = tv[g * KC + k];
#pragma unroll
              for (int i = 0; i < 4; ++i) lg[g][i] += t * pk[k][i];
            }
          }
        }
      } else {
#pragma unroll
        for (int k = 0; k < KC; ++k) add_plane(k, pk[k]);
      }
    } else {
      for (int k = 0; k < K; ++k) {
        float pr[4];
        if (protos_in_lds) {
          const float4 v = *reinterpret_cast<const float4*>(protos_lds + (size_t)k * R + r0);
          pr[0] = v.x;
          pr[1] = v.y;
          pr[2] = v.z;
          pr[3] = v.w;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) pr[i] = sh_load<DT>(protos_T, (int64_t)k * R + r0 + i);
        }
        add_plane(k, pr);
      }
    }
  };
  // workgroup-wide reduction of one value per head; every lane gets the result
  auto reduce = [&](float (&v)[GC], bool is_max) {
#pragma unroll
    for (int g = 0; g < GC; ++g) v[g] = is_max ? wave_reduce_to_last<true>(v[g]) : wave_reduce_to_last<false>(v[g]);
    __syncthreads();  // earlier readers of `red` are done
    if (lane == 63) {   // (the reduction leaves a wave's result in its last lane)
#pragma unroll
      for (int g = 0; g < GC; ++g) red[wave * GC + g] = v[g];
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < GC; ++g) {
      float a = red[g];
#pragma unroll
      for (int w = 1; w < kSHWaves; ++w) a = is_max ? fmaxf(a, red[w * GC + g]) : a + red[w * GC + g];
      v[g] = a;
    }
  };

  // With R <= 1024 a lane owns a single run of four buckets: its logits are
  // computed once and kept; otherwise each sweep recomputes them.
  const bool keep = direct || R <= kSHThreads * 4;
  float lg[GC][4];
  float mx[GC], sm[GC];
#pragma unroll
  for (int g = 0; g < GC; ++g) {
    mx[g] = -INFINITY;
    sm[g] = 0.f;
  }
  for (int r0 = tid * 4; r0 < R; r0 += kSHThreads * 4) {
    logits4(r0, lg);
#pragma unroll
    for (int g = 0; g < GC; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) mx[g] = fmaxf(mx[g], lg[g][i]);
  }
  reduce(mx, true);
  for (int r0 = tid * 4; r0 < R; r0 += kSHThreads * 4) {
    if (!keep) logits4(r0, lg);
#pragma unroll
    for (int g = 0; g < GC; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float e = expf(lg[g][i] - mx[g]);
        sm[g] += e;
        if (keep) lg[g][i] = e;   // kept for the write sweep
      }
  }
  reduce(sm, false);
  // (one reciprocal per head and a product per bucket where there were sixteen divisions a lane:
  // the last write sweep was the longest phase of the workgroup)
  float inv[GC];
#pragma unroll
  for (int g = 0; g < GC; ++g) inv[g] = 1.f / sm[g];
  for (int r0 = tid * 4; r0 < R; r0 += kSHThreads * 4) {
    if (!keep) logits4(r0, lg);
#pragma unroll
    for (int g = 0; g < GC; ++g)
#pragma unroll
      for (int i = 0; i < 4; ++i)   // now probabilities
        lg[g][i] = (g < G) ? (keep ? lg[g][i] : expf(lg[g][i] - mx[g])) * inv[g] : 0.f;
    if (parts == 0) {
      // reference layout [B,Hq,L,R]
#pragma unroll
      for (int g = 0; g < GC; ++g) {
        if (g < G) {
          const int64_t o = (((int64_t)b * Hq + kvh * G + g) * L + l) * R + r0;
          if (out_dtype == SOCKET_F32) {
            *reinterpret_cast<float4*>((float*)out + o) = make_float4(lg[g][0], lg[g][1], lg[g][2], lg[g][3]);
          } else {
            uint2 w;
            w.x = f32x2_to_bf16_bits(lg[g][0], lg[g][1]);
            w.y = f32x2_to_bf16_bits(lg[g][2], lg[g][3]);
            *reinterpret_cast<uint2*>((uint16_t*)out + o) = w;
          }
        }
      }
    } else {
      // grouped layout [B*Hkv*parts, L, R, width]: the scorer's LDS image.  Width and
      // part are compile-time in each instance below, so v[] is indexed statically
      // (with a runtime width the compiler kept it in scratch memory).
      auto write_part = [&](auto width_c, auto part_c) {
        constexpr int W = decltype(width_c)::value, PART = decltype(part_c)::value;
        if constexpr (PART * W < GC) {
          const int64_t o = ((((int64_t)pair * parts + PART) * L + l) * R + r0) * W;
          float v[4 * W];  // [bucket][head of this part]: 4 * W consecutive elements of the table
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int gg = 0; gg < W; ++gg) v[i * W + gg] = lg[PART * W + gg][i];
          if (out_dtype == SOCKET_F32) {
#pragma unroll
            for (int c = 0; c < W; ++c)
              *reinterpret_cast<float4*>((float*)out + o + 4 * c) =
                  make_float4(v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]);
          } else {
            uint32_t w[2 * W];
#pragma unroll
            for (int c = 0; c < 2 * W; ++c)
              w[c] = f32x2_to_bf16_bits(v[2 * c], v[2 * c + 1]);
            uint16_t* dst = (uint16_t*)out + o;
            if constexpr (W == 4) {
              *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
              *reinterpret_cast<uint4*>(dst + 8) = make_uint4(w[4], w[5], w[6], w[7]);
            } else if constexpr (W == 2) {
              *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
            } else {
              *reinterpret_cast<uint2*>(dst) = make_uint2(w[0], w[1]);
            }
          }
        }
      };
      using std::integral_constant;
      if (width == 4) {
        write_part(integral_constant<int, 4>{}, integral_constant<int, 0>{});
        if (parts > 1) write_part(integral_constant<int, 4>{}, integral_constant<int, 1>{});
      } else if (width == 2) {
        write_part(integral_constant<int, 2>{}, integral_constant<int, 0>{});
      } else {
        write_part(integral_constant<int, 1>{}, integral_constant<int, 0>{});
      }
    }
  }
}

// Few buckets (R <= 256) and K other than 10: a wave to a head, everything in registers.  A lane has four elements of
// the query and of every plane, and four buckets; the K sums, the maximum and the sum of exponentials are lane
// reductions, lane k makes plane k's tanh.  The kernel above leaves three of its four waves without a bucket here and
// goes through LDS and six barriers, and is bound by that chain: 7.9 us for 32 heads, 32 tables of 8 float32 planes of
// 128 dims, where this one takes 4.2 (and 6.5 with the rotation, the append and the key's hash of a decode step, which
// are 7.3 us in two launches of their own).
constexpr int kSmallR = 4 * SOCKET_WAVE;

// FT, freqs, rope_pos, rope_on, q_out: as in soft_hash_block.
template <class DT, int KM, class FT>
__device__ __forceinline__ void soft_hash_small_block(
    const int l, const int pair, const void* __restrict__ q, int64_t q_sb, int64_t q_sh, const void* __restrict__ planes,
    const void* __restrict__ protos_T, void* __restrict__ out, int out_dtype, int Hq, int Hkv, int G, int D, int L, int K, int R,
    float scale, int parts, int width, const void* __restrict__ freqs, int64_t rope_pos, bool rope_on, void* __restrict__ q_out) {
  constexpr bool kRope = !std::is_void<FT>::value;
  const int b = pair / Hkv, kvh = pair % Hkv;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool in_d = 4 * lane < D, in_r = 4 * lane < R;
  const int d0 = min(4 * lane, D - 4), r0 = min(4 * lane, R - 4);
  const int W = parts > 0 ? width : 1, members = parts > 0 ? parts * width : G;
  float pl[KM][4], pr[KM][4];
#pragma unroll
  for (int k = 0; k < KM; ++k) sh_load4<DT>(planes, ((int64_t)l * K + min(k, K - 1)) * D + d0, pl[k]);
#pragma unroll
  for (int k = 0; k < KM; ++k) sh_load4<DT>(protos_T, (int64_t)min(k, K - 1) * R + r0, pr[k]);
  float f[4];
  // (angles of row 0 for a position outside the table: a load under a condition is waited for at once)
  if constexpr (kRope) sh_load4<FT>(freqs, (rope_on ? rope_pos : 0) * D + d0, f);
  for (int m = wave; m < members; m += kSHWaves) {
    float lg[4] = {0.f, 0.f, 0.f, 0.f};
    if (m < G) {                                    // (heads that only fill a unit up are zero)
      float x[4], z = 0.f;
      sh_load4<DT>(q, b * q_sb + (int64_t)(kvh * G + m) * q_sh + d0, x);
      if constexpr (kRope) {
        if (rope_on) {
          float re, im;
          rotate_pair(x[0], x[1], f[0], f[1], re, im);
          x[0] = sh_round<DT>(re), x[1] = sh_round<DT>(im);
          rotate_pair(x[2], x[3], f[2], f[3], re, im);
          x[2] = sh_round<DT>(re), x[3] = sh_round<DT>(im);
        }
        if (l == 0 && in_d) sh_store4<DT>(q_out, ((int64_t)b * Hq + kvh * G + m) * D + d0, x);
      }
#pragma unroll
      for (int k = 0; k < KM; ++k) {
        float s = x[0] * pl[k][0];
#pragma unroll
        for (int e = 1; e < 4; ++e) s = fmaf(x[e], pl[k][e], s);
        s = group_sum<64>(in_d ? s : 0.f);
        z = lane == k ? s : z;
      }
      const float t = tanhf(z) * scale;
#pragma unroll
      for (int k = 0; k < KM; ++k)
        if (k < K) {
          const float tk = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(t), k));
#pragma unroll
          for (int i = 0; i < 4; ++i) lg[i] = fmaf(tk, pr[k][i], lg[i]);
        }
      float mx = in_r ? fmaxf(fmaxf(lg[0], lg[1]), fmaxf(lg[2], lg[3])) : -INFINITY;
      mx = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wave_reduce_to_last<true>(mx)), 63));
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        lg[i] = expf(lg[i] - mx);
        sum += lg[i];
      }
      const float inv = 1.f / group_sum<64>(in_r ? sum : 0.f);
#pragma unroll
      for (int i = 0; i < 4; ++i) lg[i] *= inv;
    }
    if (!in_r) continue;
    const int64_t unit = parts > 0 ? (int64_t)pair * parts + m / W : (int64_t)b * Hq + kvh * G + m;
    const int64_t o = ((unit * L + l) * R + r0) * W + (parts > 0 ? m % W : 0);
    if (W == 1) {
      if (out_dtype == SOCKET_F32) sh_store4<DType_f32>(out, o, lg);
      else sh_store4<DType_bf16>(out, o, lg);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (out_dtype == SOCKET_F32) ((float*)out)[o + i * W] = lg[i];
        else ((uint16_t*)out)[o + i * W] = f32_to_bf16_bits(lg[i]);
      }
    }
  }
}

template <class DT, int KM>
__global__ __launch_bounds__(kSHThreads) void soft_hash_small_kernel(
    const void* __restrict__ q, int64_t q_sb, int64_t q_sh, const void* __restrict__ planes, const void* __restrict__ protos_T,
    void* __restrict__ out, int out_dtype, int Hq, int Hkv, int G, int D, int L, int K, int R, float scale, int parts, int width) {
  soft_hash_small_block<DT, KM, void>(blockIdx.x, blockIdx.y, q, q_sb, q_sh, planes, protos_T, out, out_dtype, Hq, Hkv, G, D, L, K, R,
                                      scale, parts, width, nullptr, 0, false, nullptr);
}

template <class DT, int GC, int KC>
__global__ __launch_bounds__(kSHThreads) void soft_hash_kernel(
    const void* __restrict__ q, int64_t q_sb, int64_t q_sh, const void* __restrict__ planes,
    const void* __restrict__ protos_T, void* __restrict__ out, int out_dtype, int Hq, int Hkv, int G,
    int D, int L, int K, int R, float tanh_scale, float inv_temperature, int parts, int width,
    int protos_in_lds, int vec_ok) {
  soft_hash_block<DT, GC, KC, void>(blockIdx.x, blockIdx.y, q, q_sb, q_sh, planes, protos_T, out, out_dtype, Hq,
                                    Hkv, G, D, L, K, R, tanh_scale, inv_temperature, parts, width, protos_in_lds,
                                    vec_ok, nullptr, 0, false, nullptr);
}

// ---------------------------------------------------------------------------
// The head of a single-token decode step in one launch (bf16 or fp32, head
// dimension 128): rotary embedding of the new token's query and key, append of the key and
// value to the cache, hash of the new key with the value norm, and the soft hash
// of the rotated query (GPT-FAST/model.py:433-451 and :392-401).  Each of these
// is a few microseconds of dependent latency on its own, so as three launches
// they cost three launch floors; here they are workgroups of one grid:
//
//   blocks [0, n_key_blocks): block (pair, part) has wave w hash packed word
//     4 * part + w of the new key of (sequence, kv head) `pair`; part 0's first
//     wave also writes the K/V rows, the value norm and the cached length;
//   the rest: the soft hash's workgroups (table l, pair), which rotate the
//     queries as they stage them; those of table 0 write the rotated queries.
//
// The key's sign bits come from the same matrix-core contraction as the cache
// hashing kernel's (planes the M operand, the key column 0 of the N operand, the
// k-steps in the same order), so both give the same bits for the same key.
constexpr int kPrologueD = 128;

// Eight elements of a row, loaded and stored as they are.
template <class DT>
struct alignas(16) sh_row8 {
  uint4 w[DT::kPer16B == 8 ? 1 : 2];
};
template <class DT>
__device__ __forceinline__ void sh_unpack8(const sh_row8<DT>& r, float (&x)[8]) {
  if constexpr (DT::kPer16B == 8) {
    unpack16<DT>(r.w[0], x);
  } else {
    __builtin_memcpy(x, r.w, 32);
  }
}
template <class DT>
__device__ __forceinline__ sh_row8<DT> sh_pack8(const float (&x)[8]) {
  sh_row8<DT> r;
  if constexpr (DT::kPer16B == 8) {
    r.w[0] = make_uint4(f32x2_to_bf16_bits(x[0], x[1]), f32x2_to_bf16_bits(x[2], x[3]), f32x2_to_bf16_bits(x[4], x[5]),
                        f32x2_to_bf16_bits(x[6], x[7]));
  } else {
    __builtin_memcpy(r.w, x, 32);
  }
  return r;
}
// The eight as bf16, which is what keys are hashed in.
template <class DT>
__device__ __forceinline__ uint4 sh_bf16_of8(const sh_row8<DT>& r) {
  if constexpr (DT::kPer16B == 8) {
    return r.w[0];
  } else {
    float x[8];
    sh_unpack8<DT>(r, x);
    return sh_pack8<DType_bf16>(x).w[0];
  }
}

// DT: type of the projection, the caches, planes and prototypes.
// GC: as in soft_hash_block (bf16 only), or 0: soft_hash_mx_block or soft_hash_mx32_block with units of W heads, OT the
// output's elements; below zero: soft_hash_small_block for at most -GC planes.
// (bf16 operands on the matrix cores: four waves a SIMD.  At the three that 164 registers leave (and runs of four buckets to a
// lane), sixteen sequences of 28 heads x 48 tables took 23.4 us instead of 20.4, four of 32 x 60 11.0 instead of 10.5.)
template <class DT, int GC, class FT, int W, class OT>
__global__ __launch_bounds__(kSHThreads, GC == 0 && DT::kEnum == SOCKET_BF16 ? 4 : 1) void decode_prologue_kernel(
    const typename DT::storage* __restrict__ qkv, int64_t qkv_sb, const void* __restrict__ freqs,
    const int64_t* __restrict__ pos, int pos_stride, int64_t n_pos, typename DT::storage* __restrict__ q_out,
    typename DT::storage* __restrict__ k_cache, typename DT::storage* __restrict__ v_cache, int64_t c_sb, int64_t c_sh, int64_t c_ss,
    int32_t* __restrict__ lens, const uint16_t* __restrict__ planes_words, uint32_t* __restrict__ codes,
    uint16_t* __restrict__ v_norm, int NW, int64_t Tcap, const void* __restrict__ planes,
    const void* __restrict__ protos_T, void* __restrict__ q_table, int out_dtype, int Hq, int Hkv, int G, int L,
    int K, int R, float tanh_scale, float inv_temperature, int parts, int width, int word_blocks,
    int n_key_blocks, MxUnits units) {
  typedef typename DT::storage ST;
  constexpr int D = kPrologueD;
  constexpr bool kF32 = DT::kEnum == SOCKET_F32;
  const int bx = blockIdx.x;
  if (bx >= n_key_blocks) {
    const int i = bx - n_key_blocks;
    const int l = i % L, pair = i / L;
    const float mx = mx_scale(tanh_scale, inv_temperature);
    if constexpr (GC == 0 && kF32) {
      soft_hash_mx32_block<FT, W, DType_f32>(l, pair, units, qkv, qkv_sb, D, (const float*)planes, (const float*)protos_T, q_table, L, mx,
                                  freqs, pos, pos_stride, n_pos, q_out);
    } else if constexpr (GC == 0) {
      soft_hash_mx_block<FT, W, std::conditional_t<sizeof(OT) == 4, DType_f32, DType_bf16>>(
          l, pair, units, qkv, qkv_sb, D, (const uint16_t*)planes, (const uint16_t*)protos_T, q_table, L, mx, freqs, pos, pos_stride, n_pos, q_out);
    } else {
      const int64_t p = pos[(int64_t)(pair / Hkv) * pos_stride];
      const bool turn = p >= 0 && p < n_pos;
      if constexpr (GC < 0)
        soft_hash_small_block<DT, -GC, FT>(l, pair, qkv, qkv_sb, D, planes, protos_T, q_table, out_dtype, Hq, Hkv, G, D, L, K, R,
                                           tanh_scale * inv_temperature, parts, width, freqs, p, turn, q_out);
      else
        soft_hash_block<DT, GC, 10, FT>(l, pair, qkv, qkv_sb, D, planes, protos_T, q_table, out_dtype, Hq, Hkv, G, D, L, K, R,
                                        tanh_scale, inv_temperature, parts, width, 0, 1, freqs, p, turn, q_out);
    }
    return;
  }
  const int pair = bx / word_blocks, part = bx % word_blocks;
  const int b = pair / Hkv, kvh = pair % Hkv;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int prow = lane & 15, quarter = lane >> 4;
  const int64_t p = pos[(int64_t)b * pos_stride];
  const bool rope_on = p >= 0 && p < n_pos;               // a position outside the table is not rotated,
  const bool rows_ok = rope_on && p < Tcap;               // one outside the cache or the table writes no K/V row,
  const bool cached = (uint64_t)p < (uint64_t)Tcap;       // one outside the cache no code and no norm
  const int w = part * kSHWaves + wave;
  const bool first = part == 0 && wave == 0;
  if (w >= NW && !first) return;

  // plane fragments of this wave's word (they do not depend on the key: requested first)
  const int pbit0 = 8 * (prow >> 2) + 7 - (prow & 3);
  ShFrag pf[4][2];
  if (w < NW) {
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        const int col = w * 32 + pbit0 - 4 * mb;
        pf[ks][mb].u = reinterpret_cast<const uint4*>(planes_words)[(int64_t)col * 16 + ks * 4 + quarter];
      }
  }
  // the new key as column 0 of the N operand: lane 16 * quarter holds elements
  // 32 * ks + 8 * quarter .. + 7 of k-step ks, every other column is zero
  const ST* krow = qkv + b * qkv_sb + (int64_t)(Hq + kvh) * D;
  const ST* vrow = qkv + b * qkv_sb + (int64_t)(Hq + Hkv + kvh) * D;
  typedef sh_row8<DT> Row8;                               // eight elements as they lie in memory
  ShFrag kf[4];
  Row8 vr[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    kf[ks].u = make_uint4(0, 0, 0, 0);
    vr[ks] = Row8{};
  }
  if (prow == 0) {
    Row8 raw[4];
    float f[4][8];
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int e0 = ks * 32 + quarter * 8;
      // (all three fetched whether needed or not -- the angles from row 0 for a position outside
      // the table, the value row by every wave: loads under a condition are waited for one by one)
      raw[ks] = *reinterpret_cast<const Row8*>(krow + e0);
      sh_load8<FT>(freqs, (rope_on ? p : 0) * D + e0, f[ks]);   // ((p * D/2) + e0/2) * 2
      vr[ks] = *reinterpret_cast<const Row8*>(vrow + e0);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      if (rope_on) {
        float x[8], o[8];
        sh_unpack8<DT>(raw[ks], x);
#pragma unroll
        for (int j = 0; j < 8; j += 2) rotate_pair(x[j], x[j + 1], f[ks][j], f[ks][j + 1], o[j], o[j + 1]);
        raw[ks] = sh_pack8<DT>(o);
      }
      kf[ks].u = sh_bf16_of8<DT>(raw[ks]);
    }
    if (first && rows_ok) {
      ST* kdst = k_cache + b * c_sb + kvh * c_sh + p * c_ss;
      ST* vdst = v_cache + b * c_sb + kvh * c_sh + p * c_ss;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) {
        const int e0 = ks * 32 + quarter * 8;
        *reinterpret_cast<Row8*>(kdst + e0) = raw[ks];
        *reinterpret_cast<Row8*>(vdst + e0) = vr[ks];
      }
    }
  }
  if (first) {
    // the cached length follows the position
    if (kvh == 0 && lane == 0 && rows_ok && lens) lens[b] = (int32_t)p + 1;
    float norm2;
    if constexpr (kF32) {
      // (sixteen lanes of eight elements each, added up as the hash's launch adds them)
      float x[8];
      sh_unpack8<DT>(*reinterpret_cast<const Row8*>(vrow + 8 * prow), x);
      norm2 = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) norm2 += x[i] * x[i];
      norm2 = group_sum<16>(norm2);
    } else {
      // ||v||^2 = element (0, 0) of the value column against itself: register 0 of lane 0
      sh_f32x4 g = sh_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) g = sh_mfma(sh_bf16_of8<DT>(vr[ks]), sh_bf16_of8<DT>(vr[ks]), g);
      norm2 = g[0];
    }
    if (lane == 0 && cached) v_norm[(int64_t)pair * Tcap + p] = f32_to_f16_bits(sqrtf(norm2));
  }
  if (w < NW) {
    sh_f32x4 acc[2] = {sh_f32x4{0.f, 0.f, 0.f, 0.f}, sh_f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
        acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[ks][mb].v, kf[ks].v, acc[mb], 0, 0, 0);
    // register r of block mb in lane quarter q is the plane at bit 8q + 7 - 4mb - r
    uint32_t neg = 0;
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) neg = __builtin_amdgcn_alignbit(neg, __float_as_uint(acc[mb][r]), 31);
    const uint32_t word = (__builtin_amdgcn_readlane(neg, 0) & 0xffu) | ((__builtin_amdgcn_readlane(neg, 16) & 0xffu) << 8) |
                          ((__builtin_amdgcn_readlane(neg, 32) & 0xffu) << 16) |
                          ((__builtin_amdgcn_readlane(neg, 48) & 0xffu) << 24);
    const int cpw = 32 / K;
    const int nbits = min(cpw, L - w * cpw) * K;
    const uint32_t valid = nbits >= 32 ? 0xffffffffu : ((1u << nbits) - 1u);
    if (lane == 0 && cached) codes[((int64_t)pair * NW + w) * Tcap + p] = ~word & valid;
  }
}

}  // namespace

namespace {

// The matrix-core form takes one prototype table size, the one the models have; its bits depend on neither the
// group nor the layout, so that every way to a table gives the same one.
bool mx_serves(int D, int K, int R) { return D == kMxD && K == kMxK && R == kMxR; }

MxUnits mx_units(int B, int Hq, int Hkv, int parts) {
  const int per_seq = parts > 0 ? Hkv * parts : Hq;
  return {B * per_seq, parts, Hq, Hkv, Hq / Hkv, per_seq, 1.f / (float)per_seq, parts > 0 ? 1.f / (float)parts : 0.f};
}

int soft_hash_entry(const void* q, int dtype, int64_t q_stride_b, int64_t q_stride_h, const void* planes,
                    const void* protos_T, void* out, int out_dtype, int B, int Hq, int Hkv, int D, int L, int K,
                    int R, float tanh_scale, float inv_temperature, void* stream, int grouped) {
  SOCKET_REQUIRE(q && planes && protos_T && out, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(socket_dtype_bytes(dtype) != 0, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(out_dtype == SOCKET_F32 || out_dtype == SOCKET_BF16, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && L > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(D >= 1 && D <= kSHMaxD && K >= 1 && K <= kSHMaxK, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(Hq / Hkv <= kSHMaxG, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(R >= 4 && R % 4 == 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE((int64_t)B * Hkv <= 65535, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(socket_aligned16(out), SOCKET_ERR_ALIGN);
  int parts = 0, width = 0;
  if (grouped) {
    const int st = socket_group_shape(Hq, Hkv, &parts, &width);
    if (st != SOCKET_OK) return st;
  }
  const dim3 grid(L, B * Hkv);
  hipStream_t s = (hipStream_t)stream;
  // vector loads of four elements: everything a lane fetches starts at a multiple of four
  const int vec_ok = (D % 4 == 0 && q_stride_b % 4 == 0 && q_stride_h % 4 == 0 && socket_aligned16(q) &&
                      socket_aligned16(planes) && socket_aligned16(protos_T))
                         ? 1
                         : 0;
  const int G = Hq / Hkv;
  if (dtype == SOCKET_BF16 && mx_serves(D, K, R) && vec_ok && q_stride_b % 8 == 0 && q_stride_h % 8 == 0) {
    const MxUnits units = mx_units(B, Hq, Hkv, parts);
    const int W = grouped ? width : 1, per = kMxHeads / W;
    const dim3 mx_grid(L, (units.count + per - 1) / per);
    SOCKET_REQUIRE(mx_grid.y <= 65535, SOCKET_ERR_SHAPE);
    const float scale = mx_scale(tanh_scale, inv_temperature);
#define SOCKET_MX(WV)                                                                                                         \
  do {                                                                                                                        \
    if (out_dtype == SOCKET_F32)                                                                                              \
      hipLaunchKernelGGL((soft_hash_mx_kernel<WV, DType_f32>), mx_grid, dim3(kSHThreads), 0, s, (const uint16_t*)q, q_stride_b,  \
                         q_stride_h, (const uint16_t*)planes, (const uint16_t*)protos_T, out, units, L, scale);               \
    else                                                                                                                      \
      hipLaunchKernelGGL((soft_hash_mx_kernel<WV, DType_bf16>), mx_grid, dim3(kSHThreads), 0, s, (const uint16_t*)q, q_stride_b, \
                         q_stride_h, (const uint16_t*)planes, (const uint16_t*)protos_T, out, units, L, scale);               \
  } while (0)
    if (W == 4) SOCKET_MX(4);
    else if (W == 2) SOCKET_MX(2);
    else SOCKET_MX(1);
#undef SOCKET_MX
    SOCKET_LAUNCH_CHECK();
    return SOCKET_OK;
  }
  if (dtype == SOCKET_F32 && mx_serves(D, K, R) && vec_ok) {
    const MxUnits units = mx_units(B, Hq, Hkv, parts);
    const int W = grouped ? width : 1, per = kMxHeads / W;
    const dim3 mx_grid(L, (units.count + per - 1) / per);
    SOCKET_REQUIRE(mx_grid.y <= 65535, SOCKET_ERR_SHAPE);
    auto of_type = [&](auto dt) {
      typedef decltype(dt) OutDT;
      return W == 4 ? soft_hash_mx32_kernel<4, OutDT> : W == 2 ? soft_hash_mx32_kernel<2, OutDT> : soft_hash_mx32_kernel<1, OutDT>;
    };
    auto kern = out_dtype == SOCKET_F32 ? of_type(DType_f32{}) : of_type(DType_bf16{});
    hipLaunchKernelGGL(kern, mx_grid, dim3(kSHThreads), 0, s, (const float*)q, q_stride_b, q_stride_h, (const float*)planes,
                       (const float*)protos_T, out, units, L, mx_scale(tanh_scale, inv_temperature));
    SOCKET_LAUNCH_CHECK();
    return SOCKET_OK;
  }
  // K = 10 with a single sweep (R <= 4 buckets per lane) and vector loads: the
  // prototypes go from global memory straight into registers.  Otherwise they go
  // to LDS as fp32 when they fit in 64 KB, else they are read from global memory
  // in every sweep.
  const bool direct = K == 10 && R <= kSHThreads * 4 && vec_ok;
  if (vec_ok && R <= kSmallR && K != 10) {
    const float scale = tanh_scale * inv_temperature;
#define SOCKET_SMALL_LAUNCH(DT, KM)                                                                                          \
  hipLaunchKernelGGL((soft_hash_small_kernel<DT, KM>), grid, dim3(kSHThreads), 0, s, q, q_stride_b, q_stride_h, planes, protos_T, \
                     out, out_dtype, Hq, Hkv, G, D, L, K, R, scale, parts, width)
#define SOCKET_SMALL(DT)                       \
  do {                                         \
    if (K <= 8) SOCKET_SMALL_LAUNCH(DT, 8);    \
    else SOCKET_SMALL_LAUNCH(DT, kSHMaxK);     \
  } while (0)
    if (dtype == SOCKET_F32) SOCKET_SMALL(DType_f32);
    else if (dtype == SOCKET_BF16) SOCKET_SMALL(DType_bf16);
    else SOCKET_SMALL(DType_f16);
#undef SOCKET_SMALL
#undef SOCKET_SMALL_LAUNCH
    SOCKET_LAUNCH_CHECK();
    return SOCKET_OK;
  }
  const size_t protos_bytes = (size_t)K * R * sizeof(float);
  const int protos_in_lds = (!direct && protos_bytes <= 64 * 1024) ? 1 : 0;
  const int GC = G <= 4 ? 4 : 8;
  const size_t head_floats = (((size_t)G * D + (((size_t)K * (D + 1) + 3) / 4) * 4 + (((size_t)G * K + 3) / 4) * 4 +
                               kSHWaves * GC + 3) / 4) * 4;
  const size_t dyn_lds = head_floats * sizeof(float) + (protos_in_lds ? protos_bytes : 0);
#define SOCKET_SH_LAUNCH(DT, GCV, KCV)                                                                     \
  do {                                                                                                     \
    auto kern = soft_hash_kernel<DT, GCV, KCV>;                                                            \
    if (dyn_lds > 16 * 1024 &&                                                                             \
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, \
                            (int)dyn_lds) != hipSuccess)                                                   \
      return SOCKET_ERR_LAUNCH;                                                                            \
    hipLaunchKernelGGL(kern, grid, dim3(kSHThreads), dyn_lds, s, q, q_stride_b, q_stride_h, planes,        \
                       protos_T, out, out_dtype, Hq, Hkv, G, D, L, K, R, tanh_scale, inv_temperature,       \
                       parts, width, protos_in_lds, vec_ok);                                               \
  } while (0)
#define SOCKET_SH(DT)                                          \
  do {                                                         \
    if (direct) {                                              \
      if (GC == 4) SOCKET_SH_LAUNCH(DT, 4, 10);                \
      else SOCKET_SH_LAUNCH(DT, 8, 10);                        \
    } else {                                                   \
      if (GC == 4) SOCKET_SH_LAUNCH(DT, 4, 0);                 \
      else SOCKET_SH_LAUNCH(DT, 8, 0);                         \
    }                                                          \
  } while (0)
  if (dtype == SOCKET_F32) SOCKET_SH(DType_f32);
  else if (dtype == SOCKET_BF16) SOCKET_SH(DType_bf16);
  else SOCKET_SH(DType_f16);
#undef SOCKET_SH
#undef SOCKET_SH_LAUNCH
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

}  // namespace

extern "C" int socket_soft_hash(const void* q, int dtype, int64_t q_stride_b, int64_t q_stride_h,
                                const void* planes, const void* protos_T, void* out, int out_dtype,
                                int B, int Hq, int Hkv, int D, int L, int K, int R,
                                float tanh_scale, float inv_temperature, void* stream) {
  return soft_hash_entry(q, dtype, q_stride_b, q_stride_h, planes, protos_T, out, out_dtype, B, Hq, Hkv, D, L,
                         K, R, tanh_scale, inv_temperature, stream, 0);
}

extern "C" int socket_soft_hash_grouped(const void* q, int dtype, int64_t q_stride_b, int64_t q_stride_h,
                                        const void* planes, const void* protos_T, void* q_table,
                                        int out_dtype, int B, int Hq, int Hkv, int D, int L, int K, int R,
                                        float tanh_scale, float inv_temperature, void* stream) {
  return soft_hash_entry(q, dtype, q_stride_b, q_stride_h, planes, protos_T, q_table, out_dtype, B, Hq, Hkv, D,
                         L, K, R, tanh_scale, inv_temperature, stream, 1);
}

namespace {

int decode_prologue_entry(const void* qkv, int dtype, int64_t qkv_stride_b, const void* freqs_cis,
                                      int freqs_dtype, int64_t n_pos, const int64_t* pos, int pos_stride,
                                      void* q_out, void* k_cache, void* v_cache, int64_t cache_stride_b,
                                      int64_t cache_stride_h, int64_t cache_stride_s, int32_t* lens,
                                      const void* planes_words, void* codes, void* v_norm, const void* planes,
                                      const void* protos_T, void* q_table, int out_dtype, int grouped, int B,
                                      int Hq, int Hkv, int D, int L, int K, int R, int64_t Tcap,
                                      float tanh_scale, float inv_temperature, void* stream) {
  SOCKET_REQUIRE(qkv && freqs_cis && pos && q_out && k_cache && v_cache && planes_words && codes && v_norm &&
                     planes && protos_T && q_table,
                 SOCKET_ERR_NULL);
  // the shapes the fused launch is written for; anything else takes the separate entry points
  const bool mx = mx_serves(D, K, R), small = K != 10 && R <= kSmallR;
  SOCKET_REQUIRE((dtype == SOCKET_BF16 || dtype == SOCKET_F32) && D == kPrologueD && K >= 1 && K <= kSHMaxK, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(small || (dtype == SOCKET_BF16 ? K == 10 : mx && out_dtype == SOCKET_F32), SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(freqs_dtype == SOCKET_F32 || freqs_dtype == SOCKET_BF16, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(out_dtype == SOCKET_F32 || out_dtype == SOCKET_BF16, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && L > 0 && Tcap > 0 && n_pos > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(Hq / Hkv <= kSHMaxG, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(R >= 4 && R % 4 == 0 && R <= kSHThreads * 4, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(pos_stride == 0 || pos_stride == 1, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(qkv_stride_b % 8 == 0 && cache_stride_b % 8 == 0 && cache_stride_h % 8 == 0 &&
                     cache_stride_s % 8 == 0,
                 SOCKET_ERR_ALIGN);
  SOCKET_REQUIRE(socket_aligned16(qkv) && socket_aligned16(freqs_cis) && socket_aligned16(q_out) &&
                     socket_aligned16(k_cache) && socket_aligned16(v_cache) && socket_aligned16(planes_words) &&
                     socket_aligned16(planes) && socket_aligned16(protos_T) && socket_aligned16(q_table),
                 SOCKET_ERR_ALIGN);
  int parts = 0, width = 0;
  if (grouped) {
    const int st = socket_group_shape(Hq, Hkv, &parts, &width);
    if (st != SOCKET_OK) return st;
  }
  const int G = Hq / Hkv, GC = G <= 4 ? 4 : 8;
  const int cpw = 32 / K, NW = (L + cpw - 1) / cpw;
  const int word_blocks = (NW + kSHWaves - 1) / kSHWaves;
  const int64_t n_key_blocks = (int64_t)B * Hkv * word_blocks;
  const int64_t n_blocks = n_key_blocks + (int64_t)B * Hkv * L;
  SOCKET_REQUIRE(n_blocks < (1LL << 31), SOCKET_ERR_SHAPE);
  const size_t head_floats = (((size_t)G * D + (((size_t)K * (D + 1) + 3) / 4) * 4 + (((size_t)G * K + 3) / 4) * 4 +
                               kSHWaves * GC + 3) / 4) * 4;
  const size_t dyn_lds = head_floats * sizeof(float);
  hipStream_t s = (hipStream_t)stream;
  const MxUnits units = mx_units(B, Hq, Hkv, parts);
  const int W = grouped ? width : 1, per = kMxHeads / W;
  const int64_t blocks = mx ? n_key_blocks + (int64_t)((units.count + per - 1) / per) * L : n_blocks;
#define SOCKET_DP(DT, GCV, FT, WV, OT)                                                                                        \
  hipLaunchKernelGGL((decode_prologue_kernel<DT, GCV, FT, WV, OT>), dim3((unsigned)blocks), dim3(kSHThreads), GCV > 0 ? dyn_lds : 0, s, \
                     (const DT::storage*)qkv, qkv_stride_b, freqs_cis, pos, pos_stride, n_pos, (DT::storage*)q_out,            \
                     (DT::storage*)k_cache, (DT::storage*)v_cache, cache_stride_b, cache_stride_h, cache_stride_s, lens,       \
                     (const uint16_t*)planes_words, (uint32_t*)codes, (uint16_t*)v_norm, NW, Tcap, planes, protos_T, q_table,  \
                     out_dtype, Hq, Hkv, G, L, K, R, tanh_scale, inv_temperature, parts, width, word_blocks,                   \
                     (int)n_key_blocks, units)
#define SOCKET_DP_MX(DT, FT, OT)                  \
  do {                                            \
    if (W == 4) SOCKET_DP(DT, 0, FT, 4, OT);      \
    else if (W == 2) SOCKET_DP(DT, 0, FT, 2, OT); \
    else SOCKET_DP(DT, 0, FT, 1, OT);             \
  } while (0)
#define SOCKET_DP_FT(FT)                                                                  \
  do {                                                                                    \
    if (small && dtype == SOCKET_F32) {                                                   \
      if (K <= 8) SOCKET_DP(DType_f32, -8, FT, 1, float);                                 \
      else SOCKET_DP(DType_f32, -kSHMaxK, FT, 1, float);                                  \
    } else if (small) {                                                                   \
      if (K <= 8) SOCKET_DP(DType_bf16, -8, FT, 1, float);                                \
      else SOCKET_DP(DType_bf16, -kSHMaxK, FT, 1, float);                                 \
    } else if (dtype == SOCKET_F32) SOCKET_DP_MX(DType_f32, FT, float);                   \
    else if (mx && out_dtype == SOCKET_F32) SOCKET_DP_MX(DType_bf16, FT, float);          \
    else if (mx) SOCKET_DP_MX(DType_bf16, FT, uint16_t);                                  \
    else if (GC == 4) SOCKET_DP(DType_bf16, 4, FT, 1, float);                             \
    else SOCKET_DP(DType_bf16, 8, FT, 1, float);                                          \
  } while (0)
  if (freqs_dtype == SOCKET_F32) SOCKET_DP_FT(DType_f32);
  else SOCKET_DP_FT(DType_bf16);
#undef SOCKET_DP_FT
#undef SOCKET_DP_MX
#undef SOCKET_DP
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

}  // namespace

extern "C" int socket_decode_prologue(const void* qkv, int dtype, int64_t qkv_stride_b, const void* freqs_cis,
                                      int freqs_dtype, int64_t n_pos, const int64_t* pos, int pos_stride,
                                      void* q_out, void* k_cache, void* v_cache, int64_t cache_stride_b,
                                      int64_t cache_stride_h, int64_t cache_stride_s, int32_t* lens,
                                      const void* planes_words, void* codes, void* v_norm, const void* planes,
                                      const void* protos_T, void* q_table, int out_dtype, int grouped, int B,
                                      int Hq, int Hkv, int D, int L, int K, int R, int64_t Tcap,
                                      float tanh_scale, float inv_temperature, void* stream) {
  // (what this entry has always taken: bf16, ten planes)
  SOCKET_REQUIRE(qkv && freqs_cis && pos && q_out && k_cache && v_cache && planes_words && codes && v_norm &&
                     planes && protos_T && q_table,
                 SOCKET_ERR_NULL);
  SOCKET_REQUIRE(dtype == SOCKET_BF16 && K == 10, SOCKET_ERR_UNSUPPORTED);
  return decode_prologue_entry(qkv, dtype, qkv_stride_b, freqs_cis, freqs_dtype, n_pos, pos, pos_stride, q_out, k_cache,
                               v_cache, cache_stride_b, cache_stride_h, cache_stride_s, lens, planes_words, codes, v_norm,
                               planes, protos_T, q_table, out_dtype, grouped, B, Hq, Hkv, D, L, K, R, Tcap, tanh_scale,
                               inv_temperature, stream);
}

extern "C" int socket_decode_prologue_typed(const void* qkv, int dtype, int64_t qkv_stride_b, const void* freqs_cis,
                                      int freqs_dtype, int64_t n_pos, const int64_t* pos, int pos_stride,
                                      void* q_out, void* k_cache, void* v_cache, int64_t cache_stride_b,
                                      int64_t cache_stride_h, int64_t cache_stride_s, int32_t* lens,
                                      const void* planes_words, void* codes, void* v_norm, const void* planes,
                                      const void* protos_T, void* q_table, int out_dtype, int grouped, int B,
                                      int Hq, int Hkv, int D, int L, int K, int R, int64_t Tcap,
                                      float tanh_scale, float inv_temperature, void* stream) {
  return decode_prologue_entry(qkv, dtype, qkv_stride_b, freqs_cis, freqs_dtype, n_pos, pos, pos_stride, q_out, k_cache,
                               v_cache, cache_stride_b, cache_stride_h, cache_stride_s, lens, planes_words, codes, v_norm,
                               planes, protos_T, q_table, out_dtype, grouped, B, Hq, Hkv, D, L, K, R, Tcap, tanh_scale,
                               inv_temperature, stream);
}
