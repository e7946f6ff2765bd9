// Gated linear recurrences with a decay per head and key channel, with or without the
// delta rule, or with the generalized delta rule (the definition stands at socket_recurrence in socket_hip.h): one token per
// call for decoding, chunks of tokens on the matrix cores for prompts.  fp32 throughout;
// only the projected rows that come in and the gated rows that go out have the model's type.
//
// Chunk form.  Inside a chunk let b_t be the running sum of log g (per channel, <= 0) and
// S0 the state before the chunk.  Unrolling the recurrence,
//   o_t = (q_t e^{b_t})^T S0 + sum_{s <= t} Aqk[t,s] u_s,   Aqk[t,s] = sum_c q_tc k_sc e^{b_tc - b_sc}
//   u_t = beta_t (v_t - (k_t e^{b_t})^T S0 - sum_{s < t} Akk[t,s] u_s)     (delta rule)
//   S   = diag(e^{b_C}) S0 + sum_s (k_s e^{b_C - b_s}) u_s^T
// so with L = diag(beta) Akk (strictly lower), U = (I + L)^{-1} diag(beta) (V - K^ S0) = Ubar - W S0.
// Everything without S0 is worked out for all chunks at once (recurrence_prep_kernel); only
// U = Ubar - W S0, O = Q^ S0 + Aqk U and the update of S run in sequence over the chunks
// (recurrence_scan_kernel), independently per (sequence, head, 16 value columns).
//
// e^{b_t - b_s} must not be split as e^{b_t} e^{-b_s}: the second factor overflows under
// strong decay.  Tokens are grouped in blocks of 16 with sums pl local to the block and
// block totals tot; for s in an earlier block the exponent splits at the start of t's
// block into two parts that are both <= 0.  Inside a block the split at the block's
// start is used while its total stays above kMildDecay, else the exponent is taken per
// pair on the vector ALU.
//
// All products are v_mfma_f32_16x16x4_f32 (fp32 operands).  Its operands hold one k index
// per lane quarter; a step r of four takes k = 4 * quarter + r of a 16-wide tile, so that
// a lane's four values are one 16-byte vector ("fragment order": lane (quarter, x) holds row x,
// columns 4 quarter .. + 3 of a tile), and an accumulator (rows 4 quarter + r, column x) is
// directly the second operand of the next product.
#include <type_traits>

#include "elem.h"

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float rc_f32x4;

__device__ __forceinline__ rc_f32x4 mfma4(const float4& a, const rc_f32x4& b, rc_f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b[0], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b[1], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b[2], c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b[3], c, 0, 0, 0);
  return c;
}

// ---- what both forms share: inputs of one (sequence, head) -------------------------------

constexpr float kRcLog2e = 1.4426950408889634f;

__device__ __forceinline__ float exp2_fast(float x) { return __builtin_amdgcn_exp2f(x); }   // v_exp_f32

// log2 of a channel's decay factor for z = low-rank product + bias; a_exp = exp(a_log[h]).
__device__ __forceinline__ float log2_decay(const socket_recurrence& a, float a_exp, float z) {
  if (a.decay_kind == 2) return -a.decay_rate * kRcLog2e * sigmoid_f32(z);
  const float f = a.decay_kind == 0 ? a_exp : a.inv_tau;
  return -f * kRcLog2e * softplus_f32(a.decay_kind == 0 ? z : -z);
}

__device__ __forceinline__ float gate_act(int kind, float x) {
  const float s = sigmoid_f32(x);
  return kind == 0 ? s : x * s;
}

__device__ __forceinline__ int conv_channels(const socket_recurrence& a) { return 2 * a.Hk * a.dk + a.H * a.dv; }

constexpr int kTapsAtOnce = 4;   // rows requested together

// q | k | v channel `ch` of token t (column `col` of the projected row), after the short
// convolution and its activation.  Rows before the portion come from half `parity` of the
// convolution state.  N channels at once, N = 1 or 8 (aligned).
template <class DT, int N>
__device__ __forceinline__ void conv_input(const socket_recurrence& a, int b, int t, int col, int ch, int parity,
                                           float* out) {
  const int64_t row = b * a.proj_stride_b + col;
  if (a.taps < 1) {
    load_vec<DT, N>(a.proj, row + t * a.proj_stride_t, out);
    return;
  }
  const int n1 = a.taps - 1, C = conv_channels(a);
#pragma unroll
  for (int e = 0; e < N; ++e) out[e] = 0.f;
  for (int m0 = 0; m0 < a.taps; m0 += kTapsAtOnce) {
    float x[kTapsAtOnce][N], w[kTapsAtOnce][N];
#pragma unroll
    for (int i = 0; i < kTapsAtOnce; ++i) {
      const int m = m0 + i, tt = t - n1 + m;
#pragma unroll
      for (int e = 0; e < N; ++e) x[i][e] = w[i][e] = 0.f;
      if (m < a.taps) {
        load_vec<DType_f32, N>(a.conv_w, (int64_t)m * C + ch, w[i]);
        if (tt >= 0) load_vec<DT, N>(a.proj, row + tt * a.proj_stride_t, x[i]);
        else if (!a.fresh) load_vec<DT, N>(a.conv_state, (((int64_t)parity * a.B + b) * n1 + (tt + n1)) * C + ch, x[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < kTapsAtOnce; ++i)
#pragma unroll
      for (int e = 0; e < N; ++e) out[e] = fmaf(x[i][e], w[i][e], out[e]);
  }
#pragma unroll
  for (int e = 0; e < N; ++e) out[e] *= sigmoid_f32(out[e]);
}

// ---- one token ------------------------------------------------------------------------------

// Rows of the low-rank products of one head: the decay's dk rows, then the gate's dv rows (none
// without gate_w), y[r] = w[r, :] . x.  16 lanes per row; kRowsAtOnce rows of a lane group are
// requested before the first is summed, so that a head's matrices (which no cache holds from one
// token to the next) cost one trip to memory.
constexpr int kRowsAtOnce = 8;

// One lane's 8 elements as loaded, so that eight rows in flight take few registers.
template <class DT>
struct Raw8 {
  uint4 v[8 / DT::kPer16B];
  __device__ __forceinline__ void load(const void* p, int64_t i) {
#pragma unroll
    for (int k = 0; k < 8 / DT::kPer16B; ++k)
      v[k] = *reinterpret_cast<const uint4*>((const typename DT::storage*)p + i + k * DT::kPer16B);
  }
  __device__ __forceinline__ void zero() {
#pragma unroll
    for (int k = 0; k < 8 / DT::kPer16B; ++k) v[k] = make_uint4(0, 0, 0, 0);
  }
  __device__ __forceinline__ void get(float* out) const {
#pragma unroll
    for (int k = 0; k < 8 / DT::kPer16B; ++k) unpack16<DT>(v[k], out + k * DT::kPer16B);
  }
};

// By lanes tid = 0 .. nt - 1 (a multiple of 64).  TANH: of the decay's columns.
template <class DT, bool TANH>
__device__ __forceinline__ void low_rank_rows(const socket_recurrence& a, int h, int64_t row0, int tid, int nt, float* gs,
                                              float* gate) {
  constexpr int ROWS = DT::kPer16B == 8 ? kRowsAtOnce : kRowsAtOnce / 2;
  const int sub = tid & 15, grp = tid >> 4, ngrp = nt >> 4;
  const int n = a.dk + (a.gate_w ? a.dv : 0);
  const bool vec = a.decay_rank % 8 == 0 && a.decay_rank <= 128 && (row0 + a.decay_off) % 8 == 0 &&
                   (!a.gate_w || (a.gate_rank % 8 == 0 && a.gate_rank <= 128 && (row0 + a.gate_off) % 8 == 0));
  if (vec) {
    Raw8<DT> xd, xg;
    xd.zero();
    xg.zero();
    if (sub * 8 < a.decay_rank) xd.load(a.proj, row0 + a.decay_off + sub * 8);
    if (a.gate_w && sub * 8 < a.gate_rank) xg.load(a.proj, row0 + a.gate_off + sub * 8);
    float xt[8];
    if constexpr (TANH) {
      xd.get(xt);
#pragma unroll
      for (int e = 0; e < 8; ++e) xt[e] = tanh_f32(xt[e]);
    }
    for (int c0 = 0; c0 < n; c0 += ngrp * ROWS) {   // (all lanes take part in the sums)
      Raw8<DT> w[ROWS];
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const int c = c0 + i * ngrp + grp;
        w[i].zero();
        if (c < a.dk) {
          if (sub * 8 < a.decay_rank) w[i].load(a.decay_w, ((int64_t)h * a.dk + c) * a.decay_rank + sub * 8);
        } else if (c < n) {
          if (sub * 8 < a.gate_rank) w[i].load(a.gate_w, ((int64_t)h * a.dv + c - a.dk) * a.gate_rank + sub * 8);
        }
      }
#pragma unroll
      for (int i = 0; i < ROWS; ++i) {
        const int c = c0 + i * ngrp + grp;
        float x[8], y[8], t = 0.f;
        (c < a.dk ? xd : xg).get(x);
        if constexpr (TANH) {
#pragma unroll
          for (int e = 0; e < 8; ++e) x[e] = xt[e];      // (no gate here)
        }
        w[i].get(y);
#pragma unroll
        for (int e = 0; e < 8; ++e) t = fmaf(y[e], x[e], t);
        t = group_sum<16>(t);
        if (c < n && sub == 0) (c < a.dk ? gs : gate - a.dk)[c] = t;
      }
    }
    return;
  }
  for (int c0 = 0; c0 < n; c0 += ngrp) {
    const int c = c0 + grp;
    float t = 0.f;
    if (c < n) {
      const bool decay = c < a.dk;
      const void* w = decay ? a.decay_w : a.gate_w;
      const int rank = decay ? a.decay_rank : a.gate_rank;
      const int64_t wr = (decay ? (int64_t)h * a.dk + c : (int64_t)h * a.dv + c - a.dk) * rank;
      const int64_t xr = row0 + (decay ? a.decay_off : a.gate_off);
      for (int r = sub; r < rank; r += 16) {
        const float x = load_elem<DT>(a.proj, xr + r);
        t = fmaf(load_elem<DT>(w, wr + r), TANH && decay ? tanh_f32(x) : x, t);
      }
    }
    t = group_sum<16>(t);
    if (c < n && sub == 0) (c < a.dk ? gs : gate - a.dk)[c] = t;
  }
}

// How a workgroup's lanes cover a state: `nc` lanes of VEC columns across (nc_shift: its base-2
// logarithm, -1 if it is no power of two) and RG rows side by side.
struct StepShape {
  int nc, nc_shift, RG;
};

// One workgroup per (head, sequence); grid (heads per q / k head, q / k heads, sequences).  The
// state lives in registers: a lane owns VEC neighbouring columns of every RG-th row; sums
// over the rows go through LDS.  GENERAL: rule 1.
template <class DT, int VEC, int ROWS, bool GENERAL>
__global__ __launch_bounds__(1024) void recurrence_step_kernel(socket_recurrence a, StepShape sh) {
  extern __shared__ __attribute__((aligned(16))) float rs_lds[];
  const int hk = blockIdx.y, h = hk * gridDim.x + blockIdx.x, b = blockIdx.z;
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63;
  const int dk = a.dk, dv = a.dv;
  const bool delta = GENERAL || a.beta_off >= 0;
  float* qs = rs_lds;             // dk
  float* ks = qs + dk;            // dk
  float* gs = ks + dk;            // dk: low-rank product, then decay
  float* vs = gs + dk;            // dv
  float* gate = vs + dv;          // dv
  float* os = gate + dv;          // dv: sums over the rows
  float* red = os + dv;           // 16
  float* rates = red + 16;        // GENERAL: dk, removal rate per key channel
  float* part = rates + (GENERAL ? dk : 0);   // RG * dv
  const int RG = sh.RG;
  const int rg = sh.nc_shift >= 0 ? tid >> sh.nc_shift : tid / sh.nc;
  const int col = (tid - rg * sh.nc) * VEC;
  const bool active = rg < RG;

  // the state, requested before anything else, then the small operands of later phases
  float* Sp = a.state + ((int64_t)b * a.H + h) * dk * dv + rg * dv + col;
  float S[ROWS][VEC];
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) S[i][e] = 0.f;
    if (active && rg + i * RG < dk) load_vec<DType_f32, VEC>(Sp, i * RG * dv, S[i]);
  }
  const int64_t row0 = b * a.proj_stride_b;
  const float bias = (a.decay_bias && tid < dk) ? a.decay_bias[h * dk + tid] : 0.f;
  const float nw = tid < dv ? a.norm_w[(GENERAL && a.norm_per_head ? h * dv : 0) + tid] : 0.f;
  const float beta_z = !GENERAL && delta ? load_elem<DT>(a.proj, row0 + a.beta_off + h) : 0.f;
  const int half = nt >> 1;
  if (tid < half) {
    // half of the waves: the low-rank products
    low_rank_rows<DT, GENERAL>(a, h, row0, tid, half, gs, gate);
  } else {
    // the other half meanwhile: q, k and v through the convolution, whose inputs move up by one
    // in the other half of its state (heads that share q / k write the same values).  Both halves
    // are read, so that the loads do not wait for the position.
    const int n1 = a.taps - 1, C = conv_channels(a);
    const int64_t pos = *a.pos;
    if constexpr (GENERAL)
      for (int c = tid - half; c < dk; c += half) {
        const float z = load_elem<DT>(a.proj, row0 + a.rate_off + h * dk + c);
        rates[c] = sigmoid_f32(z + (a.rate_bias ? a.rate_bias[h * dk + c] : 0.f));
      }
    for (int i = tid - half; i < 2 * dk + dv; i += half) {
      const int which = (i >= dk) + (i >= 2 * dk);
      const int at = which == 2 ? h * dv + i - 2 * dk : hk * dk + i - which * dk;
      const int ch = which * a.Hk * dk + at;
      const float now = load_elem<DT>(a.proj, row0 + (which == 0 ? a.q_off : which == 1 ? a.k_off : a.v_off) + at);
      float y = now;
      if (!GENERAL && a.taps >= 1) {
        y = 0.f;
        const int64_t s0 = (int64_t)b * n1 * C + ch, other = (int64_t)a.B * n1 * C;
        for (int m0 = 0; m0 < a.taps; m0 += kTapsAtOnce) {
          float w[kTapsAtOnce], x0[kTapsAtOnce], x1[kTapsAtOnce];
#pragma unroll
          for (int u = 0; u < kTapsAtOnce; ++u) {
            const int m = m0 + u;
            w[u] = x0[u] = x1[u] = 0.f;
            if (m < a.taps) w[u] = a.conv_w[m * C + ch];
            if (m < n1) {
              x0[u] = load_elem<DT>(a.conv_state, s0 + m * C);
              x1[u] = load_elem<DT>(a.conv_state, s0 + other + m * C);
            }
          }
          const bool odd = pos & 1;
#pragma unroll
          for (int u = 0; u < kTapsAtOnce; ++u) {
            const int m = m0 + u;
            const float x = m < n1 ? (odd ? x1[u] : x0[u]) : now;
            y = fmaf(x, w[u], y);
            if (m >= 1 && m <= n1) store_elem<DT>(a.conv_state, s0 + (odd ? 0 : other) + (m - 1) * C, x);
          }
        }
        y *= sigmoid_f32(y);
      }
      qs[i < 2 * dk ? i : i + dk] = y;     // q | k | (decays) | v
    }
    if (!a.gate_w)
      for (int c = tid - half; c < dv; c += half) gate[c] = load_elem<DT>(a.proj, row0 + a.gate_off + h * dv + c);
  }
  const float a_exp = a.decay_kind == 0 ? exp_f32(a.a_log[h]) : 0.f;
  __syncthreads();
  if (tid < dk) gs[tid] = exp2_fast(log2_decay(a, a_exp, gs[tid] + bias));   // (dk <= 256 <= nt)
  float q_mul = a.q_scale, k_mul = 1.f;
  if (GENERAL || a.unit_qk) {
    // (every wave takes both sums for itself: no further barrier)
    float sq = 0.f, sk = 0.f;
    for (int c = lane; c < dk; c += 64) {
      sq = fmaf(qs[c], qs[c], sq);
      sk = fmaf(ks[c], ks[c], sk);
    }
    if (!GENERAL) q_mul *= rsqrt_f32(group_sum<64>(sq) + 1e-6f);
    k_mul = rsqrt_f32(group_sum<64>(sk) + 1e-6f);
  }
  __syncthreads();

  auto column_sum = [&](int c) __attribute__((always_inline)) {
    float s = 0.f;
#pragma unroll 8
    for (int r = 0; r < RG; ++r) s += part[r * dv + c];
    return s;
  };
  // decay (GENERAL: later), and what the state holds for this key
  float u[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) u[e] = 0.f;
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int row = rg + i * RG;
    if (active && row < dk) {
      const float g = gs[row], k = ks[row] * k_mul;
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        if (!GENERAL) S[i][e] *= g;
        u[e] = fmaf(S[i][e], k, u[e]);
      }
    }
  }
  if (delta) {
    if (active) store_vec<DType_f32, VEC>(part, rg * dv + col, u);
    __syncthreads();
    if (tid < dv) os[tid] = GENERAL ? column_sum(tid) : sigmoid_f32(beta_z) * (vs[tid] - column_sum(tid));   // (dv <= 256 <= nt)
    __syncthreads();
  }
  float o[VEC];
#pragma unroll
  for (int e = 0; e < VEC; ++e) o[e] = 0.f;
  float v[VEC];
  if (active) load_vec<DType_f32, VEC>(delta ? os : vs, col, u);
  if (GENERAL && active) load_vec<DType_f32, VEC>(vs, col, v);
#pragma unroll
  for (int i = 0; i < ROWS; ++i) {
    const int row = rg + i * RG;
    if (active && row < dk) {
      const float k = ks[row] * k_mul, q = qs[row] * q_mul;
      const float gone = GENERAL ? -rates[row] * k : 0.f;
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        if constexpr (GENERAL) S[i][e] = fmaf(ks[row], v[e], fmaf(gone, u[e], S[i][e] * gs[row]));
        else S[i][e] = fmaf(k, u[e], S[i][e]);
        o[e] = fmaf(S[i][e], q, o[e]);
      }
    }
  }
  if (active) store_vec<DType_f32, VEC>(part, rg * dv + col, o);   // (its last readers passed a barrier since)
#pragma unroll
  for (int i = 0; i < ROWS; ++i)
    if (active && rg + i * RG < dk) store_vec<DType_f32, VEC>(Sp, i * RG * dv, S[i]);
  __syncthreads();
  const float s = tid < dv ? column_sum(tid) : 0.f;
  const float rs = rsqrt_f32(block_sum(s * s, red) / (float)dv + a.eps);
  if (tid < dv) store_elem<DT>(a.out, ((int64_t)b * a.H + h) * dv + tid, s * rs * nw * gate_act(a.gate_kind, gate[tid]));
}

// ---- chunks of tokens -----------------------------------------------------------------------

constexpr int kPrepThreads = 1024;
constexpr int kPrepWaves = kPrepThreads / 64;
constexpr int kPrepHeadsFirst = 65535;   // chunks up to which they are the grid's y, whose limit this is
constexpr float kMildDecay = -60.f;   // a block's total log2 decay above which 2^{-pl} is safe in fp32

// Workspace of one (chunk, head, sequence), in floats.  kt / vt: 16-wide tiles of dk / dv.
// extra: what rule 1 adds to the read-out and to the state whatever the state was.
struct ChunkSpace {
  int kt, vt, nb;
  bool extra = false;
  __host__ __device__ int64_t w() const { return 0; }
  __host__ __device__ int64_t q() const { return (int64_t)nb * kt * 256; }
  __host__ __device__ int64_t kT() const { return 2 * (int64_t)nb * kt * 256; }
  __host__ __device__ int64_t u() const { return 3 * (int64_t)nb * kt * 256; }
  __host__ __device__ int64_t aqk() const { return u() + (int64_t)nb * vt * 256; }
  __host__ __device__ int64_t gamma() const { return aqk() + (int64_t)nb * nb * 256; }
  __host__ __device__ int64_t o() const { return gamma() + (int64_t)kt * 16; }
  __host__ __device__ int64_t s() const { return o() + (int64_t)nb * vt * 256; }
  __host__ __device__ int64_t size() const { return extra ? s() + (int64_t)kt * vt * 256 : o(); }
};

// Channels [0, 16 tiles) of token rows [0, 16 NB) of q, k or v into LDS rows of `pitch`
// floats; rows past the portion and channels past `width` are zero.
template <class DT>
__device__ __forceinline__ void stage_rows(const socket_recurrence& a, int b, int t_first, int n_rows, int rows, int col0,
                                           int ch0, int width, int padded, float* dst, int pitch, bool vec) {
  if (vec) {
    const int per = padded / 8;
    for (int w = threadIdx.x; w < rows * per; w += kPrepThreads) {
      const int r = w / per, c = w % per * 8;
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = 0.f;
      if (r < n_rows && c < width) conv_input<DT, 8>(a, b, t_first + r, col0 + c, ch0 + c, (int)(a.pos0 & 1), x);
      *reinterpret_cast<float4*>(dst + r * pitch + c) = make_float4(x[0], x[1], x[2], x[3]);
      *reinterpret_cast<float4*>(dst + r * pitch + c + 4) = make_float4(x[4], x[5], x[6], x[7]);
    }
  } else {
    for (int w = threadIdx.x; w < rows * padded; w += kPrepThreads) {
      const int r = w / padded, c = w % padded;
      float x = 0.f;
      if (r < n_rows && c < width) conv_input<DT, 1>(a, b, t_first + r, col0 + c, ch0 + c, (int)(a.pos0 & 1), &x);
      dst[r * pitch + c] = x;
    }
  }
}

// By one wave: the tile d = -L (strictly lower, fragment order) becomes (I + L)^{-1}, a column per lane.
__device__ __forceinline__ void invert_diagonal(float* d, int x16, int quarter) {
  float x[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    x[r] = r == x16 ? 1.f : 0.f;
#pragma unroll
    for (int s0 = 0; s0 < r; s0 += 4) {
      const float4 m = *reinterpret_cast<const float4*>(d + ((s0 >> 2) * 16 + r) * 4);
      x[r] = fmaf(m.x, x[s0], x[r]);
      if (s0 + 1 < r) x[r] = fmaf(m.y, x[s0 + 1], x[r]);
      if (s0 + 2 < r) x[r] = fmaf(m.z, x[s0 + 2], x[r]);
      if (s0 + 3 < r) x[r] = fmaf(m.w, x[s0 + 3], x[r]);
    }
  }
  if (quarter == 0)
#pragma unroll
    for (int r = 0; r < 16; ++r) d[((x16 >> 2) * 16 + r) * 4 + (x16 & 3)] = x[r];
}

// Eight channels of N inputs of token t (q, k and v of one head: columns `col` of the projected row, channels `ch`
// of the convolution) after the convolution and its activation, as conv_input gives them, every tap of every input
// requested before the first is used.  No load stands under a condition: rows before the portion come from another
// address, and rows that are nowhere are cleared where a chunk can have them.
template <class DT, int N, int TAPS>
__device__ __forceinline__ void conv_inputs(const socket_recurrence& a, int b, int t, bool at_start, const int (&col)[N],
                                            const int (&ch)[N], float (&out)[N][8]) {
  const int64_t row = b * a.proj_stride_b;
  if (a.taps < 1) {
    Raw8<DT> x[N];
#pragma unroll
    for (int s = 0; s < N; ++s) x[s].load(a.proj, row + t * a.proj_stride_t + col[s]);
#pragma unroll
    for (int s = 0; s < N; ++s) x[s].get(out[s]);
    return;
  }
  const int n1 = a.taps - 1, C = conv_channels(a);
#pragma unroll
  for (int s = 0; s < N; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) out[s][e] = 0.f;
  for (int m0 = 0; m0 < a.taps; m0 += TAPS) {
    Raw8<DT> x[N][TAPS];
#pragma unroll
    for (int i = 0; i < TAPS; ++i) {
      const int tt = t - n1 + min(m0 + i, n1);
      const bool stored = at_start && tt < 0 && !a.fresh;
      const void* from = stored ? a.conv_state : a.proj;
      const int64_t at = stored ? (((int64_t)(a.pos0 & 1) * a.B + b) * n1 + (tt + n1)) * C : row + max(tt, 0) * a.proj_stride_t;
#pragma unroll
      for (int s = 0; s < N; ++s) x[s][i].load(from, at + (stored ? ch[s] : col[s]));
    }
    if (at_start && a.fresh) {
#pragma unroll
      for (int i = 0; i < TAPS; ++i)
        if (t - n1 + m0 + i < 0)
#pragma unroll
          for (int s = 0; s < N; ++s) x[s][i].zero();
    }
#pragma unroll
    for (int s = 0; s < N; ++s) {
#pragma unroll
      for (int i0 = 0; i0 < TAPS; i0 += 2) {
        float w[2][8];
#pragma unroll
        for (int i = 0; i < 2; ++i) load_vec<DType_f32, 8>(a.conv_w, (int64_t)min(m0 + i0 + i, n1) * C + ch[s], w[i]);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (m0 + i0 + i < a.taps) {
            float y[8];
            x[s][i0 + i].get(y);
#pragma unroll
            for (int e = 0; e < 8; ++e) out[s][e] = fmaf(y[e], w[i][e], out[s][e]);
          }
        }
      }
    }
  }
#pragma unroll
  for (int s = 0; s < N; ++s)
#pragma unroll
    for (int e = 0; e < 8; ++e) out[s][e] *= sigmoid_f32(out[s][e]);
}

// Sum of the squares of a token's channels, eight consecutive ones in each of its LPR lanes, in the order in which a wave
// of one channel a lane adds them: channels 64 apart one after the other, then the butterfly, whose first three steps are
// inside a lane.
template <int LPR>
__device__ __forceinline__ float sum_of_squares(const float (&x)[8], int lane) {
  static_assert(LPR == 16 || LPR == 32, "128 or 256 channels");
  float s[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float other = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x[e]), 0x128, 0xf, 0xf, false));   // row_ror:8
    const float low = lane & 8 ? other : x[e], high = lane & 8 ? x[e] : other;
    if constexpr (LPR == 16) {
      s[e] = fmaf(high, high, low * low);
    } else {
      const float low2 = lane_xor16(low), high2 = lane_xor16(high);
      const bool upper = lane & 16;
      const float c0 = upper ? low2 : low, c1 = upper ? high2 : high, c2 = upper ? low : low2, c3 = upper ? high : high2;
      s[e] = fmaf(c3, c3, fmaf(c2, c2, fmaf(c1, c1, c0 * c0)));
    }
  }
  return group_sum<8>(((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7])));
}

// Lane j of every four lanes gives x[c] of lane c: x[c] becomes what lane c held at j.
__device__ __forceinline__ void transpose_quad(rc_f32x4& x, int lane) {
  const bool odd = lane & 1, high = lane & 2;
#pragma unroll
  for (int p = 0; p < 4; p += 2) {
    const float got = butterfly_partner<1>(odd ? x[p] : x[p + 1]);
    x[p] = odd ? got : x[p];
    x[p + 1] = odd ? x[p + 1] : got;
  }
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    const float got = butterfly_partner<2>(high ? x[p] : x[p + 2]);
    x[p] = high ? got : x[p];
    x[p + 2] = high ? x[p + 2] : got;
  }
}

// One workgroup per (chunk, head, sequence).  With 16 waves on a CU and one such workgroup (three operands and the
// tiles in LDS) nothing but the waves themselves hides a wait, so each phase asks for all it reads before it uses any:
//  * a lane's eight channels of q, k and v with all their taps, and its eight decays, in one trip to memory; unit
//    norms from those registers, running sums of the decays over 8 rows of a lane and, from its sum on, a lane 32 further
//    on (with both halves summed from zero and put together afterwards neighbours are rounded apart at the full sum's
//    magnitude: states up to four times as far from float64, 6.8e-7 where this gives 1.7e-7);
//  * the tiles of Aqk and L (a diagonal tile inverted by its own wave) and the fragments of Q^ and K^T are dealt out
//    by a counter, the long ones first;
//  * the forward substitution has its tiles in registers before it starts, and W leaves in 16-byte stores.
// A workgroup of 128 key channels with the delta rule / of 64 without, in clock cycles: 63000 / 29000 -> 47000 / 21000
// (18000 of the 47000 the first trip and its arithmetic, 13000 the tiles, 5000 the substitution); 5000 tokens of 16 heads
// of either kind 294 -> 245 us.  A chunk writes 144 KB for the scan, which 256 of them drain in about 8 us.  Holding
// the second kind to 64 registers for two workgroups a CU spilled: 63 us a pass instead of 53.
template <class DT, int NB, bool DELTA>
__global__ __launch_bounds__(kPrepThreads) void recurrence_prep_kernel(socket_recurrence a, int n_chunks, int vec, int own_v) {
  constexpr int C = 16 * NB;
  constexpr int LPR = kPrepThreads / C;          // lanes to a token: 8 channels each
  extern __shared__ __attribute__((aligned(16))) float rp_lds[];
  __shared__ int next_item;
  // (a head on one XCD, where its scan will be, while the chunks fit the grid's y)
  const bool heads_first = n_chunks <= kPrepHeadsFirst;
  const int h = heads_first ? blockIdx.x : blockIdx.y, chunk = heads_first ? blockIdx.y : blockIdx.x, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int x16 = lane & 15, quarter = lane >> 4;
  const int dk = a.dk, dv = a.dv, hk = h / (a.H / a.Hk);
  const ChunkSpace sp{(dk + 15) / 16, (dv + 15) / 16, NB};
  const int dkp = sp.kt * 16, dvp = sp.vt * 16;
  const int kp = dkp + 4, vp = dvp + 4;          // LDS pitches
  const int t_first = a.t0 + chunk * C;          // token of the portion
  const int n_rows = min(C, a.t0 + a.n - t_first);

  float* pl = rp_lds;                            // C x kp: running sum of the log2 decay inside the block
  float* tot = pl + C * kp;                      // NB x dkp
  float* beta = tot + NB * dkp;                  // C
  float* lk = beta + C;                          // DELTA: NB x NB tiles in fragment order: -L, inverses on the diagonal
  float* ks = lk + (DELTA ? NB * NB * 256 : 0);  // C x kp
  float* qs = ks + C * kp;                       // C x kp
  // C x vp; by itself where LDS allows it, else over q (without the delta rule over k as well) once that has been used
  float* vs = DELTA && own_v ? qs + C * kp : DELTA ? qs : ks;

  float* ws = (float*)a.workspace + (((int64_t)b * a.H + h) * n_chunks + chunk) * sp.size();

  // ---- inputs.  Decays: lane x of 32 (and x + 32) takes a channel over rows 0 .. 7 (and 8 .. 15) of a block
  const int spans = (dkp + 31) / 32;
  float z[8];
  auto request_decays = [&](int g) __attribute__((always_inline)) {
    const int blk = g / spans, c = (g - blk * spans) * 32 + (lane & 31), r0 = 16 * blk + 8 * (lane >> 5);
    const int64_t zc = (int64_t)h * dk + min(c, dk - 1);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int64_t zi = ((int64_t)b * a.T + t_first + min(r0 + r, n_rows - 1)) * a.H * dk + zc;
      z[r] = a.decay_z_f32 ? ((const float*)a.decay_z)[zi] : load_elem<DT>(a.decay_z, zi);
    }
  };
  if (wave < NB * spans) request_decays(wave);
  {
    const int r = tid / LPR, c = tid % LPR * 8;
    const bool row_ok = r < n_rows;
    const int t = t_first + min(r, n_rows - 1);
    constexpr int N = 3;
    const int width[N] = {dk, dk, dv};
    const int col0[N] = {a.q_off + hk * dk, a.k_off + hk * dk, a.v_off + h * dv};
    const int ch0[N] = {hk * dk, a.Hk * dk + hk * dk, 2 * a.Hk * dk + h * dv};
    float x[N][8];
    if (vec) {
      int col[N], ch[N];
#pragma unroll
      for (int s = 0; s < N; ++s) {
        const int in = c < width[s] ? c : 0;
        col[s] = col0[s] + in;
        ch[s] = ch0[s] + in;
      }
      const bool at_start = t_first < a.taps - 1;
      if (DELTA && own_v) {
        conv_inputs<DT, 3, DT::kPer16B == 8 ? 4 : 2>(a, b, t, at_start, col, ch, x);
      } else {
        const int col2[2] = {col[0], col[1]}, ch2[2] = {ch[0], ch[1]};
        float y[2][8];
        conv_inputs<DT, 2, 2>(a, b, t, at_start, col2, ch2, y);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          x[0][e] = y[0][e];
          x[1][e] = y[1][e];
          x[2][e] = 0.f;
        }
      }
    } else {
      stage_rows<DT>(a, b, t_first, n_rows, C, col0[0], ch0[0], dk, dkp, qs, kp, false);
      stage_rows<DT>(a, b, t_first, n_rows, C, col0[1], ch0[1], dk, dkp, ks, kp, false);
      if (DELTA && own_v) stage_rows<DT>(a, b, t_first, n_rows, C, col0[2], ch0[2], dv, dvp, vs, vp, false);
      __syncthreads();
      // (a lane's own eight channels, which it writes again below; those past the width are zero)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[0][e] = c < dkp ? qs[r * kp + c + e] : 0.f;
        x[1][e] = c < dkp ? ks[r * kp + c + e] : 0.f;
        x[2][e] = DELTA && own_v && c < dvp ? vs[r * vp + c + e] : 0.f;
      }
    }
#pragma unroll
    for (int s = 0; s < N; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[s][e] = row_ok && c < width[s] ? x[s][e] : 0.f;
    float mul[2] = {a.q_scale, 1.f};
    if (a.unit_qk) {
      mul[0] *= rsqrt_f32(sum_of_squares<LPR>(x[0], lane) + 1e-6f);
      mul[1] = rsqrt_f32(sum_of_squares<LPR>(x[1], lane) + 1e-6f);
    }
    auto put = [&](float* to, const float* y, float m) __attribute__((always_inline)) {
      *reinterpret_cast<float4*>(to) = make_float4(y[0] * m, y[1] * m, y[2] * m, y[3] * m);
      *reinterpret_cast<float4*>(to + 4) = make_float4(y[4] * m, y[5] * m, y[6] * m, y[7] * m);
    };
    if (c < dkp) {
      put(qs + r * kp + c, x[0], mul[0]);
      put(ks + r * kp + c, x[1], mul[1]);
    }
    if (DELTA && own_v && c < dvp) put(vs + r * vp + c, x[2], 1.f);
  }
  const float a_exp = a.decay_kind == 0 ? exp_f32(a.a_log[h]) : 0.f;
  for (int g = wave; g < NB * spans; g += kPrepWaves) {
    if (g != wave) request_decays(g);
    const int blk = g / spans, c = (g - blk * spans) * 32 + (lane & 31), r0 = 16 * blk + 8 * (lane >> 5);
    const float bias = a.decay_bias && c < dk ? a.decay_bias[h * dk + c] : 0.f;
    // (a block's sixteen rows are summed one after the other: the upper half's lanes go on from the lower half's sum)
    float half = 0.f;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      z[r] = r0 + r < n_rows && c < dk ? log2_decay(a, a_exp, z[r] + bias) : 0.f;
      half += z[r];
    }
    const float before = lane_xor32(half);
    float sum = lane < 32 ? 0.f : before;
    if (c < dkp) {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        sum += z[r];
        pl[(r0 + r) * kp + c] = sum;
      }
      if (lane >= 32) tot[blk * dkp + c] = sum;
    }
  }
  if (tid < C)
    beta[tid] = (DELTA && tid < n_rows)
                    ? sigmoid_f32(load_elem<DT>(a.proj, b * a.proj_stride_b + (t_first + tid) * a.proj_stride_t + a.beta_off + h))
                    : 0.f;
  if (tid == 0) next_item = 0;
  __syncthreads();

  for (int c = tid; c < dkp; c += kPrepThreads) {
    float s = 0.f;
    for (int m = 0; m < NB; ++m) s += tot[m * dkp + c];
    ws[sp.gamma() + c] = exp2_fast(s);
  }

  // Aqk and -L, tile (I, J): lane (quarter, x) holds row x of block I against keys
  // 4 quarter + r of block J (the transposed product, which leaves fragment order)
  auto pair_tile = [&](int I, int J) __attribute__((always_inline)) {
    const int t = 16 * I + x16, s = 16 * J + x16;
    rc_f32x4 aq = {0.f, 0.f, 0.f, 0.f}, ak = {0.f, 0.f, 0.f, 0.f};
    bool mild = true;
    if (I == J) {
      bool low = false;
      for (int c = lane; c < dkp; c += 64) low |= tot[I * dkp + c] < kMildDecay;
      mild = __builtin_amdgcn_ballot_w64(low) == 0;
    }
    if (mild) {
#pragma unroll 2
      for (int j = 0; j < sp.kt; ++j) {
        const int c = 16 * j + 4 * quarter;
        float4 kk = *reinterpret_cast<const float4*>(ks + s * kp + c);
        const float4 ps = *reinterpret_cast<const float4*>(pl + s * kp + c);
        const float4 pt = *reinterpret_cast<const float4*>(pl + t * kp + c);
        const float4 qt = *reinterpret_cast<const float4*>(qs + t * kp + c);
        float4 kt = make_float4(0.f, 0.f, 0.f, 0.f);
        if (DELTA) kt = *reinterpret_cast<const float4*>(ks + t * kp + c);
        float4 e = make_float4(-ps.x, -ps.y, -ps.z, -ps.w);
#pragma unroll
        for (int m = 0; m < NB - 1; ++m) {
          if (m >= J && m < I) {
            const float4 tm = *reinterpret_cast<const float4*>(tot + m * dkp + c);
            e.x += tm.x;
            e.y += tm.y;
            e.z += tm.z;
            e.w += tm.w;
          }
        }
        kk.x *= exp2_fast(e.x);
        kk.y *= exp2_fast(e.y);
        kk.z *= exp2_fast(e.z);
        kk.w *= exp2_fast(e.w);
        const float4 f = make_float4(exp2_fast(pt.x), exp2_fast(pt.y), exp2_fast(pt.z), exp2_fast(pt.w));
        aq = mfma4(kk, rc_f32x4{qt.x * f.x, qt.y * f.y, qt.z * f.z, qt.w * f.w}, aq);
        if (DELTA) ak = mfma4(kk, rc_f32x4{kt.x * f.x, kt.y * f.y, kt.z * f.z, kt.w * f.w}, ak);
      }
    } else {
      // Strong decay inside the block: four channels of the rows at a time.  (16 heads x 5000 tokens with every tile such a
      // one: 393 us for the branch, 390 with mild tiles; five matrix products split at the middle of ever smaller groups of
      // rows are no faster.)
      for (int c = 0; c < dkp; c += 4) {
        const float4 p = *reinterpret_cast<const float4*>(pl + t * kp + c);
        const float4 q = *reinterpret_cast<const float4*>(qs + t * kp + c);
        float4 kt = make_float4(0.f, 0.f, 0.f, 0.f);
        if (DELTA) kt = *reinterpret_cast<const float4*>(ks + t * kp + c);
        float4 k[4], ps[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          k[r] = *reinterpret_cast<const float4*>(ks + (16 * J + 4 * quarter + r) * kp + c);
          ps[r] = *reinterpret_cast<const float4*>(pl + (16 * J + 4 * quarter + r) * kp + c);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float w = (&k[r].x)[e] * exp2_fast(fminf((&p.x)[e] - (&ps[r].x)[e], 0.f));
            aq[r] = fmaf((&q.x)[e], w, aq[r]);
            if (DELTA) ak[r] = fmaf((&kt.x)[e], w, ak[r]);
          }
      }
    }
    const float bt = DELTA ? beta[t] : 0.f;
    float4 q4, k4;
    float* q4p = &q4.x;
    float* k4p = &k4.x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int sr = 16 * J + 4 * quarter + r;
      q4p[r] = sr <= t ? aq[r] : 0.f;
      k4p[r] = sr < t ? -bt * ak[r] : 0.f;
    }
    *reinterpret_cast<float4*>(ws + sp.aqk() + (I * NB + J) * 256 + lane * 4) = q4;
    if (DELTA) {
      float* d = lk + (I * NB + J) * 256;
      *reinterpret_cast<float4*>(d + lane * 4) = k4;
      if (I == J) {
        // (I + L_II)^{-1}, a column per lane; the tile is this wave's own until the barrier
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        invert_diagonal(d, x16, quarter);
      }
    }
  };
  auto q_fragment = [&](int w) __attribute__((always_inline)) {
    const int ct = w / NB, rt = w % NB;
    const int t = 16 * rt + x16, c = 16 * ct + 4 * quarter;
    float4 e = *reinterpret_cast<const float4*>(pl + t * kp + c);
    const float4 q = *reinterpret_cast<const float4*>(qs + t * kp + c);
#pragma unroll
    for (int m = 0; m < NB - 1; ++m) {
      if (m < rt) {
        const float4 tm = *reinterpret_cast<const float4*>(tot + m * dkp + c);
        e.x += tm.x;
        e.y += tm.y;
        e.z += tm.z;
        e.w += tm.w;
      }
    }
    *reinterpret_cast<float4*>(ws + sp.q() + (rt * sp.kt + ct) * 256 + lane * 4) =
        make_float4(q.x * exp2_fast(e.x), q.y * exp2_fast(e.y), q.z * exp2_fast(e.z), q.w * exp2_fast(e.w));
  };
  auto k_fragment = [&](int w) __attribute__((always_inline)) {
    const int ct = w / NB, rt = w % NB;
    const int c = 16 * ct + x16;
    float after = 0.f;
#pragma unroll
    for (int m = 0; m < NB; ++m) after += m >= rt ? tot[m * dkp + c] : 0.f;
    float4 o;
    float* op = &o.x;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = 16 * rt + 4 * quarter + r;
      op[r] = ks[t * kp + c] * exp2_fast(after - pl[t * kp + c]);
    }
    *reinterpret_cast<float4*>(ws + sp.kT() + (ct * NB + rt) * 256 + lane * 4) = o;
  };

  // ---- tiles (the diagonal ones first), then fragments of Q^ and K^T (for the update), one of each to an item
  constexpr int kTiles = NB * (NB + 1) / 2;
  const int items = kTiles + NB * sp.kt;
  for (int item = wave;;) {
    if (item >= items) break;   // (an item past the end is the wave's last)
    if (item < kTiles) {
      int I = item, J = item;
      if (item >= NB) {
        I = 1;
        J = item - NB;
        while (J >= I) J -= I++;
      }
      pair_tile(I, J);
    } else {
      q_fragment(item - kTiles);
      k_fragment(item - kTiles);
    }
    int got = 0;
    if (lane == 0) got = atomicAdd(&next_item, 1);
    item = kPrepWaves + __builtin_amdgcn_readfirstlane(got);
  }
  __syncthreads();
  if (!DELTA || !own_v) {
    stage_rows<DT>(a, b, t_first, n_rows, C, a.v_off + h * dv, 2 * a.Hk * dk + h * dv, dv, dvp, vs, vp, vec);
    __syncthreads();
  }

  // ---- Ubar = T beta V and W = T beta K^, a 16-column tile per wave: forward substitution over
  // the blocks; a finished block's accumulator is the next product's operand
  const int n_tiles = DELTA ? sp.vt + sp.kt : sp.vt;
  for (int tile = wave; tile < n_tiles; tile += kPrepWaves) {
    const bool is_v = !DELTA || tile < sp.vt;
    const int ct = is_v ? tile : tile - sp.vt;
    const int c = 16 * ct + x16;
    rc_f32x4 X[NB];
    float4 m[DELTA ? kTiles : 1];
    if constexpr (DELTA) {
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int J = 0; J <= I; ++J)
          m[I * (I + 1) / 2 + J] = *reinterpret_cast<const float4*>(lk + (I * NB + J) * 256 + lane * 4);
    }
    if (is_v) {
#pragma unroll
      for (int I = 0; I < NB; ++I)
#pragma unroll
        for (int r = 0; r < 4; ++r) X[I][r] = vs[(16 * I + 4 * quarter + r) * vp + c];
    } else {
      float before = 0.f;
#pragma unroll
      for (int I = 0; I < NB; ++I) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * I + 4 * quarter + r;
          X[I][r] = ks[t * kp + c] * exp2_fast(before + pl[t * kp + c]);
        }
        before += tot[I * dkp + c];
      }
    }
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      if constexpr (DELTA) {
        rc_f32x4 acc;
        const float4 bt = *reinterpret_cast<const float4*>(beta + 16 * I + 4 * quarter);
        acc[0] = bt.x * X[I][0];
        acc[1] = bt.y * X[I][1];
        acc[2] = bt.z * X[I][2];
        acc[3] = bt.w * X[I][3];
#pragma unroll
        for (int J = 0; J < I; ++J) acc = mfma4(m[I * (I + 1) / 2 + J], X[J], acc);
        X[I] = mfma4(m[I * (I + 1) / 2 + I], acc, rc_f32x4{0.f, 0.f, 0.f, 0.f});
      }
      if (is_v) {
        *reinterpret_cast<rc_f32x4*>(ws + sp.u() + (I * sp.vt + ct) * 256 + lane * 4) = X[I];
      } else {
        rc_f32x4 y = X[I];
        transpose_quad(y, lane);
        *reinterpret_cast<rc_f32x4*>(ws + sp.w() + (I * sp.kt + ct) * 256 + ((x16 >> 2) * 16 + 4 * quarter + (x16 & 3)) * 4) = y;
      }
    }
  }
}

// ---- chunks of the generalized delta rule ---------------------------------------------------
//
// With y_t = S_{t-1}^T n_t, c_t = a_t * n_t and b_t the running sum of log g,
//   y_t = (n_t e^{b_{t-1}})^T S0 + sum_{s < t} M[t,s] v_s - L[t,s] y_s
//   o_t = (q_t e^{b_t})^T S0 + sum_{s <= t} Aqk[t,s] v_s - Aqc[t,s] y_s
//   S   = diag(e^{b_C}) S0 + sum_s (k_s e^{b_C - b_s}) v_s^T - (c_s e^{b_C - b_s}) y_s^T
// where M, L pair n_t e^{b_{t-1}} with k_s e^{-b_s}, c_s e^{-b_s}, and Aqk, Aqc pair q_t e^{b_t} with
// them.  With U = -Y the sequential part is the delta rule's, U = Ubar - W S0, O = Q^ S0 + Aqc U,
// S = diag(e^{b_C}) S0 + C^T U, plus two terms that do not depend on S0: Obar = Aqk V and Sbar = K^T V.
// W = (I + L)^{-1} (n e^{b-}), Ubar = -(I + L)^{-1} M V.
//
// A token's log2 decay is bounded (decay kind 2), so a chunk's sum stays far inside fp32's exponent
// range and e^{b_t - b_s} is taken as e^{b_t} e^{-b_s} (the host checks the bound).
constexpr int kGeneralItems = 2;         // (row, 4 channels) pieces per lane
constexpr float kMaxChunkDecay = 100.f;  // log2; exponents of that size and their products are normal numbers

template <class DT, int NB>
__global__ __launch_bounds__(kPrepThreads) void general_prep_kernel(socket_recurrence a, int vec, int late_v) {
  constexpr int C = 16 * NB;
  extern __shared__ __attribute__((aligned(16))) float rp_lds[];
  const int chunk = blockIdx.x, h = blockIdx.y, b = blockIdx.z;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int x16 = lane & 15, quarter = lane >> 4;
  const int dk = a.dk, dv = a.dv;
  const ChunkSpace sp{(dk + 15) / 16, (dv + 15) / 16, NB, true};
  const int dkp = sp.kt * 16, dvp = sp.vt * 16;
  const int kp = dkp + 4, vp = dvp + 4;          // LDS pitches
  const int t_first = a.t0 + chunk * C;
  const int n_rows = min(C, a.t0 + a.n - t_first);

  float* qs = rp_lds;                            // C x kp: q, then q e^b
  float* us = qs + C * kp;                       // C x kp: log2 decay, its running sum in the block, then n e^{b-}
  float* ks = us + C * kp;                       // C x kp: k, then k e^{-b}
  float* cs = ks + C * kp;                       // C x kp: rates, then a n e^{-b}
  float* vs = late_v ? qs : cs + C * kp;         // C x vp; late_v (wide heads): over q once that has been used
  float* tot = cs + C * kp + (late_v ? 0 : C * vp);   // NB x dkp
  float* lk = tot + NB * dkp;                    // tiles (I, J) in fragment order: -L, inverses on the diagonal
  float* mk = lk + NB * NB * 256;                // M
  float* ak = mk + NB * NB * 256;                // Aqk
  float* kn = ak + NB * NB * 256;                // C: 1 / |k|

  float* ws = (float*)a.workspace + (((int64_t)b * a.H + h) * gridDim.x + chunk) * sp.size();

  // ---- inputs
  stage_rows<DT>(a, b, t_first, n_rows, C, a.q_off + h * dk, h * dk, dk, dkp, qs, kp, vec);
  stage_rows<DT>(a, b, t_first, n_rows, C, a.k_off + h * dk, a.Hk * dk + h * dk, dk, dkp, ks, kp, vec);
  stage_rows<DT>(a, b, t_first, n_rows, C, a.rate_off + h * dk, 0, dk, dkp, cs, kp, vec && a.rate_off % 8 == 0);
  if (!late_v) stage_rows<DT>(a, b, t_first, n_rows, C, a.v_off + h * dv, 2 * a.Hk * dk + h * dv, dv, dvp, vs, vp, vec);
#pragma unroll 4
  for (int w = tid; w < C * dkp; w += kPrepThreads) {
    const int r = w / dkp, c = w % dkp;
    float g = 0.f;
    if (r < n_rows && c < dk) {
      const int64_t zi = ((int64_t)b * a.T + t_first + r) * a.H * dk + h * dk + c;
      g = log2_decay(a, 0.f, (a.decay_z_f32 ? ((const float*)a.decay_z)[zi] : load_elem<DT>(a.decay_z, zi)) +
                                 (a.decay_bias ? a.decay_bias[h * dk + c] : 0.f));
    }
    us[r * kp + c] = g;
  }
  __syncthreads();

  // ---- norms of the keys; running sums of the log2 decay inside each block
  for (int r = wave; r < C; r += kPrepWaves) {
    float sk = 0.f;
    for (int c = lane; c < dkp; c += 64) sk = fmaf(ks[r * kp + c], ks[r * kp + c], sk);
    sk = group_sum<64>(sk);
    if (lane == 0) kn[r] = rsqrt_f32(sk + 1e-6f);
  }
  for (int w = tid; w < NB * dkp; w += kPrepThreads) {
    const int blk = w / dkp, c = w % dkp;
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      s += us[(blk * 16 + r) * kp + c];
      us[(blk * 16 + r) * kp + c] = s;
    }
    tot[blk * dkp + c] = s;
  }
  __syncthreads();

  // ---- the four scaled operands, in place (a row's sums are read by the row after it: registers between)
  const int quads = dkp / 4;
  float4 nq[kGeneralItems], nu[kGeneralItems], nk[kGeneralItems], nc[kGeneralItems];
#pragma unroll
  for (int it = 0; it < kGeneralItems; ++it) {
    const int w = tid + it * kPrepThreads, r = w / quads, c = w % quads * 4;
    if (r >= C) continue;
    float4 off = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int m = 0; m < (r >> 4); ++m) {
      const float4 tm = *reinterpret_cast<const float4*>(tot + m * dkp + c);
      off.x += tm.x;
      off.y += tm.y;
      off.z += tm.z;
      off.w += tm.w;
    }
    const float4 in = *reinterpret_cast<const float4*>(us + r * kp + c);
    const float4 ex = (r & 15) ? *reinterpret_cast<const float4*>(us + (r - 1) * kp + c) : make_float4(0.f, 0.f, 0.f, 0.f);
    const float4 q = *reinterpret_cast<const float4*>(qs + r * kp + c), k = *reinterpret_cast<const float4*>(ks + r * kp + c);
    const float4 z = *reinterpret_cast<const float4*>(cs + r * kp + c);
    const float n = kn[r];
    const float* offp = &off.x;
    const float* inp = &in.x;
    const float* exp_ = &ex.x;
    const float* qp = &q.x;
    const float* kq = &k.x;
    const float* zp = &z.x;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float bt = offp[e] + inp[e], grow = exp2_fast(-bt), u = kq[e] * n;
      const float rate = sigmoid_f32(zp[e] + (a.rate_bias && c + e < dk ? a.rate_bias[h * dk + c + e] : 0.f));
      (&nq[it].x)[e] = qp[e] * a.q_scale * exp2_fast(bt);
      (&nu[it].x)[e] = u * exp2_fast(offp[e] + exp_[e]);
      (&nk[it].x)[e] = kq[e] * grow;
      (&nc[it].x)[e] = rate * u * grow;
    }
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kGeneralItems; ++it) {
    const int w = tid + it * kPrepThreads, r = w / quads, c = w % quads * 4;
    if (r >= C) continue;
    *reinterpret_cast<float4*>(qs + r * kp + c) = nq[it];
    *reinterpret_cast<float4*>(us + r * kp + c) = nu[it];
    *reinterpret_cast<float4*>(ks + r * kp + c) = nk[it];
    *reinterpret_cast<float4*>(cs + r * kp + c) = nc[it];
  }
  __syncthreads();

  // ---- tile (I, J) of the four products, against k in one wave and against c in another: lane
  // (quarter, x) holds row x of block I against tokens 4 quarter + r of block J
  for (int item = wave; item < NB * (NB + 1); item += kPrepWaves) {
    const bool with_k = item & 1;
    int I = 0, J = item >> 1;
    while (J > I) J -= ++I;
    const int t = 16 * I + x16, s = 16 * J + x16;
    const float* right = with_k ? ks : cs;
    rc_f32x4 aq = {0.f, 0.f, 0.f, 0.f}, au = {0.f, 0.f, 0.f, 0.f};
    for (int j = 0; j < sp.kt; ++j) {
      const int c = 16 * j + 4 * quarter;
      const float4 kk = *reinterpret_cast<const float4*>(right + s * kp + c);
      const float4 qt = *reinterpret_cast<const float4*>(qs + t * kp + c);
      const float4 ut = *reinterpret_cast<const float4*>(us + t * kp + c);
      aq = mfma4(kk, rc_f32x4{qt.x, qt.y, qt.z, qt.w}, aq);
      au = mfma4(kk, rc_f32x4{ut.x, ut.y, ut.z, ut.w}, au);
    }
    float4 q4, u4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int sr = 16 * J + 4 * quarter + r;
      (&q4.x)[r] = sr <= t ? aq[r] : 0.f;
      (&u4.x)[r] = sr < t ? (with_k ? au[r] : -au[r]) : 0.f;
    }
    const int at = (I * NB + J) * 256 + lane * 4;
    if (with_k) {
      *reinterpret_cast<float4*>(ak + at) = q4;
      *reinterpret_cast<float4*>(mk + at) = u4;
    } else {
      *reinterpret_cast<float4*>(ws + sp.aqk() + at) = q4;
      *reinterpret_cast<float4*>(lk + at) = u4;
    }
  }

  // ---- Q^ and C^T fragments, the chunk's total decay
  auto total = [&](int c) __attribute__((always_inline)) {
    float s = 0.f;
#pragma unroll
    for (int m = 0; m < NB; ++m) s += tot[m * dkp + c];
    return exp2_fast(s);
  };
  for (int item = wave; item < 2 * NB * sp.kt; item += kPrepWaves) {
    const bool is_q = item < NB * sp.kt;
    const int w = is_q ? item : item - NB * sp.kt;
    if (is_q) {
      const int rt = w / sp.kt, ct = w % sp.kt;
      *reinterpret_cast<float4*>(ws + sp.q() + (rt * sp.kt + ct) * 256 + lane * 4) =
          *reinterpret_cast<const float4*>(qs + (16 * rt + x16) * kp + 16 * ct + 4 * quarter);
    } else {
      const int ct = w / NB, rt = w % NB;
      const int c = 16 * ct + x16;
      const float after = total(c);
      float4 o;
#pragma unroll
      for (int r = 0; r < 4; ++r) (&o.x)[r] = cs[(16 * rt + 4 * quarter + r) * kp + c] * after;
      *reinterpret_cast<float4*>(ws + sp.kT() + (ct * NB + rt) * 256 + lane * 4) = o;
    }
  }
  for (int c = tid; c < dkp; c += kPrepThreads) ws[sp.gamma() + c] = total(c);
  __syncthreads();

  if (wave < NB) invert_diagonal(lk + (wave * NB + wave) * 256, x16, quarter);
  if (late_v) stage_rows<DT>(a, b, t_first, n_rows, C, a.v_off + h * dv, 2 * a.Hk * dk + h * dv, dv, dvp, vs, vp, vec);
  __syncthreads();

  // ---- a 16-column tile per wave: Ubar with Obar, W, then the tiles of Sbar
  const int solves = sp.vt + sp.kt;
  for (int item = wave; item < solves + sp.kt * sp.vt; item += kPrepWaves) {
    if (item >= solves) {
      const int j = (item - solves) / sp.vt, ct = (item - solves) % sp.vt;
      const int c = 16 * j + x16;
      const float after = total(c);
      rc_f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        float4 k;
        rc_f32x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = 16 * I + 4 * quarter + r;
          (&k.x)[r] = ks[t * kp + c] * after;
          v[r] = vs[t * vp + 16 * ct + x16];
        }
        acc = mfma4(k, v, acc);
      }
      *reinterpret_cast<rc_f32x4*>(ws + sp.s() + (j * sp.vt + ct) * 256 + lane * 4) = acc;
      continue;
    }
    const bool is_v = item < sp.vt;
    const int ct = is_v ? item : item - sp.vt;
    const int c = 16 * ct + x16;
    rc_f32x4 X[NB], B[NB];
#pragma unroll
    for (int I = 0; I < NB; ++I)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int t = 16 * I + 4 * quarter + r;
        B[I][r] = is_v ? vs[t * vp + c] : us[t * kp + c];
      }
#pragma unroll
    for (int I = 0; I < NB; ++I) {
      rc_f32x4 acc = {0.f, 0.f, 0.f, 0.f}, o = {0.f, 0.f, 0.f, 0.f};
      if (is_v) {
#pragma unroll
        for (int J = 0; J <= I; ++J) {
          acc = mfma4(*reinterpret_cast<const float4*>(mk + (I * NB + J) * 256 + lane * 4), B[J], acc);
          o = mfma4(*reinterpret_cast<const float4*>(ak + (I * NB + J) * 256 + lane * 4), B[J], o);
        }
        *reinterpret_cast<rc_f32x4*>(ws + sp.o() + (I * sp.vt + ct) * 256 + lane * 4) = o;
      } else {
        acc = B[I];
      }
#pragma unroll
      for (int J = 0; J < I; ++J)
        acc = mfma4(*reinterpret_cast<const float4*>(lk + (I * NB + J) * 256 + lane * 4), X[J], acc);
      X[I] = mfma4(*reinterpret_cast<const float4*>(lk + (I * NB + I) * 256 + lane * 4), acc, rc_f32x4{0.f, 0.f, 0.f, 0.f});
      if (is_v) {
        *reinterpret_cast<rc_f32x4*>(ws + sp.u() + (I * sp.vt + ct) * 256 + lane * 4) = -X[I];
      } else {
        float* w = ws + sp.w() + (I * sp.kt + ct) * 256;
#pragma unroll
        for (int r = 0; r < 4; ++r) w[((x16 >> 2) * 16 + 4 * quarter + r) * 4 + (x16 & 3)] = X[I][r];
      }
    }
  }
}

constexpr int kScanThreads = 512;
constexpr int kScanWaves = 4;     // of either kind

// The chunks of one (16 value columns, head, sequence) in order, by two kinds of waves, one of each on a SIMD:
//  * wave w of the first four has state tiles w, w + 4, ... and, with the delta rule, row block w of U = Ubar - W S;
//  * wave w of the others reads row block w out, O = Q^ S + Aqk U, which nothing later waits for: it takes S and U into
//    registers as soon as they are there and works a barrier behind the first kind, whose waits its products fill.
// S and (DELTA) U pass through LDS, S in two copies so that one is read while the next is written; without the delta
// rule U is what the preparation left, and a chunk has one barrier instead of two.  KT: 16-row state tiles.
// EXTRA: rule 1's additions to the read-outs and the state.
// The chain state -> U -> state bounds it: its products are dependent, with an LDS exchange after each half.  Four waves
// that did both, fragments one chunk ahead, took 245 us for 5000 tokens x 16 heads x 128 key channels with the delta rule and
// 116 for 64 without; these 204 and 108 (eight waves alone 229 and 127, with fragments two chunks ahead 212 and 109, with a
// chunk's state tiles asked for together and the first kind's products first the rest).  Read-outs a barrier behind: 32
// chunks of 16 heads of 128 x 128 with the delta rule 70.8 -> 66.9 us, of 64 x 128 without 40.0 -> 39.0.  Two accumulators in turn
// for every chain: 69.3.  Parts of it left out, under a tracer and with one head of keys for all (70.8): without the matrix products 42,
// without the fragments' loads 65, without the read-outs 44; without the delta rule 38.7: 23.8, 36.8, 18.5.
template <int KT, int NB, bool DELTA, bool EXTRA>
__global__ __launch_bounds__(kScanThreads, 2) void recurrence_scan_kernel(socket_recurrence a, int n_chunks) {
  constexpr int C = 16 * NB;
  constexpr int OWN = (KT + kScanWaves - 1) / kScanWaves;
  __shared__ __attribute__((aligned(16))) float s_lds[2][KT * 256];
  __shared__ __attribute__((aligned(16))) float u_lds[DELTA ? 1 : 2][NB * 256];
  // workgroups go to the XCDs round-robin by id: the slices of one (sequence, head) share an
  // XCD (whose L2 then serves their common W, Q^ and K^T) when the heads are a multiple of 8
  const int bh_n = a.B * a.H;
  const int slice = blockIdx.x / bh_n, bh = blockIdx.x % bh_n;
  const int h = bh % a.H, b = bh / a.H;
  const int lane = threadIdx.x & 63, id = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = id & (kScanWaves - 1);
  const bool reads_out = id >= kScanWaves;
  const int x16 = lane & 15, quarter = lane >> 4;
  const ChunkSpace sp{(a.dk + 15) / 16, (a.dv + 15) / 16, NB, EXTRA};
  const int kt = sp.kt;
  const int col = 16 * slice + x16;
  const bool col_ok = col < a.dv;
  const bool rows_mine = wave < NB;
  const int wb = rows_mine ? wave : 0;
  const float* ws = (const float*)a.workspace + (int64_t)bh * n_chunks * sp.size();
  const uint32_t l4 = lane * 4;
  auto tile = [&](const float* at) __attribute__((always_inline)) { return *reinterpret_cast<const float4*>(at + l4); };
  auto acc_tile = [&](const float* at) __attribute__((always_inline)) { return *reinterpret_cast<const rc_f32x4*>(at + l4); };
  // Loads return in the order of their requests, and a wait counts those made since: the first chunks' are made in the
  // order in which the loop makes them (the compiler, left to itself, mixed them and waited in the loop for all).
  auto in_order = [] __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
  auto chunk_at = [&](int n) __attribute__((always_inline)) { return ws + (int64_t)min(n, n_chunks - 1) * sp.size(); };
  // A fragment's registers take a later chunk's as soon as it has been used: every load has the time of two chunks to
  // arrive (where registers hold two, one chunk otherwise).
  constexpr int SETS = NB == 4 ? 2 : 1;

  if (reads_out) {
    float4 fq[SETS][KT], fa[SETS][NB];
    rc_f32x4 fo[SETS] = {};
    auto q_tile = [&](const float* c, int j) __attribute__((always_inline)) {
      return tile(c + sp.q() + (wb * kt + (j < kt ? j : kt - 1)) * 256);     // (tiles past dk meet zero state)
    };
    auto a_tile = [&](const float* c, int J) __attribute__((always_inline)) {
      return tile(c + sp.aqk() + (wb * NB + (J <= wb ? J : wb)) * 256);
    };
#pragma unroll
    for (int p = 0; p < SETS; ++p) {
      const float* c = chunk_at(p);
#pragma unroll
      for (int j = 0; j < KT; ++j) fq[p][j] = q_tile(c, j);
      in_order();
      if (EXTRA) fo[p] = acc_tile(c + sp.o() + (wb * sp.vt + slice) * 256);
#pragma unroll
      for (int J = 0; J < NB; ++J) fa[p][J] = a_tile(c, J);
      in_order();
    }
    rc_f32x4 x[KT], u[NB];
    auto take_state = [&](const float* from) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < KT; ++j) x[j] = acc_tile(from + j * 256);
    };
    auto take_u = [&](const float* from) __attribute__((always_inline)) {
#pragma unroll
      for (int J = 0; J < NB; ++J) u[J] = acc_tile(from + J * 256);
    };
    __syncthreads();   // the first state
    if (rows_mine) {
      take_state(s_lds[0]);
      if (!DELTA) take_u(u_lds[0]);
    }
    __syncthreads();   // the first U; without the delta rule the second state
    auto chunk = [&](int n, auto half) __attribute__((always_inline)) {
      constexpr int at = decltype(half)::value, p = at % SETS, next = DELTA ? 0 : at ^ 1;
      const float* nx = chunk_at(n + SETS);
      const bool more = n + 1 < n_chunks;
      rc_f32x4 o = fo[p];
      if (rows_mine) {
#pragma unroll
        for (int j = 0; j < KT; ++j) {
          o = mfma4(fq[p][j], x[j], o);
          fq[p][j] = q_tile(nx, j);
        }
        if (EXTRA) fo[p] = acc_tile(nx + sp.o() + (wb * sp.vt + slice) * 256);
        in_order();
        if (DELTA) take_u(u_lds[0]);
      }
      if (DELTA) __syncthreads();   // the next state complete, this U read
      if (rows_mine) {
#pragma unroll
        for (int J = 0; J < NB; ++J) {
          if (J <= wave) o = mfma4(fa[p][J], u[J], o);
          fa[p][J] = a_tile(nx, J);
        }
        in_order();
        if (more) {
          take_state(s_lds[at ^ 1]);
          if (!DELTA) take_u(u_lds[next]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int t = n * C + 16 * wave + 4 * quarter + r;
          if (t < a.n && col_ok) a.o_buf[(((int64_t)b * a.n + t) * a.H + h) * a.dv + col] = o[r];
        }
      }
      if (more) __syncthreads();   // the next U complete, without the delta rule the state after the next; those taken read
    };
    for (int n = 0; n + 1 < n_chunks; n += 2) {
      chunk(n, std::integral_constant<int, 0>{});
      chunk(n + 1, std::integral_constant<int, 1>{});
    }
    if (n_chunks & 1) chunk(n_chunks - 1, std::integral_constant<int, 0>{});
    return;
  }

  float* Sg = a.state + (int64_t)bh * a.dk * a.dv;
  rc_f32x4 S[OWN];
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int j = wave + i * kScanWaves;
    S[i] = rc_f32x4{0.f, 0.f, 0.f, 0.f};
    if (!a.fresh && j < kt && col_ok) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * j + 4 * quarter + r;
        if (row < a.dk) S[i][r] = Sg[(int64_t)row * a.dv + col];
      }
    }
    if (j < KT) {
      *reinterpret_cast<rc_f32x4*>(s_lds[0] + j * 256 + lane * 4) = S[i];
      if (j >= kt) *reinterpret_cast<rc_f32x4*>(s_lds[1] + j * 256 + lane * 4) = S[i];   // (zero, and written by nobody later)
    }
  }
  float4 fw[SETS][DELTA ? KT : 1], fk[SETS][OWN][NB], fg[SETS][OWN];
  rc_f32x4 fu[2], fs[SETS][EXTRA ? OWN : 1];
  auto w_tile = [&](const float* c, int j) __attribute__((always_inline)) {
    return tile(c + sp.w() + (wb * kt + (j < kt ? j : kt - 1)) * 256);
  };
  auto own = [&](int i) __attribute__((always_inline)) { return min(wave + i * kScanWaves, kt - 1); };
  auto k_tile = [&](const float* c, int i, int I) __attribute__((always_inline)) { return tile(c + sp.kT() + (own(i) * NB + I) * 256); };
  auto gammas = [&](const float* c, int i) __attribute__((always_inline)) {
    return *reinterpret_cast<const float4*>(c + sp.gamma() + 16 * own(i) + (uint32_t)(4 * quarter));
  };
  auto u_tile = [&](const float* c) __attribute__((always_inline)) { return acc_tile(c + sp.u() + (wb * sp.vt + slice) * 256); };
  auto publish = [&](float* to, const rc_f32x4& u) __attribute__((always_inline)) {
    if (rows_mine) *reinterpret_cast<rc_f32x4*>(to + wave * 256 + lane * 4) = u;
  };
  auto s_tile = [&](const float* c, int i) __attribute__((always_inline)) { return acc_tile(c + sp.s() + (own(i) * sp.vt + slice) * 256); };
#pragma unroll
  for (int p = 0; p < SETS; ++p) {
    const float* c = chunk_at(p);
    if (DELTA) {
#pragma unroll
      for (int j = 0; j < KT; ++j) fw[p][j] = w_tile(c, j);
      in_order();
    }
    if (DELTA) fu[p] = u_tile(c);
    in_order();
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      fg[p][i] = gammas(c, i);
      if (EXTRA) fs[p][i] = s_tile(c, i);
#pragma unroll
      for (int I = 0; I < NB; ++I) fk[p][i][I] = k_tile(c, i, I);
      in_order();
    }
  }
  if (!DELTA) {
    publish(u_lds[0], u_tile(ws));
    fu[1] = u_tile(chunk_at(1));
    fu[0] = u_tile(chunk_at(2));
  }
  __syncthreads();   // the first state
  __builtin_amdgcn_s_setprio(1);   // (the other kind's products go where these leave the matrix core free)
  auto chunk = [&](int n, auto half) __attribute__((always_inline)) {
    constexpr int at = decltype(half)::value, p = at % SETS;
    const float* nx = chunk_at(n + SETS);
    const float* Sn = s_lds[at];
    rc_f32x4 ub[NB];
    if constexpr (DELTA) {
      if (rows_mine) {
        rc_f32x4 y = {0.f, 0.f, 0.f, 0.f}, x[KT];
#pragma unroll
        for (int j = 0; j < KT; ++j) x[j] = acc_tile(Sn + j * 256);
        __builtin_amdgcn_sched_barrier(0);     // (every tile asked for before the first product)
#pragma unroll
        for (int j = 0; j < KT; ++j) {
          y = mfma4(fw[p][j], x[j], y);
          fw[p][j] = w_tile(nx, j);
        }
        rc_f32x4 u = fu[p];
#pragma unroll
        for (int r = 0; r < 4; ++r) u[r] -= y[r];
        publish(u_lds[0], u);
        in_order();
        fu[p] = u_tile(nx);
      }
      __syncthreads();   // U complete
    } else {
      // (U comes from memory: the next chunk's is laid down beside this one's)
      publish(u_lds[DELTA ? 0 : at ^ 1], fu[at ^ 1]);
      in_order();
      fu[at ^ 1] = u_tile(chunk_at(n + 3));
    }
#pragma unroll
    for (int I = 0; I < NB; ++I) ub[I] = acc_tile(u_lds[DELTA ? 0 : at] + I * 256);
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
      const int j = wave + i * kScanWaves;
      S[i][0] *= fg[p][i].x;
      S[i][1] *= fg[p][i].y;
      S[i][2] *= fg[p][i].z;
      S[i][3] *= fg[p][i].w;
      fg[p][i] = gammas(nx, i);
      if (EXTRA) {
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] += fs[p][i][r];
        fs[p][i] = s_tile(nx, i);
      }
#pragma unroll
      for (int I = 0; I < NB; ++I) {
        S[i] = mfma4(fk[p][i][I], ub[I], S[i]);
        fk[p][i][I] = k_tile(nx, i, I);
      }
      if (j < kt) *reinterpret_cast<rc_f32x4*>(s_lds[at ^ 1] + j * 256 + lane * 4) = S[i];
    }
    __syncthreads();   // the next state complete, U and this one read
  };
  for (int n = 0; n + 1 < n_chunks; n += 2) {
    chunk(n, std::integral_constant<int, 0>{});
    chunk(n + 1, std::integral_constant<int, 1>{});
  }
  if (n_chunks & 1) chunk(n_chunks - 1, std::integral_constant<int, 0>{});
#pragma unroll
  for (int i = 0; i < OWN; ++i) {
    const int j = wave + i * kScanWaves;
    if (j < kt && col_ok) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * j + 4 * quarter + r;
        if (row < a.dk) Sg[(int64_t)row * a.dv + col] = S[i][r];
      }
    }
  }
}

// The read-outs' norm and gate: LPH lanes per (token, head), V neighbouring values each and
// LPH * V apart.
template <class DT, int LPH, int V>
__global__ __launch_bounds__(256) void recurrence_out_kernel(socket_recurrence a) {
  const int sub = threadIdx.x % LPH;
  const int64_t w = (int64_t)blockIdx.x * (256 / LPH) + threadIdx.x / LPH;
  const bool live = w < (int64_t)a.B * a.n * a.H;    // (every lane takes part in the sum)
  const int64_t wl = live ? w : 0;
  const int h = (int)(wl % a.H), dv = a.dv;
  const int64_t bt = wl / a.H;
  const int t = (int)(bt % a.n), b = (int)(bt / a.n);
  const float* o = a.o_buf + wl * dv;
  float ss = 0.f;
  for (int c = sub * V; c < dv; c += LPH * V) {
    float x[V];
    load_vec<DType_f32, V>(o, c, x);
#pragma unroll
    for (int e = 0; e < V; ++e) ss = fmaf(x[e], x[e], ss);
  }
  const float rs = rsqrt_f32(group_sum<LPH>(ss) / (float)dv + a.eps);
  if (!live) return;
  const int64_t dst = ((int64_t)b * a.T + a.t0 + t) * a.H * dv + (int64_t)h * dv;
  const int64_t gsrc = a.gate_w ? dst : b * a.proj_stride_b + (a.t0 + t) * a.proj_stride_t + a.gate_off + h * dv;
  for (int c = sub * V; c < dv; c += LPH * V) {
    float x[V], g[V], nw[V];
    load_vec<DType_f32, V>(o, c, x);
    load_vec<DT, V>(a.gate_w ? a.gate_z : a.proj, gsrc + c, g);
    load_vec<DType_f32, V>(a.norm_w, (a.norm_per_head ? h * dv : 0) + c, nw);
#pragma unroll
    for (int e = 0; e < V; ++e) x[e] = x[e] * rs * nw[e] * gate_act(a.gate_kind, g[e]);
    store_vec<DT, V>(a.out, dst + c, x);
  }
}

// The last taps - 1 inputs of a portion (older ones from the state where the portion is shorter).
// One lane per channel, rows in ascending order: row m reads row m + T of the same half at most.
template <class DT>
__global__ __launch_bounds__(256) void conv_tail_kernel(socket_recurrence a) {
  const int C = conv_channels(a), ch = blockIdx.x * 256 + threadIdx.x, b = blockIdx.y;
  if (ch >= C) return;
  const int qk = a.Hk * a.dk, n1 = a.taps - 1;
  const int col = ch < qk ? a.q_off + ch : (ch < 2 * qk ? a.k_off + ch - qk : a.v_off + ch - 2 * qk);
  const int64_t from = ((int64_t)(a.pos0 & 1) * a.B + b) * n1 * C + ch;
  const int64_t to = ((int64_t)((a.pos0 + a.T) & 1) * a.B + b) * n1 * C + ch;
  for (int m = 0; m < n1; ++m) {
    const int t = a.T - n1 + m;
    float x = 0.f;
    if (t >= 0) x = load_elem<DT>(a.proj, b * a.proj_stride_b + t * a.proj_stride_t + col);
    else if (!a.fresh) x = load_elem<DT>(a.conv_state, from + (int64_t)(t + n1) * C);
    store_elem<DT>(a.conv_state, to + (int64_t)m * C, x);
  }
}

template <class DT>
__global__ __launch_bounds__(256) void tanh_rows_kernel(const void* x, int64_t x_stride, void* y, int64_t items, int cols) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < items) store_elem<DT>(y, i, tanh_f32(load_elem<DT>(x, i / cols * x_stride + i % cols)));
}

int chunk_blocks(int dk, int rule) { return dk <= (rule == 1 ? 64 : 128) ? 4 : 2; }

int check_recurrence(const socket_recurrence* p) {
  SOCKET_REQUIRE(p && p->proj && p->state && p->out && p->norm_w, SOCKET_ERR_NULL);
  const socket_recurrence& a = *p;
  SOCKET_REQUIRE(a.dtype == SOCKET_F32 || a.dtype == SOCKET_BF16, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(a.B > 0 && a.B <= 65535 && a.T > 0 && a.H > 0 && a.H <= 65535 && a.Hk > 0 && a.H % a.Hk == 0 && a.dk > 0 && a.dv > 0,
                 SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(a.dk <= 256 && a.dv <= 256, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE((a.taps < 1 || a.conv_w) && (a.taps <= 1 || a.conv_state), SOCKET_ERR_NULL);
  SOCKET_REQUIRE(a.taps >= 0 && a.taps <= 32, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(a.rule == 0 || a.rule == 1, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(a.rule == 1 ? a.decay_kind == 2 : (a.decay_kind == 0 || a.decay_kind == 1) && !a.decay_tanh, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(a.rule == 0 || (a.H == a.Hk && a.taps == 0 && !a.gate_w && a.decay_tanh && a.rate_off >= 0), SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(a.rule == 0 || (a.decay_rate >= 0.f && a.decay_rate * kRcLog2e * 16 * chunk_blocks(a.dk, 1) <= kMaxChunkDecay),
                 SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(a.gate_kind == 0 || a.gate_kind == 1, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(a.decay_kind != 0 || a.a_log, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(socket_aligned16(a.state) && socket_aligned16(a.proj), SOCKET_ERR_ALIGN);
  return SOCKET_OK;
}

template <class DT>
int launch_step(const socket_recurrence& a, hipStream_t s) {
  const int vec = a.dv % 4 == 0 ? 4 : 1;
  const int nc = a.dv / vec;
  // lanes enough to hold the state in at most 16 registers each where 1024 allow it
  int nt = 256;
  auto rows_of = [&](int n) { const int rg = n / nc; return (a.dk + rg - 1) / rg; };
  const int want = 16 / vec;
  while (nt < 1024 && rows_of(nt) > want) nt *= 2;
  const int rows = rows_of(nt);
  StepShape sh{nc, -1, nt / nc};
  if ((nc & (nc - 1)) == 0)
    for (sh.nc_shift = 0; (1 << sh.nc_shift) < nc; ++sh.nc_shift) {}
  const bool general = a.rule == 1;
  const size_t lds = (size_t)((general ? 4 : 3) * a.dk + 3 * a.dv + 16 + sh.RG * a.dv) * 4;
  SOCKET_REQUIRE(lds <= 48 * 1024, SOCKET_ERR_UNSUPPORTED);
  const dim3 grid((unsigned)(a.H / a.Hk), (unsigned)a.Hk, (unsigned)a.B), block((unsigned)nt);
#define SOCKET_STEP(V, R)                                                                                        \
  do {                                                                                                           \
    if (general) hipLaunchKernelGGL((recurrence_step_kernel<DT, V, R, true>), grid, block, lds, s, a, sh);       \
    else hipLaunchKernelGGL((recurrence_step_kernel<DT, V, R, false>), grid, block, lds, s, a, sh);              \
  } while (0)
  if (vec == 4) {
    if (rows <= 4) SOCKET_STEP(4, 4);
    else if (rows <= 8) SOCKET_STEP(4, 8);
    else if (rows <= 16) SOCKET_STEP(4, 16);
    else return SOCKET_ERR_UNSUPPORTED;
  } else {
    if (rows <= 16) SOCKET_STEP(1, 16);
    else if (rows <= 32) SOCKET_STEP(1, 32);
    else if (rows <= 64) SOCKET_STEP(1, 64);
    else return SOCKET_ERR_UNSUPPORTED;
  }
#undef SOCKET_STEP
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

template <class DT, int NB, bool DELTA>
int launch_prep(const socket_recurrence& a, int n_chunks, bool vec, hipStream_t s) {
  constexpr int C = 16 * NB;
  constexpr size_t kStatic = 64;
  const ChunkSpace sp{(a.dk + 15) / 16, (a.dv + 15) / 16, NB};
  const int dkp = sp.kt * 16, dvp = sp.vt * 16, kp = dkp + 4, vp = dvp + 4;
  const size_t limit = (size_t)socket_device_limits().max_lds_per_block;
  const size_t fixed = (size_t)(C * kp + NB * dkp + C + (DELTA ? NB * NB * 256 : 0)) * 4, qk = (size_t)2 * C * kp * 4;
  // what shares LDS with V once it is through: q, or q and k where nothing reads k after the fragments
  const size_t over = (size_t)(DELTA ? C * kp : 2 * C * kp) * 4, v = (size_t)C * vp * 4;
  const int own_v = DELTA && dvp <= kPrepThreads / C * 8 && fixed + qk + v + kStatic <= limit ? 1 : 0;
  const size_t lds = fixed + qk + (own_v ? v : v > over ? v - over : 0);
  SOCKET_REQUIRE(lds + kStatic <= limit, SOCKET_ERR_UNSUPPORTED);
  auto kern = recurrence_prep_kernel<DT, NB, DELTA>;
  if (lds > 48 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return SOCKET_ERR_LAUNCH;
  const unsigned heads = (unsigned)a.H, chunks = (unsigned)n_chunks;
  const bool heads_first = n_chunks <= kPrepHeadsFirst;
  const dim3 grid(heads_first ? heads : chunks, heads_first ? chunks : heads, (unsigned)a.B);
  hipLaunchKernelGGL(kern, grid, dim3(kPrepThreads), lds, s, a, n_chunks, vec ? 1 : 0, own_v);
  return SOCKET_OK;
}

template <class DT, int NB>
int launch_prep(const socket_recurrence& a, int n_chunks, bool vec, bool delta, hipStream_t s) {
  return delta ? launch_prep<DT, NB, true>(a, n_chunks, vec, s) : launch_prep<DT, NB, false>(a, n_chunks, vec, s);
}

template <class DT, int NB>
int launch_general_prep(const socket_recurrence& a, int n_chunks, bool vec, hipStream_t s) {
  constexpr int C = 16 * NB;
  const int dkp = (a.dk + 15) / 16 * 16, dvp = (a.dv + 15) / 16 * 16;
  const size_t limit = (size_t)socket_device_limits().max_lds_per_block, own_v = (size_t)C * (dvp + 4) * 4;
  size_t lds = (size_t)(4 * C * (dkp + 4) + NB * dkp + 3 * NB * NB * 256 + C) * 4;
  const int late_v = lds + own_v > limit && dvp <= dkp ? 1 : 0;
  if (!late_v) lds += own_v;
  SOCKET_REQUIRE(lds <= limit, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(C * dkp / 4 <= kGeneralItems * kPrepThreads, SOCKET_ERR_UNSUPPORTED);
  auto kern = general_prep_kernel<DT, NB>;
  if (lds > 48 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return SOCKET_ERR_LAUNCH;
  hipLaunchKernelGGL(kern, dim3((unsigned)n_chunks, (unsigned)a.H, (unsigned)a.B), dim3(kPrepThreads), lds, s, a, vec ? 1 : 0,
                     late_v);
  return SOCKET_OK;
}

template <int NB, bool DELTA, bool EXTRA = false>
int launch_scan(const socket_recurrence& a, int n_chunks, hipStream_t s) {
  const int kt = (a.dk + 15) / 16, slices = (a.dv + 15) / 16;
  const dim3 grid((unsigned)((int64_t)slices * a.B * a.H)), block(kScanThreads);
#define SOCKET_SCAN(KT) hipLaunchKernelGGL((recurrence_scan_kernel<KT, NB, DELTA, EXTRA>), grid, block, 0, s, a, n_chunks)
  if constexpr (NB == 4) {
    if (kt <= 2) SOCKET_SCAN(2);
    else if (kt <= 4) SOCKET_SCAN(4);
    else if (kt <= 6) SOCKET_SCAN(6);
    else SOCKET_SCAN(8);
  } else {
    if (EXTRA && kt <= 8) SOCKET_SCAN(8);
    else if (kt <= 12) SOCKET_SCAN(12);
    else SOCKET_SCAN(16);
  }
#undef SOCKET_SCAN
  return SOCKET_OK;
}

}  // namespace

extern "C" int socket_recurrence_step(const socket_recurrence* args, void* stream) {
  const int rc = check_recurrence(args);
  if (rc != SOCKET_OK) return rc;
  const socket_recurrence& a = *args;
  SOCKET_REQUIRE(a.pos && a.decay_w && a.decay_rank > 0, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(a.T == 1 && !a.fresh, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(!a.gate_w || a.gate_rank > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(socket_aligned16(a.decay_w) && (!a.gate_w || socket_aligned16(a.gate_w)), SOCKET_ERR_ALIGN);
  hipStream_t s = (hipStream_t)stream;
  return a.dtype == SOCKET_F32 ? launch_step<DType_f32>(a, s) : launch_step<DType_bf16>(a, s);
}

extern "C" int socket_recurrence_chunk(int dk, int rule) { return 16 * chunk_blocks(dk, rule); }

extern "C" size_t socket_recurrence_workspace_bytes(int B, int n, int H, int dk, int dv, int rule) {
  if (B <= 0 || n <= 0 || H <= 0 || dk <= 0 || dv <= 0) return 0;
  const int nb = chunk_blocks(dk, rule), C = 16 * nb;
  const ChunkSpace sp{(dk + 15) / 16, (dv + 15) / 16, nb, rule == 1};
  return (size_t)B * H * ((n + C - 1) / C) * sp.size() * sizeof(float);
}

extern "C" int socket_recurrence_scan(const socket_recurrence* args, void* stream) {
  const int rc = check_recurrence(args);
  if (rc != SOCKET_OK) return rc;
  const socket_recurrence& a = *args;
  SOCKET_REQUIRE(a.decay_z && a.o_buf && a.workspace && (!a.gate_w || a.gate_z), SOCKET_ERR_NULL);
  SOCKET_REQUIRE(a.t0 >= 0 && a.n > 0 && a.t0 + a.n <= a.T && a.pos0 >= 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(a.workspace_bytes >= socket_recurrence_workspace_bytes(a.B, a.n, a.H, a.dk, a.dv, a.rule), SOCKET_ERR_WORKSPACE);
  SOCKET_REQUIRE(socket_aligned16(a.workspace), SOCKET_ERR_ALIGN);
  hipStream_t s = (hipStream_t)stream;
  const int nb = chunk_blocks(a.dk, a.rule), C = 16 * nb, n_chunks = (a.n + C - 1) / C;
  const int per = 8;
  const bool vec = a.dk % 8 == 0 && a.dv % 8 == 0 && a.q_off % per == 0 && a.k_off % per == 0 && a.v_off % per == 0 &&
                   a.proj_stride_b % per == 0 && a.proj_stride_t % per == 0 &&
                   (a.taps < 1 || socket_aligned16(a.conv_w)) && (a.taps <= 1 || socket_aligned16(a.conv_state));
  const bool delta = a.beta_off >= 0;
  int st;
  if (a.rule == 1) {
    if (nb == 4)
      st = a.dtype == SOCKET_F32 ? launch_general_prep<DType_f32, 4>(a, n_chunks, vec, s)
                                 : launch_general_prep<DType_bf16, 4>(a, n_chunks, vec, s);
    else
      st = a.dtype == SOCKET_F32 ? launch_general_prep<DType_f32, 2>(a, n_chunks, vec, s)
                                 : launch_general_prep<DType_bf16, 2>(a, n_chunks, vec, s);
  } else if (nb == 4)
    st = a.dtype == SOCKET_F32 ? launch_prep<DType_f32, 4>(a, n_chunks, vec, delta, s) : launch_prep<DType_bf16, 4>(a, n_chunks, vec, delta, s);
  else
    st = a.dtype == SOCKET_F32 ? launch_prep<DType_f32, 2>(a, n_chunks, vec, delta, s) : launch_prep<DType_bf16, 2>(a, n_chunks, vec, delta, s);
  if (st != SOCKET_OK) return st;
  SOCKET_LAUNCH_CHECK();
  if (a.rule == 1) st = nb == 4 ? launch_scan<4, true, true>(a, n_chunks, s) : launch_scan<2, true, true>(a, n_chunks, s);
  else if (nb == 4) st = delta ? launch_scan<4, true>(a, n_chunks, s) : launch_scan<4, false>(a, n_chunks, s);
  else st = delta ? launch_scan<2, true>(a, n_chunks, s) : launch_scan<2, false>(a, n_chunks, s);
  if (st != SOCKET_OK) return st;
  SOCKET_LAUNCH_CHECK();
  const int64_t items = (int64_t)a.B * a.n * a.H;
  SOCKET_REQUIRE((items + 3) / 4 < (1LL << 31), SOCKET_ERR_SHAPE);
  const bool v8 = vec && a.gate_off % 8 == 0 && socket_aligned16(a.out) && socket_aligned16(a.o_buf) &&
                  socket_aligned16(a.norm_w) && (!a.gate_w || socket_aligned16(a.gate_z));
#define SOCKET_OUT(DT, LPH, V)                                                                                    \
  hipLaunchKernelGGL((recurrence_out_kernel<DT, LPH, V>), dim3((unsigned)((items + 256 / LPH - 1) / (256 / LPH))), \
                     dim3(256), 0, s, a)
  if (a.dtype == SOCKET_F32) {
    if (v8) SOCKET_OUT(DType_f32, 16, 8);
    else SOCKET_OUT(DType_f32, 64, 1);
  } else {
    if (v8) SOCKET_OUT(DType_bf16, 16, 8);
    else SOCKET_OUT(DType_bf16, 64, 1);
  }
#undef SOCKET_OUT
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

extern "C" int socket_tanh_rows(const void* x, int64_t x_stride, void* y, int dtype, int64_t rows, int cols, void* stream) {
  SOCKET_REQUIRE(x && y, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(dtype == SOCKET_F32 || dtype == SOCKET_BF16, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(rows > 0 && cols > 0 && x_stride >= cols, SOCKET_ERR_SHAPE);
  const int64_t items = rows * cols;
  SOCKET_REQUIRE((items + 255) / 256 < (1LL << 31), SOCKET_ERR_SHAPE);
  const dim3 grid((unsigned)((items + 255) / 256)), block(256);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == SOCKET_F32) hipLaunchKernelGGL((tanh_rows_kernel<DType_f32>), grid, block, 0, s, x, x_stride, y, items, cols);
  else hipLaunchKernelGGL((tanh_rows_kernel<DType_bf16>), grid, block, 0, s, x, x_stride, y, items, cols);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

extern "C" int socket_recurrence_conv_tail(const socket_recurrence* args, void* stream) {
  const int rc = check_recurrence(args);
  if (rc != SOCKET_OK) return rc;
  const socket_recurrence& a = *args;
  if (a.taps <= 1) return SOCKET_OK;
  const int C = 2 * a.Hk * a.dk + a.H * a.dv;
  const dim3 grid((unsigned)((C + 255) / 256), (unsigned)a.B), block(256);
  hipStream_t s = (hipStream_t)stream;
  if (a.dtype == SOCKET_F32) hipLaunchKernelGGL((conv_tail_kernel<DType_f32>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((conv_tail_kernel<DType_bf16>), grid, block, 0, s, a);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}
