// A (b, h) row's attention over a short index list by one workgroup: shared by the launch that reads the list from memory
// (attend.hip) and the one that selects it first (topk.hip).
#pragma once
#include "socket_common.h"

namespace {

__device__ __forceinline__ float fast_exp(float x) { return __expf(x); }

// Merge (m, l, acc) pairs of an online softmax.
template <int E>
__device__ __forceinline__ void merge_state(float& m, float& l, float* acc, float m2, float l2,
                                            const float* acc2) {
  const float nm = fmaxf(m, m2);
  const float s1 = (m == nm) ? 1.f : fast_exp(m - nm);
  const float s2 = (m2 == nm) ? 1.f : fast_exp(m2 - nm);
  l = l * s1 + l2 * s2;
#pragma unroll
  for (int i = 0; i < E; ++i) acc[i] = acc[i] * s1 + acc2[i] * s2;
  m = nm;
}

constexpr int kRowWaves = 16, kRowUnroll = 8;
template <class DT>
constexpr int row_entries(int D) { return kRowWaves * (SOCKET_WAVE / (D / DT::kPer16B)) * kRowUnroll; }

// All kRowWaves waves: softmax(q k^T scale) v over the rows list[0, len) of k / v (base addresses of the row's kv head, element
// strides between rows), entries that are negative or not below kv_rows left out; len <= width <= row_entries<DT>(D).  The
// list may lie in LDS.  `lds` is the caller's alone.  0 / 0 = NaN where nothing is attended, as in the reference.
template <class DT, int D>
__device__ __forceinline__ void row_attend(const typename DT::storage* q, const typename DT::storage* k, int64_t k_ss,
                                           const typename DT::storage* v, int64_t v_ss, const int32_t* list, int len, int width,
                                           int kv_rows, float sm_scale, float (*lds)[D + 2], typename DT::storage* out) {
  constexpr int E = DT::kPer16B, LPR = D / E, RPW = SOCKET_WAVE / LPR;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int slot = lane / LPR, chunk = lane % LPR;
  const typename DT::storage* kbase = k + chunk * E;
  const typename DT::storage* vbase = v + chunk * E;
  const uint4 qw = *reinterpret_cast<const uint4*>(q + chunk * E);
  int idx[kRowUnroll];
#pragma unroll
  for (int u = 0; u < kRowUnroll; ++u) {         // (past the list: its last entry, not live)
    const int e = (u * kRowWaves + wave) * RPW + slot;
    idx[u] = list[min(e, width - 1)];
    if (e >= len || idx[u] >= kv_rows) idx[u] = -1;
  }
  uint4 kr[kRowUnroll], vr[kRowUnroll];
#pragma unroll
  for (int u = 0; u < kRowUnroll; ++u) {
    kr[u] = vr[u] = make_uint4(0, 0, 0, 0);
    if (idx[u] >= 0) {
      kr[u] = *reinterpret_cast<const uint4*>(kbase + (int64_t)idx[u] * k_ss);
      vr[u] = *reinterpret_cast<const uint4*>(vbase + (int64_t)idx[u] * v_ss);
    }
  }
  float qf[E], sc[kRowUnroll], m = -INFINITY, l = 0.f, acc[E];
  unpack16<DT>(qw, qf);
#pragma unroll
  for (int i = 0; i < E; ++i) acc[i] = 0.f;
#pragma unroll
  for (int u = 0; u < kRowUnroll; ++u) {
    float kf[E];
    unpack16<DT>(kr[u], kf);
    float d = fmaf(qf[0], kf[0], qf[1] * kf[1]);
#pragma unroll
    for (int i = 2; i < E; ++i) d = fmaf(qf[i], kf[i], d);
    d = group_sum<LPR>(d);
    sc[u] = idx[u] >= 0 ? d * sm_scale : -INFINITY;
    m = fmaxf(m, sc[u]);
  }
#pragma unroll
  for (int u = 0; u < kRowUnroll; ++u) {
    const float p = idx[u] >= 0 ? fast_exp(sc[u] - m) : 0.f;
    float vf[E];
    unpack16<DT>(vr[u], vf);
    l += p;
#pragma unroll
    for (int i = 0; i < E; ++i) acc[i] += p * vf[i];
  }
  // row slots inside the wave, then the waves through LDS
#pragma unroll
  for (int d = LPR; d < SOCKET_WAVE; d <<= 1) {
    auto partner = [&](float x) { return d == 16 ? lane_xor16(x) : d == 32 ? lane_xor32(x) : __shfl_xor(x, d, SOCKET_WAVE); };
    const float m2 = partner(m), l2 = partner(l);
    float a2[E];
#pragma unroll
    for (int i = 0; i < E; ++i) a2[i] = partner(acc[i]);
    merge_state<E>(m, l, acc, m2, l2, a2);
  }
  if (lane < LPR) {
#pragma unroll
    for (int i = 0; i < E; ++i) lds[wave][chunk * E + i] = acc[i];
    if (chunk == 0) {
      lds[wave][D] = m;
      lds[wave][D + 1] = l;
    }
  }
  __syncthreads();
  if (tid >= D) return;
  float M = -INFINITY, sum = 0.f, val = 0.f;
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) M = fmaxf(M, lds[w][D]);
#pragma unroll
  for (int w = 0; w < kRowWaves; ++w) {
    const float f = lds[w][D] == M ? 1.f : fast_exp(lds[w][D] - M);
    sum += lds[w][D + 1] * f;
    val += lds[w][tid] * f;
  }
  store_elem<DT>(out, tid, val / sum);
}

}  // namespace
