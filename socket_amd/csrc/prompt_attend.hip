// Prompt attention for the head widths that carry most models: 64 and 128 dims, and 128 + 64
// shared dims with 128 value dims, in 16-bit types.  The operands are those of chunk_attend.hip
// (which serves every other shape): chunks of the position axis or one endless chunk, keys of the
// portion from its own rows and older ones from a ring, query heads of a kv head packed as rows.
//
// A workgroup of four waves takes 128 query rows of one kv head, 32 rows per wave.  Both products
// are v_mfma_f32_32x32x16 in the transposed orientation (the query row is the N index: lane x holds
// row x % 32 in every accumulator):
//   S^T[key, row] = K . Q^T,   O^T[dim, row] = V^T . P^T
// so a row's maximum and sum are over a lane's own registers and one lane swap, and the weights a
// lane computes are the operand it has to supply.  K and V tiles of 64 keys go from global memory
// straight into LDS, one tile ahead, in their own [key][dim] order: the 16-byte pieces of a row are
// placed at piece ^ f(key) so that both the K fragments (one row per lane) and the transposing
// reads of V (ds_read_b64_tr_b16: 16 lanes name four keys x 16 dims and receive four keys of one
// dim each) spread over all banks.  No transposition through registers, one barrier per tile.
//
// What bounds it: the matrix pipes and, per score, one exponential (three with a soft cap) and some
// five other vector operations on the same SIMD; two workgroups per CU (64 KB of LDS each, at most
// 256 registers) let one's softmax run beside the other's products.  32 rows per wave: a K fragment
// of 1 KB feeds one 32-cycle product, which is what the LDS delivers.  Measured (causal, bf16, repeated calls; in
// brackets chunk_attend.hip's kernel): 32 heads over 8 kv heads of 128, cap 30, 8000 tokens 795 (1017) us, 660 TFLOP/s;
// 32 heads of 128 + 64 shared dims, 8000 tokens 798 (1538) us, 821; without a cap 6001 tokens 307 us (961 TFLOP/s; 385 us
// within a prompt pass) with weights rounded to 16 bits, 399 (740) in two terms, 495 (596) in three.  A rescale that
// waits until a maximum has grown by 2^8 takes 297 us instead of 307, but then a row's largest weight is rounded (error
// against float64 2.08e-3 instead of 2.02e-3) and depends on the wave's other rows.
#include "mma_tiles.h"

namespace {

constexpr int kPaRows = 32 * kPaWaves;
constexpr float kPaMaxCap = 60.f;   // exp(60) * 2^31 keys < 3.4e38, exp(-60) > 1.2e-38

// D: key dims, D2: dims of a second key segment that all heads share (with it the output may be gated),
// DV: value dims.  TERMS: weights enter the second product as a sum of so many 16-bit numbers; three of bf16 hold all
// 24 bits of a 32-bit weight.  CAPPED: scores pass softcap tanh(s / softcap), which bounds them, so that exp(score) needs no running
// maximum: p = exp(cap - 2 cap / (exp(2 s / cap) + 1)).  POS: token t sees the keys up to positions[t]
// instead of pos0 + t (one endless chunk, a.k_from = 0).
template <class DT, int D, int D2, int DV, int TERMS, bool CAPPED, bool POS>
__global__ __launch_bounds__(64 * kPaWaves, 2) void prompt_attend_kernel(socket_chunk_attention a, const int64_t* positions, int first_round) {
  constexpr int CK = D / 8, CK2 = D2 / 8, CV = DV / 8;            // 16-byte pieces per row
  constexpr int KS = D / 16, KS2 = D2 / 16, DB = DV / 32;
  constexpr int kK2 = kPaKeys * D * 2, kV = kK2 + kPaKeys * D2 * 2, kStage = kV + kPaKeys * DV * 2;   // places in a stage
  extern __shared__ __attribute__((aligned(16))) unsigned char pa_lds[];

  const int Gq = a.H / a.G;
  // kv heads are neighbours in the launch order: with eight of them each XCD's L2 serves one head's
  // keys.  Later tiles see more keys and come first.  Where every workgroup is at work at once, two to a CU (first_round: the
  // tiles that make one for every CU; 0: more or fewer than that), the second ones come shortest first: the CU with the
  // longest tile has the shortest as well, and all end together (2 x 2048 tokens of 16 heads over caches of 4096 to 8192
  // keys, weights in three terms: 335 us with the longest first throughout, 296).
  const int heads = a.G * a.B, tiles = gridDim.x / heads;
  const int hb = blockIdx.x % heads, nth = blockIdx.x / heads;
  const int tile = first_round > 0 && nth >= first_round ? nth - first_round : tiles - 1 - nth;
  const int g = hb % a.G, b = hb / a.G;
  const int64_t R = (int64_t)a.T * Gq, r0 = (int64_t)tile * kPaRows;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 31, half = lane >> 5;

  // (positions as 32-bit offsets from the first key of the tile's first chunk)
  const int64_t base = POS ? 0 : (a.pos0 + r0 / Gq) / a.chunk * a.chunk;
  const int64_t wr0 = min(r0 + wave * 32, R - 1), wr1 = min(r0 + wave * 32 + 31, R - 1);
  int end = (int)(a.pos0 + min(r0 + kPaRows - 1, R - 1) / Gq - base) + 1;   // keys [0, end)
  int iw0 = (int)(a.pos0 + wr0 / Gq - base), iw1 = (int)(a.pos0 + wr1 / Gq - base);
  const int cw0 = iw0 / a.chunk * a.chunk, cw1 = iw1 / a.chunk * a.chunk;   // (base is a chunk's start)
  const bool wave_live = r0 + wave * 32 < R;

  const char* k_new = (const char*)a.k_new + (b * a.k_stride_b + g * a.k_stride_g) * 2;
  const char* v_new = (const char*)a.v_new + (b * a.v_stride_b + g * a.v_stride_g) * 2;
  const char* k_ring = (const char*)a.k_ring + (b * a.ring_stride_b + g * a.ring_stride_g) * 2;
  const char* v_ring = (const char*)a.v_ring + (b * a.ring_stride_b + g * a.ring_stride_g) * 2;
  const char* k2 = D2 ? (const char*)a.k2 + b * a.k2_stride_b * 2 : nullptr;
  const int64_t k_st = a.k_stride_t * 2, v_st = a.v_stride_t * 2, r_ss = a.ring_stride_s * 2, k2_st = a.k2_stride_t * 2;

  uint4 qf[KS + KS2];
  int row_i, row_c;                          // position and chunk start of the lane's row; nothing visible: i < c
  const int64_t r = r0 + wave * 32 + col;
  {
    const bool live = r < R;
    const int64_t t = (live ? r : 0) / Gq;
    row_i = live ? (int)(a.pos0 + t - base) : -1;
    if (POS && live) row_i = (int)max((int64_t)-1, min(positions[t], a.pos0 + a.T - 1));
    row_c = live && !POS ? row_i / a.chunk * a.chunk : 0;
    const uint16_t* q = (const uint16_t*)a.q + b * a.q_stride_b + t * a.q_stride_t + (g * Gq + (live ? r : 0) % Gq) * a.q_stride_h;
#pragma unroll
    for (int ks = 0; ks < KS + KS2; ++ks) qf[ks] = live ? *reinterpret_cast<const uint4*>(q + 16 * ks + 8 * half) : make_uint4(0, 0, 0, 0);
  }
  // (the fragments must have arrived before the first copy is issued: the compiler's own counts
  // do not include the copies and would drain them on every trip)
#pragma unroll
  for (int ks = 0; ks < KS + KS2; ++ks) asm volatile("" ::"v"(qf[ks].x), "v"(qf[ks].y), "v"(qf[ks].z), "v"(qf[ks].w));

  if constexpr (POS) {      // what the tile's and the wave's rows see, from the positions themselves
    int* ends = reinterpret_cast<int*>(pa_lds);
    int lo = row_i < 0 && r >= R ? INT32_MAX : row_i, hi = row_i;
#pragma unroll
    for (int step = 32; step > 0; step >>= 1) {
      lo = min(lo, __shfl_xor(lo, step, 64));
      hi = max(hi, __shfl_xor(hi, step, 64));
    }
    iw0 = __builtin_amdgcn_readfirstlane(lo);
    iw1 = __builtin_amdgcn_readfirstlane(hi);
    if (lane == 0) ends[wave] = hi + 1;
    __syncthreads();
    end = __builtin_amdgcn_readfirstlane(max(max(ends[0], ends[1]), max(ends[2], ends[3])));
    __syncthreads();        // (the places are the first tile's)
  }
  static_assert(kPaWaves == 4, "ends");

  pa_f32x16 o[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) o[db] = pa_f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
  float l = 0.f, m = -INFINITY;
  // (the largest weight: the later terms of small weights would leave fp16's range if it were 1)
  constexpr float kUnit = DT::kEnum == SOCKET_F16 && TERMS > 1 ? 16384.f : 1.f;
  const float c1 = CAPPED ? 2.f * kPaLog2e * a.scale / a.softcap : a.scale * kPaLog2e;
  const float c2 = a.softcap * kPaLog2e;

  // Keys j0 .. j0 + 63 into a stage.  Keys past the end are copies of the last one (a live row; masked below).
  auto copy_keys = [&](int j0, int stage) __attribute__((always_inline)) {
    unsigned char* st = pa_lds + stage * kStage;
    const int64_t first = base + j0;
    if (j0 + kPaKeys <= end && first >= a.k_from) {      // (uniform)
      pa_copy_tile<CK>(k_new + (first - a.k_from) * k_st, k_st, st, wave, lane);
      if constexpr (D2 > 0) pa_copy_tile<CK2>(k2 + first * k2_st, k2_st, st + kK2, wave, lane);
      pa_copy_tile<CV>(v_new + (first - a.k_from) * v_st, v_st, st + kV, wave, lane);
    } else {
      auto pos = [&](int key) { return base + min(j0 + key, end - 1); };
      auto row = [&](int key, const char* fresh, int64_t stride, const char* ring) {
        const int64_t j = pos(key);
        return j >= a.k_from ? fresh + (j - a.k_from) * stride : ring + (j % a.chunk) * r_ss;
      };
      pa_copy_rows<CK>([&](int key) { return row(key, k_new, k_st, k_ring); }, st, wave, lane);
      if constexpr (D2 > 0) pa_copy_rows<CK2>([&](int key) { return k2 + pos(key) * k2_st; }, st + kK2, wave, lane);
      pa_copy_rows<CV>([&](int key) { return row(key, v_new, v_st, v_ring); }, st + kV, wave, lane);
    }
  };

  const int k_swz = pa_swizzle<CK>(col);      // (of K row `col` of a 32-key block)

  if (end > 0) copy_keys(0, 0);
  int stage = 0;
  for (int j0 = 0; j0 < end; j0 += kPaKeys, stage ^= 1) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();     // this tile has landed for every wave, the other stage has been consumed
    if (j0 + kPaKeys < end) copy_keys(j0 + kPaKeys, stage ^ 1);
    if (!wave_live || j0 > iw1 || j0 + kPaKeys - 1 < cw0) continue;   // (wave-uniform)
    const bool open = j0 + kPaKeys - 1 <= iw0 && j0 >= cw1;
    const uint4* kt = reinterpret_cast<const uint4*>(pa_lds + stage * kStage);
    const unsigned char* vt = pa_lds + stage * kStage + kV;

    pa_f32x16 s[2];
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) s[nb] = pa_f32x16{0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int nb = 0; nb < 2; ++nb) s[nb] = PaType<DT>::mfma(kt[(nb * 32 + col) * CK + ((2 * ks + half) ^ k_swz)], qf[ks], s[nb]);
    if constexpr (D2 > 0) {
      const uint4* kt2 = reinterpret_cast<const uint4*>(pa_lds + stage * kStage + kK2);
#pragma unroll
      for (int ks = 0; ks < KS2; ++ks)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
          s[nb] = PaType<DT>::mfma(kt2[(nb * 32 + col) * CK2 + ((2 * ks + half) ^ pa_swizzle<CK2>(col))], qf[KS + ks], s[nb]);
    }

    // register i of block nb: key j0 + 32 nb + 8 (i / 4) + 4 half + i % 4
    if (!open) {
      const int first = j0 + 4 * half;
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const int j = first + 32 * nb + 8 * (i >> 2) + (i & 3);
          if (!(j <= row_i && j >= row_c)) s[nb][i] = -INFINITY;
        }
    }
    if constexpr (CAPPED) {
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          const float t = __builtin_amdgcn_exp2f(s[nb][i] * c1);
          float p = __builtin_amdgcn_exp2f(fmaf(-2.f * c2, __builtin_amdgcn_rcpf(t + 1.f), c2));
          if (!open && s[nb][i] == -INFINITY) p = 0.f;
          s[nb][i] = p;
          l += p;
        }
    } else {
      float mb = s[0][0];
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) mb = fmaxf(mb, s[nb][i]);
      mb = fmaxf(mb, lane_xor32(mb)) * c1;      // (c1 > 0)
      // The shift is the row's own maximum so far, whatever the wave's other rows do: the largest weight is a power of two, which
      // rounds exactly, and lanes whose maximum stays multiply by 1.
      const float mn = fmaxf(m, mb);
      if (__builtin_amdgcn_ballot_w64(mn > m) != 0) {
        const float alpha = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(m - mn);
        m = mn;
        l *= alpha;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
          for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
      }
      const float shift = m == -INFINITY ? 0.f : m;
      const bool large = fabsf(shift) > 1048576.f;
      if (__builtin_amdgcn_ballot_w64(large) == 0) {
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[nb][i] = __builtin_amdgcn_exp2f(fmaf(s[nb][i], c1, -shift)) * kUnit;
      } else {        // scores so large that the product's rounding matters: round it as the maximum's was
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            s[nb][i] = __builtin_amdgcn_exp2f(large ? pa_scaled_minus(s[nb][i], c1, shift) : fmaf(s[nb][i], c1, -shift)) * kUnit;
      }
#pragma unroll
      for (int nb = 0; nb < 2; ++nb)
#pragma unroll
        for (int i = 0; i < 16; ++i) l += s[nb][i];
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {          // 16 keys: registers 8 (kk % 2) .. + 7 of block kk / 2
      uint4 p[TERMS];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float x = s[kk >> 1][8 * (kk & 1) + 2 * i], y = s[kk >> 1][8 * (kk & 1) + 2 * i + 1];
#pragma unroll
        for (int n = 0; n < TERMS; ++n) {     // (what is left after a term is exact)
          const uint32_t w = PaType<DT>::pack2(x, y);
          (&p[n].x)[i] = w;
          x -= PaType<DT>::low(w);
          y -= PaType<DT>::high(w);
        }
      }
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const uint4 vf = pa_values<CV>(vt, 16 * kk, db, lane);
#pragma unroll
        for (int n = 0; n < TERMS; ++n) o[db] = PaType<DT>::mfma(vf, p[n], o[db]);
      }
    }
  }

  l += lane_xor32(l);
  if (r >= R) return;
  const float inv = l > 0.f || l != l ? 1.f / l : 0.f;     // (a row that sees nothing is zero)
  const int64_t t = r / Gq, h = g * Gq + r % Gq;
  uint16_t* out = (uint16_t*)a.out + (((int64_t)b * a.T + t) * a.H + h) * DV;
  const int64_t g0 = b * a.gate_stride_b + t * a.gate_stride_t + h * DV;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int i = 0; i < 16; i += 4) {
      const int d = db * 32 + 2 * i + 4 * half;
      float x[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) x[e] = o[db][i + e] * inv;
      if (D2 > 0 && a.gate) {
        float gate[4];
        load_vec<DType_bf16, 4>(a.gate, g0 + d, gate);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] *= sigmoid_f32(gate[e]);
      }
      *reinterpret_cast<uint2*>(out + d) = make_uint2(PaType<DT>::pack2(x[0], x[1]), PaType<DT>::pack2(x[2], x[3]));
    }
}

template <class DT, int D, int D2, int DV, int TERMS, bool CAPPED, bool POS = false>
int pa_launch(const socket_chunk_attention& a, const int64_t* positions, hipStream_t s) {
  const int64_t rows = (int64_t)a.T * (a.H / a.G);
  const int64_t n = (rows + kPaRows - 1) / kPaRows * a.G * a.B;
  SOCKET_REQUIRE(n < (1LL << 31), SOCKET_ERR_SHAPE);
  constexpr int lds = 2 * kPaKeys * (D + D2 + DV) * 2;
  auto kern = prompt_attend_kernel<DT, D, D2, DV, TERMS, CAPPED, POS>;
  if constexpr (lds > 65536) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
      return SOCKET_ERR_LAUNCH;
  }
  const int cus = socket_device_limits().cu_count, heads = a.G * a.B;
  const int first_round = n > cus && n <= 2 * (int64_t)cus ? (cus + heads - 1) / heads : 0;
  hipLaunchKernelGGL(kern, dim3((unsigned)n), dim3(64 * kPaWaves), lds, s, a, positions, first_round);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

template <class DT, int D, int TERMS>
int pa_terms(const socket_chunk_attention& a, const int64_t* positions, hipStream_t s) {
  return positions ? pa_launch<DT, D, 0, D, TERMS, false, true>(a, positions, s) : pa_launch<DT, D, 0, D, TERMS, false>(a, nullptr, s);
}

template <class DT, int D>
int pa_plain(const socket_chunk_attention& a, const int64_t* positions, int terms, hipStream_t s) {
  if constexpr (DT::kEnum == SOCKET_BF16) {
    if (a.softcap > 0.f) return pa_launch<DT, D, 0, D, 2, true>(a, nullptr, s);
    if (terms == 2) return pa_launch<DT, D, 0, D, 2, false>(a, nullptr, s);
  }
  return terms == 1 ? pa_terms<DT, D, 1>(a, positions, s) : pa_terms<DT, D, 3>(a, positions, s);
}

template <class DT>
int pa_run(const socket_chunk_attention& a, const int64_t* positions, int terms, hipStream_t s) {
  if constexpr (DT::kEnum == SOCKET_BF16) {
    if (a.k2) return pa_launch<DT, 128, 64, 128, 2, false>(a, nullptr, s);
  }
  return a.D == 64 ? pa_plain<DT, 64>(a, positions, terms, s) : pa_plain<DT, 128>(a, positions, terms, s);
}

}  // namespace

// Whether the shape is one of this file's; alignment and the checks of the entry points are the caller's.
bool prompt_attend_fits(const socket_chunk_attention& a) {
  if (!(a.scale > 0.f) || a.softcap < 0.f || a.softcap > kPaMaxCap) return false;
  if (a.dtype == SOCKET_F16 && a.softcap > 0.f) return false;     // (exp(cap) leaves the type)
  // (a tile's keys are addressed with 32-bit offsets from its first)
  const int64_t far = INT32_MAX / (2 * kPaKeys);
  for (int64_t st : {a.k_stride_t, a.v_stride_t, a.k2_stride_t})
    if (st < 0 || st > far) return false;
  if (a.k2) return a.D == 128 && a.D2 == 64 && a.Dv == 128 && a.softcap == 0.f && a.dtype == SOCKET_BF16;
  return (a.D == 64 || a.D == 128) && a.Dv == a.D && !a.gate;
}

// terms: 1 or 3, or 2 as chunk_attend.hip's kernel has them (bf16, no positions); a capped score or a shared segment
// always takes 2.
int prompt_attend_launch(const socket_chunk_attention& a, const int64_t* positions, int terms, hipStream_t s) {
  return a.dtype == SOCKET_F16 ? pa_run<DType_f16>(a, positions, terms, s) : pa_run<DType_bf16>(a, positions, terms, s);
}
