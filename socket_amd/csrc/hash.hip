// K1: key hashing.  codes = pack(sign(keys . planes^T)) with the value norm fused.
//
// Replaces hard_hash_keys + pack_bits (GPT-FAST/model.py:403-413): the einsum
// that materialises [B,S,Hkv,L,P] projections, the bool compare and the int16
// weighted sum become one MFMA contraction with a sign-bit epilogue.
//
// The hyperplanes are pre-ordered (socket_permute_planes) so that column
// w*32 + p of the contraction is the plane whose sign is bit p of packed word w.
// With planes as the M operand and keys as the N operand of
// v_mfma_f32_16x16x32_bf16, accumulator register r of lane x holds
//   plane row 4*(x/16) + r of a 16-plane block,  key x%16,
// so each lane has sign bits of ITS key in its own registers: they are shifted
// into a byte one v_alignbit per register, the four lane quarters are OR-ed into
// the 32-bit word, and lane x ends up with the packed word of key x of the
// 64-key tile, stored as one 256-byte run of the table-major code cache.  No
// compares, no ballots, no LDS round trip.  The 16x16x32 shape is chosen for the
// key loads: its N operand wants 64 consecutive bytes of a row from four lanes,
// so a load instruction touches 16 rows x one 64-byte sector (the 32x32x16 shape
// touches 64 lines for 16 bytes each, eight times over).
//
// A wave owns 64 consecutive keys of one (b, kv head) (four 16-key blocks) at a
// time and keeps their fragments in registers for the whole column sweep; the
// planes sit in LDS (all NW words when NW*8 KB fits, which L=60 x P=10 exactly
// does at 160 KB) and workgroups are persistent, so the planes are fetched once
// per CU, not once per tile.
#include "socket_common.h"

#include <type_traits>

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;

constexpr int kHashThreads = 512;
constexpr int kHashWaves = kHashThreads / SOCKET_WAVE;
constexpr int kKeysPerWave = 64;
constexpr int kD = 128;
constexpr int kKSteps = kD / 32;      // MFMA k-steps (16x16x32)
constexpr int kKeyBlocks = kKeysPerWave / 16;

union Frag {
  uint4 u;
  bf16x8 v;
};

// 8 consecutive elements starting at `p` as a bf16x8 fragment.
template <class DT>
__device__ __forceinline__ uint4 load_frag8(const typename DT::storage* p);
template <>
__device__ __forceinline__ uint4 load_frag8<DType_bf16>(const uint16_t* p) {
  return *reinterpret_cast<const uint4*>(p);
}
template <>
__device__ __forceinline__ uint4 load_frag8<DType_f32>(const float* p) {
  const float4 a = *reinterpret_cast<const float4*>(p);
  const float4 c = *reinterpret_cast<const float4*>(p + 4);
  uint4 r;
  r.x = f32x2_to_bf16_bits(a.x, a.y);
  r.y = f32x2_to_bf16_bits(a.z, a.w);
  r.z = f32x2_to_bf16_bits(c.x, c.y);
  r.w = f32x2_to_bf16_bits(c.z, c.w);
  return r;
}
template <>
__device__ __forceinline__ uint4 load_frag8<DType_f16>(const uint16_t* p) {
  const uint4 raw = *reinterpret_cast<const uint4*>(p);
  float f[8];
  unpack16<DType_f16>(raw, f);
  uint4 r;
  r.x = f32x2_to_bf16_bits(f[0], f[1]);
  r.y = f32x2_to_bf16_bits(f[2], f[3]);
  r.z = f32x2_to_bf16_bits(f[4], f[5]);
  r.w = f32x2_to_bf16_bits(f[6], f[7]);
  return r;
}

// A cache position handed over on the device (per-sequence positions) is not
// checked by the host: rows that would land outside [0, Tcap) are dropped.
__device__ __forceinline__ bool in_cache(int pos, int64_t Tcap) { return (uint64_t)(int64_t)pos < (uint64_t)Tcap; }

// LDS placement of the planes: row `col` is 16 groups of 16 bytes, group g stored
// at slot g ^ plane_swizzle(col).  A fragment read has sixteen lanes on sixteen
// columns {4..7} + 8j (or {0..3} + 8j) at one group; the swizzle sends those to
// sixteen different slots, i.e. all 64 banks once.
__device__ __forceinline__ int plane_swizzle(int col) { return (col & 3) | (((col >> 3) & 3) << 2); }

// Sum of squares of 8 consecutive elements starting at p (fp32).
template <class DT>
__device__ __forceinline__ float sumsq8(const typename DT::storage* p) {
  float s = 0.f;
  if (DT::kPer16B == 8) {
    float f[8];
    unpack16<DT>(*reinterpret_cast<const uint4*>(p), f);
#pragma unroll
    for (int i = 0; i < 8; ++i) s += f[i] * f[i];
  } else {
    float f[4];
    unpack16<DT>(*reinterpret_cast<const uint4*>(p), f);
#pragma unroll
    for (int i = 0; i < 4; ++i) s += f[i] * f[i];
    unpack16<DT>(*reinterpret_cast<const uint4*>((const char*)p + 16), f);
#pragma unroll
    for (int i = 0; i < 4; ++i) s += f[i] * f[i];
  }
  return s;
}

// Persistent: the grid is sized to the CU count and every wave walks the 64-key
// tiles tile = first, first + stride, ...; the plane slice is loaded into LDS once
// per workgroup (all of it when NW*8 KB fits) and amortised over all of them.
// NARROW: rows of D < 128 elements, which end in zeros.  (Without the test of every piece 8 x 2500 bf16 rows of 60 x 10 planes
// take 13.6 us instead of 14.0.)
template <class DT, bool NARROW>
__global__ __launch_bounds__(kHashThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void hash_keys_kernel(
    const void* __restrict__ k_, const void* __restrict__ v_, int64_t k_sb, int64_t k_sh,
    int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss,
    const uint16_t* __restrict__ planes_words,  // bf16 [NW*32, 128]
    uint32_t* __restrict__ codes, uint16_t* __restrict__ v_norm,
    const int32_t* __restrict__ pos_b, int t0, int Hkv, int S, int D, int L, int P, int NW, int64_t Tcap,
    int tiles_per_row, int n_tiles, int wc, int words_per_wg) {
  typedef typename DT::storage ST;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  // planes slice in LDS: [wc*32 columns][128] bf16, 16-byte groups XOR-swizzled
  // by column so the per-lane fragment reads (stride 256 B) spread over banks.
  uint4* plds = reinterpret_cast<uint4*>(lds_raw);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int first_tile = blockIdx.x * kHashWaves + wave;
  const int tile_stride = gridDim.x * kHashWaves;
  const int cpw = 32 / P;

  // gridDim.y splits the packed words between workgroups when there are too
  // few key tiles to occupy the chip
  const int word_begin = blockIdx.y * words_per_wg;
  const int word_end = min(NW, word_begin + words_per_wg);

  for (int w0 = word_begin; w0 < word_end; w0 += wc) {
    const int nw = min(wc, word_end - w0);
    __syncthreads();
    {
      // fill: nw*32 columns x 16 groups of 16 bytes, eight loads in flight per lane
      const uint4* src = reinterpret_cast<const uint4*>(planes_words) + (int64_t)w0 * 32 * 16;
      const int total = nw * 32 * 16;
      constexpr int U = 8;
      int i0 = tid;
      for (; i0 + (U - 1) * kHashThreads < total; i0 += U * kHashThreads) {
        uint4 x[U];
#pragma unroll
        for (int u = 0; u < U; ++u) x[u] = src[i0 + u * kHashThreads];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = i0 + u * kHashThreads;
          const int col = i >> 4, grp = i & 15;
          plds[col * 16 + (grp ^ plane_swizzle(col))] = x[u];
        }
      }
      for (; i0 < total; i0 += kHashThreads) {
        const int col = i0 >> 4, grp = i0 & 15;
        plds[col * 16 + (grp ^ plane_swizzle(col))] = src[i0];
      }
    }
    __syncthreads();

    // Key fragments (the N operand of v_mfma_f32_16x16x32_bf16): for key block nb
    // and k-step ks, lane x holds key nb*16 + x%16, elements 32*ks + 8*(x/16) .. +7,
    // so the four lanes x, x+16, x+32, x+48 read 64 consecutive bytes of one row:
    // a load instruction touches 16 rows x one 64-byte sector each.
    auto load_rows = [&](const void* base_, int64_t sb, int64_t sh, int64_t ss, int tile,
                         Frag (&dst)[kKeyBlocks][kKSteps]) {
      const int pair = tile / tiles_per_row;
      const int s0 = (tile % tiles_per_row) * kKeysPerWave;
      const ST* base = (const ST*)base_ + (pair / Hkv) * sb + (pair % Hkv) * sh;
#pragma unroll
      for (int nb = 0; nb < kKeyBlocks; ++nb) {
        const int srow = s0 + nb * 16 + (lane & 15);
        const bool ok = srow < S;
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks) {
          const int d = ks * 32 + (lane >> 4) * 8;
          dst[nb][ks].u = ok && (!NARROW || d < D) ? load_frag8<DT>(base + (int64_t)srow * ss + d) : make_uint4(0, 0, 0, 0);
        }
      }
    };
    // bf16 values: their norms come from the matrix core too (see below), from
    // fragments requested together with the keys'
    constexpr bool kNormByMfma = DT::kEnum == SOCKET_BF16;
    const bool want_norm = v_ != nullptr && w0 == 0;  // only the workgroups that own word 0
    Frag kfrag[kKeyBlocks][kKSteps];

    for (int tile = first_tile; tile < n_tiles; tile += tile_stride) {
      const int pair = tile / tiles_per_row;
      const int s0 = (tile % tiles_per_row) * kKeysPerWave;
      const int b = pair / Hkv, h = pair % Hkv;
      const int pos0 = pos_b ? pos_b[b] : t0;
      load_rows(k_, k_sb, k_sh, k_ss, tile, kfrag);
      Frag vfrag[kKeyBlocks][kKSteps];
      if (kNormByMfma && want_norm) load_rows(v_, v_sb, v_sh, v_ss, tile, vfrag);

      const int prow = lane & 15, quarter = lane >> 4;
      // fused value norm, bf16 values (once per tile; done first so that the value
      // fragments are not live across the contraction)
      if (kNormByMfma) {
        // ||v||^2 is the diagonal of V V^T: the value fragments against themselves.
        // Element (i, i) of a 16 x 16 block sits in register i % 4 of lane
        // 16 * (i / 4) + i, so sixteen lanes of the wave hold the sixteen norms and
        // store them; no cross-lane reduction.  (bf16 products are exact in fp32.)
        if (want_norm) {
          uint16_t* vn = v_norm + (int64_t)pair * Tcap + pos0;
          const int r = prow - 4 * quarter;
#pragma unroll
          for (int nb = 0; nb < kKeyBlocks; ++nb) {
            f32x4 g = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ks = 0; ks < kKSteps; ++ks)
              g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vfrag[nb][ks].v, vfrag[nb][ks].v, g, 0, 0, 0);
            const float d = r == 0 ? g[0] : r == 1 ? g[1] : r == 2 ? g[2] : g[3];
            const int srow = s0 + nb * 16 + prow;
            if (r >= 0 && r < 4 && srow < S && in_cache(pos0 + srow, Tcap)) vn[srow] = f32_to_f16_bits(sqrtf(d));
          }
        }
      }

      uint32_t* codes_pair = codes + (int64_t)pair * NW * Tcap;
      // Planes are the M operand: accumulator register r of lane x is plane row
      // 4*(x/16) + r of its 16-plane block against key x%16.  A lane shifts the sign
      // bits of its eight accumulators (two plane blocks x four registers) into a
      // byte, one v_alignbit each; byte q of the word comes from lane quarter q.
      // Block mb, register r, quarter q therefore lands at bit 8q + 7 - 4mb - r, and
      // the lane fetches for plane row i of block mb the plane column that belongs
      // at that bit, so the word comes out in the packed order.
      const int pbit0 = 8 * (prow >> 2) + 7 - (prow & 3);  // block 0; block 1 is 4 lower
      // Byte q of a key's word is made in lane quarter q, and a lane makes one byte
      // for each of the four key blocks: a 4 x 4 byte transpose between the quarters,
      // done on whole words in two exchanges (lanes x ^ 16, then x ^ 32) with a
      // byte-select each.  Afterwards lane x holds the word of key s0 + x.
      const uint32_t sel1 = (quarter & 1) ? 0x03070105u : 0x06020400u;
      const uint32_t sel2 = (quarter & 2) ? 0x03020706u : 0x05040100u;
      // plane fragments of one packed word: [k-step][plane block], straight from LDS
      auto load_planes = [&](int ww, Frag (&pf)[kKSteps][2]) {
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks) {
          const int grp = ks * 4 + quarter;
#pragma unroll
          for (int mb = 0; mb < 2; ++mb) {
            const int col = ww * 32 + pbit0 - 4 * mb;
            pf[ks][mb].u = plds[col * 16 + (grp ^ plane_swizzle(col))];
          }
        }
      };
      auto do_word = [&](int ww, const Frag (&pf)[kKSteps][2]) {
        f32x4 acc[2][kKeyBlocks];
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int nb = 0; nb < kKeyBlocks; ++nb) acc[mb][nb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
          for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int nb = 0; nb < kKeyBlocks; ++nb)  // (blocks past the last key hold zeros: no branch here)
              acc[mb][nb] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[ks][mb].v, kfrag[nb][ks].v, acc[mb][nb], 0, 0, 0);
        const int w = w0 + ww;
        const int nbits = min(cpw, L - w * cpw) * P;
        const uint32_t valid = nbits >= 32 ? 0xffffffffu : ((1u << nbits) - 1u);
        // sign bits (set = negative projection; an accumulator that starts at +0 never
        // becomes -0, so "sign clear" is exactly "projection >= 0"); byte nb of `neg`
        // is this quarter's byte for key block nb
        uint32_t neg = 0;
#pragma unroll
        for (int nb = kKeyBlocks - 1; nb >= 0; --nb)
#pragma unroll
          for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int r = 0; r < 4; ++r) neg = __builtin_amdgcn_alignbit(neg, __float_as_uint(acc[mb][nb][r]), 31);
        const uint32_t t = lane_xor16(neg, quarter & 1);
        const uint32_t x = __builtin_amdgcn_perm(t, neg, sel1);   // two blocks x this pair of quarters
        const uint32_t u = lane_xor32(x, quarter & 2);
        const uint32_t word = __builtin_amdgcn_perm(u, x, sel2);  // block `quarter` x all four quarters
        if (s0 + lane < S && in_cache(pos0 + s0 + lane, Tcap)) codes_pair[(int64_t)w * Tcap + pos0 + s0 + lane] = ~word & valid;
      };
      // two fragment sets: the next word's LDS reads are in flight during the
      // current word's contraction
      Frag pfa[kKSteps][2], pfb[kKSteps][2];
      load_planes(0, pfa);
      for (int ww = 0; ww < nw; ww += 2) {
        if (ww + 1 < nw) load_planes(ww + 1, pfb);
        do_word(ww, pfa);
        if (ww + 1 < nw) {
          if (ww + 2 < nw) load_planes(ww + 2, pfa);
          do_word(ww + 1, pfb);
        }
      }

      // fused value norm for the other element types (once per tile)
      if (!kNormByMfma && want_norm) {
        // they keep their precision: 16 lanes per row, 4 rows per pass
        const ST* vbase = (const ST*)v_ + b * v_sb + h * v_sh;
        uint16_t* vn = v_norm + (int64_t)pair * Tcap + pos0;
        const int sub = lane >> 4, part = lane & 15;
        // all sixteen row groups' loads are issued before the first is reduced
        float ss[kKeysPerWave / 4];
#pragma unroll
        for (int g = 0; g < kKeysPerWave / 4; ++g) {
          const int srow = s0 + g * 4 + sub;
          ss[g] = (srow < S && (!NARROW || part * 8 < D)) ? sumsq8<DT>(vbase + (int64_t)srow * v_ss + part * 8) : 0.f;
        }
#pragma unroll
        for (int g = 0; g < kKeysPerWave / 4; ++g) {
          const int srow = s0 + g * 4 + sub;
          float t = ss[g];
#pragma unroll
          for (int x = 1; x < 16; x <<= 1) t += __shfl_xor(t, x, SOCKET_WAVE);
          if (part == 0 && srow < S && in_cache(pos0 + srow, Tcap)) vn[srow] = f32_to_f16_bits(sqrtf(t));
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Streamed variant for large launches (prefill).
//
// The roles are turned round: the PLANES are stationary in registers and the
// keys stream through LDS.  Wave i of the eight owns packed words i, i + 8 and
// i + 16 (96 plane rows = 96 registers per lane, loaded once per kernel), and all
// eight waves read the same 128-key tile, which arrives by direct global -> LDS
// loads (no registers, no LDS store instructions) one tile ahead of the
// contraction: the memory latency that the register-staged kernel above exposes
// once per tile is hidden behind a whole tile of MFMA work.  Values come the same
// way; wave i takes the norms of key block i of the tile from the Gram diagonal.
//
// LDS image of a tile: row r (256 bytes) holds its sixteen 16-byte chunks at slot
// chunk ^ (r & 15); the lane that fetches slot s of row r asks global memory for
// chunk s ^ (r & 15), so the image needs no pass of its own, and the sixteen
// lanes of a fragment read (sixteen consecutive rows, one chunk) hit sixteen
// different slots.
constexpr int kStreamTile = 128;                       // keys per tile, at most
// LDS of a stage: bf16 keys, and the values where they come straight into LDS
constexpr int stream_stage_bytes(int dtype, int D, int tile) { return (dtype == SOCKET_BF16 ? 2 : 1) * tile * D * 2; }
constexpr int kStreamWordsPerWave = 3;
constexpr int kStreamMaxWords = kStreamWordsPerWave * kHashWaves;

// Keys of other types have to be rounded to bf16 on the way, and their value norms are fp32 sums: their tiles (64 keys of
// 128 dims, so that the registers suffice) are loaded into registers a tile ahead, eight elements of a row to a lane, and
// from there go on into the caches, into the norms and, rounded, into the same LDS image.
// The whole append of 8 pairs, 20 words, us before (staged, the copy a launch of its own): 128 dims, 3000 / 12000 / 50000 tokens
// fp16 27.6 / 59.9 / 211 -> 15.8 / 36.5 / 118, fp32 36 / 86 / 312 -> 20.8 / 55 / 196 (89 % of a copy's rate);
// 64 dims fp16 24 / 45 / 153 -> 9.7 / 20 / 65, fp32 26 / 58 / 200 -> 12.6 / 31 / 107.  bf16, whose lengths were a launch of
// their own and whose tiles were 128 keys always: 20.8 / 35.8 / 118 -> 14.7 / 33.9 / 115.
//
// D: 128, or 64 (half the contraction: the planes' other half is zero).  kTile: 128 or 64 keys.  STORE: the tile's rows also go on
// into k_cache / v_cache (element strides c_sb, c_sh, c_ss) at their positions: an append then
// reads its keys and values once.
template <class DT, int D, int kTile, bool STORE>
__global__ __launch_bounds__(kHashThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void hash_keys_stream_kernel(
    const typename DT::storage* __restrict__ k_, const typename DT::storage* __restrict__ v_, int64_t k_sb, int64_t k_sh,
    int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss,
    const uint16_t* __restrict__ planes_words,  // bf16 [NW*32, 128]
    uint32_t* __restrict__ codes, uint16_t* __restrict__ v_norm,
    const int32_t* __restrict__ pos_b, int t0, int Hkv, int S, int L, int P, int NW, int64_t Tcap,
    int tiles_per_row, int n_tiles, typename DT::storage* __restrict__ k_cache, typename DT::storage* __restrict__ v_cache,
    int64_t c_sb, int64_t c_sh, int64_t c_ss, int32_t* __restrict__ lens, int B) {
  typedef typename DT::storage ST;
  constexpr bool kDma = DT::kEnum == SOCKET_BF16;
  constexpr int kKSteps = D / 32, CH = D / 8, kRows = 64 / CH;      // k-steps; 8-element pieces of a row; rows of a wave's copy
  constexpr int kStreamTileBytes = kTile * D * 2, kStreamStageBytes = stream_stage_bytes(DT::kEnum, D, kTile);
  constexpr int kPieces = kTile / kRows / kHashWaves;
  // where piece c of row r goes: sixteen consecutive rows at one piece must hit sixteen different 16-byte
  // slots of the banks (rows of 128 bytes start half a bank line apart by the row's parity)
  auto place = [](int r, int c) { return c ^ (CH == 16 ? (r & 15) : ((r >> 1) & 7)); };
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  // (the wave index as a scalar: every address that depends on it -- this wave's
  // words of the code cache above all -- then stays out of the vector registers;
  // with it in a VGPR the kernel spilled three registers, and each reload in the
  // middle of a tile came with a vmcnt(0) that also waited for the NEXT tile's
  // copies, so the copies never overlapped the contraction)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int prow = lane & 15, quarter = lane >> 4;
  const int cpw = 32 / P;
  const bool with_values = v_ != nullptr;

  // this wave's plane rows, in the operand order of the sign-bit epilogue (see
  // hash_keys_kernel): register set [j][k-step][plane block]
  const int pbit0 = 8 * (prow >> 2) + 7 - (prow & 3);
  Frag preg[kStreamWordsPerWave][kKSteps][2];
  {
    const uint4* planes16 = reinterpret_cast<const uint4*>(planes_words);
#pragma unroll
    for (int j = 0; j < kStreamWordsPerWave; ++j) {
      const int w = wave + kHashWaves * j;
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
          const int col = w * 32 + pbit0 - 4 * mb;
          preg[j][ks][mb].u = w < NW ? planes16[(int64_t)col * (kD / 8) + ks * 4 + quarter] : make_uint4(0, 0, 0, 0);
        }
    }
  }
  const uint32_t sel1 = (quarter & 1) ? 0x03070105u : 0x06020400u;
  const uint32_t sel2 = (quarter & 2) ? 0x03020706u : 0x05040100u;
  // (a copy's rows are all the same modulo 16, so a lane's piece is too)
  const int lane_at = lane / CH * (int)(c_ss / 8) + place(kRows * wave + lane / CH, lane % CH);

  // eight elements of a row as they lie in memory
  struct alignas(16) Row8 {
    uint4 w[DT::kPer16B == 8 ? 1 : 2];
  };
  Row8 kreg[kDma ? 1 : kPieces], vreg[kDma ? 1 : kPieces];
  auto load_row8 = [&](const ST* p) __attribute__((always_inline)) {
    typedef uint32_t u32x4_s __attribute__((ext_vector_type(4)));
    Row8 r;
#pragma unroll
    for (int i = 0; i < (int)(sizeof(Row8) / 16); ++i) {
      const u32x4_s v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_s*>(p) + i);
      r.w[i] = make_uint4(v.x, v.y, v.z, v.w);
    }
    return r;
  };
  // this wave's pieces of a tile (rows kRows p .. of piece p), keys and values: into LDS, or into registers
  auto issue_tile = [&](int tile, int stage) __attribute__((always_inline)) {
    const int pair = tile / tiles_per_row;
    const int s0 = (tile % tiles_per_row) * kTile;
    const int b = pair / Hkv, h = pair % Hkv;
    const ST* kbase = k_ + b * k_sb + h * k_sh;
    const ST* vbase = with_values ? v_ + b * v_sb + h * v_sh : nullptr;
    unsigned char* dst = lds_raw + (size_t)stage * kStreamStageBytes;
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
      const int p = wave + kHashWaves * q;
      const int row = kRows * p + lane / CH;
      const int srow = min(s0 + row, S - 1);  // rows past the end re-read the last one; never stored
      if constexpr (kDma) {
        const int chunk = place(kRows * wave + lane / CH, lane % CH);
        lds_dma16_stream(kbase + (int64_t)srow * k_ss + chunk * 8, dst + p * 1024);
        if (with_values) lds_dma16_stream(vbase + (int64_t)srow * v_ss + chunk * 8, dst + kStreamTileBytes + p * 1024);
      } else {
        kreg[q] = load_row8(kbase + (int64_t)srow * k_ss + lane % CH * 8);
        if (with_values) vreg[q] = load_row8(vbase + (int64_t)srow * v_ss + lane % CH * 8);
      }
    }
  };

  int tile = blockIdx.x;
  if (tile < n_tiles) issue_tile(tile, 0);
  if (STORE && lens && blockIdx.x == 0)
    for (int b = tid; b < B; b += kHashThreads) lens[b] = t0 + S;
  for (int it = 0; tile < n_tiles; tile += gridDim.x, ++it) {
    const int stage = it & 1;
    const int next = tile + gridDim.x;
    const int pair = tile / tiles_per_row;
    const int s0 = (tile % tiles_per_row) * kTile;
    const int pos0 = pos_b ? pos_b[pair / Hkv] : t0;
    if constexpr (!kDma) {
      // out of the registers: rounded keys into the stage (left by every wave before the last barrier), rows into the
      // caches, norms
      uint4* image = reinterpret_cast<uint4*>(lds_raw + (size_t)stage * kStreamStageBytes);
#pragma unroll
      for (int q = 0; q < kPieces; ++q) {
        const int r = kRows * (wave + kHashWaves * q) + lane / CH, c = lane % CH;
        image[r * CH + place(r, c)] = load_frag8<DT>(reinterpret_cast<const ST*>(kreg[q].w));
        if constexpr (STORE) {
          if (s0 + r < S) {
            const int64_t at = (int64_t)(pair / Hkv) * c_sb + (pair % Hkv) * c_sh + (int64_t)(pos0 + s0 + r) * c_ss + c * 8;
            *reinterpret_cast<Row8*>(k_cache + at) = kreg[q];
            *reinterpret_cast<Row8*>(v_cache + at) = vreg[q];
          }
        }
        if (with_values) {
          const float t = group_sum<CH>(sumsq8<DT>(reinterpret_cast<const ST*>(vreg[q].w)));
          if (c == 0 && s0 + r < S && in_cache(pos0 + s0 + r, Tcap)) v_norm[(int64_t)pair * Tcap + pos0 + s0 + r] = f32_to_f16_bits(sqrtf(t));
        }
      }
    }
    // One barrier per tile: behind it every wave's pieces of this tile are in place
    // AND every wave is done with the previous tile, whose stage the next tile's
    // loads may therefore overwrite while this one is contracted.
    if constexpr (kDma) wait_vmcnt(0);
    __syncthreads();
    if (next < n_tiles) issue_tile(next, stage ^ 1);

    const uint4* ktile = reinterpret_cast<const uint4*>(lds_raw + (size_t)stage * kStreamStageBytes);
    const uint4* vtile = ktile + kStreamTileBytes / 16;
    // chunk c of row r of a tile (r & 15 == prow for every row this lane reads)
    auto frag_at = [&](const uint4* t, int r, int c) { return t[r * CH + place(prow, c)]; };

    if constexpr (STORE && kDma) {
      // this wave's pieces of the tile on into the caches, whole rows of 256 (128) bytes
      const int64_t c0 = (int64_t)(pair / Hkv) * c_sb + (pair % Hkv) * c_sh + (int64_t)(pos0 + s0 + kRows * wave) * c_ss;
#pragma unroll
      for (int q = 0; q < kPieces; ++q)
        if (s0 + kRows * (wave + kHashWaves * q) + lane / CH < S) {
          const int64_t at = c0 + (int64_t)(kRows * kHashWaves * q) * c_ss;
          reinterpret_cast<uint4*>(k_cache + at)[lane_at] = ktile[(wave + kHashWaves * q) * 64 + lane];
          reinterpret_cast<uint4*>(v_cache + at)[lane_at] = vtile[(wave + kHashWaves * q) * 64 + lane];
        }
    }

    if (kDma && with_values && wave < kTile / 16) {
      // ||v||^2 = diagonal of V V^T (see hash_keys_kernel), key block `wave` of the tile
      Frag vf[kKSteps];
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) vf[ks].u = frag_at(vtile, wave * 16 + prow, ks * 4 + quarter);
      f32x4 g = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < kKSteps; ++ks) g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[ks].v, vf[ks].v, g, 0, 0, 0);
      const int r = prow - 4 * quarter;
      const float d = r == 0 ? g[0] : r == 1 ? g[1] : r == 2 ? g[2] : g[3];
      const int srow = s0 + wave * 16 + prow;
      if (r >= 0 && r < 4 && srow < S && in_cache(pos0 + srow, Tcap))
        v_norm[(int64_t)pair * Tcap + pos0 + srow] = f32_to_f16_bits(sqrtf(d));
    }

    uint32_t* codes_pair = codes + (int64_t)pair * NW * Tcap;
    // The tile's 16-key blocks go through in pairs, the next pair's
    // fragments on their way from LDS while the current pair is contracted.  A
    // 64-key group is taken high blocks first, (3,2) then (1,0), so that the sign
    // bits shift into `neg` in the byte order the transpose expects.
    auto pair_block = [](int pp) { return (pp >> 1) * 4 + ((pp & 1) ? 0 : 2); };  // lower block of pair pp
    auto load_pair = [&](int pp, Frag (&kf)[2][kKSteps]) {
      const int nb0 = pair_block(pp);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks)
          kf[i][ks].u = frag_at(ktile, (nb0 + i) * 16 + prow, ks * 4 + quarter);
    };
    auto tile_body = [&](auto nwords_c) {
      constexpr int NWD = decltype(nwords_c)::value;
      uint32_t neg[NWD];
#pragma unroll
      for (int j = 0; j < NWD; ++j) neg[j] = 0;
      auto do_pair = [&](int pp, const Frag (&kf)[2][kKSteps]) {
#pragma unroll
        for (int j = 0; j < NWD; ++j) {
          f32x4 acc[2][2];
#pragma unroll
          for (int mb = 0; mb < 2; ++mb)
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[mb][i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
              for (int i = 0; i < 2; ++i)
                acc[mb][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(preg[j][ks][mb].v, kf[i][ks].v, acc[mb][i], 0, 0, 0);
          // sign bits -> this quarter's byte per key block (higher block first)
#pragma unroll
          for (int i = 1; i >= 0; --i)
#pragma unroll
            for (int mb = 0; mb < 2; ++mb)
#pragma unroll
              for (int r = 0; r < 4; ++r) neg[j] = __builtin_amdgcn_alignbit(neg[j], __float_as_uint(acc[mb][i][r]), 31);
          if (pp & 1) {
            // all four blocks of the 64-key group are in: 4 x 4 byte transpose between
            // the quarters (as in hash_keys_kernel), lane x gets key x's word
            const int w = wave + kHashWaves * j;
            const int nbits = min(cpw, L - w * cpw) * P;
            const uint32_t valid = nbits >= 32 ? 0xffffffffu : ((1u << nbits) - 1u);
            const uint32_t t = lane_xor16(neg[j], quarter & 1);
            const uint32_t x = __builtin_amdgcn_perm(t, neg[j], sel1);
            const uint32_t u = lane_xor32(x, quarter & 2);
            const uint32_t word = __builtin_amdgcn_perm(u, x, sel2);
            const int key = s0 + (pp >> 1) * kKeysPerWave + lane;
            if (key < S && in_cache(pos0 + key, Tcap)) codes_pair[(int64_t)w * Tcap + pos0 + key] = ~word & valid;
          }
        }
      };
      Frag kfa[2][kKSteps], kfb[2][kKSteps];
      load_pair(0, kfa);
#pragma unroll
      for (int pp = 0; pp < kTile / 32; pp += 2) {
        load_pair(pp + 1, kfb);
        do_pair(pp, kfa);
        if (pp + 2 < kTile / 32) load_pair(pp + 2, kfa);
        do_pair(pp + 1, kfb);
      }
    };
    // (uniform per wave: waves 0 .. NW % 8 - 1 own one word more than the others)
    const int my_words = wave < NW ? (NW - wave + kHashWaves - 1) / kHashWaves : 0;
    if (my_words == 3) tile_body(std::integral_constant<int, 3>{});
    else if (my_words == 2) tile_body(std::integral_constant<int, 2>{});
    else if (my_words == 1) tile_body(std::integral_constant<int, 1>{});
  }
}

// ---------------------------------------------------------------------------
// Direct variant for few rows (a decode step's, a short block's): nothing in LDS, no wave waits for another.
//
// The rows of all (b, kv head) pairs are numbered through and cut into tiles of NB 16-row blocks, so that a
// decode step's handful shares one contraction whatever pairs it belongs to.  A wave makes ONE packed word of a
// tile: its plane fragments and its keys are requested together, straight into registers, and the whole kernel is
// one trip to memory, 8 NB products and a store.  (The staged kernel above pays a trip for the planes, a barrier, a trip
// for the keys, and reads the planes' LDS image through for every tile.)  The last row of the grid has the values' norms
// and, where `k_cache` is given, the rows' copies and the lengths.
// A decode step's 8 rows, 32 tables of 8 planes: 3.5 us where the staged kernel takes 6.4 (float32); 512 rows of 60 x
// 10: 3.5 against 10.8 (bf16).
// Same k-steps in the same order on the same fragments as above: the bits are equal.
constexpr int kDirectWaves = 4, kDirectThreads = kDirectWaves * SOCKET_WAVE;

template <class DT, int NB>
__global__ __launch_bounds__(kDirectThreads) void hash_keys_direct_kernel(
    const void* __restrict__ k_, const void* __restrict__ v_, int64_t k_sb, int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh,
    int64_t v_ss, const uint16_t* __restrict__ planes_words, uint32_t* __restrict__ codes, uint16_t* __restrict__ v_norm,
    const int32_t* __restrict__ pos_b, int t0, int Hkv, int S, int D, int L, int P, int NW, int64_t Tcap, int n_rows,
    int word_groups, void* __restrict__ k_cache, void* __restrict__ v_cache, int64_t c_sb, int64_t c_sh, int64_t c_ss,
    int32_t* __restrict__ lens, int B) {
  typedef typename DT::storage ST;
  constexpr int kTile = 16 * NB;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int prow = lane & 15, quarter = lane >> 4;
  const int row0 = blockIdx.x * kTile;
  struct Where {
    int b, h, s;
  };
  auto where = [&](int row) {
    const unsigned r = min(row, n_rows - 1), pair = r / (unsigned)S;
    return Where{(int)(pair / (unsigned)Hkv), (int)(pair % (unsigned)Hkv), (int)(r - pair * S)};
  };
  auto start = [&](const void* base, const Where& at, int64_t sb, int64_t sh, int64_t ss) {
    return (const ST*)base + at.b * sb + at.h * sh + at.s * ss;
  };
  auto fragments = [&](const ST* row, Frag (&dst)[kKSteps]) {
#pragma unroll
    for (int ks = 0; ks < kKSteps; ++ks) {
      const int d = ks * 32 + quarter * 8;           // (a narrower head's row ends in zeros)
      dst[ks].u = make_uint4(0, 0, 0, 0);
      if (ks * 32 < D) {                             // (the same for every lane)
        const uint4 x = load_frag8<DT>(row + min(d, D - 8));
        if (d < D) dst[ks].u = x;
      }
    }
  };

  if ((int)blockIdx.y == word_groups) {
    constexpr bool kNormByMfma = DT::kEnum == SOCKET_BF16;
    if (v_ && kNormByMfma) {                         // (the Gram diagonal, as in the kernel above)
      for (int nb = wave; nb < NB; nb += kDirectWaves) {
        const int row = row0 + nb * 16 + prow;
        const Where at = where(row);
        Frag vf[kKSteps];
        fragments(start(v_, at, v_sb, v_sh, v_ss), vf);
        f32x4 g = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < kKSteps; ++ks) g = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf[ks].v, vf[ks].v, g, 0, 0, 0);
        const int r = prow - 4 * quarter, pos = (pos_b ? pos_b[at.b] : t0) + at.s;
        const float d = r == 0 ? g[0] : r == 1 ? g[1] : r == 2 ? g[2] : g[3];
        if (r >= 0 && r < 4 && row < n_rows && in_cache(pos, Tcap))
          v_norm[((int64_t)at.b * Hkv + at.h) * Tcap + pos] = f32_to_f16_bits(sqrtf(d));
      }
    } else if (v_) {
      float ss[NB];
#pragma unroll
      for (int g = 0; g < NB; ++g) {
        const ST* row = start(v_, where(row0 + (wave * NB + g) * 4 + quarter), v_sb, v_sh, v_ss);
        const float x = sumsq8<DT>(row + min(prow * 8, D - 8));
        ss[g] = prow * 8 < D ? x : 0.f;
      }
#pragma unroll
      for (int g = 0; g < NB; ++g) {
        const int row = row0 + (wave * NB + g) * 4 + quarter;
        const Where at = where(row);
        float t = ss[g];
#pragma unroll
        for (int x = 1; x < 16; x <<= 1) t += __shfl_xor(t, x, SOCKET_WAVE);
        const int pos = (pos_b ? pos_b[at.b] : t0) + at.s;
        if (prow == 0 && row < n_rows && in_cache(pos, Tcap))
          v_norm[((int64_t)at.b * Hkv + at.h) * Tcap + pos] = f32_to_f16_bits(sqrtf(t));
      }
    }
    if (k_cache) {
      if (lens && blockIdx.x == 0)
        for (int b = tid; b < B; b += kDirectThreads) lens[b] = t0 + S;
      constexpr int E = DT::kPer16B, U = 2;
      const int per = D / E, n = min(kTile, n_rows - row0) * per;
      for (int i0 = tid; i0 < n; i0 += U * kDirectThreads) {
        uint4 x[U], y[U];
        int64_t to[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int i = min(i0 + u * kDirectThreads, n - 1), d = i % per * E;
          const Where at = where(row0 + i / per);
          x[u] = *reinterpret_cast<const uint4*>(start(k_, at, k_sb, k_sh, k_ss) + d);
          y[u] = *reinterpret_cast<const uint4*>(start(v_, at, v_sb, v_sh, v_ss) + d);
          to[u] = at.b * c_sb + at.h * c_sh + (t0 + at.s) * c_ss + d;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          if (i0 + u * kDirectThreads >= n) break;
          *reinterpret_cast<uint4*>((ST*)k_cache + to[u]) = x[u];
          *reinterpret_cast<uint4*>((ST*)v_cache + to[u]) = y[u];
        }
      }
    }
    return;
  }

  const int w = blockIdx.y * kDirectWaves + wave;
  if (w >= NW) return;
  const int pbit0 = 8 * (prow >> 2) + 7 - (prow & 3);      // (plane row of each accumulator register: see above)
  Frag pf[kKSteps][2], kf[NB][kKSteps];
#pragma unroll
  for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
      pf[ks][mb].u = reinterpret_cast<const uint4*>(planes_words)[(int64_t)(w * 32 + pbit0 - 4 * mb) * 16 + ks * 4 + quarter];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) fragments(start(k_, where(row0 + nb * 16 + prow), k_sb, k_sh, k_ss), kf[nb]);
  const int row = row0 + (NB == 4 ? lane : prow);          // whose word this lane stores
  const Where at = where(row);
  const int pos = (pos_b ? pos_b[at.b] : t0) + at.s;
  uint32_t neg = 0;
#pragma unroll
  for (int nb = NB - 1; nb >= 0; --nb) {
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ks = 0; ks < kKSteps; ++ks)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
        acc[mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pf[ks][mb].v, kf[nb][ks].v, acc[mb], 0, 0, 0);
#pragma unroll
    for (int mb = 0; mb < 2; ++mb)
#pragma unroll
      for (int r = 0; r < 4; ++r) neg = __builtin_amdgcn_alignbit(neg, __float_as_uint(acc[mb][r]), 31);
  }
  uint32_t word;
  if constexpr (NB == 4) {                                 // (the byte transpose of the kernel above)
    const uint32_t t = lane_xor16(neg, quarter & 1);
    const uint32_t x = __builtin_amdgcn_perm(t, neg, (quarter & 1) ? 0x03070105u : 0x06020400u);
    const uint32_t u = lane_xor32(x, quarter & 2);
    word = __builtin_amdgcn_perm(u, x, (quarter & 2) ? 0x03020706u : 0x05040100u);
  } else {
    static_assert(NB == 1, "one block, or four whose bytes fill a word");
    word = neg << (8 * quarter);
    word |= lane_xor16(word, quarter & 1);
    word |= lane_xor32(word, quarter & 2);
  }
  const int cpw = 32 / P, nbits = min(cpw, L - w * cpw) * P;
  const uint32_t valid = nbits >= 32 ? 0xffffffffu : ((1u << nbits) - 1u);
  if ((NB == 4 || quarter == 0) && row < n_rows && in_cache(pos, Tcap))
    codes[(((int64_t)at.b * Hkv + at.h) * NW + w) * Tcap + pos] = ~word & valid;
}

// Keys and values [B,Hkv,S,D] (any strides, whole 16-byte pieces) into rows t0 .. of the caches; the lengths
// become t0 + S.  A lane moves kCopyPieces pieces of each, requested together; a wave's stores are whole rows.
constexpr int kCopyPieces = 4;
template <class DT>
__global__ __launch_bounds__(256) void copy_rows_kernel(const void* __restrict__ k, const void* __restrict__ v, int64_t k_sb,
                                                        int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss,
                                                        void* __restrict__ k_cache, void* __restrict__ v_cache, int64_t c_sb,
                                                        int64_t c_sh, int64_t c_ss, int32_t* __restrict__ lens, int t0, int B,
                                                        int Hkv, int S, int D) {
  typedef typename DT::storage ST;
  constexpr int E = DT::kPer16B;
  if (lens && blockIdx.x == 0 && blockIdx.y == 0)
    for (int b = threadIdx.x; b < B; b += 256) lens[b] = t0 + S;
  const int b = blockIdx.y / Hkv, h = blockIdx.y % Hkv, per = D / E;
  const ST* kp = (const ST*)k + b * k_sb + h * k_sh;
  const ST* vp = (const ST*)v + b * v_sb + h * v_sh;
  const int64_t c0 = b * c_sb + h * c_sh, n = (int64_t)S * per, i0 = (int64_t)blockIdx.x * 256 * kCopyPieces + threadIdx.x;
  uint4 x[kCopyPieces], y[kCopyPieces];
#pragma unroll
  for (int u = 0; u < kCopyPieces; ++u) {
    const int64_t i = min(i0 + u * 256, n - 1);
    const int s = (int)(i / per), d = (int)(i % per) * E;
    x[u] = *reinterpret_cast<const uint4*>(kp + s * k_ss + d);
    y[u] = *reinterpret_cast<const uint4*>(vp + s * v_ss + d);
  }
#pragma unroll
  for (int u = 0; u < kCopyPieces; ++u) {
    const int64_t i = i0 + u * 256;
    if (i >= n) break;
    const int64_t at = c0 + (t0 + i / per) * c_ss + i % per * E;
    *reinterpret_cast<uint4*>((ST*)k_cache + at) = x[u];
    *reinterpret_cast<uint4*>((ST*)v_cache + at) = y[u];
  }
}

template <class PT>
__global__ void permute_planes_kernel(const void* __restrict__ planes_, uint16_t* __restrict__ out,
                                      int L, int P, int D, int NW) {
  typedef typename PT::storage ST;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (int64_t)NW * 32 * D) return;
  const int d = (int)(i % D);
  const int colw = (int)(i / D);
  const int w = colw / 32, p = colw % 32;
  const int cpw = 32 / P;
  const int l = w * cpw + p / P;
  uint16_t r = 0;
  if (p < cpw * P && l < L) {
    const int k = P - 1 - (p % P);
    const ST* planes = (const ST*)planes_;
    const int64_t src = ((int64_t)l * P + k) * D + d;
    float f;
    if (PT::kEnum == SOCKET_F32) f = ((const float*)planes)[src];
    else if (PT::kEnum == SOCKET_BF16) f = bf16_bits_to_f32(((const uint16_t*)planes)[src]);
    else f = f16_bits_to_f32(((const uint16_t*)planes)[src]);
    r = f32_to_bf16_bits(f);
  }
  out[i] = r;
}

__global__ void unpack_codes_kernel(const uint32_t* __restrict__ codes, int16_t* __restrict__ out,
                                    int Hkv, int L, int P, int t0, int T, int64_t Tcap, int NW,
                                    int64_t osb, int64_t osh, int64_t osl, int64_t ost) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int pair = blockIdx.y;
  if (t >= T) return;
  const int b = pair / Hkv, h = pair % Hkv;
  const int cpw = 32 / P;
  const uint32_t mask = (1u << P) - 1u;
  const uint32_t* src = codes + (int64_t)pair * NW * Tcap + t0 + t;
  int16_t* dst = out + b * osb + h * osh + (int64_t)t * ost;
  for (int w = 0; w < NW; ++w) {
    const uint32_t word = src[(int64_t)w * Tcap];
    for (int j = 0; j < cpw && w * cpw + j < L; ++j)
      dst[(int64_t)(w * cpw + j) * osl] = (int16_t)((word >> (j * P)) & mask);
  }
}

__global__ void pack_codes_kernel(const int16_t* __restrict__ in, int64_t isb, int64_t ish,
                                  int64_t isl, int64_t ist, uint32_t* __restrict__ codes, int Hkv,
                                  int L, int P, int t0, int T, int64_t Tcap, int NW) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int pair = blockIdx.y;
  if (t >= T) return;
  const int b = pair / Hkv, h = pair % Hkv;
  const int cpw = 32 / P;
  const uint32_t mask = (1u << P) - 1u;
  const int16_t* src = in + b * isb + h * ish + (int64_t)t * ist;
  uint32_t* dst = codes + (int64_t)pair * NW * Tcap + t0 + t;
  for (int w = 0; w < NW; ++w) {
    uint32_t word = 0;
    for (int j = 0; j < cpw && w * cpw + j < L; ++j)
      word |= ((uint32_t)(uint16_t)src[(int64_t)(w * cpw + j) * isl] & mask) << (j * P);
    dst[(int64_t)w * Tcap] = word;
  }
}

int words_per_key(int L, int P) {
  if (P < 1 || P > 16 || L < 1) return 0;
  const int cpw = 32 / P;
  return (L + cpw - 1) / cpw;
}

}  // namespace

extern "C" int socket_words_per_key(int L, int P) { return words_per_key(L, P); }

extern "C" int socket_permute_planes(const void* planes, int planes_dtype, int L, int P, int D,
                                     void* planes_words, void* stream) {
  SOCKET_REQUIRE(planes && planes_words, SOCKET_ERR_NULL);
  const int NW = words_per_key(L, P);
  SOCKET_REQUIRE(NW > 0 && D > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(socket_dtype_bytes(planes_dtype) != 0, SOCKET_ERR_UNSUPPORTED);
  const int64_t n = (int64_t)NW * 32 * D;
  const int threads = 256;
  const dim3 grid((unsigned)((n + threads - 1) / threads));
  hipStream_t s = (hipStream_t)stream;
  uint16_t* out = (uint16_t*)planes_words;
  if (planes_dtype == SOCKET_F32)
    hipLaunchKernelGGL((permute_planes_kernel<DType_f32>), grid, dim3(threads), 0, s, planes, out, L, P, D, NW);
  else if (planes_dtype == SOCKET_BF16)
    hipLaunchKernelGGL((permute_planes_kernel<DType_bf16>), grid, dim3(threads), 0, s, planes, out, L, P, D, NW);
  else
    hipLaunchKernelGGL((permute_planes_kernel<DType_f16>), grid, dim3(threads), 0, s, planes, out, L, P, D, NW);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

namespace {

// Keys (and values) as hash_keys and cache_append have them; k_cache: the rows also go there.
struct HashRows {
  const void *k, *v;
  int dtype;
  int64_t k_sb, k_sh, k_ss, v_sb, v_sh, v_ss;
  const void* planes_words;
  uint32_t* codes;
  uint16_t* v_norm;
  const int32_t* pos_b;
  int t0, B, Hkv, S, D, L, P, NW;
  int64_t Tcap;
  void *k_cache, *v_cache;
  int64_t c_sb, c_sh, c_ss;
};

int64_t stream_tiles(const HashRows& a, int tile) { return (int64_t)a.B * a.Hkv * ((a.S + tile - 1) / tile); }

// Keys of a tile: 128, halves where that leaves CUs idle or (rows of 128 dims that go through the registers) is more than
// the registers hold.
int stream_tile(const HashRows& a, const SocketDeviceLimits& lim) {
  if (a.dtype != SOCKET_BF16 && a.D == 128) return kStreamTile / 2;
  return stream_tiles(a, kStreamTile) >= lim.cu_count ? kStreamTile : kStreamTile / 2;
}


// Whether the variant with the planes in registers serves: rows of 128 or 64 dims, up to 24 words, and so many rows that what
// a workgroup fetches once, all planes (160 KB at 20 words), no longer outweighs what the direct variant fetches for
// every tile and word.  The whole append of 8 pairs, us, direct / streamed: 128 dims, 20 words, bf16 4000 rows 8.7 / 9.3, 6216
// 10.4 / 9.8, 8800 13.1 / 10.4; fp16 2400 7.1 / 9.7, 4000 10.2 / 9.9, 8800 13.0 / 10.7; fp32 2400 8.8 / 11.2, 4000 12.5 / 12.2;
// 8 words, bf16 2400 5.4 / 6.0, 4000 6.5 / 6.2, 6216 9.3 / 6.4.  64 dims, 20 words, 2400 rows: 6.4 / 6.0, 6.4 / 6.2, 7.3 / 6.7;
// 6216: 7.5 / 6.4, 8.3 / 6.4, 10.1 / 7.5.  (The staged variant is behind from 5000 rows on: 24000 rows, 128 dims, 20 words,
// with the copy 21.0 / 14.7, 27.5 / 15.7, 35.5 / 20.8.)  Many pairs of few rows each leave most of a tile empty: not
// unless every CU has a tile of 128 all the same.
bool streams(const HashRows& a, const SocketDeviceLimits& lim) {
  if ((a.D != 128 && a.D != 64) || a.NW > kStreamMaxWords) return false;
  const int tile = stream_tile(a, lim);
  if (2 * stream_stage_bytes(a.dtype, a.D, tile) > lim.max_lds_per_block) return false;
  const int64_t rows = (int64_t)a.B * a.Hkv * a.S;
  return stream_tiles(a, kStreamTile) >= lim.cu_count ||
         (rows >= (a.D == 64 ? 2048 : 4096 + 128 * a.NW) && 2 * rows >= stream_tiles(a, tile) * tile);
}

template <class DT, int D, int kTile, bool STORE>
int launch_stream_of(const HashRows& a, const SocketDeviceLimits& lim, int32_t* lens, hipStream_t s) {
  typedef typename DT::storage ST;
  const int tiles_per_row = (a.S + kTile - 1) / kTile;
  const int64_t n_tiles = (int64_t)a.B * a.Hkv * tiles_per_row;
  const size_t lds = 2 * (size_t)stream_stage_bytes(DT::kEnum, D, kTile);
  auto kern = hash_keys_stream_kernel<DT, D, kTile, STORE>;
  if (lds > 48 * 1024 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return SOCKET_ERR_LAUNCH;
  const int n_wg = (int)(n_tiles < lim.cu_count ? n_tiles : lim.cu_count);
  hipLaunchKernelGGL(kern, dim3(n_wg), dim3(kHashThreads), lds, s, (const ST*)a.k, (const ST*)a.v, a.k_sb, a.k_sh, a.k_ss, a.v_sb,
                     a.v_sh, a.v_ss, (const uint16_t*)a.planes_words, a.codes, a.v_norm, a.pos_b, a.t0, a.Hkv, a.S, a.L, a.P, a.NW,
                     a.Tcap, tiles_per_row, (int)n_tiles, (ST*)a.k_cache, (ST*)a.v_cache, a.c_sb, a.c_sh, a.c_ss, lens, a.B);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

template <bool STORE>
int launch_stream(const HashRows& a, const SocketDeviceLimits& lim, int32_t* lens, hipStream_t s) {
  const bool half = stream_tile(a, lim) < kStreamTile;
#define SOCKET_STREAM(DT, D)                                                                             \
  return half ? launch_stream_of<DT, D, kStreamTile / 2, STORE>(a, lim, lens, s)                         \
              : launch_stream_of<DT, D, kStreamTile, STORE>(a, lim, lens, s)
  if (a.D == 64) {
    if (a.dtype == SOCKET_BF16) SOCKET_STREAM(DType_bf16, 64);
    if (a.dtype == SOCKET_F16) SOCKET_STREAM(DType_f16, 64);
    SOCKET_STREAM(DType_f32, 64);
  }
  if (a.dtype == SOCKET_BF16) SOCKET_STREAM(DType_bf16, 128);
  if (a.dtype == SOCKET_F16) return launch_stream_of<DType_f16, 128, kStreamTile / 2, STORE>(a, lim, lens, s);
  return launch_stream_of<DType_f32, 128, kStreamTile / 2, STORE>(a, lim, lens, s);
#undef SOCKET_STREAM
}

// Few enough rows for the direct variant.  Its time grows with rows x words, since a wave fetches its tile's keys and
// its word's planes for itself; the staged variant's hardly does below a few tiles per CU.  Hashing 8 pairs' rows with 20
// words, bf16 of 128 dims, direct / staged: 8192 rows 10.4 / 11.8 us, 12288 13.5 / 12.1; with 8 words 24576 rows 11.3 / 12.0.
// The lines cross between 180k (float32) and 260k words; with the copy in the same launch (one fewer) between 270k and
// 400k.  Where the streamed kernel serves and has at least half of every tile it is ahead of both (32768 rows, 8 words:
// 7.0 against 14.5 direct).
bool goes_direct(const HashRows& a, const SocketDeviceLimits& lim, bool streamed) {
  const int64_t rows = (int64_t)a.B * a.Hkv * a.S;
  if (streamed) {
    const int tile = stream_tile(a, lim);
    if (2 * rows >= stream_tiles(a, tile) * tile) return false;
  }
  return rows * a.NW <= (a.k_cache ? 256 : 176) * 1024 && a.NW <= 65536;      // (a grid's y)
}

int launch_direct(const HashRows& a, const SocketDeviceLimits& lim, int32_t* lens, hipStream_t s) {
  const int n_rows = a.B * a.Hkv * a.S, groups = (a.NW + kDirectWaves - 1) / kDirectWaves;
  const int rows_of = (a.v || a.k_cache) ? 1 : 0;
  // four blocks to a tile once that still gives every CU a workgroup
  const bool wide = (int64_t)((n_rows + 63) / 64) * groups >= lim.cu_count;
  const int tile = wide ? 64 : 16;
  const dim3 grid((n_rows + tile - 1) / tile, groups + rows_of);
#define SOCKET_DIRECT(DT, NB)                                                                                             \
  hipLaunchKernelGGL((hash_keys_direct_kernel<DT, NB>), grid, dim3(kDirectThreads), 0, s, a.k, a.v, a.k_sb, a.k_sh, a.k_ss, \
                     a.v_sb, a.v_sh, a.v_ss, (const uint16_t*)a.planes_words, a.codes, a.v_norm, a.pos_b, a.t0, a.Hkv, a.S, \
                     a.D, a.L, a.P, a.NW, a.Tcap, n_rows, groups, a.k_cache, a.v_cache, a.c_sb, a.c_sh, a.c_ss, lens, a.B)
#define SOCKET_DIRECT_DT(DT)           \
  do {                                 \
    if (wide) SOCKET_DIRECT(DT, 4);    \
    else SOCKET_DIRECT(DT, 1);         \
  } while (0)
  if (a.dtype == SOCKET_BF16) SOCKET_DIRECT_DT(DType_bf16);
  else if (a.dtype == SOCKET_F16) SOCKET_DIRECT_DT(DType_f16);
  else SOCKET_DIRECT_DT(DType_f32);
#undef SOCKET_DIRECT_DT
#undef SOCKET_DIRECT
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

int launch_staged(const HashRows& a, const SocketDeviceLimits& lim, hipStream_t s) {
  const int tiles_per_row = (a.S + kKeysPerWave - 1) / kKeysPerWave;
  const int64_t n_tiles64 = (int64_t)a.B * a.Hkv * tiles_per_row;
  SOCKET_REQUIRE(n_tiles64 < (1LL << 31), SOCKET_ERR_SHAPE);
  const int n_tiles = (int)n_tiles64, NW = a.NW;
  // plane slice: every word when they all fit in LDS (one slice, loaded once per
  // workgroup), else as many as fit; one persistent workgroup per CU
  int wc = lim.max_lds_per_block / (32 * kD * 2);
  if (wc < 1) wc = 1;
  if (wc > NW) wc = NW;
  int n_wg = (n_tiles + kHashWaves - 1) / kHashWaves;
  if (n_wg > lim.cu_count) n_wg = lim.cu_count;
  int wsplit = lim.cu_count / n_wg;  // > 1 only when the tiles leave CUs idle
  if (wsplit > NW) wsplit = NW;
  if (wsplit < 1) wsplit = 1;
  const int words_per_wg = (NW + wsplit - 1) / wsplit;
  wsplit = (NW + words_per_wg - 1) / words_per_wg;
  if (wc > words_per_wg) wc = words_per_wg;
  const size_t lds = (size_t)wc * 32 * kD * 2;
  const dim3 grid(n_wg, wsplit);
#define SOCKET_HASH_LAUNCH(DT)                                                                     \
  do {                                                                                             \
    auto kern = a.D == kD ? hash_keys_kernel<DT, false> : hash_keys_kernel<DT, true>;              \
    if (lds > 48 * 1024 &&                                                                         \
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern),                                   \
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)   \
      return SOCKET_ERR_LAUNCH;                                                                    \
    hipLaunchKernelGGL(kern, grid, dim3(kHashThreads), lds, s, a.k, a.v, a.k_sb, a.k_sh, a.k_ss,   \
                       a.v_sb, a.v_sh, a.v_ss, (const uint16_t*)a.planes_words, a.codes, a.v_norm, \
                       a.pos_b, a.t0, a.Hkv, a.S, a.D, a.L, a.P, NW, a.Tcap, tiles_per_row, n_tiles, \
                       wc, words_per_wg);                                                          \
  } while (0)
  if (a.dtype == SOCKET_BF16) SOCKET_HASH_LAUNCH(DType_bf16);
  else if (a.dtype == SOCKET_F16) SOCKET_HASH_LAUNCH(DType_f16);
  else SOCKET_HASH_LAUNCH(DType_f32);
#undef SOCKET_HASH_LAUNCH
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

int check_hash_rows(const HashRows& a) {
  SOCKET_REQUIRE(a.k && a.planes_words && a.codes, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(a.v == nullptr || a.v_norm != nullptr, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(a.NW > 0 && a.B > 0 && a.Hkv > 0 && a.S > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(a.t0 >= 0 && (a.pos_b != nullptr || (int64_t)a.t0 + a.S <= a.Tcap), SOCKET_ERR_SHAPE);
  const int eb = socket_dtype_bytes(a.dtype);
  SOCKET_REQUIRE(eb != 0, SOCKET_ERR_UNSUPPORTED);
  const int per16 = 16 / eb;
  SOCKET_REQUIRE(socket_aligned16(a.k) && socket_aligned16(a.planes_words) && a.k_sb % per16 == 0 && a.k_sh % per16 == 0 &&
                     a.k_ss % per16 == 0,
                 SOCKET_ERR_ALIGN);
  if (a.v)
    SOCKET_REQUIRE(socket_aligned16(a.v) && a.v_sb % per16 == 0 && a.v_sh % per16 == 0 && a.v_ss % per16 == 0, SOCKET_ERR_ALIGN);
  // (tile + grid size stays an int)
  SOCKET_REQUIRE((int64_t)a.B * a.Hkv * ((a.S + kStreamTile / 2 - 1) / (kStreamTile / 2)) < (1LL << 30), SOCKET_ERR_SHAPE);
  return SOCKET_OK;
}

}  // namespace

extern "C" int socket_hash_keys(const void* k, const void* v, int dtype, int64_t k_stride_b,
                                int64_t k_stride_h, int64_t k_stride_s, int64_t v_stride_b,
                                int64_t v_stride_h, int64_t v_stride_s, const void* planes_words,
                                uint32_t* codes, uint16_t* v_norm, const int32_t* pos_b, int t0,
                                int B, int Hkv, int S, int D, int L, int P, int64_t Tcap,
                                void* stream) {
  SOCKET_REQUIRE(k && planes_words && codes, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(v == nullptr || v_norm != nullptr, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(D == kD, SOCKET_ERR_UNSUPPORTED);
  const HashRows a = {k, v, dtype, k_stride_b, k_stride_h, k_stride_s, v_stride_b, v_stride_h, v_stride_s, planes_words, codes,
                      v_norm, pos_b, t0, B, Hkv, S, D, L, P, words_per_key(L, P), Tcap, nullptr, nullptr, 0, 0, 0};
  const int st = check_hash_rows(a);
  if (st != SOCKET_OK) return st;
  const SocketDeviceLimits& lim = socket_device_limits();
  const bool streamed = streams(a, lim);
  if (goes_direct(a, lim, streamed)) return launch_direct(a, lim, nullptr, (hipStream_t)stream);
  return streamed ? launch_stream<false>(a, lim, nullptr, (hipStream_t)stream) : launch_staged(a, lim, (hipStream_t)stream);
}

extern "C" int socket_hash_rows(const void* k, const void* v, int dtype, int64_t k_stride_b, int64_t k_stride_h,
                                int64_t k_stride_s, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_s,
                                const void* planes_words, uint32_t* codes, uint16_t* v_norm, const int32_t* pos_b, int t0,
                                int B, int Hkv, int S, int D, int L, int P, int64_t Tcap, void* stream) {
  SOCKET_REQUIRE(D > 0 && D <= kD && D % 8 == 0, SOCKET_ERR_UNSUPPORTED);
  const HashRows a = {k, v, dtype, k_stride_b, k_stride_h, k_stride_s, v_stride_b, v_stride_h, v_stride_s, planes_words, codes,
                      v_norm, pos_b, t0, B, Hkv, S, D, L, P, words_per_key(L, P), Tcap, nullptr, nullptr, 0, 0, 0};
  const int st = check_hash_rows(a);
  if (st != SOCKET_OK) return st;
  hipStream_t s = (hipStream_t)stream;
  const SocketDeviceLimits& lim = socket_device_limits();
  const bool streamed = streams(a, lim);
  if (goes_direct(a, lim, streamed)) return launch_direct(a, lim, nullptr, s);
  if (!streamed) return launch_staged(a, lim, s);
  return launch_stream<false>(a, lim, nullptr, s);
}

extern "C" int socket_cache_append(const void* k, const void* v, int dtype, int64_t k_stride_b, int64_t k_stride_h,
                                   int64_t k_stride_s, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_s,
                                   const void* planes_words, void* k_cache, void* v_cache, int64_t cache_stride_b,
                                   int64_t cache_stride_h, int64_t cache_stride_s, uint32_t* codes, uint16_t* v_norm,
                                   int32_t* lens, int t0, int B, int Hkv, int S, int D, int L, int P, int64_t Tcap,
                                   void* stream) {
  SOCKET_REQUIRE(k && v && k_cache && v_cache, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(D > 0 && D <= kD && D % 8 == 0, SOCKET_ERR_UNSUPPORTED);
  HashRows a = {k, v, dtype, k_stride_b, k_stride_h, k_stride_s, v_stride_b, v_stride_h, v_stride_s, planes_words, codes,
                v_norm, nullptr, t0, B, Hkv, S, D, L, P, words_per_key(L, P), Tcap, k_cache, v_cache, cache_stride_b,
                cache_stride_h, cache_stride_s};
  const int st = check_hash_rows(a);
  if (st != SOCKET_OK) return st;
  const int per16 = 16 / socket_dtype_bytes(dtype);
  SOCKET_REQUIRE(socket_aligned16(k_cache) && socket_aligned16(v_cache) && cache_stride_b % per16 == 0 &&
                     cache_stride_h % per16 == 0 && cache_stride_s % per16 == 0,
                 SOCKET_ERR_ALIGN);
  SOCKET_REQUIRE((int64_t)B * Hkv <= 65535 && cache_stride_s >= 0 && cache_stride_s < (1 << 28), SOCKET_ERR_SHAPE);
  hipStream_t s = (hipStream_t)stream;
  const SocketDeviceLimits& lim = socket_device_limits();
  const bool streamed = streams(a, lim);
  if (goes_direct(a, lim, streamed)) return launch_direct(a, lim, lens, s);
  if (streamed) return launch_stream<true>(a, lim, lens, s);
  // the rows' copy and the lengths
  const int64_t pieces = (int64_t)S * (D / per16);
  const dim3 grid((unsigned)((pieces + 256 * kCopyPieces - 1) / (256 * kCopyPieces)), (unsigned)(B * Hkv));
#define SOCKET_COPY(DT)                                                                                                    \
  hipLaunchKernelGGL((copy_rows_kernel<DT>), grid, dim3(256), 0, s, k, v, k_stride_b, k_stride_h, k_stride_s, v_stride_b,  \
                     v_stride_h, v_stride_s, k_cache, v_cache, cache_stride_b, cache_stride_h, cache_stride_s, lens, t0, B, \
                     Hkv, S, D)
  if (dtype == SOCKET_F32) SOCKET_COPY(DType_f32);
  else SOCKET_COPY(DType_bf16);      // (16-bit rows are moved as they are)
#undef SOCKET_COPY
  SOCKET_LAUNCH_CHECK();
  // Rows past what the caches of the chip hold are read back from where the copy has put them, whole heads in order,
  // rather than a token apart; fewer are nearer where they came from.  float32, 128 dims, 60 x 10 planes, the whole
  // append, caller's rows / cache: 8 x 2500 rows (20 MB) 31.3 / 32.5 us, 8 x 10000 62.7 / 61.9, 8 x 24000 147 / 142,
  // 8 x 60000 382 / 358.
  if ((int64_t)B * Hkv * S * D * (16 / per16) * 2 > (128ll << 20)) {
    const int64_t first = (int64_t)t0 * cache_stride_s * (16 / per16);
    a.k = (const char*)k_cache + first, a.v = (const char*)v_cache + first;
    a.k_sb = a.v_sb = cache_stride_b, a.k_sh = a.v_sh = cache_stride_h, a.k_ss = a.v_ss = cache_stride_s;
  }
  return launch_staged(a, lim, s);
}

extern "C" int socket_unpack_codes(const uint32_t* codes, int16_t* out, int B, int Hkv, int L, int P,
                                   int t0, int T, int64_t Tcap, int64_t out_stride_b,
                                   int64_t out_stride_h, int64_t out_stride_l, int64_t out_stride_t,
                                   void* stream) {
  SOCKET_REQUIRE(codes && out, SOCKET_ERR_NULL);
  const int NW = words_per_key(L, P);
  SOCKET_REQUIRE(NW > 0 && B > 0 && Hkv > 0 && T > 0 && t0 >= 0 && (int64_t)t0 + T <= Tcap,
                 SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE((int64_t)B * Hkv <= 65535, SOCKET_ERR_SHAPE);
  dim3 grid((T + 255) / 256, B * Hkv);
  hipLaunchKernelGGL(unpack_codes_kernel, grid, dim3(256), 0, (hipStream_t)stream, codes, out, Hkv, L,
                     P, t0, T, Tcap, NW, out_stride_b, out_stride_h, out_stride_l, out_stride_t);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

extern "C" int socket_pack_codes(const int16_t* in, int64_t in_stride_b, int64_t in_stride_h,
                                 int64_t in_stride_l, int64_t in_stride_t, uint32_t* codes, int B,
                                 int Hkv, int L, int P, int t0, int T, int64_t Tcap, void* stream) {
  SOCKET_REQUIRE(codes && in, SOCKET_ERR_NULL);
  const int NW = words_per_key(L, P);
  SOCKET_REQUIRE(NW > 0 && B > 0 && Hkv > 0 && T > 0 && t0 >= 0 && (int64_t)t0 + T <= Tcap,
                 SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE((int64_t)B * Hkv <= 65535, SOCKET_ERR_SHAPE);
  dim3 grid((T + 255) / 256, B * Hkv);
  hipLaunchKernelGGL(pack_codes_kernel, grid, dim3(256), 0, (hipStream_t)stream, in, in_stride_b,
                     in_stride_h, in_stride_l, in_stride_t, codes, Hkv, L, P, t0, T, Tcap, NW);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}
