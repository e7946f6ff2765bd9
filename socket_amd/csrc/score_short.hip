// K2: soft-collision scorer, calls with few tokens per CU (the persistent and the tiled launches: score.hip).
#include "score_entry.h"

namespace {

// ---------------------------------------------------------------------------
// The scorer of the packed cache for calls with few tokens per CU: every lane owns TPL tokens of one tile and nothing else.
//
// Such a call is bound by what a workgroup does once, not per token: the whole table passes through its LDS (491 KB of
// bf16 at L60 x P10 for four heads, which a CU pulls from its L2 in some 5 us) and every step of that is a trip to the L2.
// So the code words of a lane's tokens all sit in registers before the first lookup -- no code load ever shares a wait
// with the table copies -- and the copies of two slices are in flight while one is gathered from.  Tokens are dealt one to
// a lane over all sixteen waves, and a second one only where they do not suffice: with the four to a lane that the
// persistent kernel's loads want, 1000 tokens would leave twelve waves idle and the gathers of the rest exposed.
// us against the launches that served these calls before (8 rows, caches that hold the operands):
//   L60 x P10 bf16   4096 tokens 8.4 (18.3)   9001: 9.6 (16.3)   24001: 12.4 (16.8)   32771: 14.6 (17.5)   49153: 17.7 (17.8)
//            fp32               12.5 (38.9)        13.5 (26.2)         15.9 (27.1)          18.4 (27.5)          22.7 (25.9)
//   L32 x P8  bf16               4.8 (8.3)          5.2 (8.8)           6.1 (9.0)            7.5 (10.2)           8.9 (9.9)
// Past some 500 tokens per CU the lookups add to that (their LDS reads and the copies' LDS writes share one port).
// Measured and dropped: entries gathered from the L2 without LDS (64 cycles a load: 10.7 / 25.7 us at 4096 / 24001 tokens
// bf16; fp32 13.1 at 4096), four tokens to a lane (+2 us), the loop unrolled over the words (the same to 0.9 us slower:
// its code is fetched from the L2 as it runs).
// Needs: grouped table, entries of 2 or 4 heads, every packed word full, at most kShortWords words.
// Row r of (sequence, kv head, part of the head group) is workgroups r, r + rows, ...: with rows a multiple or a divisor
// of 8 each row stays on as few XCDs as it can, whose L2 then serves its table to all its workgroups.
// ---------------------------------------------------------------------------
constexpr int kShortLanes = 1024;     // lanes of a workgroup
constexpr int kShortWords = 20;      // packed words of a key at most
constexpr int kShortBuffers = 3;
constexpr int kShortSlice = 48 << 10;  // bytes of a full slice: three 1 KB copies a wave

template <int GP, class TT, int PT, int TPL>
__global__ __launch_bounds__(kShortLanes) void score_short_kernel(
    const typename TT::elem* __restrict__ q_table, const uint32_t* __restrict__ codes,
    const uint16_t* __restrict__ v_norm, const int32_t* __restrict__ lens, float* __restrict__ scores,
    int Hq, int Hkv, int G, int T, int64_t Tcap, int64_t score_stride, int NW, int hsplit, int rows, int tile_tokens,
    uint32_t bf16_one, int fill_masked) {
  typedef typename TT::elem TE;
  constexpr int CPW = 32 / PT, EB = GP * (int)sizeof(TE), kWaves = kShortLanes / 64;
  constexpr int kTable = EB << PT, kWord = CPW * kTable;       // bytes of a table, of a word's tables
  constexpr int C = kShortSlice / kWord;                       // words of a slice
  constexpr int kCopies = kShortSlice / (kWaves * 1024);
  static_assert(C * kWord == kShortSlice && kCopies * kWaves * 1024 == kShortSlice, "slices are whole words and whole copies");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  const Bf16Select sel = make_bf16_select(bf16_one);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int row = blockIdx.x % rows, tile = blockIdx.x / rows;
  const int part = row % hsplit, pair = row / hsplit, b = pair / Hkv;
  const int geff = min(GP, G - part * GP);
  const int len = lens ? max(0, min(lens[b], T)) : T;
  const int start = tile * tile_tokens, end = min(start + tile_tokens, T);
  const int tok = start + tid;                        // the lane's first token; group i: kShortLanes i further
  float* out = scores + (int64_t)(b * Hq + (pair % Hkv) * G + part * GP) * score_stride;

  float acc[TPL][GP], vn[TPL];
#pragma unroll
  for (int i = 0; i < TPL; ++i) {
    vn[i] = 0.f;
#pragma unroll
    for (int g = 0; g < GP; ++g) acc[i][g] = 0.f;
  }

  if (start < len) {
    const char* table = reinterpret_cast<const char*>(q_table) + (int64_t)row * NW * kWord;
    const int table_bytes = NW * kWord;
    // this wave's share of slice `s` (as much of it as there is) -> LDS buffer `buf`
    auto copy_slice = [&](int s, int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int k = 0; k < kCopies; ++k) {
        const int o = (k * kWaves + wave) * 1024;
        if (s * kShortSlice + o < table_bytes) lds_dma16(table + s * kShortSlice + o + lane * 16, lds_raw + buf * kShortSlice + o);
      }
    };
    // groups of the wave that have a token (uniform)
    const int groups = min(TPL, max(0, (min(end, len) - start - wave * 64 + kShortLanes - 1) / kShortLanes));
    // (a lane without a token reads the tile's first, and stores nothing)
    // (a vector register file index that is the same in all lanes: the loop below is a few hundred bytes of code that stay
    // in the instruction cache, where a loop unrolled over the words would be fetched from the L2 as it runs)
    typedef uint32_t words_t __attribute__((ext_vector_type(32)));
    static_assert(kShortWords <= 32, "words_t");
    words_t word[TPL];
    uint16_t vraw[TPL] = {};
#pragma unroll
    for (int i = 0; i < TPL; ++i) {
      if (i >= groups) break;
      const int at = tok + i * kShortLanes < end ? tok + i * kShortLanes : start;
      const uint32_t* cw = codes + (int64_t)pair * NW * Tcap + at;
#pragma unroll
      for (int w = 0; w < kShortWords; ++w)
        if (w < NW) word[i][w] = __builtin_nontemporal_load(cw + (int64_t)w * Tcap);
      vraw[i] = v_norm[(int64_t)pair * Tcap + at];
    }
    for (int s = 0; s < kShortBuffers - 1; ++s) copy_slice(s, s);
    // The first two slices, the codes and the norms have landed; from here on the only memory operations in flight are
    // copies, which retire in order: a wait that leaves the copies of the slice after it in flight is a wait for a slice.
    wait_vmcnt(0);
    __syncthreads();
    copy_slice(kShortBuffers - 1, kShortBuffers - 1);
    int buf = 0;
    for (int s = 0, w = 0; w < NW; ++s) {
      if (s > 0) {
        // (a short last slice: everything is waited for)
        if ((s + 2) * C <= NW) wait_vmcnt(kCopies);
        else wait_vmcnt(0);
        __syncthreads();
        copy_slice(s + kShortBuffers - 1, buf);      // (into the buffer every wave has just left)
        buf = buf + 1 == kShortBuffers ? 0 : buf + 1;
      }
      const int wend = min(w + C, NW);
      if (groups == 0) {
        w = wend;
        continue;
      }
      const unsigned char* tw = lds_raw + buf * kShortSlice;
#pragma unroll 1
      for (; w < wend; ++w, tw += kWord) {
        RawEntry<EB> ent[CPW][TPL];
        static_for<TPL>([&](auto ii) __attribute__((always_inline)) {
          constexpr int i = decltype(ii)::value;
          if (i >= groups) return;
          const uint32_t x = word[i][w];
#pragma unroll
          for (int j = 0; j < CPW; ++j) ent[j][i] = load_entry<EB>(tw + j * kTable + __builtin_amdgcn_ubfe(x, j * PT, PT) * EB);
        });
        static_for<TPL>([&](auto ii) __attribute__((always_inline)) {
          constexpr int i = decltype(ii)::value;
          if (i >= groups) return;
#pragma unroll
          for (int j = 0; j < CPW; ++j) accumulate<GP>(acc[i], ent[j][i], (const TT*)nullptr, sel);
        });
      }
    }
#pragma unroll
    for (int i = 0; i < TPL; ++i) vn[i] = f16_bits_to_f32((uint16_t)vraw[i]);
  }
  // (without the fill, positions at or past the length may stay as they are)
  const int written = fill_masked ? end : min(end, len);
#pragma unroll
  for (int i = 0; i < TPL; ++i) {
    if (tok + i * kShortLanes >= written) break;
#pragma unroll
    for (int g = 0; g < GP; ++g) {
      if (g >= geff) break;
      __builtin_nontemporal_store(tok + i * kShortLanes < len ? acc[i][g] * vn[i] : -INFINITY,
                                  out + (int64_t)g * score_stride + tok + i * kShortLanes);
    }
  }
}

}  // namespace

// Whether the kernel serves this call: the operands it is written for, and so few tokens that one round of workgroups holds
// them all.  Two tokens to a lane are as far as it pays: at that a workgroup's lookups take as long as the passage of the
// table, and the persistent kernel, which keeps four to a lane, is as fast (8 rows of 65535 tokens, L60 x P10: bf16 20.2
// against 18.4 us, 49153: 17.7 against 17.8; fp32 25.7 against 27.0; a group of 7 heads, 65535: bf16 19.8 against 24.0).
bool socket_score_short_serves(const ScoreArgs& a, size_t elem_bytes) {
  const SocketDeviceLimits& lim = socket_device_limits();
  const int G = a.Hq / a.Hkv;
  if (!a.grouped || a.row_range || G < 2 || (a.P != 8 && a.P != 10) || a.R != 1 << a.P) return false;
  const int cpw = 32 / a.P;
  if (a.L % cpw != 0 || a.L / cpw > kShortWords || lim.max_lds_per_block < kShortBuffers * kShortSlice) return false;
  const int width = G == 2 ? 2 : 4, hsplit = (G + width - 1) / width;
  const int64_t rows = (int64_t)a.B * a.Hkv * hsplit;
  return rows <= lim.cu_count && lim.cu_count / rows * (hsplit > 1 || elem_bytes == 4 ? 2 * kShortLanes : kShortLanes * 7 / 4) >= a.T;
}

namespace {

template <int GP, class TT, int PT, int TPL>
int launch_score_short(const ScoreArgs& a) {
  const SocketDeviceLimits& lim = socket_device_limits();
  const int G = a.Hq / a.Hkv, hsplit = (G + GP - 1) / GP;
  auto kern = score_short_kernel<GP, TT, PT, TPL>;
  constexpr int lds_bytes = kShortBuffers * kShortSlice;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes) != hipSuccess)
    return SOCKET_ERR_LAUNCH;
  // every row in as many equal tiles, whole waves of them, as there are CUs for it
  const int rows = a.B * a.Hkv * hsplit, per_row = lim.cu_count / rows;
  const int tile_tokens = ((a.T + per_row - 1) / per_row + 63) / 64 * 64;
  const int tiles = (a.T + tile_tokens - 1) / tile_tokens;
  hipLaunchKernelGGL(kern, dim3(rows * tiles), dim3(kShortLanes), lds_bytes, a.stream, (const typename TT::elem*)a.q_probs, a.codes,
                     a.v_norm, a.lens, a.scores, a.Hq, a.Hkv, G, a.T, a.Tcap, a.score_stride, a.L / (32 / PT), hsplit, rows,
                     tile_tokens, 0x3f80u, (a.flags & SOCKET_SCORE_SKIP_MASKED) ? 0 : 1);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

template <int GP, class TT, int PT>
int dispatch_short_p(const ScoreArgs& a) {
  const SocketDeviceLimits& lim = socket_device_limits();
  const int64_t rows = (int64_t)a.B * a.Hkv * ((a.Hq / a.Hkv + GP - 1) / GP);
  if (lim.cu_count / rows * kShortLanes >= a.T) return launch_score_short<GP, TT, PT, 1>(a);
  return launch_score_short<GP, TT, PT, 2>(a);
}

template <int GP, class TT>
int dispatch_short(const ScoreArgs& a) {
  return a.P == 10 ? dispatch_short_p<GP, TT, 10>(a) : dispatch_short_p<GP, TT, 8>(a);
}

}  // namespace

int socket_score_short(const ScoreArgs& a, size_t elem_bytes) {
  const bool two = a.Hq / a.Hkv == 2;
  if (elem_bytes == 4) return two ? dispatch_short<2, TabF32>(a) : dispatch_short<4, TabF32>(a);
  return two ? dispatch_short<2, TabBF16>(a) : dispatch_short<4, TabBF16>(a);
}

extern "C" int socket_score_lanes_serve(int B, int Hq, int Hkv, int T, int q_dtype, int L, int P, int R) {
  if (B <= 0 || Hq <= 0 || Hkv <= 0 || T <= 0 || Hq % Hkv != 0 || Hq / Hkv > 8 || L <= 0 || P < 1 || P > 16 || R <= 0) return -1;
  if (q_dtype != SOCKET_F32 && q_dtype != SOCKET_BF16) return -1;
  ScoreArgs a{};
  a.B = B; a.Hq = Hq; a.Hkv = Hkv; a.L = L; a.P = P; a.R = R; a.T = T;
  a.grouped = 1;
  return socket_score_short_serves(a, q_dtype == SOCKET_F32 ? 4 : 2) ? 1 : 0;
}
