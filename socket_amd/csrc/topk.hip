// K3: per-row top-k select with the "equal scores -> lower index first" rule,
// fused with the [sink | window | heavy] index-list assembly of
// GPT-FAST/kernels/sparse.py:57-95.
//
// Scores are mapped to order-preserving 32-bit keys and paired with the
// complemented index into 64-bit composites (key << 32 | ~index), so "larger
// composite" is exactly "higher score, then lower index" and all composites of a
// row are distinct.
//
// select_list_kernel, workgroups of 1024 lanes (512 where rows outnumber the CUs), selects in two ways:
//  * pooled: a superset of the row's m winners, at most kPoolCap composites, is
//    formed and the m-th largest located in it by range refinement -- a 2048-bin
//    LDS histogram over [lo, hi] (initially the pool's min / max, so the bins
//    spread over the values that occur and LDS atomics rarely collide), then the
//    bin holding the m-th becomes the new range, until it holds at most kCandCap
//    entries.  Because the composites are distinct, ties need no special case.
//    The pool is the whole row when that fits; otherwise everything at or above a
//    threshold estimated from a fixed sample of the row and aimed at about 2m
//    entries, found in one streaming pass over the row (compacted in LDS, then
//    held in registers).  Where CUs are to spare several workgroups share a row:
//    each streams its share against the same threshold and appends what passes
//    to the row's list in memory, and the last to arrive selects from that list,
//    in the same launch.  A pool that comes out shorter than m or longer than
//    kPoolCap (the sample misjudged the row, or one key value is massively
//    repeated) is dropped and the row redone from scratch: the result is always
//    exact, only the time differs.
//  * from scratch: the same refinement over the row itself, one pass per level
//    (the row stays in L2), until the m-th key's bin holds at most kCandCap keys;
//    one more pass collects the keys above the bin and the bin's own.  A single
//    key value with more than kCandCap copies (mass ties) is resolved by a
//    histogram over index ranges (lowest indices win).  The scorer can hand over
//    the row's key range, which saves the first pass.
// Either way the winners are put in order without a full sort: their level-0
// histogram bins already order them coarsely and a bin seldom holds more than a
// few, so each winner goes to (#winners in higher bins) + (#bin-mates beating
// it); crowded bins fall back to an in-LDS bitonic sort whose short exchange
// distances stay in registers and wave shuffles.  In the pooled path the first
// refinement pass is that level-0 histogram: every entry keeps the slot its
// bin's counter handed it, the scan that finds the m-th bin turns the counters
// into offsets, and when that one pass isolates the bin (the usual case) the
// winners are grouped by bin with no second count.
#include <utility>

#include "attend_row.h"


namespace {

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / SOCKET_WAVE;
constexpr int kBins = 2048;
constexpr int kCandCap = 2048;           // entries of the k-th bin kept in LDS
constexpr int kMaxBinForCounting = 128;  // larger bins are sorted, not rank-counted

constexpr int kBatch = kThreads * 16;  // scores a workgroup filters per batch (16 per lane)
constexpr int kPoolCap = 8192;         // composites pooled per row
constexpr int kMaxParts = 16;          // workgroups that share one row at most

typedef unsigned long long u64;

// Four consecutive scores.  Rows start on any multiple of four bytes (a row pitch of odd length is what a caller's
// [B,Hq,T] tensor has); the hardware takes 16-byte loads at such addresses, and a wave's 1024 bytes then touch nine
// 128-byte lines instead of eight (32 rows of 20881 / 32771 scores, us against a score at a time: 13.5 / 13.6 against
// 15.9 / 17.9).
typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// The key of minus infinity, which scores of masked positions are.
constexpr uint32_t kMaskedKey = 0x007fffffu;

// f(0) to f(N - 1), each index a constant from the start.  (An array that an unrolled loop indexes may still be one vector
// when registers are given out.  The slots of select_from_pool were one of eight registers, which the half workgroup moved to
// scratch and back around every entry, 80 spilled registers in all.  us, that loop / this: masked rows, 512 of 8192 23.2 / 10.5,
// 512 of 32768 29.2 / 20.7, 700 of 9000 32.6 / 21.3, 448 of 98304 48.7 / 41.1; unmasked, 448 of 98304 38.1 / 37.7.)
template <int I>
struct IntTag {
  static constexpr int value = I;
};
template <int... I, class F>
__device__ __forceinline__ void for_indices(std::integer_sequence<int, I...>, F&& f) {
  (f(IntTag<I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void for_constant(F&& f) {
  for_indices(std::make_integer_sequence<int, N>{}, f);
}

template <bool B>
struct BoolTag {
  static constexpr bool value = B;
};

struct SelectShared {
  u64 lo, hi;           // current key / composite range (inclusive)
  int need;             // winners still to take from inside [lo, hi]
  int bin_count;        // entries in the bin holding the k-th
  int done;
  int fill_above, fill_cand, fill_pool;
  int idx_star;         // mass ties: largest index taken among the ties
  int found_bin, found_before, found_count;
  u64 wmin[kWaves], wmax[kWaves];
  int wsum[kWaves];
  int wflag[kWaves];
  uint32_t kmin, kmax;  // key range of the pool
  int base;             // where this workgroup's entries go in the row's shared list
  int last;             // this workgroup is the last of its row to arrive
  int crowded;          // a bin above the k-th holds more than kMaxBinForCounting entries
};

__device__ __forceinline__ u64 composite(uint32_t key, int idx) {
  return ((u64)key << 32) | (u64)(0xffffffffu - (uint32_t)idx);
}
__device__ __forceinline__ int32_t composite_index(u64 c) {
  return (int32_t)(0xffffffffu - (uint32_t)(c & 0xffffffffull));
}

// Minimum and maximum over the 64 lanes, left in lane 63 (the same six steps as
// the prefix sum; lanes a step does not reach take the identity).
__device__ __forceinline__ void wave_minmax_to_last(uint32_t& kmin, uint32_t& kmax) {
#define SOCKET_MINMAX_STEP(ctrl, rows)                                                                        \
  kmin = min(kmin, (uint32_t)__builtin_amdgcn_update_dpp((int)0xffffffffu, (int)kmin, ctrl, rows, 0xf, false)); \
  kmax = max(kmax, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)kmax, ctrl, rows, 0xf, false));
  SOCKET_MINMAX_STEP(0x111, 0xf)   // row_shr:1
  SOCKET_MINMAX_STEP(0x112, 0xf)   // row_shr:2
  SOCKET_MINMAX_STEP(0x114, 0xf)   // row_shr:4
  SOCKET_MINMAX_STEP(0x118, 0xf)   // row_shr:8
  SOCKET_MINMAX_STEP(0x142, 0xa)   // row_bcast:15 into rows 1 and 3
  SOCKET_MINMAX_STEP(0x143, 0xc)   // row_bcast:31 into rows 2 and 3
#undef SOCKET_MINMAX_STEP
}

__device__ __forceinline__ u64 shfl_xor_u64(u64 v, int mask) {
  const uint32_t lo = (uint32_t)__shfl_xor((int)(uint32_t)v, mask, SOCKET_WAVE);
  const uint32_t hi = (uint32_t)__shfl_xor((int)(uint32_t)(v >> 32), mask, SOCKET_WAVE);
  return ((u64)hi << 32) | lo;
}

// Sum of sums[0, wave) of W <= 16 waves: every wave scans all of them, one to a lane.  (One LDS read a wave; each lane reading
// them one after another was 256 reads a workgroup, 0.4 us of each of the two or three calls of a selection.)
template <int W>
__device__ __forceinline__ int earlier_waves(const int* sums, int lane, int wave) {
  static_assert(W <= 16 && (W & (W - 1)) == 0, "a row of 16 lanes");
  int v = sums[lane & (W - 1)];
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);   // row_shr:1
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);   // row_shr:2
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);   // row_shr:4
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);   // row_shr:8
  const int w = __builtin_amdgcn_readfirstlane(wave);
  const int s = __builtin_amdgcn_readlane(v, (w + 63) & 63);        // (lane w - 1)
  return w > 0 ? s : 0;
}

// All THREADS lanes.  Ranks the bins from the top (descending != 0) or from the
// bottom, kBins / THREADS per lane, and publishes in `sh` the bin where the
// running count first reaches `need`, the count ranked before it and its own.
// With OFFSETS every bin's counter is replaced by `entries ranked before the bin |
// its own count << 16` (each lane rewrites the bins it read, nobody else's), and
// sh.crowded is raised (never cleared here) when a bin ranked wholly before the
// found one holds more than kMaxBinForCounting entries.
// `on_found(bin, ranked before it, its count)` runs in the one lane that finds the
// bin, before the closing barrier: what it writes to `sh` every lane sees afterwards.
struct NoFoundAction {
  __device__ void operator()(int, int, int) const {}
};
template <int THREADS, bool OFFSETS = false, class F = NoFoundAction>
__device__ __forceinline__ void find_bin(uint32_t* hist, int need, int descending, SelectShared& sh,
                                         int tid, F&& on_found = F()) {
  constexpr int PER = kBins / THREADS;
  const int lane = tid & 63, wave = tid >> 6;
  int c[PER], mine = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int r = tid * PER + i;
    c[i] = (int)hist[descending ? (kBins - 1 - r) : r];
    mine += c[i];
  }
  const int incl_w = wave_incl_scan(mine, lane);
  if (lane == 63) sh.wsum[wave] = incl_w;
  __syncthreads();
  int run = incl_w - mine + earlier_waves<THREADS / SOCKET_WAVE>(sh.wsum, lane, wave);
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (run < need && need <= run + c[i]) {
      const int r = tid * PER + i;
      sh.found_bin = descending ? (kBins - 1 - r) : r;
      sh.found_before = run;
      sh.found_count = c[i];
      on_found(descending ? (kBins - 1 - r) : r, run, c[i]);
    }
    if constexpr (OFFSETS) {
      const int r = tid * PER + i;
      hist[descending ? (kBins - 1 - r) : r] = (uint32_t)run | ((uint32_t)c[i] << 16);
      if (c[i] > kMaxBinForCounting && run + c[i] < need) sh.crowded = 1;
    }
    run += c[i];
  }
  __syncthreads();
}

// Visit row[begin:n) once, 16 bytes per lane per load and eight loads in flight
// per lane (a lone workgroup per row has to cover the memory latency itself).
template <int THREADS, class F>
__device__ __forceinline__ void for_each_in(const float* row, int begin, int n, int tid, F&& f) {
  constexpr int U = 8;
  const int n4 = n & ~3;   // begin is a multiple of 4
  constexpr int kStride = THREADS * 4;
  int i = begin + tid * 4;
  for (; i + (U - 1) * kStride < n4; i += U * kStride) {
    f32x4_any x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) x[u] = *reinterpret_cast<const f32x4_any*>(row + i + u * kStride);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      f(i + u * kStride, x[u].x);
      f(i + u * kStride + 1, x[u].y);
      f(i + u * kStride + 2, x[u].z);
      f(i + u * kStride + 3, x[u].w);
    }
  }
  for (; i < n4; i += kStride) {
    const f32x4_any x = *reinterpret_cast<const f32x4_any*>(row + i);
    f(i, x.x);
    f(i + 1, x.y);
    f(i + 2, x.z);
    f(i + 3, x.w);
  }
  for (int t = max(n4, begin) + tid; t < n; t += THREADS) f(t, row[t]);
}

// Append `value` to a list if `take`: one LDS atomic per wave, positions handed
// out by a ballot prefix count.  Safe under divergence (only active lanes vote).
__device__ __forceinline__ void wave_append(bool take, u64 value, int* cursor, u64* list, int cap) {
  const u64 mask = __ballot(take);
  if (mask == 0) return;
  const int lane = threadIdx.x & 63;
  const int leader = __ffsll((long long)mask) - 1;
  int base = 0;
  if (lane == leader) base = atomicAdd(cursor, __popcll(mask));
  base = __builtin_amdgcn_readlane(base, leader);   // (leader is wave-uniform: a scalar read, no LDS crossbar)
  if (take) {
    const int p = base + __popcll(mask & ((1ull << lane) - 1ull));
    if (p < cap) list[p] = value;
  }
}

// Bitonic sort of buf[0:np] (np a power of two) into descending order by the
// whole workgroup.  Lane t owns elements [t*E, (t+1)*E): exchange
// distances below E stay in registers, below 64*E go through wave shuffles, and
// only the longer ones through LDS with a barrier.  Callers sync before and get
// a synced buffer back.
template <int E, int THREADS>
__device__ __forceinline__ void sort_desc_impl(u64* buf, int np, int tid) {
  const bool active = tid * E < np;
  u64 r[E];
  auto load = [&]() {
#pragma unroll
    for (int e = 0; e < E; ++e) r[e] = active ? buf[tid * E + e] : 0ull;
  };
  auto store = [&]() {
    if (active) {
#pragma unroll
      for (int e = 0; e < E; ++e) buf[tid * E + e] = r[e];
    }
  };
  auto reg_stages = [&](int k, int jstart) {
    for (int j = jstart; j >= E; j >>= 1) {  // partner in another lane of the wave
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const int i = tid * E + e;
        const u64 other = shfl_xor_u64(r[e], j / E);
        const bool lower = (i & j) == 0, desc = (i & k) == 0;
        const u64 mx = r[e] > other ? r[e] : other;
        const u64 mn = r[e] > other ? other : r[e];
        r[e] = (lower == desc) ? mx : mn;
      }
    }
#pragma unroll
    for (int j = E / 2; j >= 1; j >>= 1) {  // partner in this lane
      if (j > jstart) continue;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        if (e & j) continue;
        const int p = e | j;
        const bool desc = ((tid * E + e) & k) == 0;
        const u64 a = r[e], c = r[p];
        const u64 mx = a > c ? a : c, mn = a > c ? c : a;
        r[e] = desc ? mx : mn;
        r[p] = desc ? mn : mx;
      }
    }
  };
  const int span = 64 * E;  // distances below this never leave the wave
  load();
  for (int k = 2; k <= np && k <= span; k <<= 1) reg_stages(k, k >> 1);
  store();
  __syncthreads();
  for (int k = 2 * span; k <= np; k <<= 1) {
    for (int j = k >> 1; j >= span; j >>= 1) {
      for (int i = tid; i < np; i += THREADS) {
        const int p = i ^ j;
        if (p > i) {
          const u64 a = buf[i], c = buf[p];
          const bool desc = (i & k) == 0;
          if (desc ? (a < c) : (a > c)) {
            buf[i] = c;
            buf[p] = a;
          }
        }
      }
      __syncthreads();
    }
    load();
    reg_stages(k, span >> 1);
    store();
    __syncthreads();
  }
}

template <int THREADS>
__device__ __forceinline__ void sort_desc(u64* buf, int np, int tid) {
  if (np <= THREADS) sort_desc_impl<1, THREADS>(buf, np, tid);
  else if (np == 2 * THREADS) sort_desc_impl<2, THREADS>(buf, np, tid);
  else if (np == 4 * THREADS) sort_desc_impl<4, THREADS>(buf, np, tid);
  else if (np == 8 * THREADS) sort_desc_impl<8, THREADS>(buf, np, tid);
  else sort_desc_impl<16, THREADS>(buf, np, tid);
}

__device__ __forceinline__ int next_pow2_dev(int x) {
  return x <= 1 ? 1 : 1 << (32 - __clz(x - 1));
}

// Row length n and heavy budget m of a row of sequence b (m clipped to the room
// the list row leaves after the sink / window part), and that part's length.
__device__ __forceinline__ void row_shape(const int32_t* lens, const int32_t* budgets, int b, int T,
                                          int M, int sink, int window, int write_base, int list_width,
                                          int& n, int& m, int& nbase) {
  n = lens ? max(0, min(lens[b], T)) : T;
  m = budgets ? budgets[b] : M;
  m = max(0, min(min(m, M), n));
  nbase = 0;
  if (write_base) {
    const int s_e = max(0, min(sink, n));
    const int w_e = max(0, min(window, n));
    const int win_start = max(n - w_e, s_e);
    nbase = s_e + ((w_e > 0 && win_start < n) ? n - win_start : 0);
    if (nbase == 0) nbase = 1;
  }
  m = max(0, min(nbase + m, list_width) - nbase);
}

// What the list holds for a position.
template <bool MASKED>
__device__ __forceinline__ int32_t listed(int32_t at, const uint8_t* ok) {
  if constexpr (MASKED) return at >= 0 && ok[at] ? at : -1;
  else return at;
}

// Sink / window part of a list row, its length and the -1 padding.
template <bool MASKED>
__device__ __forceinline__ void write_list_base(int32_t* out, int n, int m, int nbase, int sink,
                                                int window, int write_base, int list_width,
                                                int32_t* len_out, const uint8_t* ok, int tid, int nthreads) {
  if (write_base) {
    const int s_e = max(0, min(sink, n));
    const int w_e = max(0, min(window, n));
    const int win_start = max(n - w_e, s_e);
    if (s_e + ((w_e > 0 && win_start < n) ? n - win_start : 0) == 0) {
      if (tid == 0 && list_width > 0) out[0] = listed<MASKED>(n - 1, ok);
    } else {
      for (int i = tid; i < nbase && i < list_width; i += nthreads)
        out[i] = listed<MASKED>(i < s_e ? i : win_start + (i - s_e), ok);
    }
  }
  const int total = min(nbase + m, list_width);
  for (int i = total + tid; i < list_width; i += nthreads) out[i] = -1;
  if (len_out && tid == 0) *len_out = total;
}

// Smallest shift for which [lo, hi] maps onto at most kBins bins.
// (In closed form: span >> shift < kBins = 2^11 as soon as shift >= bits(span) - 11.
// Counting the shift up in a loop cost 40-odd trips of 64-bit shifts per call for
// composites, on every wave: 1.5-2 us a call with four waves to a SIMD.)
__device__ __forceinline__ int range_shift(u64 lo, u64 hi) {
  static_assert(kBins == 2048, "range_shift assumes 2^11 bins");
  const u64 span = hi - lo;
  const int bits = span ? 64 - __clzll((long long)span) : 0;
  return bits > 11 ? bits - 11 : 0;
}

// Bin of a composite in the histogram that starts at lo0.  Where positions may be masked it starts at the lowest one
// that is not: the others lie below it, and every place that bins counts them in the lowest bin (a difference that wraps is
// no bin, and there can be thousands of them above the m-th entry of a row that has fewer allowed positions than m).
template <bool MASKED>
__device__ __forceinline__ int level0_bin(u64 v, u64 lo0, int shift0) {
  return MASKED && v < lo0 ? 0 : (int)((v - lo0) >> shift0);
}

// Final step of both paths.  buf[0:n_above) holds the winners above the k-th
// bin, cand[0:ncand) the k-th bin's entries of which the best `need` win; the
// n_above + need winners are written in descending order at out[0:...).
// Winners are placed by their level-0 bin with counting ranks
// when `counting_ok` (tmp then has 2 * cap_above slots) and no bin is crowded,
// else by the bitonic sort.  All lanes; callers sync before; no barrier at
// the end.
template <bool MASKED, int THREADS>
__device__ __forceinline__ void order_and_write(u64* buf, int n_above, u64* cand, int ncand, int need,
                                                u64 lo0, int shift0, u64* tmp, uint32_t* hist,
                                                SelectShared& sh, bool counting_ok, int32_t* out,
                                                const uint8_t* ok, int tid, bool placed = false) {
  const int lane = tid & 63, wave = tid >> 6;
  // ---- the k-th bin: rank its entries, the best `need` follow the winners ----------
  if (ncand <= kMaxBinForCounting || need == ncand) {
    // (by the last lanes: the first have most of the winners)
    for (int i = THREADS - 1 - tid; i < ncand; i += THREADS) {
      const u64 v = cand[i];
      int r = 0;
#pragma unroll 4
      for (int j = 0; j < ncand; ++j) r += cand[j] > v;
      if (r < need) out[n_above + r] = listed<MASKED>(composite_index(v), ok);
    }
  } else {
    const int npc = next_pow2_dev(ncand);
    for (int i = ncand + tid; i < npc; i += THREADS) cand[i] = 0ull;
    __syncthreads();
    sort_desc<THREADS>(cand, npc, tid);
    for (int i = tid; i < need; i += THREADS) out[n_above + i] = listed<MASKED>(composite_index(cand[i]), ok);
  }
  if (n_above == 0) return;

  // ---- winners above the bin ----------------------------------------------------------
  if (placed) {
    // `buf` holds them grouped by level-0 bin already, hist[bin] = offset | population << 16
    for (int p = tid; p < n_above; p += THREADS) {
      const u64 v = buf[p];
      const uint32_t h = hist[level0_bin<MASKED>(v, lo0, shift0)];
      const int s0 = (int)(h & 0xffffu), c = (int)(h >> 16);
      int r = 0;
      for (int q = s0; q < s0 + c; ++q) r += buf[q] > v;
      out[s0 + r] = listed<MASKED>(composite_index(v), ok);
    }
    return;
  }
  if (counting_ok) {
    for (int i = tid; i < kBins; i += THREADS) hist[i] = 0;
    __syncthreads();
    for (int i = tid; i < n_above; i += THREADS) {
      const int bin = level0_bin<MASKED>(buf[i], lo0, shift0);
      const uint32_t slot = atomicAdd(&hist[bin], 1u);
      tmp[i] = ((u64)bin << 32) | slot;  // parked until the offsets are known
    }
    __syncthreads();
    // descending exclusive scan over the bins, PER per lane; crowded-bin check
    constexpr int PER = kBins / THREADS;
    int c[PER], mine = 0, full = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      c[i] = (int)hist[kBins - 1 - PER * tid - i];
      mine += c[i];
      full |= c[i] > kMaxBinForCounting;
    }
    const int incl_w = wave_incl_scan(mine, lane);
    const int crowded = __any(full);
    if (lane == 63) sh.wsum[wave] = incl_w;
    if (lane == 0) sh.wflag[wave] = crowded;
    __syncthreads();
    int base = 0, any_crowded = 0;
    for (int w = 0; w < (THREADS / SOCKET_WAVE); ++w) {
      if (w < wave) base += sh.wsum[w];
      any_crowded |= sh.wflag[w];
    }
    int excl = base + incl_w - mine;
    __syncthreads();
    if (!any_crowded) {
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        hist[kBins - 1 - PER * tid - i] = (uint32_t)excl | ((uint32_t)c[i] << 16);  // offset | population << 16
        excl += c[i];
      }
      __syncthreads();
      u64* grouped = tmp + n_above;
      for (int i = tid; i < n_above; i += THREADS) {
        const int bin = (int)(tmp[i] >> 32);
        const int slot = (int)(tmp[i] & 0xffffffffull);
        grouped[(hist[bin] & 0xffffu) + slot] = buf[i];
      }
      __syncthreads();
      for (int p = tid; p < n_above; p += THREADS) {
        const u64 v = grouped[p];
        const uint32_t h = hist[level0_bin<MASKED>(v, lo0, shift0)];
        const int s0 = (int)(h & 0xffffu), c = (int)(h >> 16);
        int r = 0;
        for (int q = s0; q < s0 + c; ++q) r += grouped[q] > v;
        out[s0 + r] = listed<MASKED>(composite_index(v), ok);
      }
      return;
    }
  }
  const int np = next_pow2_dev(n_above);
  for (int i = n_above + tid; i < np; i += THREADS) buf[i] = 0ull;
  __syncthreads();
  sort_desc<THREADS>(buf, np, tid);
  for (int j = tid; j < n_above; j += THREADS) out[j] = listed<MASKED>(composite_index(buf[j]), ok);
}

// ---------------------------------------------------------------------------
// threshold from a sample
// ---------------------------------------------------------------------------
// A pool of kPoolCap composites can be relied on to hold a row's m winners when
// it is filled with everything above a threshold aimed at max(2m, 1024) entries.
__host__ __device__ __forceinline__ bool sampling_ok(int m) {
  const int target = 2 * m > 1024 ? 2 * m : 1024;
  return target + target / 2 <= kPoolCap;
}

// All THREADS lanes; returns (to every lane) a key tau such that about
// max(2m, 1024) of the row's n scores have keys >= tau.  The estimate comes from
// a fixed sample of the row -- runs of 64 consecutive scores at evenly spaced
// places, 4096 scores in all (16384 for rows beyond 262144) -- whose r-th largest
// key is located with the same histogram refinement as everywhere else; tau is
// the lower edge of its bin.  Every workgroup that calls this for a row gets the
// same tau.  Needs n > kPoolCap; clears hist itself (nobody may be using it).  When
// it returns every lane has passed the barrier that follows the last read of hist.
constexpr int kSample = 4096, kLongSample = 16384;
template <int THREADS>
constexpr int kSampleVecs = kLongSample / 4 / THREADS;   // groups of four per lane at most

// The sample's scores, requested ahead of the row's first batches: what is asked for first arrives first.
template <int THREADS>
__device__ __forceinline__ void request_sample(const float* row, int n, f32x4_any (&x)[kSampleVecs<THREADS>], int tid) {
  const int nsample = n <= 262144 ? kSample : kLongSample;
  const int nq = nsample / 4 / THREADS;  // 1 or 4 (1024 lanes), 2 or 8 (512 lanes)
  const int shift = nsample == kSample ? 6 : 8;          // runs of 64 scores, 2^shift of them
#pragma unroll
  for (int j = 0; j < kSampleVecs<THREADS>; ++j) {
    if (j < nq) {
      const int q = j * THREADS + tid;
      const int at = (int)(((int64_t)(q >> 4) * n >> shift) & ~3ll) + (q & 15) * 4;
      x[j] = *reinterpret_cast<const f32x4_any*>(row + at);
    }
  }
}

template <int THREADS, bool MASKED>
__device__ __forceinline__ uint32_t sample_threshold(const f32x4_any (&x)[kSampleVecs<THREADS>], int n, int m, uint32_t* hist,
                                                     SelectShared& sh, int tid) {
  constexpr int kMaxQ = kSampleVecs<THREADS>;
  const int lane = tid & 63, wave = tid >> 6;
  const int nsample = n <= 262144 ? kSample : kLongSample;
  const int nq = nsample / 4 / THREADS;
  uint32_t key[kMaxQ * 4];
  for (int i = tid; i < kBins; i += THREADS) hist[i] = 0;   // (no one uses hist before this call)
#pragma unroll
  for (int j = 0; j < kMaxQ; ++j) {
    if (j < nq) {
#pragma unroll
      for (int c = 0; c < 4; ++c) key[j * 4 + c] = score_to_key(x[j][c]);
    }
  }
  uint32_t kmin = 0xffffffffu, kmax = 0u;
#pragma unroll
  for (int j = 0; j < kMaxQ; ++j) {
    if (j < nq) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (!MASKED || key[j * 4 + c] > kMaskedKey) kmin = min(kmin, key[j * 4 + c]);
        kmax = max(kmax, key[j * 4 + c]);
      }
    }
  }
  wave_minmax_to_last(kmin, kmax);
  if (lane == 63) {
    sh.wmin[wave] = kmin;
    sh.wmax[wave] = kmax;
  }
  __syncthreads();   // (also: hist is zero everywhere)
  // every wave reduces the waves' extremes for itself
  kmin = (uint32_t)sh.wmin[lane & (THREADS / SOCKET_WAVE - 1)];
  kmax = (uint32_t)sh.wmax[lane & (THREADS / SOCKET_WAVE - 1)];
  wave_minmax_to_last(kmin, kmax);
  const uint32_t smax = (uint32_t)__builtin_amdgcn_readlane((int)kmax, 63);
  const uint32_t smin = min((uint32_t)__builtin_amdgcn_readlane((int)kmin, 63), smax);
  const int target = max(2 * m, 1024);
  const int r = (int)min((int64_t)nsample, ((int64_t)target * nsample + n - 1) / n);
  const int fine = max(4, r / 8);  // a bin this small pins tau well enough
  for (int iter = 0; iter < 4; ++iter) {
    // the first pass takes its range from the sample's extremes, the later ones from
    // what the pass before published
    const uint32_t lo = iter ? (uint32_t)sh.lo : smin, hi = iter ? (uint32_t)sh.hi : smax;
    const int need_in = iter ? sh.need : r;
    const int shift = range_shift(lo, hi);
    if (iter) {
      for (int i = tid; i < kBins; i += THREADS) hist[i] = 0;
      __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < kMaxQ; ++j) {
      if (j < nq) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const uint32_t k = MASKED ? max(key[j * 4 + c], smin) : key[j * 4 + c];
          if (k >= lo && k <= hi) atomicAdd(&hist[(k - lo) >> shift], 1u);
        }
      }
    }
    __syncthreads();
    find_bin<THREADS>(hist, need_in, 1, sh, tid, [&](int bin, int before, int count) {
      const uint32_t blo = lo + ((uint32_t)bin << shift);
      const uint32_t bspan = (shift == 0) ? 0u : ((1u << shift) - 1u);
      sh.lo = blo;
      sh.hi = (hi - blo < bspan) ? hi : blo + bspan;
      sh.need = need_in - before;
      sh.done = (count <= fine || shift == 0) ? 1 : 0;
    });
    if (sh.done) break;
  }
  return (uint32_t)sh.lo;
}

// ---------------------------------------------------------------------------
// rows
// ---------------------------------------------------------------------------
// Agent-wide coherent accesses without a fence (written through / read past this
// die's caches): what workgroups of one row on different dies exchange.
__device__ __forceinline__ void store_coherent(u64* p, u64 v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 load_coherent(const u64* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// from a pool in registers, kPoolCap / THREADS entries per lane
// ---------------------------------------------------------------------------
// A row of at most kPoolCap scores, all of it (past its end: zeros, which no load asks the memory for).
template <int THREADS>
__device__ __forceinline__ void request_row(const float* row, int n, f32x4_any (&x)[kPoolCap / THREADS / 4], int tid) {
  const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(row), 0, n * 4, 0x00027000);
#pragma unroll
  for (int u = 0; u < kPoolCap / THREADS / 4; ++u)
    x[u] = __builtin_bit_cast(f32x4_any, __builtin_amdgcn_raw_buffer_load_b128(src, (u * THREADS + tid) * 16, 0, 0));
}

// Its entries, four neighbours to a lane and group, and the range of the keys that this lane holds.
template <bool MASKED, int THREADS>
__device__ __forceinline__ void pool_row(const f32x4_any (&x)[kPoolCap / THREADS / 4], int n, u64 (&pv)[kPoolCap / THREADS],
                                         uint32_t& have, uint32_t& kmin, uint32_t& kmax, int tid) {
#pragma unroll
  for (int u = 0; u < kPoolCap / THREADS; ++u) {
    const int i = ((u >> 2) * THREADS + tid) * 4 + (u & 3);
    const uint32_t k = score_to_key(x[u >> 2][u & 3]);
    if (i < n) {
      if (!MASKED || k > kMaskedKey) kmin = min(kmin, k);
      kmax = max(kmax, k);
      have |= 1u << u;
    }
    pv[u] = composite(k, i);
  }
}

// All lanes: the m best of the pool's entries, in order, at heavy[0:m).  have: bit u where pv[u] is one; kmin / kmax: the
// range of this lane's keys; hist is zero, sh's counters and range are as select_list_kernel sets them, and a barrier lies behind both.
template <bool MASKED, int THREADS>
__device__ __forceinline__ void select_from_pool(const u64 (&pv)[kPoolCap / THREADS], uint32_t have, uint32_t kmin, uint32_t kmax, int m,
                                                 uint32_t* hist, SelectShared& sh, u64* buf, u64* cand, u64* tmp, int cap_above,
                                                 bool counting_ok, int32_t* heavy, const uint8_t* ok, int tid) {
  constexpr int U = kPoolCap / THREADS;
  static_assert(U <= 32, "a bit each");
  const int lane = tid & (SOCKET_WAVE - 1);
  // range of the pooled composites, from their keys (the high halves): any range
  // that holds them all serves the refinement
  wave_minmax_to_last(kmin, kmax);
  if (lane == 63) {
    atomicMin(&sh.kmin, kmin);
    atomicMax(&sh.kmax, kmax);
  }
  __syncthreads();
  const u64 lo0 = (u64)(MASKED ? min(sh.kmin, sh.kmax) : sh.kmin) << 32, hi0 = ((u64)sh.kmax << 32) | 0xffffffffull;
  const int shift0 = range_shift(lo0, hi0);
  // refinement on the composites; they are distinct, so it ends with a bin of
  // at most kCandCap entries (ties need no special case here).
  // The first pass covers every entry, and every entry keeps the slot that its
  // bin's counter hands out.  When that pass already isolates the k-th bin (the
  // usual case) the bins' counters, turned into offsets by the same scan that
  // finds the bin, and those slots place every winner next to the others of its
  // bin and the k-th bin's entries in their list with no further counting.
  {
    uint32_t slot2[U / 2] = {};   // 16 bits per entry  (hist is zero: cleared ahead of the pool)
    for_constant<U>([&](auto i) __attribute__((always_inline)) {
      constexpr int u = decltype(i)::value;
      if (have >> u & 1) {
        const uint32_t sl = atomicAdd(&hist[level0_bin<MASKED>(pv[u], lo0, shift0)], 1u);
        slot2[u >> 1] |= sl << (16 * (u & 1));
      }
    });
    __syncthreads();
    find_bin<THREADS, true>(hist, m, 1, sh, tid, [&](int bin, int before, int count) {
      const u64 blo = lo0 + ((u64)bin << shift0);
      const u64 bspan = (shift0 == 0) ? 0ull : ((1ull << shift0) - 1ull);
      sh.lo = MASKED && bin == 0 ? 0ull : blo;
      sh.hi = (hi0 - blo < bspan) ? hi0 : blo + bspan;
      sh.need = m - before;
      sh.done = (count <= kCandCap || shift0 == 0) ? 1 : 0;
    });
    if (sh.done && !sh.crowded) {
      const int fb = sh.found_bin, need = sh.need, ncand = min(sh.found_count, kCandCap);
      for_constant<U>([&](auto i) __attribute__((always_inline)) {
        constexpr int u = decltype(i)::value;
        if (have >> u & 1) {
          const u64 v = pv[u];
          const int bin = level0_bin<MASKED>(v, lo0, shift0);
          const int sl = (int)((slot2[u >> 1] >> (16 * (u & 1))) & 0xffffu);
          if (bin > fb) buf[(int)(hist[bin] & 0xffffu) + sl] = v;
          else if (bin == fb && sl < kCandCap) cand[sl] = v;
        }
      });
      __syncthreads();
      order_and_write<MASKED, THREADS>(buf, m - need, cand, ncand, need, lo0, shift0, tmp, hist, sh, counting_ok, heavy,
                                       ok, tid, true);
      return;
    }
  }
  for (int iter = 1; iter < 8 && !sh.done; ++iter) {
    const u64 lo = sh.lo, hi = sh.hi;
    const int need_in = sh.need;
    const int shift = range_shift(lo, hi);
    for (int i = tid; i < kBins; i += THREADS) hist[i] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const u64 v = pv[u];
      if ((have >> u & 1) && v >= lo && v <= hi) atomicAdd(&hist[(int)((v - lo) >> shift)], 1u);
    }
    __syncthreads();
    find_bin<THREADS>(hist, need_in, 1, sh, tid);
    if (tid == 0) {
      const u64 blo = lo + ((u64)sh.found_bin << shift);
      const u64 bspan = (shift == 0) ? 0ull : ((1ull << shift) - 1ull);
      sh.lo = blo;
      sh.hi = (hi - blo < bspan) ? hi : blo + bspan;
      sh.need = need_in - sh.found_before;
      sh.done = (sh.found_count <= kCandCap || shift == 0) ? 1 : 0;
    }
    __syncthreads();
    if (sh.done) break;
  }
  const u64 blo = sh.lo, bhi = sh.hi;
  const int need = sh.need;
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const u64 v = pv[u];
    const bool in = have >> u & 1;
    wave_append(in && v > bhi, v, &sh.fill_above, buf, cap_above);
    wave_append(in && v >= blo && v <= bhi, v, &sh.fill_cand, cand, kCandCap);
  }
  __syncthreads();
  order_and_write<MASKED, THREADS>(buf, m - need, cand, min(sh.fill_cand, kCandCap), need, lo0, shift0, tmp, hist, sh,
                                   counting_ok, heavy, ok, tid);
}

// `parts` workgroups per row (blockIdx.x = row * parts + part).  With parts > 1
// each filters its share of the row against the same sampled threshold (every
// part works it out for itself from the same sample), appends what passes to the
// row's list in `loc` (a stretch reserved with one atomic add on row_count), and
// the last part to arrive (row_done) selects from that list; the others leave.
// row_count and row_done are zero on entry and zero again on exit.
// The pooled composites are held in registers, kPoolCap / THREADS per lane, from the moment
// the pool is complete; LDS holds them only while they are being compacted.
// MASKED: a byte per score says whether its position may be listed; positions that may not become -1 in the list, and
// their scores are minus infinity.  Those are kept out of the ranges that the histograms are laid over (they count in
// the lowest bin): with them in, half the bins lie between minus infinity and the lowest score, and rows with a masked end
// took two passes more (56 rows of 4135, part of each masked: 19.1 us against 8.9).
template <bool MASKED, int THREADS>
__global__ __launch_bounds__(THREADS, 4) void select_list_kernel(
    const float* __restrict__ scores, const uint8_t* __restrict__ allowed, int64_t score_stride, const int32_t* __restrict__ lens,
    const int32_t* __restrict__ budgets, const uint32_t* __restrict__ row_range, int range_parts,
    int Hq, int T, int M, int sink, int window, int write_base, int32_t* __restrict__ sparse_list,
    int64_t list_stride, int list_width, int32_t* __restrict__ sparse_len, int cap_above,
    int counting_ok, int use_pool, int pool_slots, int parts, u64* __restrict__ loc,
    int32_t* __restrict__ row_count, unsigned int* __restrict__ row_done) {
  __shared__ uint32_t hist[kBins];
  __shared__ SelectShared sh;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds_raw[];
  u64* buf = reinterpret_cast<u64*>(lds_raw);  // winners                  [cap_above]
  u64* cand = buf + cap_above;                 // entries of the k-th bin  [kCandCap]
  // What passes the filter [pool_slots]: kPoolCap for rows beyond that.  In the half workgroup it lies over the rest,
  // which nothing writes before every lane holds its entries of the pool in registers.
  constexpr bool kPoolOver = THREADS < kThreads;
  u64* pool = kPoolOver ? buf : cand + kCandCap;
  u64* tmp = kPoolOver ? cand + kCandCap : pool + pool_slots;   // counting placement [2*cap_above] if counting_ok

  const int rowi = blockIdx.x / parts, part = blockIdx.x % parts;
  const int b = rowi / Hq;
  const int tid = threadIdx.x;
  const int lane = tid & (SOCKET_WAVE - 1);
  const int wave = tid / SOCKET_WAVE;
  int n, m, nbase;
  row_shape(lens, budgets, b, T, M, sink, window, write_base, list_width, n, m, nbase);
  const float* row = scores + (int64_t)rowi * score_stride;
  int32_t* out = sparse_list + (int64_t)rowi * list_stride;
  const uint8_t* ok = MASKED ? allowed + (int64_t)rowi * T : nullptr;
  auto list_base = [&]() __attribute__((always_inline)) {
    if (part == 0)
      write_list_base<MASKED>(out, n, m, nbase, sink, window, write_base, list_width,
                              sparse_len ? sparse_len + rowi : nullptr, ok, tid, THREADS);
  };
  if (m == 0) {
    list_base();
    return;
  }
  int32_t* heavy = out + nbase;

  // ================================ pooled select ======================================
  if (use_pool) {
    if (tid == 0) {
      sh.fill_above = 0;
      sh.fill_cand = 0;
      sh.fill_pool = 0;
      sh.kmin = 0xffffffffu;
      sh.kmax = 0u;
      sh.crowded = 0;
    }
    int total = -1;  // uniform; stays -1 when no pool could be formed
    uint32_t kmin = 0xffffffffu, kmax = 0u;  // key range of what this lane holds
    constexpr int U = kPoolCap / THREADS;
    u64 pv[U];                               // of the pool, this lane's
    uint32_t have = 0;                       // bit u: pv[u] is an entry
    if (n <= kPoolCap) {  // the whole row, by one workgroup
      if (part != 0) return;
      f32x4_any x[U / 4];
      request_row<THREADS>(row, n, x, tid);
      list_base();
      pool_row<MASKED, THREADS>(x, n, pv, have, kmin, kmax, tid);
      total = n;
      for (int i = tid; i < kBins; i += THREADS) hist[i] = 0;   // for the first refinement pass
      __syncthreads();
    } else if (sampling_ok(m)) {
      // This part's share of the row; the last part also takes the one to three
      // scores past the last multiple of four.
      const int n4 = n & ~3;
      const int chunk = (((n + parts - 1) / parts) + 3) & ~3;
      const int begin = min(part * chunk, n4), e4 = min(begin + chunk, n4);
      const int tail_end = (part == parts - 1) ? n : e4;
      // In batches of 16 scores per lane (four 16-byte loads, all in flight
      // together); the first two batches are requested before the threshold is
      // worked out, each further one two batches ahead of the one being filtered.  A
      // wave counts what passes in its batch, reserves a stretch of the pool with
      // one LDS atomic and writes its entries there: no barrier in the loop.
      constexpr int kLoads = 4, kStep = THREADS * 4 * kLoads;
      auto fetch = [&](int base, float4 (&x)[kLoads]) {
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
          // (past the end: the share's last four, fetched and ignored -- a load under
          // a condition would make every wait in the loop a wait for all loads)
          const int i0 = max(min(base + (u * THREADS + tid) * 4, e4 - 4), 0);
          const f32x4_any v = __builtin_nontemporal_load(reinterpret_cast<const f32x4_any*>(row + i0));
          x[u] = make_float4(v.x, v.y, v.z, v.w);
        }
      };
      // One batch of one wave.  Each of a lane's 16 scores is tested on the float (keys only for the pool): x passes when
      // it is not below the float whose key is tau.  A tau above +inf's key or below -inf's is no float's key and is
      // widened to that infinity (the pool only has to hold everything at or above tau; more is allowed).  A lane counts
      // its own; a scan over the lanes and one LDS atomic give it its stretch of the pool, which it fills in order: some
      // nine vector instructions a score, where ranking the lanes of every score's ballot took twenty (us, before / now: 32
      // rows of 32771 11.8 / 11.4, 256 of 65536 18.1 / 17.9, 448 of 98304 39.7 / 37.8).  A batch that would run past the
      // pool is counted but not written (the row is then redone from scratch anyway).
      auto filter_batch = [&](auto full, int base, const float4 (&x)[kLoads], float tau_f) {
        constexpr bool FULL = decltype(full)::value;   // every lane's 16 scores are inside the share
        int mine = 0;
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
          const float xs[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
          const bool in = FULL || base + (u * THREADS + tid) * 4 < e4;
#pragma unroll
          for (int c = 0; c < 4; ++c) mine += in && !(xs[c] < tau_f) ? 1 : 0;
        }
        const int upto = wave_incl_scan(mine, lane);
        const int total = __builtin_amdgcn_readlane(upto, 63);
        if (total == 0) return;  // uniform
        int at = 0;
        if (lane == 0) at = atomicAdd(&sh.fill_pool, total);
        at = __builtin_amdgcn_readfirstlane(at);
        if (at + total > kPoolCap) return;  // uniform
        const uint32_t cidx = 0xffffffffu - (uint32_t)(base + tid * 4);
        uint32_t addr = (uint32_t)(uintptr_t)(pool + at + upto - mine);
#pragma unroll
        for (int u = 0; u < kLoads; ++u) {
          const float xs[4] = {x[u].x, x[u].y, x[u].z, x[u].w};
          const bool in = FULL || base + (u * THREADS + tid) * 4 < e4;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            if (in && !(xs[c] < tau_f)) {
              // the two halves of the entry from wherever they are, in one write
              // (a 64-bit store would first copy them into a register pair)
              asm volatile("ds_write2_b32 %0, %1, %2 offset1:1"
                           :: "v"(addr), "v"(cidx - (uint32_t)(u * THREADS * 4 + c)), "v"(__float_as_uint(xs[c]))
                           : "memory");
              addr += 8;
            }
          }
        }
      };
      auto filter = [&](int base, const float4 (&x)[kLoads], float tau_f) {
        if (base >= e4) return;  // uniform
        if (base + kStep <= e4) filter_batch(BoolTag<true>{}, base, x, tau_f);
        else filter_batch(BoolTag<false>{}, base, x, tau_f);
      };
      float4 b0[kLoads], b1[kLoads], b2[kLoads];
      f32x4_any sample[kSampleVecs<THREADS>];
      request_sample<THREADS>(row, n, sample, tid);
      const float tail = e4 + lane < tail_end ? row[e4 + lane] : 0.f;     // (of wave 0)
      __builtin_amdgcn_sched_barrier(0);
      fetch(begin, b0);
      fetch(begin + kStep, b1);
      list_base();
      const uint32_t tau = sample_threshold<THREADS, MASKED>(sample, n, m, hist, sh, tid);
      for (int i = tid; i < kBins; i += THREADS) hist[i] = 0;   // for the first refinement pass
      const float tau_f = tau >= 0xff800000u ? INFINITY : tau <= 0x007fffffu ? -INFINITY
                          : __uint_as_float((tau & 0x80000000u) ? (tau & 0x7fffffffu) : ~tau);
      for (int base = begin; base < e4; base += 3 * kStep) {
        fetch(base + 2 * kStep, b2);
        filter(base, b0, tau_f);
        fetch(base + 3 * kStep, b0);
        filter(base + kStep, b1, tau_f);
        fetch(base + 4 * kStep, b1);
        filter(base + 2 * kStep, b2, tau_f);
      }
      __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the pool writes above are not the compiler's to wait for
      if (wave == 0) {
        const int i = e4 + lane;
        wave_append(i < tail_end && !(tail < tau_f), composite(__float_as_uint(tail), i), &sh.fill_pool, pool, kPoolCap);
      }
      __syncthreads();
      // (an entry of the pool: the score's bits over the complemented index)
      auto keyed = [](u64 e) {
        return ((u64)score_to_key(__uint_as_float((uint32_t)(e >> 32))) << 32) | (e & 0xffffffffull);
      };
      const int got = sh.fill_pool;   // what passed here, also when it is more than the pool holds
      if (parts == 1) {
        if (got >= m && got <= kPoolCap) {
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (tid + u * THREADS < got) pv[u] = keyed(pool[tid + u * THREADS]);
          total = got;
        }
      } else {
        if (tid == 0) sh.base = atomicAdd(&row_count[rowi], got);
        __syncthreads();
        const int at = sh.base;
        u64* mine = loc + (int64_t)rowi * kPoolCap;
        if (at + got <= kPoolCap) {   // (a row whose parts pass more than the list holds is redone from scratch)
          for (int i = tid; i < got; i += THREADS) store_coherent(mine + at + i, keyed(pool[i]));
        }
        // Every lane waits until its written-through stores have been acknowledged,
        // the barrier collects the lanes, and only then is the ticket drawn: whoever
        // draws the last one can read every part's entries.
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();
        if (tid == 0) sh.last = draw_ticket(&row_done[rowi], (unsigned int)(parts - 1)) == (unsigned int)(parts - 1);
        __syncthreads();
        if (!sh.last) return;
        const int sum = __hip_atomic_load(&row_count[rowi], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __syncthreads();
        if (tid == 0) __hip_atomic_store(&row_count[rowi], 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (sum >= m && sum <= kPoolCap) {
#pragma unroll
          for (int u = 0; u < U; ++u)
            if (tid + u * THREADS < sum) pv[u] = load_coherent(mine + tid + u * THREADS);
          total = sum;
        }
      }
      if (total >= 0) {
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (tid + u * THREADS < total) {
            have |= 1u << u;
            const uint32_t k = (uint32_t)(pv[u] >> 32);
            if (!MASKED || k > kMaskedKey) kmin = min(kmin, k);
            kmax = max(kmax, k);
          }
      }
    } else {
      if (part != 0) return;   // no threshold can be relied on: one workgroup selects from scratch
      list_base();
    }
    if (total >= 0) {
      select_from_pool<MASKED, THREADS>(pv, have, kmin, kmax, m, hist, sh, buf, cand, tmp, cap_above, counting_ok != 0, heavy, ok, tid);
      return;
    }
  } else {
    if (part != 0) return;
    list_base();
  }

  // ================================ from scratch ======================================
  // ---- key range of the row -----------------------------------------------------
  {
    uint32_t kmin = 0xffffffffu, kmax = 0u;
    if (row_range) {
      const uint32_t* rr = row_range + (int64_t)rowi * range_parts * 2;
      for (int i = tid; i < range_parts; i += THREADS) {
        kmin = min(kmin, rr[2 * i]);
        kmax = max(kmax, rr[2 * i + 1]);
      }
    } else {
      for_each_in<THREADS>(row, 0, n, tid, [&](int, float x) {
        const uint32_t k = score_to_key(x);
        kmin = min(kmin, k);
        kmax = max(kmax, k);
      });
    }
    wave_minmax_to_last(kmin, kmax);
    if (lane == 63) {
      sh.wmin[wave] = kmin;
      sh.wmax[wave] = kmax;
    }
    __syncthreads();
    if (tid == 0) {
      kmin = 0xffffffffu;
      kmax = 0u;
      for (int w = 0; w < (THREADS / SOCKET_WAVE); ++w) {
        kmin = min(kmin, (uint32_t)sh.wmin[w]);
        kmax = max(kmax, (uint32_t)sh.wmax[w]);
      }
      sh.lo = kmin;
      sh.hi = max(kmin, kmax);
      sh.need = m;
      sh.done = 0;
      sh.fill_above = 0;
      sh.fill_cand = 0;
      sh.idx_star = 0x7fffffff;
    }
    __syncthreads();
  }
  const uint32_t lo0 = (uint32_t)sh.lo;
  const int shift0 = range_shift(sh.lo, sh.hi);

  // ---- range refinement -------------------------------------------------------
  for (int iter = 0; iter < 4; ++iter) {
    const uint32_t lo = (uint32_t)sh.lo, hi = (uint32_t)sh.hi;
    const int need_in = sh.need;
    const int shift = range_shift(lo, hi);
    for (int i = tid; i < kBins; i += THREADS) hist[i] = 0;
    __syncthreads();
    for_each_in<THREADS>(row, 0, n, tid, [&](int, float x) {
      const uint32_t k = score_to_key(x);
      if (k >= lo && k <= hi) atomicAdd(&hist[(k - lo) >> shift], 1u);
    });
    __syncthreads();
    find_bin<THREADS>(hist, need_in, 1, sh, tid);
    if (tid == 0) {
      const uint32_t blo = lo + ((uint32_t)sh.found_bin << shift);
      const uint32_t bspan = (shift == 0) ? 0u : ((1u << shift) - 1u);
      sh.lo = blo;
      sh.hi = (hi - blo < bspan) ? hi : blo + bspan;
      sh.need = need_in - sh.found_before;
      sh.bin_count = sh.found_count;
      sh.done = (sh.found_count <= kCandCap || shift == 0) ? 1 : 0;
    }
    __syncthreads();
    if (sh.done) break;
  }

  const uint32_t blo = (uint32_t)sh.lo, bhi = (uint32_t)sh.hi;
  const int need = sh.need;  // keys to take from [blo, bhi]
  const int bin_count = sh.bin_count;
  const bool mass_ties = bin_count > kCandCap;  // then blo == bhi

  if (mass_ties) {
    // Take the `need` lowest indices among the keys equal to blo: histogram over
    // index ranges, then an in-order walk of the one range that straddles.
    const int binw = (n + kBins - 1) / kBins;
    for (int i = tid; i < kBins; i += THREADS) hist[i] = 0;
    __syncthreads();
    for_each_in<THREADS>(row, 0, n, tid, [&](int i, float x) {
      if (score_to_key(x) == blo) atomicAdd(&hist[i / binw], 1u);
    });
    __syncthreads();
    find_bin<THREADS>(hist, need, 0, sh, tid);
    if (wave == 0) {
      int rest = need - sh.found_before;  // >= 1 ties to take inside this index range
      const int i0 = sh.found_bin * binw, i1 = min(n, i0 + binw);
      int star = i0;
      for (int base = i0; base < i1 && rest > 0; base += SOCKET_WAVE) {
        const int i = base + lane;
        const bool eq = (i < i1) && (score_to_key(row[min(i, i1 - 1)]) == blo);
        const u64 mask = __ballot(eq);
        const int c = __popcll(mask);
        if (c >= rest) {
          u64 mm = mask;  // its rest-th set bit is the last tie taken
          for (int r = 1; r < rest; ++r) mm &= mm - 1;
          star = base + (__ffsll((long long)mm) - 1);
          rest = 0;
        } else {
          rest -= c;
        }
      }
      if (lane == 0) sh.idx_star = star;
    }
    __syncthreads();
  }

  // ---- collect ------------------------------------------------------------------
  const int idx_star = sh.idx_star;
  for_each_in<THREADS>(row, 0, n, tid, [&](int i, float x) {
    const uint32_t k = score_to_key(x);
    const u64 v = composite(k, i);
    const bool in_bin = k >= blo && k <= bhi;
    // mass ties: the ties with the lowest indices are winners outright (there can
    // be more of them than the candidate list holds)
    wave_append(k > bhi || (mass_ties && in_bin && i <= idx_star), v, &sh.fill_above, buf, cap_above);
    wave_append(!mass_ties && in_bin, v, &sh.fill_cand, cand, kCandCap);
  });
  __syncthreads();
  // mass ties: all m winners are in buf and there are no candidates
  const int ncand = mass_ties ? 0 : min(sh.fill_cand, kCandCap);
  const int n_above = mass_ties ? m : m - need;
  order_and_write<MASKED, THREADS>(buf, n_above, cand, ncand, mass_ties ? 0 : need, (u64)lo0 << 32, shift0 + 32, tmp, hist,
                  sh, counting_ok != 0, heavy, ok, tid);
}

// A short row's selection and its attention in one launch, a workgroup to a (b, h) row: the list stays in LDS.  Rows of at
// most kPoolCap scores whose list is one pass of row_attend, no more rows than CUs.  What bounds it is a chain of short
// phases on one CU; what it saves is a launch, and the list's way to memory and back.  Two launches / one, us: fp32, 32 rows
// of 4096, 196 entries 13.0 / 10.7, 128 rows 15.4 / 12.3, 256 rows of 2000, 168 entries 17.2 / 13.5; bf16, 32 rows of 8000, 504
// entries 15.7 / 13.9, 256 rows of 8192 27.2 / 20.9.  From one row up, where the two spread a row over many CUs: fp32, 1 / 8 rows of
// 4096 11.7 / 9.9 and 12.6 / 10.4; bf16, 1 / 8 rows of 8000, 504 entries 13.9 / 12.7 and 14.5 / 12.9, of 8192, 508 entries of 64 dims 16.4 / 14.8.
constexpr int kFuseList = 512;      // entries of a list at most
template <class DT, int D>
__global__ __launch_bounds__(kThreads, 4) void select_attend_kernel(
    const float* __restrict__ scores, int64_t score_stride, const int32_t* __restrict__ lens, const int32_t* __restrict__ budgets,
    int Hq, int T, int M, int sink, int window, int list_width, const typename DT::storage* __restrict__ q_,
    const typename DT::storage* __restrict__ k_, const typename DT::storage* __restrict__ v_, int64_t q_sb, int64_t q_sh, int64_t k_sb,
    int64_t k_sh, int64_t k_ss, int64_t v_sb, int64_t v_sh, int64_t v_ss, int G, int kv_rows, float sm_scale,
    typename DT::storage* __restrict__ out, int64_t out_sb, int64_t out_sh) {
  static_assert(kRowWaves * SOCKET_WAVE == kThreads, "one workgroup serves both parts");
  __shared__ uint32_t hist[kBins];
  __shared__ SelectShared sh;
  __shared__ u64 buf[kFuseList], cand[kCandCap], tmp[2 * kFuseList];
  __shared__ int32_t list[kFuseList];
  __shared__ float waves[kRowWaves][D + 2];
  const int b = blockIdx.x / Hq, h = blockIdx.x % Hq, kvh = h / G, tid = threadIdx.x;
  int n, m, nbase;
  row_shape(lens, budgets, b, T, M, sink, window, 1, list_width, n, m, nbase);
  if (m > 0) {
    const float* row = scores + (int64_t)blockIdx.x * score_stride;
    if (tid == 0) {
      sh.fill_above = 0;
      sh.fill_cand = 0;
      sh.kmin = 0xffffffffu;
      sh.kmax = 0u;
      sh.crowded = 0;
    }
    u64 pv[kPoolCap / kThreads];
    uint32_t have = 0, kmin = 0xffffffffu, kmax = 0u;
    f32x4_any x[kPoolCap / kThreads / 4];
    request_row<kThreads>(row, n, x, tid);
    for (int i = tid; i < kBins; i += kThreads) hist[i] = 0;
    write_list_base<false>(list, n, m, nbase, sink, window, 1, list_width, nullptr, nullptr, tid, kThreads);
    pool_row<false, kThreads>(x, n, pv, have, kmin, kmax, tid);
    __syncthreads();
    select_from_pool<false, kThreads>(pv, have, kmin, kmax, m, hist, sh, buf, cand, tmp, kFuseList, true, list + nbase, nullptr, tid);
  } else {
    write_list_base<false>(list, n, m, nbase, sink, window, 1, list_width, nullptr, nullptr, tid, kThreads);
  }
  __syncthreads();
  row_attend<DT, D>(q_ + b * q_sb + h * q_sh, k_ + b * k_sb + kvh * k_sh, k_ss, v_ + b * v_sb + kvh * v_sh, v_ss, list,
                    min(nbase + m, list_width), list_width, kv_rows, sm_scale, waves, out + b * out_sb + h * out_sh);
}

int next_pow2(int x) {
  int p = 1;
  while (p < x) p <<= 1;
  return p;
}

// Workgroups per row.  One workgroup streams its row at what one CU can pull
// (about 35 GB/s: 3.7 us per 32768 scores); sharing a row between several costs
// about 3 us for the exchange through memory, more when the launch then fills
// every CU (each part works out the threshold from the same sample, and each
// needs a CU to itself for its LDS).  Measured on 256 CUs with top-k 2048: two
// parts never pay; 8 or 32 rows gain from 49152 / 65536 scores up (9.5 and 7.6 us
// at 131072), 64 rows from 98304 up, 128 rows never.
int row_parts(int rows, int T, int m_max) {
  if (!(T > kPoolCap && m_max > 0 && sampling_ok(m_max))) return 1;
  const int cus = socket_device_limits().cu_count;
  int p = cus / rows;
  p = p < kMaxParts ? p : kMaxParts;
  p = p < T / kBatch ? p : T / kBatch;
  if (p < 3) return 1;
  const double saved = (double)T * (p - 1) / p;                 // scores a workgroup no longer streams
  return saved >= 24576.0 + 49152.0 * rows * p / cus ? p : 1;
}

struct SplitLayout {
  size_t off_loc, off_count, off_done, total;
};

// per row: a list of kPoolCap composites, its length, the arrivals
SplitLayout split_layout(int rows) {
  SplitLayout l;
  size_t o = 0;
  auto take = [&](size_t bytes) {
    const size_t at = o;
    o += (bytes + 255) / 256 * 256;
    return at;
  };
  l.off_count = take((size_t)rows * sizeof(int32_t));     // the two counter arrays first: they are
  l.off_done = take((size_t)rows * sizeof(uint32_t));     // what has to be zero on entry
  l.off_loc = take((size_t)rows * kPoolCap * sizeof(u64));
  l.total = o;
  return l;
}

}  // namespace

extern "C" size_t socket_select_workspace_bytes(int B, int Hq, int T, int M) {
  if (B <= 0 || Hq <= 0 || T <= 0 || M < 0) return 0;
  if (row_parts(B * Hq, T, M < T ? M : T) < 2) return 0;
  return split_layout(B * Hq).total;
}

extern "C" size_t socket_select_workspace_zero_bytes(int B, int Hq, int T, int M) {
  if (socket_select_workspace_bytes(B, Hq, T, M) == 0) return 0;
  return split_layout(B * Hq).off_loc;
}

namespace {

int select_entry(const float* scores, const uint8_t* allowed, int64_t score_stride, const int32_t* lens,
                                  const int32_t* budgets, const uint32_t* row_range, int range_parts,
                                  int B, int Hq, int T, int M, int sink, int window, int write_base,
                                  int32_t* sparse_list, int64_t list_stride, int list_width,
                                  int32_t* sparse_len, void* workspace, size_t workspace_bytes,
                                  void* stream) {
  SOCKET_REQUIRE(scores && sparse_list, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(B > 0 && Hq > 0 && T > 0 && M >= 0 && sink >= 0 && window >= 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(score_stride >= T && list_width >= 0 && list_stride >= list_width, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(row_range == nullptr || range_parts > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(M <= SOCKET_TOPK_MAX_M, SOCKET_ERR_UNSUPPORTED);
  const int rows = B * Hq;
  SOCKET_REQUIRE(rows <= 65535, SOCKET_ERR_SHAPE);
  const int m_max = M < T ? M : T;
  const int cap_above = next_pow2(m_max > 0 ? m_max : 1);
  const SocketDeviceLimits& lim = socket_device_limits();
  const size_t lds_max = (size_t)lim.max_lds_per_block;
  const size_t lds_static = kBins * 4 + sizeof(SelectShared) + 256;
  size_t lds = (size_t)(cap_above + kCandCap) * sizeof(u64);
  SOCKET_REQUIRE(lds + lds_static <= lds_max, SOCKET_ERR_UNSUPPORTED);
  hipStream_t s = (hipStream_t)stream;

  // extras as LDS allows: the pool (where a pooled select can apply at all), then
  // counting placement (2 * cap_above more slots)
  // (rows of at most kPoolCap scores are pooled whole, straight into registers)
  int use_pool = 0, counting_ok = 0, pool_slots = 0;
  if (T <= kPoolCap) {
    use_pool = 1;
  } else if (sampling_ok(m_max) && lds + (size_t)kPoolCap * sizeof(u64) + lds_static <= lds_max) {
    use_pool = 1;
    pool_slots = kPoolCap;
    lds += (size_t)kPoolCap * sizeof(u64);
  }
  if (lds + (size_t)2 * cap_above * sizeof(u64) + lds_static <= lds_max) {
    counting_ok = 1;
    lds += (size_t)2 * cap_above * sizeof(u64);
  }

  // rows shared between workgroups exchange their entries through the workspace
  int parts = (workspace && use_pool) ? row_parts(rows, T, m_max) : 1;
  u64* loc = nullptr;
  int32_t* row_count = nullptr;
  unsigned int* row_done = nullptr;
  if (parts > 1) {
    const SplitLayout l = split_layout(rows);
    SOCKET_REQUIRE(workspace_bytes >= l.total, SOCKET_ERR_WORKSPACE);
    SOCKET_REQUIRE(socket_aligned16(workspace), SOCKET_ERR_ALIGN);
    char* ws = (char*)workspace;
    loc = (u64*)(ws + l.off_loc);
    row_count = (int32_t*)(ws + l.off_count);
    row_done = (unsigned int*)(ws + l.off_done);
  }
  SOCKET_REQUIRE((int64_t)rows * parts <= 0x7fffffff, SOCKET_ERR_SHAPE);

  // More rows than CUs: workgroups of half the lanes, and so little LDS that a CU holds two of them, so that one's
  // barriers and waits are the other's work and no last round leaves most CUs idle.  Whole / half workgroups, us: 260 rows
  // of 65536 33.1 / 26.9, 264 of 131072 53.0 / 47.0, 288 of 12000 21.3 / 14.9, 320 of 32768 25.7 / 19.7, 448 of 16384 to
  // 98304 40.3 / 36.6, 512 of 32768 28.3 / 20.2, 2048 of up to 20000 81.3 / 54.8; rows pooled whole, 448 of 3000 12.6 / 9.0,
  // 512 of 4096 13.2 / 9.4, 512 of 8192 16.6 / 12.7, 1280 of 2000 28.2 / 18.8.  Rows that all have a CU to themselves keep
  // its 16 waves (32 to 256 of 4096: 7.0 to 7.3 / 7.3 to 7.5); budgets past 2048 need more LDS than half of a CU's.
  const bool half = use_pool && parts == 1 && rows > lim.cu_count && 3 * cap_above + kCandCap <= kPoolCap;
  if (half && pool_slots > 0) lds = (size_t)kPoolCap * sizeof(u64);
  auto kern = half ? (allowed ? select_list_kernel<true, kThreads / 2> : select_list_kernel<false, kThreads / 2>)
                   : (allowed ? select_list_kernel<true, kThreads> : select_list_kernel<false, kThreads>);
  if (lds > 32 * 1024 &&
      hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                          hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return SOCKET_ERR_LAUNCH;
  hipLaunchKernelGGL(kern, dim3(rows * parts), dim3(half ? kThreads / 2 : kThreads), lds, s, scores, allowed, score_stride, lens, budgets,
                     row_range, range_parts, Hq, T, M, sink, window, write_base, sparse_list,
                     list_stride, list_width, sparse_len, cap_above, counting_ok, use_pool, pool_slots, parts,
                     loc, row_count, row_done);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

}  // namespace

extern "C" int socket_select_list(const float* scores, int64_t score_stride, const int32_t* lens,
                                  const int32_t* budgets, const uint32_t* row_range, int range_parts,
                                  int B, int Hq, int T, int M, int sink, int window, int write_base,
                                  int32_t* sparse_list, int64_t list_stride, int list_width,
                                  int32_t* sparse_len, void* workspace, size_t workspace_bytes,
                                  void* stream) {
  return select_entry(scores, nullptr, score_stride, lens, budgets, row_range, range_parts, B, Hq, T, M, sink, window, write_base,
                      sparse_list, list_stride, list_width, sparse_len, workspace, workspace_bytes, stream);
}

extern "C" int socket_select_list_allowed(const float* scores, int64_t score_stride, const uint8_t* allowed, int B, int Hq, int T, int M,
                                          int sink, int window, int32_t* sparse_list, int64_t list_stride, int list_width,
                                          int32_t* sparse_len, void* workspace, size_t workspace_bytes, void* stream) {
  SOCKET_REQUIRE(allowed, SOCKET_ERR_NULL);
  return select_entry(scores, allowed, score_stride, nullptr, nullptr, nullptr, 0, B, Hq, T, M, sink, window, 1, sparse_list,
                      list_stride, list_width, sparse_len, workspace, workspace_bytes, stream);
}

extern "C" int socket_select_attend_fits(int B, int Hq, int D, int T, int list_width, int dtype) {
  const int eb = socket_dtype_bytes(dtype);
  if (eb == 0 || B <= 0 || Hq <= 0 || T <= 0 || list_width <= 0 || (D != 64 && D != 128)) return 0;
  const int most = eb == 4 ? row_entries<DType_f32>(D) : row_entries<DType_bf16>(D);
  return T <= kPoolCap && list_width <= most && list_width <= kFuseList && (int64_t)B * Hq <= socket_device_limits().cu_count;
}

extern "C" int socket_select_attend(const float* scores, int64_t score_stride, const int32_t* lens, const int32_t* budgets, int T,
                                    int M, int sink, int window, int list_width, const void* q, const void* k, const void* v,
                                    int dtype, int64_t q_stride_b, int64_t q_stride_h, int64_t k_stride_b, int64_t k_stride_h,
                                    int64_t k_stride_s, int64_t v_stride_b, int64_t v_stride_h, int64_t v_stride_s, void* out,
                                    int64_t out_stride_b, int64_t out_stride_h, int B, int Hq, int Hkv, int D, int kv_rows,
                                    void* stream) {
  SOCKET_REQUIRE(scores && q && k && v && out, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(B > 0 && Hq > 0 && Hkv > 0 && Hq % Hkv == 0 && T > 0 && kv_rows > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(M >= 0 && sink >= 0 && window >= 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(score_stride >= T && list_width > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE(M <= SOCKET_TOPK_MAX_M, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(socket_select_attend_fits(B, Hq, D, T, list_width, dtype), SOCKET_ERR_UNSUPPORTED);
  const int per16 = 16 / socket_dtype_bytes(dtype);
  SOCKET_REQUIRE(socket_aligned16(q) && socket_aligned16(k) && socket_aligned16(v), SOCKET_ERR_ALIGN);
  for (int64_t st : {q_stride_b, q_stride_h, k_stride_b, k_stride_h, k_stride_s, v_stride_b, v_stride_h, v_stride_s})
    SOCKET_REQUIRE(st % per16 == 0, SOCKET_ERR_ALIGN);
#define SOCKET_SA(DT, DD)                                                                                                          \
  hipLaunchKernelGGL((select_attend_kernel<DT, DD>), dim3(B * Hq), dim3(kThreads), 0, (hipStream_t)stream, scores, score_stride, lens, \
                     budgets, Hq, T, M, sink, window, list_width, (const DT::storage*)q, (const DT::storage*)k, (const DT::storage*)v, \
                     q_stride_b, q_stride_h, k_stride_b, k_stride_h, k_stride_s, v_stride_b, v_stride_h, v_stride_s, Hq / Hkv,      \
                     kv_rows, 1.0f / sqrtf((float)D), (DT::storage*)out, out_stride_b, out_stride_h)
#define SOCKET_SA_D(DT)             \
  do {                              \
    if (D == 128) SOCKET_SA(DT, 128); \
    else SOCKET_SA(DT, 64);         \
  } while (0)
  if (dtype == SOCKET_F32) SOCKET_SA_D(DType_f32);
  else if (dtype == SOCKET_F16) SOCKET_SA_D(DType_f16);
  else SOCKET_SA_D(DType_bf16);
#undef SOCKET_SA_D
#undef SOCKET_SA
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}
