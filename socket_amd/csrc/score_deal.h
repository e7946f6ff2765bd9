// How the persistent scorer (score.hip) shares the cached tokens out among its workgroups.
#pragma once
#include "score_stretch.h"
#include "socket_common.h"

namespace {

// Tokens [start, end) of row (b, vp); end <= the sequence's length; start == end: none.
struct ScoreTile {
  int b, vp, start, end;
};

// Tokens are counted in units of UNIT, tiles have up to UNITS units.  Rows are (sequence, kv head) pairs, each as long as
// its sequence, laid end to end in units.  The row space is cut into equal stretches, and the tiles of a stretch -- every
// row segment in ceil(n / UNITS) tiles of equal size, the head parts of a tile next to each other -- are dealt in turn to
// the workgroups that share the stretch:
//   spread == 0: a stretch per workgroup (it walks consecutive tiles of one row); workgroup
//     n of N takes stretch (n % 8) * N / 8 + n / 8, so that neighbouring stretches, the
//     tiles of one row, sit on one XCD (workgroup n runs on XCD n % 8) and share its L2;
//   spread == 1: a stretch per XCD, its tiles dealt round to its workgroups.  They then work
//     on neighbouring tiles at any moment: few tables are live in the XCD's L2 however many
//     rows its stretch holds, and the parts of a wide head group, which read the same
//     codes, read them at the same time -- the second read is served by the L2.
//     The tiles are then as small as the rounds they take allow (even_out below): dealt at their full size, a little
//     more than one round took two, and all but a few workgroups stood idle in the last.  us of the scorer, full
//     tiles / even ones: 8 sequences x 28 heads of 4, 60 tables x 1024, 40000 tokens 67.8 / 52.4, 81920: 101.5 / 95.0,
//     32768 and 65536 (whole rounds) 39.0 / 38.8 and 72.4 / 72.1, ragged 57344: 65.4 / 49.8; 4 x 28 heads, 48 tables,
//     131072 ragged 56.5 / 42.5; 8 x 32 heads, 65536 ragged 70.1 / 55.7; 32 tables x 256, 8 x 28 heads, 16384 tokens 13.8 / 13.5,
//     65536 ragged 31.3 / 27.9.
// (One wave ranks the lengths of up to 64 sequences.)
template <int UNIT, int UNITS>
struct ScoreDeal {
  int B, Hkv, hsplit, gsize;
  int len_l, u_l;                  // lane l: cached length of sequence l, and its units
  int row_b, row_kvh, row_a, left; // where the stretch stands: sequence, kv head, unit; units left
  int skip;                        // tiles of the stretch before this workgroup's next
  int units;                       // of a tile at most

  __device__ __forceinline__ ScoreDeal(const int32_t* lens, int B_, int Hkv_, int hsplit_, int T, int spread)
      : B(B_), Hkv(Hkv_), hsplit(hsplit_), len_l(0), row_b(0), row_kvh(0), row_a(0) {
    const int lane = threadIdx.x & 63;
    if (lane < B) len_l = lens ? max(0, min(lens[lane], T)) : T;
    u_l = (len_l + UNIT - 1) / UNIT;
    const int incl = wave_incl_scan(u_l);
    const int nwg = gridDim.x;
    const bool by_xcd = (nwg & 7) == 0;
    const int slot = by_xcd ? (int)(blockIdx.x >> 3) : (int)blockIdx.x;
    const int group = !spread ? (by_xcd ? (int)(blockIdx.x & 7) * (nwg >> 3) + slot : slot) : by_xcd ? (int)(blockIdx.x & 7) : 0;
    gsize = !spread ? 1 : by_xcd ? nwg >> 3 : nwg;
    // (What comes before the first copy is a chain of scalar instructions that nothing hides, a 64-bit division some 150 of
    // them; with two of those, and divisions by the one or two parts, a launch took 0.3 to 0.9 us longer.)
    const uint32_t total = (uint32_t)(__builtin_amdgcn_readlane(incl, 63) * Hkv);
    const ScoreStretch mine = score_stretch(total, (uint32_t)group, (uint32_t)(!spread ? nwg : by_xcd ? 8 : 1));
    const int x0 = (int)mine.start;
    left = (int)mine.size;
    skip = spread ? slot : 0;
    if (left > 0) {
      row_b = __popcll(__builtin_amdgcn_ballot_w64(incl * Hkv <= x0));
      const uint32_t ub = (uint32_t)__builtin_amdgcn_readlane(u_l, row_b);
      const uint32_t rem = (uint32_t)(x0 - (__builtin_amdgcn_readlane(incl, row_b) - (int)ub) * Hkv);
      row_kvh = (int)(rem / ub);
      row_a = (int)(rem - row_kvh * ub);
    }
    units = UNITS;
    if (spread) even_out(incl, x0);
  }

  // The fewest units to a tile that need no more rounds than full tiles do, where at least an eighth of these would stand
  // idle.  The count is 0.2 to 0.9 us that nothing hides: a few sequences one after another with a size to each lane, more of
  // them a lane each and the size found by halves.  (Row after row, 0.15 us a row, it was left out past 64 rows in all and
  // given up after 12 of a stretch.)  us of the scorer, full tiles / row after row / this, 60 tables x 1024 unless stated:
  // 32 x 4 kv heads of 7, 12000 ragged 67.9 / 67.1 / 53.2, 20000 ragged 87 / 90 / 79, 6000 full 38.0 / 37.7 / 38.6; 20 x 4, 12000 57.5 /
  // 57.7 / 47.1; 9 x 8, 20000 ragged 65.8 / 66.0 / 48.0, 12000 ragged 38.9 / 38.7 / 39.6; 16 x 4, most of 20000 short 41.4 / 46.7 /
  // 38.5, 64 x 1 the same way 43.6 / 33.1 / 38.7; 16 x 8, 6000 full 37.6 / 37.4 / 38.4; 1 x 4, 8000 cached of 131072 22.1 / 15.9 / 16.2.
  // Tiles of up to kPassage tokens cost the passage of the table and little else, and a stretch without longer sequences is
  // not counted: 8 x 8 kv heads of 4 with 300 / 2000 / 4000 cached of 16384, full tiles 18.0 / 19.0 / 25.3, even ones with the
  // count 19.2 / 19.8 / 20.4; 16 x 4 of 7, 48 tables, of 98304: 19.0 / 19.8 / 23.1 and 20.4 / 20.8 / 22.1.
  static constexpr int kPassage = 2048;
  static constexpr int kFewSequences = 4;
  __device__ __forceinline__ void even_out(int incl, int x0) {
    if (left <= 0 || left >= 1 << 16 || left * hsplit % (UNITS * gsize) == 0) return;
    // lane l: the rows of sequence l in the stretch: units of the first, whole ones, units of the last
    const int base = (incl - u_l) * Hkv;
    const int p = max(x0 - base, 0), q = min(x0 + left - base, u_l * Hkv);
    if (__builtin_amdgcn_ballot_w64(p < q && len_l > kPassage) == 0) return;
    int head = 0, whole = 0, tail = 0;
    if (p < q) {
      const int first = quotient(p, u_l), last = quotient(q, u_l);
      tail = q - last * u_l;
      head = first == last ? q - p : (first + 1) * u_l - p;
      whole = last - first - 1;
      if (first == last) whole = tail = 0;
    }
    const float headf = (float)head, rowf = (float)u_l, tailf = (float)tail;
    const auto fits = [&](int full) __attribute__((always_inline)) { return (full + gsize - 1) / gsize * gsize; };
    unsigned long long here = __builtin_amdgcn_ballot_w64(p < q);
    if (__popcll(here) <= kFewSequences) {
      // sequence after sequence, a size to each lane
      const int most = min((int)(threadIdx.x & 63), UNITS - 1) + 1;
      int n = 0;
      for (; here; here &= here - 1) {
        const int l = __ffsll(here) - 1;
        auto of = [&](float v) __attribute__((always_inline)) {
          return tiles_of(__builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), l)), most);
        };
        n += of(headf) + __builtin_amdgcn_readlane(whole, l) * of(rowf) + of(tailf);
      }
      const int full = __builtin_amdgcn_readlane(n, UNITS - 1) * hsplit, fit = fits(full);
      if (full * 8 <= fit * 7) units = (int)__ffsll((unsigned long long)__builtin_amdgcn_ballot_w64(n * hsplit <= fit));
      return;
    }
    // all sequences at once, the size found by halves
    auto tiles = [&](int most) __attribute__((always_inline)) {
      const int n = tiles_of(headf, most) + whole * tiles_of(rowf, most) + tiles_of(tailf, most);
      return __builtin_amdgcn_readlane(wave_incl_scan(n), 63) * hsplit;
    };
    const int full = tiles(UNITS), fit = fits(full);
    if (full * 8 > fit * 7) return;
    static_assert((UNITS & (UNITS - 1)) == 0, "halves");
#pragma unroll
    for (int step = UNITS / 2; step > 0; step >>= 1)
      if (tiles(units - step) <= fit) units -= step;
  }

  // n / most rounded up (exact below 2^16: the half keeps the quotient 1 / 32 and more from a whole number)
  static __device__ __forceinline__ int tiles_of(float n, int most) {
    const float r = __builtin_amdgcn_rcpf((float)most);
    return (int)fmaf(n, r, ((float)most - 0.5f) * r);
  }
  // a / b for small quotients (the float's is one off at most)
  static __device__ __forceinline__ int quotient(int a, int b) {
    const int q = (int)((float)a * __builtin_amdgcn_rcpf((float)b)), r = a - q * b;
    return q + (r >= b ? 1 : 0) - (r < 0 ? 1 : 0);
  }

  __device__ __forceinline__ int length(int b) const { return __builtin_amdgcn_readlane(len_l, b); }

  __device__ __forceinline__ ScoreTile next() {
    ScoreTile t{0, 0, 0, 0};
    while (left > 0) {
      const int ub = __builtin_amdgcn_readlane(u_l, row_b);
      const int n = min(ub - row_a, left);               // units of this row inside the stretch
      int k = (n + UNITS - 1) / UNITS;
      if (units != UNITS) {
        asm volatile("");      // (a branch, not a choice between two results: a workgroup walks past many rows)
        k = __builtin_amdgcn_readfirstlane(tiles_of((float)n, units));
      }
      const int cnt = k * hsplit;
      if (skip < cnt) {
        const int sz = (n + k - 1) / k;
        const int j = skip >> (hsplit - 1);      // (one part or two)
        t.b = row_b;
        t.vp = row_kvh * hsplit + (skip & (hsplit - 1));
        t.start = (row_a + j * sz) * UNIT;
        t.end = min((row_a + min((j + 1) * sz, n)) * UNIT, __builtin_amdgcn_readlane(len_l, row_b));
        skip += gsize;
        return t;
      }
      skip -= cnt;
      left -= n;
      row_a = 0;
      if (++row_kvh == Hkv) {
        row_kvh = 0;
        do ++row_b;
        while (row_b < B && __builtin_amdgcn_readlane(u_l, row_b) == 0);
      }
    }
    return t;
  }
};

// Positions past each sequence's cached length: -inf.  (The scored tiles wrote it up to the next multiple of four.)
__device__ __forceinline__ void score_fill_past(float* scores, int64_t score_stride, int len_l, int B, int Hq, int T) {
  for (int row = blockIdx.x; row < B * Hq; row += gridDim.x) {
    const int len = __builtin_amdgcn_readlane(len_l, row / Hq);
    float* dst = scores + (int64_t)row * score_stride;
    for (int t = ((len + 3) & ~3) + (int)threadIdx.x * 4; t < T; t += (int)blockDim.x * 4) {
      if (t + 4 <= T) {
        store_stream16(dst + t, -INFINITY, -INFINITY, -INFINITY, -INFINITY);
      } else {
        for (int i = t; i < T; ++i) dst[i] = -INFINITY;
      }
    }
  }
}

}  // namespace
