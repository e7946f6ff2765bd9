// Soft-collision scores on the reference's own operand layout: one int16 bucket
// code per (query head, table, token), [B,H,L,T], a table of probabilities
// [B,H,L,R], a mask byte and a value norm per (head, token).
//
// Replaces soft_hash_collision of the reference's extension (the call is
// GPT-FAST/kernels/sparse.py:40-49, the kernel GPT-FAST/kernels/soft_hash_collision.cu:25-54)
// and its fp16 variant (GPT-FAST/kernels/soft_hash_score/soft_hash_score.cu:7-42):
//   out[b,h,t] = allowed ? (sum_l table[b,h,l, code[b,h,l,t]]) * v[b,h,t] : -inf
// summed over l in ascending order in fp32; codes outside [0, R) add nothing.
//
// This layout costs 2 L + 9 bytes of HBM per (head, token) -- eight times the
// packed per-kv-head cache of score.hip at G = 4 -- and the launch is bound by
// that stream if the tables stay out of its way.  A workgroup therefore keeps a
// tile of tokens of one (b, h) row and walks the tables in LDS-sized
// slices (two slices of 30 fp32 tables at L60 x R1024; one slice for fp16), copied
// straight from memory into LDS while the first codes are on their way, and
// serves several such tiles under each slice; a thread fetches the codes of its
// consecutive tokens with one load per table (wherever the row starts) and gathers
// with one branch a wave and table (is any of its codes outside?).  It has eight tokens, 16-byte loads, six tables ahead of their use;
// four or two where rows are short, 8- or 4-byte loads, 12 or 24 tables ahead.
#include <atomic>

#include "socket_common.h"

namespace {

// Consecutive tokens of a thread: eight where rows are long, four or two where a row's tokens have to be dealt out wide to
// occupy the chip.
constexpr int kTokensPerThread = 8;
// tables whose codes are in flight per lane: 96 bytes of them either way
constexpr int ahead(int tpt) { return 48 / tpt; }
constexpr size_t kCollideLdsSlack = 1024;

struct Bf16Entry {
  uint16_t bits;
};
__device__ __forceinline__ float entry_to_f32(float x) { return x; }
__device__ __forceinline__ float entry_to_f32(uint16_t x) { return f16_bits_to_f32(x); }
__device__ __forceinline__ float entry_to_f32(Bf16Entry x) { return bf16_bits_to_f32(x.bits); }

// Value norm i of an array of any of the three types (widening changes no value).
__device__ __forceinline__ float norm_at(const void* v, int dtype, int64_t i) {
  if (dtype == SOCKET_F32) return ((const float*)v)[i];
  const uint16_t u = ((const uint16_t*)v)[i];
  return dtype == SOCKET_F16 ? f16_bits_to_f32(u) : bf16_bits_to_f32(u);
}

// Vectors of a thread's eight tokens.  Rows of the reference's layout start wherever T puts them, odd rows of an odd T on an
// odd pair of bytes; global loads take such addresses as they are, and a wave's 1024 contiguous bytes touch nine 128-byte
// lines instead of eight.  (32 rows, L60 x R1024, us against a code at a time: fp32 tables at 2051 / 4135 / 9003 / 20881 / 32771
// tokens 26 / 32 / 31 / 33 / 50 against 71 / 80 / 79 / 101 / 168, bf16 24 / 29 / 26 / 28 / 41 against 60 / 69 / 68 / 88 / 147;
// rows on 16-byte boundaries are as fast as before.)
template <int TPT>
struct Vectors;
template <>
struct Vectors<8> {
  typedef uint32_t codes __attribute__((ext_vector_type(4), aligned(2)));      // 16-bit codes or norms
  typedef uint32_t bytes __attribute__((ext_vector_type(2), aligned(1)));      // mask bytes
  typedef float floats __attribute__((ext_vector_type(4), aligned(4)));
  static __device__ __forceinline__ uint32_t word(const codes& c, int i) { return c[i]; }
  static __device__ __forceinline__ uint32_t mask(const bytes& b, int i) { return (i < 4 ? b.x : b.y) >> (8 * (i & 3)); }
};
template <>
struct Vectors<4> {
  typedef uint32_t codes __attribute__((ext_vector_type(2), aligned(2)));
  typedef uint32_t bytes __attribute__((aligned(1)));
  typedef float floats __attribute__((ext_vector_type(4), aligned(4)));
  static __device__ __forceinline__ uint32_t word(const codes& c, int i) { return c[i]; }
  static __device__ __forceinline__ uint32_t mask(bytes b, int i) { return b >> (8 * i); }
};
template <>
struct Vectors<2> {
  typedef uint32_t codes __attribute__((aligned(2)));
  typedef uint16_t bytes __attribute__((aligned(1)));
  typedef float floats __attribute__((ext_vector_type(2), aligned(4)));
  static __device__ __forceinline__ uint32_t word(codes c, int) { return c; }
  static __device__ __forceinline__ uint32_t mask(bytes b, int i) { return (uint32_t)b >> (8 * i); }
};

// an entry as it is read from LDS
template <class QT>
using entry_bits_t = std::conditional_t<sizeof(QT) == 4, uint32_t, uint16_t>;

// Byte address of entry `code` of the table at `base` in LDS: the low or high code of a word, one instruction.
template <int EB>
__device__ __forceinline__ uint32_t entry_address(uint32_t codes, bool high, uint32_t base) {
  uint32_t a;
  if (high) asm("v_mad_u32_u16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(a) : "v"(codes), "n"(EB), "s"(base));
  else asm("v_mad_u32_u16 %0, %1, %2, %3" : "=v"(a) : "v"(codes), "n"(EB), "s"(base));
  return a;
}

// ct: tables per LDS slice.  INLDS false: a single table exceeds LDS, gather from global memory.
// A workgroup serves `chunks` consecutive tiles of `tile` <= THREADS x TPT tokens under every
// slice it brings into LDS; with more than one slice the running sums of a tile
// wait in `out` between slices (each thread re-reads what it wrote itself), which
// costs 8 bytes per token and slice against the 2 L + 9 of the stream and keeps
// the order of the fp32 adds.
// The thread at a row's end whose tokens would run past it takes the row's last TPT (its loads stay inside the row)
// and leaves those that its neighbour owns alone: it neither stores their sums nor their scores.
// WIDE false: rows of fewer than eight tokens, element by element.
// STREAM: the codes are loaded with the streaming hint (a code array too large to
// stay in the memory-side cache from one call to the next; WIDE only).
template <typename QT, int THREADS, int TPT, bool WIDE, bool INLDS, bool STREAM>
__global__ __launch_bounds__(THREADS) void collision_i16_kernel(
    const QT* __restrict__ q_probs, const int16_t* __restrict__ key_buckets,
    const uint8_t* __restrict__ allowed, const void* __restrict__ v_hist, int v_dtype, float* __restrict__ out,
    int rows, int L, int R, int T, int tile, int ct, int chunks) {
  extern __shared__ __attribute__((aligned(16))) unsigned char collide_lds[];
  QT* table = reinterpret_cast<QT*>(collide_lds);
  typedef Vectors<TPT> V;
  typedef typename V::codes codes_t;
  typedef typename V::floats floats_t;
  constexpr int F = sizeof(floats_t) / sizeof(float);
  // row r is workgroups r, r + rows, ...: on one XCD, or few, whose L2 then fetches its table once for all its tiles
  // (with the tiles of a row next to each other every XCD fetched every table: 32 rows, L60 x R1024, fp32, 32768 tokens
  // 42.6 us against 38.5, 1000 tokens 20.9 against 13.8, both with the copy into LDS, which is the smaller part)
  const int bh = blockIdx.x % rows, part = blockIdx.x / rows;
  const QT* qp = q_probs + (int64_t)bh * L * R;
  const int16_t* kb = key_buckets + (int64_t)bh * L * T;

  // the codes of a thread's tokens from t0 on for table l, as loaded (two per word; WIDE: all of them exist; else -1 where no
  // token is)
  auto codes_of = [&](int l, int t0) -> codes_t {
    const int16_t* row = kb + (int64_t)l * T + t0;
    if (WIDE && !STREAM) return *reinterpret_cast<const codes_t*>(row);
    if (WIDE) return __builtin_nontemporal_load(reinterpret_cast<const codes_t*>(row));
    uint32_t u[TPT / 2];
#pragma unroll
    for (int i = 0; i < TPT / 2; ++i) {
      const uint32_t lo = (t0 + 2 * i < T) ? (uint16_t)row[2 * i] : 0xffffu;
      const uint32_t hi = (t0 + 2 * i + 1 < T) ? (uint16_t)row[2 * i + 1] : 0xffffu;
      u[i] = lo | (hi << 16);
    }
    codes_t c;
    __builtin_memcpy(&c, u, sizeof(c));
    return c;
  };
  // `skip`: how many of the tokens belong to the thread before (only ever above zero at a row's end)
  auto load_partial = [&](int64_t o, int t0, int skip, float (&sum)[TPT]) {
    if (WIDE && skip == 0) {
#pragma unroll
      for (int v = 0; v < TPT; v += F) {
        const floats_t a = *reinterpret_cast<const floats_t*>(out + o + v);
#pragma unroll
        for (int i = 0; i < F; ++i) sum[v + i] = a[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < TPT; ++i) sum[i] = (i >= skip && t0 + i < T) ? out[o + i] : 0.f;
    }
  };
  auto store_row = [&](int64_t o, int t0, int skip, const float (&x)[TPT]) {
    if (WIDE && skip == 0) {
#pragma unroll
      for (int v = 0; v < TPT; v += F) {
        floats_t a;
#pragma unroll
        for (int i = 0; i < F; ++i) a[i] = x[v + i];
        *reinterpret_cast<floats_t*>(out + o + v) = a;
      }
    } else {
#pragma unroll
      for (int i = 0; i < TPT; ++i)
        if (i >= skip && t0 + i < T) out[o + i] = x[i];
    }
  };
  auto finish = [&](int64_t o, int t0, int skip, const float (&sum)[TPT]) {
    float res[TPT];
    if (WIDE) {
      const typename V::bytes ok = *reinterpret_cast<const typename V::bytes*>(allowed + o);
      float vh[TPT];
      if (v_dtype == SOCKET_F32) {      // (uniform)
#pragma unroll
        for (int v = 0; v < TPT; v += F) {
          const floats_t a = *reinterpret_cast<const floats_t*>((const float*)v_hist + o + v);
#pragma unroll
          for (int i = 0; i < F; ++i) vh[v + i] = a[i];
        }
      } else {
        const codes_t c = *reinterpret_cast<const codes_t*>((const uint16_t*)v_hist + o);
#pragma unroll
        for (int i = 0; i < TPT; ++i) {
          const uint16_t bits = (uint16_t)(V::word(c, i >> 1) >> (16 * (i & 1)));
          vh[i] = v_dtype == SOCKET_F16 ? f16_bits_to_f32(bits) : bf16_bits_to_f32(bits);
        }
      }
#pragma unroll
      for (int i = 0; i < TPT; ++i) res[i] = (V::mask(ok, i) & 0xffu) ? sum[i] * vh[i] : -INFINITY;
    } else {
#pragma unroll
      for (int i = 0; i < TPT; ++i)
        res[i] = t0 + i < T && allowed[o + i] ? sum[i] * norm_at(v_hist, v_dtype, o + i) : -INFINITY;
    }
    store_row(o, t0, skip, res);
  };

  constexpr int kAhead = ahead(TPT);
  codes_t ring[kAhead];
  auto fill_ring = [&](int l0, int nt, int t0) __attribute__((always_inline)) {
#pragma unroll
    for (int a = 0; a < kAhead; ++a) ring[a] = codes_of(l0 + min(a, nt - 1), t0);
  };
  struct Where {
    int own, t0;      // the thread's first token of a tile, and where its loads start; own < 0: it has none
  };
  auto where = [&](int c) __attribute__((always_inline)) {
    const int first = (part * chunks + c) * tile, own = first + (int)threadIdx.x * TPT;
    if (own >= min(first + tile, T)) return Where{-1, 0};
    return Where{own, WIDE ? min(own, T - TPT) : own};
  };
  const int step = INLDS ? ct : L;   // (without LDS: one pass over all tables)
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  const uint16_t last_code = (uint16_t)(min(R, 32768) - 1);      // (as 16 bits without a sign, anything above is no code)
  const uint32_t table_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) QT*)table;
  for (int l0 = 0; l0 < L; l0 += step) {
    const int nt = min(step, L - l0);
    const Where w0 = where(0);
    if (w0.own >= 0) fill_ring(l0, nt, w0.t0);     // (on their way while the slice comes)
    if (INLDS) {
      __syncthreads();   // the previous slice has been consumed
      const int bytes = nt * R * (int)sizeof(QT);
      const char* src = reinterpret_cast<const char*>(qp + (int64_t)l0 * R);
      if (((uintptr_t)src & 15) == 0 && bytes % 16 == 0) {
        // straight into LDS, all of it under way at once (through registers every 16 KB were a trip to memory)
        const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
        for (int o = wave * 1024; o < bytes; o += THREADS * 16)
          if (o + lane * 16 < bytes) lds_dma16(src + o + lane * 16, collide_lds + o);
        wait_vmcnt(0);
      } else {
        for (int i = threadIdx.x; i < nt * R; i += THREADS) table[i] = qp[(int64_t)l0 * R + i];
      }
      __syncthreads();
    }
    for (int c = 0; c < chunks; ++c) {
      const Where at = c ? where(c) : w0;
      if (at.own < 0) continue;
      const int t0 = at.t0, skip = at.own - t0;
      const int64_t o = (int64_t)bh * T + t0;
      float sum[TPT];
      if (l0 == 0) {
#pragma unroll
        for (int i = 0; i < TPT; ++i) sum[i] = 0.f;
      } else {
        load_partial(o, t0, skip, sum);
        // (waited for here: left to the first use in the loop, the wait is there in every turn, for nearly all codes in flight)
#pragma unroll
        for (int i = 0; i < TPT; ++i) asm volatile("" : "+v"(sum[i]));
      }
      // A ring of kAhead code words per lane stays in flight (one 16-byte load per lane
      // would leave the stream waiting on latency): slot a always holds table lb + a;
      // the loop is unrolled by the ring's depth, so a slot is a fixed set of registers
      // and the wait before its use counts exactly the loads behind it.
      if (c) fill_ring(l0, nt, t0);
      for (int lb = 0; lb < nt; lb += kAhead) {
#pragma unroll
        for (int a = 0; a < kAhead; ++a) {
          const int l = lb + a;
          if (l >= nt) break;
          const codes_t cur = ring[a];
          // (past the slice: its last table again, unused)
          auto refill = [&]() __attribute__((always_inline)) { ring[a] = codes_of(l0 + min(l + kAhead, nt - 1), t0); };
          // Without a branch: a stray code reads entry 0 and adds +0.0 instead (x + 0.0 == x; the sums start at +0.0, so no
          // -0.0 can be lost).
          auto add_any = [&]() __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < TPT; ++i) {
              const int r = (int)(int16_t)((i & 1) ? (V::word(cur, i >> 1) >> 16) : (V::word(cur, i >> 1) & 0xffffu));
              const bool hit = r >= 0 && r < R;
              const int rr = hit ? r : 0;
              const float e = entry_to_f32(INLDS ? table[l * R + rr] : qp[(int64_t)(l0 + l) * R + rr]);
              sum[i] += hit ? e : 0.f;
            }
          };
          if constexpr (INLDS && WIDE) {
            // One test for all codes of the wave: the sums of codes that are all inside take less than five vector
            // instructions a code, where a test of each took nine and 1.8 times the code.  The vector ALUs were what the
            // launch waited for, two waves to each of them at 512 lanes (us before / now, with the wait below: 32 rows of
            // 32768 tokens, L60 x R1024, bf16 35.6 / 30.5, fp32 43.0 / 33.7; 9001 tokens, bf16 17.1 / 15.1).  Where one is outside
            // each code is tested by one comparison more (a hundredth of the codes outside, us with a test of each / with the
            // branch's old form / now: 32 rows of 4448, L32 x R256, fp32 8.1 / 9.6 / 8.2, 32768, L60 x R1024 31.6 / 32.6 / 27.4).
            const uint32_t base = table_at + (uint32_t)(l * R) * (uint32_t)sizeof(QT);
            u16x2 most = {0, 0};
            uint32_t at[TPT];
#pragma unroll
            for (int i = 0; i < TPT; i += 2) {
              const uint32_t w = V::word(cur, i >> 1);
              most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, w));
              at[i] = entry_address<sizeof(QT)>(w, false, base);
              at[i + 1] = entry_address<sizeof(QT)>(w, true, base);
            }
            const u16x2 outside = __builtin_elementwise_sub_sat(most, u16x2{last_code, last_code});
            auto add = [&](auto all) __attribute__((always_inline)) {
              bool hit[TPT];
              // (codes from memory are asked for at once; from a cache it is not worth the copy of those in work, and slower by 3 to
              // 6 %: us behind the addresses / at once: 32 rows of 131072, L48 x R1024, fp32 88.0 / 86.6, 64 rows of 65536, L32 x R256 63.6 / 61.5;
              // 32 rows of 32768, L60 x R1024 26.5 / 27.2)
              if constexpr (STREAM) refill();
#pragma unroll
              for (int i = 0; i < TPT; ++i) {
                hit[i] = decltype(all)::value || (uint16_t)(V::word(cur, i >> 1) >> (16 * (i & 1))) <= last_code;
                at[i] = hit[i] ? at[i] : base;
              }
              __builtin_amdgcn_sched_barrier(0);     // (the codes have been used: their registers take the next)
              if constexpr (!STREAM) refill();
              entry_bits_t<QT> e[TPT];
#pragma unroll
              for (int i = 0; i < TPT; ++i) e[i] = *(const __attribute__((address_space(3))) entry_bits_t<QT>*)(uintptr_t)at[i];
#pragma unroll
              for (int i = 0; i < TPT; ++i) sum[i] += hit[i] ? entry_to_f32(__builtin_bit_cast(QT, e[i])) : 0.f;
            };
            if (__builtin_expect(__ballot(__builtin_bit_cast(uint32_t, outside) != 0) != 0, 0)) add(std::false_type{});
            else add(std::true_type{});
          } else {
            refill();
            add_any();
          }
        }
      }
      if (l0 + nt >= L) finish(o, t0, skip, sum);
      else store_row(o, t0, skip, sum);
    }
  }
}

template <typename QT>
int launch_collision_i16(const QT* q_probs, const int16_t* key_buckets, const uint8_t* allowed,
                         const void* v_hist, int v_dtype, float* out, int B, int H, int L, int R, int T,
                         hipStream_t stream) {
  const SocketDeviceLimits& lim = socket_device_limits();
  const size_t per_table = (size_t)R * sizeof(QT);
  const size_t budget = (size_t)lim.max_lds_per_block - kCollideLdsSlack;
  int ct = (int)(budget / per_table);
  if (ct > L) ct = L;
  if (ct > 0) {   // slices of equal size
    const int slices = (L + ct - 1) / ct;
    ct = (L + slices - 1) / slices;
  }
  const size_t lds = (size_t)ct * per_table;
  const int cus = lim.cu_count;
  const bool wide = T >= kTokensPerThread;
  // Rows short enough that two (or four) tokens to a lane hold them in one round of workgroups, each row in as many equal
  // tiles as there are CUs for it: with eight to a lane most waves would have no token and the rest a long chain of lookups.
  // us at two / four / eight tokens to a lane, L60 x R1024:
  //   32 rows   fp32  1000 tokens 14.9 / 15.3 / 20.2   4135 16.7 / 16.7 / 20.9   9001 20.0 / 18.3 / 22.0   16384 24.6 / 22.3 / 23.8
  //             bf16              10.4 / 11.5 / 16.9        12.7 / 13.8 / 20.2        15.5 / 15.1 / 20.7         19.6 / 18.5 / 23.1
  //   28 rows, L32 x R256, fp32: 4135 tokens 7.5 / 7.6 / 9.2, 16384 13.0 / 11.6 / 12.5
  // Two pay while half of the lanes at most have a token, four while a quarter of the lanes is spare (32 rows, 24576 tokens:
  // 24.8 / 26.4 at four / eight, bf16; 32768: 30.9 / 30.5, fp32 35.2 / 33.6).
  const int64_t per_row = cus / ((int64_t)B * H);
  const int few = !wide || ct == 0 ? 0 : per_row * 1024 >= T ? 2 : per_row * 1024 * 3 >= T ? 4 : 0;
  // Lanes of a workgroup of eight tokens each.  It pulls its row's whole table through LDS with them, which is quicker the
  // more there are; 512 of them hold a tile of 4096 tokens and run its lookups as fast (32 rows of 32768, L60 x R1024, at 512 /
  // 1024 lanes of eight / four tokens: bf16 30.5 / 30.9, fp32 33.6 / 35.2).  A row of at most 4608
  // tokens has no use for 512: one workgroup of 1024 holds it, or all but nothing.  Rows of at most 2048 tokens come here where
  // they outnumber the CUs; 256 lanes hold each of them, which pays where
  // tables share a CU's LDS (us at 256 / 1024 lanes, L32 x R256, fp32: 448 rows x 1000 14.8 / 15.4, 1024 rows x 1000 18.8 / 23.4)
  // and does not where one fills it (L60 x R1024, fp32: 257 rows x 1000 62 / 47, 1024 x 1000 183 / 121).
  // Rows that a workgroup of 1024 lanes to each of their CUs holds are cut into that many equal tiles, whole waves of them, or
  // CUs go without (56 rows of 20001, L48 x R1024, bf16: 28.8 us against 39.3 with tiles of as many tokens as the lanes hold).
  const bool even = wide && ct > 0 && !few && per_row > 0 && T > 256 * kTokensPerThread && T <= per_row * 1024 * kTokensPerThread;
  const int wave_tokens = SOCKET_WAVE * kTokensPerThread;
  auto tiles_of = [&](int th) { return (T + th * kTokensPerThread - 1) / (th * kTokensPerThread); };
  int threads = 1024;
  int tile = threads * kTokensPerThread;
  if (few) tile = (int)((T + per_row - 1) / per_row + 127) / 128 * 128;
  else if (even) tile = (int)((T + per_row - 1) / per_row + wave_tokens - 1) / wave_tokens * wave_tokens;
  if (T <= 256 * kTokensPerThread) threads = 256;
  else if (T > 4608 && (even ? tile <= 512 * kTokensPerThread : (int64_t)tiles_of(512) * B * H <= cus)) threads = 512;
  if (!few && !even) tile = threads * kTokensPerThread;
  const int tiles = (T + tile - 1) / tile;
  // tiles per workgroup: as many as leave two workgroups per CU (they amortise the
  // slices a workgroup pulls through LDS), at most 8
  int chunks = (int)((int64_t)tiles * B * H / (2 * (int64_t)lim.cu_count));
  chunks = chunks < 1 || few ? 1 : chunks > 8 ? 8 : chunks;
  if (chunks > tiles) chunks = tiles;
  const int64_t n_wg = (int64_t)((tiles + chunks - 1) / chunks) * B * H;
  SOCKET_REQUIRE(n_wg < (1LL << 31), SOCKET_ERR_SHAPE);
  dim3 grid((unsigned)n_wg);
  // (measured: 2 GB of codes gain 10 % from the hint, 135 MB that the cache still holds from the last call lose 7 %)
  const bool stream_codes = (int64_t)B * H * L * T * (int64_t)sizeof(int16_t) > (192ll << 20);
#define SOCKET_COLLIDE(TH, N, V, LD, ST)                                                                     \
  do {                                                                                                \
    auto kern = collision_i16_kernel<QT, TH, N, V, LD, ST>;                                                 \
    if (lds > 64 * 1024) {                                                                            \
      static std::atomic<size_t> granted{0};                                                          \
      if (granted.load(std::memory_order_acquire) < lds) {                                            \
        if (hipFuncSetAttribute(reinterpret_cast<const void*>(kern),                                  \
                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)budget) != hipSuccess) \
          return SOCKET_ERR_LAUNCH;                                                                   \
        granted.store(budget, std::memory_order_release);                                             \
      }                                                                                               \
    }                                                                                                 \
    hipLaunchKernelGGL(kern, grid, dim3(TH), lds, stream, q_probs, key_buckets, allowed, v_hist, v_dtype, out, B * H, L, R, T, tile, ct, chunks); \
  } while (0)
#define SOCKET_COLLIDE_W(TH, LD)                                                      \
  do {                                                                                \
    if (stream_codes) SOCKET_COLLIDE(TH, kTokensPerThread, true, LD, true);           \
    else SOCKET_COLLIDE(TH, kTokensPerThread, true, LD, false);                       \
  } while (0)
  if (!wide) {      // (fewer than eight tokens: one narrow workgroup a row)
    if (ct > 0) SOCKET_COLLIDE(256, kTokensPerThread, false, true, false);
    else SOCKET_COLLIDE(256, kTokensPerThread, false, false, false);
  } else if (few == 2) {
    SOCKET_COLLIDE(1024, 2, true, true, false);
  } else if (few == 4) {
    if (stream_codes) SOCKET_COLLIDE(1024, 4, true, true, true);
    else SOCKET_COLLIDE(1024, 4, true, true, false);
  } else if (ct > 0) {
    if (threads == 256) SOCKET_COLLIDE_W(256, true);
    else if (threads == 512) SOCKET_COLLIDE_W(512, true);
    else SOCKET_COLLIDE_W(1024, true);
  } else {
    if (threads == 256) SOCKET_COLLIDE_W(256, false);
    else if (threads == 512) SOCKET_COLLIDE_W(512, false);
    else SOCKET_COLLIDE_W(1024, false);
  }
#undef SOCKET_COLLIDE_W
#undef SOCKET_COLLIDE
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

// The rest of a row [sink | window | heavy] whose heavy entries are in place: the sink and window positions
// (the last position if there are none), -1 for every position that is not allowed, and the length.  For rows whose
// window is long (the others are written by the selection's launch): a workgroup takes kFinishEntries of a row.  100000
// positions x 32 rows, the whole operator over four small tables: 39 us, 61 with one workgroup of the selection's launch to a row.
constexpr int kFinishEntries = 4096;

__global__ __launch_bounds__(256) void finish_list_kernel(int32_t* __restrict__ list, int32_t* __restrict__ list_len,
                                                          const uint8_t* __restrict__ allowed, int T, int sink, int window,
                                                          int heavy) {
  const int start = max(T - window, sink), nwin = window > 0 && start < T ? T - start : 0, base = sink + nwin > 0 ? sink + nwin : 1;
  int32_t* row = list + (int64_t)blockIdx.x * (base + heavy);
  const uint8_t* ok = allowed + (int64_t)blockIdx.x * T;
  const int first = blockIdx.y * kFinishEntries;
  for (int i = first + threadIdx.x; i < min(first + kFinishEntries, base + heavy); i += 256) {
    const int at = i >= base ? row[i] : sink + nwin == 0 ? T - 1 : i < sink ? i : start + (i - sink);
    row[i] = ok[min(max(at, 0), T - 1)] ? at : -1;
  }
  if (first == 0 && threadIdx.x == 0) list_len[blockIdx.x] = base + heavy;
}

}  // namespace

extern "C" int socket_soft_hash_collision(const float* q_probs, const int16_t* key_buckets,
                                          const uint8_t* allowed, const float* v_hist, float* out,
                                          int B, int H, int L, int R, int T, void* stream) {
  SOCKET_REQUIRE(q_probs && key_buckets && allowed && v_hist && out, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(B > 0 && H > 0 && L > 0 && R > 0 && T > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE((int64_t)B * H <= 65535, SOCKET_ERR_SHAPE);
  return launch_collision_i16<float>(q_probs, key_buckets, allowed, v_hist, SOCKET_F32, out, B, H, L, R, T,
                                     (hipStream_t)stream);
}

extern "C" int socket_soft_hash_collision_typed(const void* q_probs, int q_dtype, const int16_t* key_buckets,
                                                const uint8_t* allowed, const void* v_hist, int v_dtype, float* out,
                                                int B, int H, int L, int R, int T, void* stream) {
  SOCKET_REQUIRE(q_probs && key_buckets && allowed && v_hist && out, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(socket_dtype_bytes(q_dtype) != 0 && socket_dtype_bytes(v_dtype) != 0, SOCKET_ERR_UNSUPPORTED);
  SOCKET_REQUIRE(B > 0 && H > 0 && L > 0 && R > 0 && T > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE((int64_t)B * H <= 65535, SOCKET_ERR_SHAPE);
  hipStream_t s = (hipStream_t)stream;
  if (q_dtype == SOCKET_F32)
    return launch_collision_i16<float>((const float*)q_probs, key_buckets, allowed, v_hist, v_dtype, out, B, H, L, R, T, s);
  if (q_dtype == SOCKET_F16)
    return launch_collision_i16<uint16_t>((const uint16_t*)q_probs, key_buckets, allowed, v_hist, v_dtype, out, B, H, L, R, T, s);
  return launch_collision_i16<Bf16Entry>((const Bf16Entry*)q_probs, key_buckets, allowed, v_hist, v_dtype, out, B, H, L, R, T, s);
}

extern "C" int socket_finish_list(int32_t* list, int32_t* list_len, const uint8_t* allowed, int rows, int T, int sink, int window,
                                  int heavy, void* stream) {
  SOCKET_REQUIRE(list && list_len && allowed, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(rows > 0 && T > 0 && sink >= 0 && window >= 0 && sink <= T && window <= T && heavy >= 0, SOCKET_ERR_SHAPE);
  const int64_t width = (int64_t)sink + window + heavy + 1;      // (at least the row's)
  SOCKET_REQUIRE(width < INT32_MAX - kFinishEntries, SOCKET_ERR_SHAPE);
  const unsigned parts = (unsigned)((width + kFinishEntries - 1) / kFinishEntries);
  SOCKET_REQUIRE(parts <= 65535, SOCKET_ERR_SHAPE);
  hipLaunchKernelGGL(finish_list_kernel, dim3((unsigned)rows, parts), dim3(256), 0, (hipStream_t)stream, list, list_len, allowed, T, sink,
                     window, heavy);
  SOCKET_LAUNCH_CHECK();
  return SOCKET_OK;
}

extern "C" int socket_soft_hash_score_f16(const uint16_t* q_probs, const int16_t* key_buckets,
                                          const uint16_t* v_norm, const uint8_t* allowed, float* out,
                                          int B, int H, int L, int R, int T, void* stream) {
  SOCKET_REQUIRE(q_probs && key_buckets && allowed && v_norm && out, SOCKET_ERR_NULL);
  SOCKET_REQUIRE(B > 0 && H > 0 && L > 0 && R > 0 && T > 0, SOCKET_ERR_SHAPE);
  SOCKET_REQUIRE((int64_t)B * H <= 65535, SOCKET_ERR_SHAPE);
  return launch_collision_i16<uint16_t>(q_probs, key_buckets, allowed, v_norm, SOCKET_F16, out, B, H, L, R, T,
                                        (hipStream_t)stream);
}
