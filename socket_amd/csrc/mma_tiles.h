// What the prompt attention kernels share: 32x32 matrix products in 16-bit types, tiles of 64 keys copied from
// global memory straight into LDS, and transposing reads of them.
#pragma once
#include "elem.h"

namespace {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 pa_bf16x8;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 pa_f16x8;
typedef float pa_f32x16 __attribute__((ext_vector_type(16)));
typedef short pa_s16x4 __attribute__((ext_vector_type(4)));

template <class DT>
struct PaType;
template <>
struct PaType<DType_bf16> {
  static __device__ __forceinline__ pa_f32x16 mfma(const uint4& a, const uint4& b, pa_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(pa_bf16x8, a), __builtin_bit_cast(pa_bf16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{lo, hi}, bf2));
  }
  static __device__ __forceinline__ float low(uint32_t w) { return __uint_as_float(w << 16); }
  static __device__ __forceinline__ float high(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
};
template <>
struct PaType<DType_f16> {
  static __device__ __forceinline__ pa_f32x16 mfma(const uint4& a, const uint4& b, pa_f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(pa_f16x8, a), __builtin_bit_cast(pa_f16x8, b), c, 0, 0, 0);
  }
  static __device__ __forceinline__ uint32_t pack2(float lo, float hi) {
    typedef _Float16 h2 __attribute__((ext_vector_type(2)));
    typedef float f2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{lo, hi}, h2));
  }
  static __device__ __forceinline__ float low(uint32_t w) { return f16_bits_to_f32((uint16_t)(w & 0xffffu)); }
  static __device__ __forceinline__ float high(uint32_t w) { return f16_bits_to_f32((uint16_t)(w >> 16)); }
};

constexpr int kPaKeys = 64;      // keys of a tile
constexpr int kPaWaves = 4;
constexpr float kPaLog2e = 1.4426950408889634f;

// x * c rounded, then less m: not contracted, so that the largest score gives exactly zero.
__device__ __forceinline__ float pa_scaled_minus(float x, float c, float m) {
#pragma clang fp contract(off)
  const float y = x * c;
  return y - m;
}

// Where a row's 16-byte pieces go (CH of them): piece ^ pa_swizzle(key).  Sixteen keys at one piece
// must fall on sixteen 16-byte bank groups (rows of 128 bytes start half a bank line apart by the
// key's parity), and the four keys x 64 bytes of a transposing read on all of them.
template <int CH>
__device__ __forceinline__ int pa_swizzle(int key) {
  if constexpr (CH == 16) return ((key & 3) << 2) | ((key >> 2) & 3);
  else return (((key >> 1) & 1) << 2) | (((key >> 2) & 1) << 1) | ((key >> 3) & 1);
}

// 16 bytes per lane from base + off into LDS (see lds_dma16); `base` is the same for the whole wave.
__device__ __forceinline__ void pa_dma16(const char* base, uint32_t off, void* lds_dst) {
  const uint32_t at = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds_dst);
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %2\n\t"
      "s_nop 0\n\t"
      "global_load_lds_dwordx4 %1, %3\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(off), "s"(at), "s"(base)
      : "memory");
}

// A tile of CH-piece rows into LDS: wave `wave` of kPaWaves issues its share of the copies.  row(key)
// tells where a key's row starts, or the rows are `stride` bytes apart from `first` on.
template <int CH, class ROW>
__device__ __forceinline__ void pa_copy_rows(ROW row, unsigned char* tile, int wave, int lane) {
  constexpr int N = kPaKeys * CH / 64 / kPaWaves;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int s = (wave * N + i) * 64 + lane, key = s / CH, piece = s % CH ^ pa_swizzle<CH>(key);
    lds_dma16(row(key) + piece * 16, tile + (wave * N + i) * 1024);
  }
}
template <int CH>
__device__ __forceinline__ void pa_copy_tile(const char* first, int64_t stride, unsigned char* tile, int wave, int lane) {
  constexpr int N = kPaKeys * CH / 64 / kPaWaves;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int s = (wave * N + i) * 64 + lane, key = s / CH, piece = s % CH ^ pa_swizzle<CH>(key);
    pa_dma16(first, (uint32_t)(key * (int)stride + piece * 16), tile + (wave * N + i) * 1024);
  }
}

// V^T fragment of 32 dims x 16 keys from a tile of CH-piece rows: keys key0 .. + 15 in the order of the
// accumulators (lane half h: 4 h .. + 3, 8 + 4 h .. + 3), dims 32 db .. + 31.  Lane i of a group of 16 names key
// i / 4 of four and dims 4 (i % 4) .. + 3; groups are (dims 0-15 | 16-31) x (h = 0 | 1).
template <int CH>
__device__ __forceinline__ uint4 pa_values(const unsigned char* tile, int key0, int db, int lane) {
  const int v_key = 4 * (lane >> 5) + ((lane >> 2) & 3), v_piece = 2 * ((lane >> 4) & 1) + ((lane >> 1) & 1);
  uint2 v[2];
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const int key = key0 + 8 * e + v_key;
    const int at = key * CH * 16 + (((4 * db + v_piece) ^ pa_swizzle<CH>(key)) << 4) + (lane & 1) * 8;
    v[e] = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) pa_s16x4*)(tile + at)));
  }
  return make_uint4(v[0].x, v[0].y, v[1].x, v[1].y);
}

}  // namespace
