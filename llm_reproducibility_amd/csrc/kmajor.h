// Operand tiles that lie the other way round (K-major: a row-major right operand [K,N], the transposed left operand of a weight
// gradient), in place: a slice of 64 k is 64 rows of the tile's columns, direct loads bring those rows into LDS, and
// ds_read_b64_tr_b16 hands out the MFMA fragments -- 16 lanes read 4 rows x 16 columns and each receives the 4 k of one
// column.  The same elements reach the same MFMA slots as from a [N,K] operand, hence the same bits.
//
// A row of COLS columns is COLS / 8 chunks of 16 bytes; row k keeps chunk c at position c ^ swizzle(k).  A fragment read
// touches rows 8g .. 8g+3 (then 8g+4 .. 8g+7) of two neighbouring chunks per lane group g: the swizzle leaves the two chunks
// side by side and spreads rows that would meet in the same banks (all of them from 128 columns on; every second row of 64
// columns, every fourth of 32) over the row.
#pragma once
#include "common.h"

namespace tbik {
namespace kmajor {

typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

template <int COLS>
__device__ __forceinline__ int swizzle(int k) {
  static_assert(COLS == 32 || COLS == 64 || COLS == 128 || COLS == 256, "rows of 4 to 32 chunks");
  const int g = (k >> 3) & 1;
  return COLS >= 128 ? 2 * ((k & 3) + 4 * g) : COLS == 64 ? 2 * (((k >> 1) & 1) + 2 * g) : 2 * g;
}

// Byte offset (from the tile's first column, row stride ld elements) of what this lane's direct load number `load` of a
// slice brings: linear LDS position load * 64 + lane of the slice's 64 rows.  Columns past `cols` (a multiple of eight) are
// clamped to the last chunk.
template <int COLS>
__device__ __forceinline__ uint32_t load_offset(int load, int lane, int64_t ld, int cols) {
  constexpr int CH = COLS / 8;
  const int q = load * 64 + lane, k = q / CH;
  return (uint32_t)((k * ld + min(((q % CH) ^ swizzle<COLS>(k)) * 8, cols - 8)) * 2);
}
// row of the slice that direct load `load` puts behind this lane
template <int COLS>
__device__ __forceinline__ int load_row(int load, int lane) { return (load * 64 + lane) / (COLS / 8); }

// LDS byte offset of this lane's fragment of the 16 columns of MFMA tile `tile` (of the whole COLS), k step 0 of the slice
template <int COLS>
__device__ __forceinline__ uint32_t frag_offset(int tile, int lane) {
  const int l = lane & 15, g = lane >> 4, k = 8 * g + (l >> 2);
  return (uint32_t)(k * COLS * 2 + ((2 * tile) ^ swizzle<COLS>(k)) * 16 + ((l >> 1) & 1) * 16 + (l & 1) * 8);
}
// the fragment: 8 k of this lane's column, k step kk (32 k each)
template <int COLS>
__device__ __forceinline__ bf16x8 read(uint8_t* tile, uint32_t offset, int kk) {
  __attribute__((address_space(3))) uint8_t* p = (__attribute__((address_space(3))) uint8_t*)tile + offset + kk * (32 * COLS * 2);
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 4 * COLS * 2));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

}  // namespace kmajor
}  // namespace tbik
