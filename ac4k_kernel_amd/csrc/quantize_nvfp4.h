// Parts of the nvfp4 quantizers that the kernels of quantize.hip and of the attention front end share.
#pragma once

#include "ac4k_common.h"

namespace ac4k {

// Elements [k, k + 8) of a row of K >= 8 that starts at any element: one 16-byte load at 2-byte alignment (the target
// allows it).  A row's last, partial vector is loaded eight elements before the row's end instead - nothing behind the
// row is read - and row_tail_u4 moves its elements into place, zeros behind them.
__device__ __forceinline__ uint4 ld_row_u4(const uint16_t *row, int64_t k, int64_t K) {
  const u32x4 v = *reinterpret_cast<const u32x4_elem *>(row + (k + 8 <= K ? k : K - 8));
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint4 row_tail_u4(uint4 v, int64_t k, int64_t K) {
  if (k < K && k + 8 > K) {
    const unsigned __int128 w = __builtin_bit_cast(unsigned __int128, v) >> (16 * (int)(k + 8 - K));
    v = __builtin_bit_cast(uint4, w);
  }
  return v;
}
__device__ __forceinline__ uint4 ld_elem_u4(const uint16_t *p) {
  const u32x4 v = *reinterpret_cast<const u32x4_elem *>(p);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// first row that the group of eight rows from row0 on reads and writes (row0 < R)
__device__ __forceinline__ int64_t crossmajor_rows(int64_t row0, int64_t R) { return row0 + 8 <= R ? row0 : R - 8; }

// bf16 component j (0..7) of a 16-byte vector as float
__device__ __forceinline__ float bf16_comp(const uint4 &v, int j) {
  const uint32_t w = (j >> 1) == 0 ? v.x : (j >> 1) == 1 ? v.y : (j >> 1) == 2 ? v.z : v.w;
  return (j & 1) ? bf16_hi(w) : bf16_lo(w);
}

// element-wise |bf16| maximum of two vectors of eight
__device__ __forceinline__ uint4 absmax_bf16x8_pairwise(uint4 acc, uint4 v) {
  auto mx = [](uint32_t a, uint32_t b) {
    const u16x2 r = __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b & 0x7fff7fffu));
    return __builtin_bit_cast(uint32_t, r);
  };
  return make_uint4(mx(acc.x, v.x), mx(acc.y, v.y), mx(acc.z, v.z), mx(acc.w, v.w));
}
__device__ __forceinline__ uint32_t u16_comp(const uint4 &v, int j) {
  const uint32_t w = (j >> 1) == 0 ? v.x : (j >> 1) == 1 ? v.y : (j >> 1) == 2 ? v.z : v.w;
  return (j & 1) ? (w >> 16) : (w & 0xffffu);
}

// source position inside a 32-group (nvfp4) or 16-group (fp8) of output position p
__device__ __forceinline__ int nvfp4_swizzle_src(int p) { return ((p & 7) >> 1) * 8 + (p >> 3) * 2 + (p & 1); }
__device__ __forceinline__ int fp8_swizzle_src(int p) { return ((p & 3) >> 1) * 8 + (p >> 2) * 2 + (p & 1); }

// Rows along the contiguous dim, blocks along the strided one: a lane quantizes the 16 positions of block kb (0..3) of
// 64-chunk cc for the eight rows from group0 on (quads of lanes hold the four blocks of a chunk).  out: rows of Kp / 2
// packed bytes; sfcol: the scale dwords of this chunk, one per row, pad rows included.
template <bool SWIZZLE>
__device__ __forceinline__ void nvfp4_crossmajor_lane(uint8_t *out, uint32_t *sfcol, const uint16_t *in, int64_t sK, int64_t R,
                                                      int64_t K, int64_t Kp, int64_t cc, int64_t group0, int kb, float alpha,
                                                      const float *lut) {
  const bool rows_valid = group0 < R;
  const int64_t row0 = rows_valid ? crossmajor_rows(group0, R) : group0;  // first of the lane's eight rows
  const uint16_t *src = in + row0;

  uint4 v[16];
  uint4 m8 = make_uint4(0, 0, 0, 0);
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int p = (kb & 1) * 16 + i;  // output position inside the 32-group
    const int64_t k = cc * 64 + (kb >> 1) * 32 + (SWIZZLE ? nvfp4_swizzle_src(p) : p);
    v[i] = make_uint4(0, 0, 0, 0);
    if (rows_valid && k < K) v[i] = ld_elem_u4(src + k * sK);
  }
#pragma unroll
  for (int i = 0; i < 16; ++i) m8 = absmax_bf16x8_pairwise(m8, v[i]);

  uint32_t code[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float o = nvfp4_block_scale(bf16_bits_to_f32(u16_comp(m8, j)), alpha, lut, code[j]);
    if (!rows_valid) code[j] = 0;  // pad rows carry zero scales
    float f0[8], f1[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      f0[i] = bf16_comp(v[i], j) * o;
      f1[i] = bf16_comp(v[8 + i], j) * o;
    }
    const uint2 packed = (o != o) ? make_uint2(0x77777777u, 0x77777777u) : make_uint2(f32x8_to_e2m1x8(f0), f32x8_to_e2m1x8(f1));
    if (rows_valid)
      *reinterpret_cast<uint2 *>(out + (row0 + j) * (Kp / 2) + cc * 32 + kb * 8) = packed;
  }
  // scale dword of (row, chunk) = the codes of the four lanes of the quad; lane kb stores rows 2kb, 2kb+1
  uint32_t sfw[8];
#pragma unroll
  for (int j = 0; j < 8; ++j)
    sfw[j] = dpp_u32<0x00>(code[j]) | (dpp_u32<0x55>(code[j]) << 8) | (dpp_u32<0xAA>(code[j]) << 16) |
             (dpp_u32<0xFF>(code[j]) << 24);
  const uint2 mine = kb == 0 ? make_uint2(sfw[0], sfw[1])
                   : kb == 1 ? make_uint2(sfw[2], sfw[3])
                   : kb == 2 ? make_uint2(sfw[4], sfw[5]) : make_uint2(sfw[6], sfw[7]);
  if (row0 == group0) {
    *reinterpret_cast<uint2 *>(sfcol + row0 + 2 * kb) = mine;
  } else {  // group moved back to end at R: the pad rows of its place in the grid are zeros
    sfcol[row0 + 2 * kb] = mine.x;
    sfcol[row0 + 2 * kb + 1] = mine.y;
    if (group0 + 2 * kb >= R) sfcol[group0 + 2 * kb] = 0u;
    if (group0 + 2 * kb + 1 >= R) sfcol[group0 + 2 * kb + 1] = 0u;
  }
}

}  // namespace ac4k
