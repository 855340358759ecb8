// What the linear kernels of linear.hip and linear_fused.hip share.
#pragma once

#include "ac4k_common.h"

namespace ac4k {

// --- output / bias element types -------------------------------------------
template <int DT>
struct Elem;
template <>
struct Elem<AC4K_DTYPE_BF16> {
  using T = uint16_t;
  static __device__ __forceinline__ float load(const void *p, int64_t i) {
    return bf16_bits_to_f32(static_cast<const uint16_t *>(p)[i]);
  }
  // round to nearest even, NaN stays NaN: v_cvt_pk_bf16_f32
  static __device__ __forceinline__ T cvt(float f) { return __builtin_bit_cast(uint16_t, (__bf16)f); }
  static __device__ __forceinline__ uint32_t cvt2(float lo, float hi) {
    typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  }
};
template <>
struct Elem<AC4K_DTYPE_FP16> {
  using T = _Float16;
  static __device__ __forceinline__ float load(const void *p, int64_t i) {
    return (float)static_cast<const _Float16 *>(p)[i];
  }
  static __device__ __forceinline__ T cvt(float f) { return (_Float16)f; }
  static __device__ __forceinline__ uint32_t cvt2(float lo, float hi) {
    const f16x2 v = {(_Float16)lo, (_Float16)hi};
    return __builtin_bit_cast(uint32_t, v);
  }
};
template <>
struct Elem<AC4K_DTYPE_FP32> {
  using T = float;
  static __device__ __forceinline__ float load(const void *p, int64_t i) {
    return static_cast<const float *>(p)[i];
  }
  static __device__ __forceinline__ T cvt(float f) { return f; }
  static __device__ __forceinline__ uint32_t cvt2(float lo, float) { return __float_as_uint(lo); }  // unused: 4-byte outputs are not packed
};
constexpr int BIAS_NONE = 3;

// dword `w` (8 nibbles) times block scale `sc` (both halves of `sc2` hold candidates, HI picks)
template <bool HI>
__device__ __forceinline__ f16x8 decode_dword(uint32_t w, f16x2 sc2) {
  const f16x2 sc = HI ? (f16x2){sc2.y, sc2.y} : (f16x2){sc2.x, sc2.x};
  f16x2 d0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0) * sc;
  f16x2 d1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1) * sc;
  f16x2 d2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2) * sc;
  f16x2 d3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3) * sc;
  return (f16x8){d0.x, d0.y, d1.x, d1.y, d2.x, d2.y, d3.x, d3.y};
}

// --- 16 weight rows per workgroup ------------------------------------------------
constexpr int R16_ROWS = 16, R16_WAVES = 8, R16_STEP = 128;
// A launch carries fewer than 2^32 threads along a grid dim and drops the rest without an error: weights of up to 2^27 - 16 rows.
static inline bool rows16_grid_ok(int64_t N) { return ceil_div(N, R16_ROWS) * (64 * R16_WAVES) < (1ll << 32); }

// End of these kernels: the sums of the eight waves in the order of the waves, scale, bias, store.
template <int D_DT, int BIAS_DT, int MT>
__device__ __forceinline__ void rows16_finish(const f32x4 (&acc)[MT][2], float4 (*part)[MT][64], void *out, const void *bias, float scale,
                                              int64_t M, int64_t N, int64_t n0) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  // lane (r, g): activation row r of tile i, weight rows 4 g .. 4 g + 3
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const f32x4 v = acc[i][0] + acc[i][1];
    part[wave][i][lane] = make_float4(v[0], v[1], v[2], v[3]);
  }
  __syncthreads();
  if (wave >= MT) return;
  float4 v = part[0][wave][lane];
#pragma unroll
  for (int q = 1; q < R16_WAVES; ++q) {
    const float4 o = part[q][wave][lane];
    v.x += o.x, v.y += o.y, v.z += o.z, v.w += o.w;
  }
  const int m = wave * 16 + r;
  const int64_t n = n0 + g * 4;
  if (m >= (int)M || n >= N) return;
  using DE = Elem<D_DT>;
  float o[4] = {v.x * scale, v.y * scale, v.z * scale, v.w * scale};
  if constexpr (BIAS_DT != BIAS_NONE) {
#pragma unroll
    for (int q = 0; q < 4; ++q) o[q] += n + q < N ? Elem<BIAS_DT>::load(bias, n + q) : 0.0f;
  }
  typename DE::T *dst = static_cast<typename DE::T *>(out) + (int64_t)m * N + n;
  if ((N & 3) == 0 && ((uintptr_t)out & 15) == 0) {
    if constexpr (sizeof(typename DE::T) == 2)
      *reinterpret_cast<uint2 *>(dst) = make_uint2(DE::cvt2(o[0], o[1]), DE::cvt2(o[2], o[3]));
    else
      *reinterpret_cast<float4 *>(dst) = make_float4(o[0], o[1], o[2], o[3]);
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (n + q < N) dst[q] = DE::cvt(o[q]);
  }
}

// quantize and linear in one launch (linear_fused.hip); rows16 kernels fit the shape and the operands are on 16 bytes
struct FusedArgs {
  void *D;
  const uint16_t *X;       // [M, K] bf16; null: the activation is in X_q, X_sf and X_gs (M <= 16)
  uint8_t *X_q, *X_sf;     // the quantized activation, for the caller
  float *X_gs;
  const uint8_t *B;
  const uint32_t *B_sf;
  const float *B_gs;
  const void *bias;
  int64_t M, N, K, Mp, Np;
};
constexpr int64_t FUSED_ELEMS = 16384;  // of the activation
int launch_fused_rows16(const FusedArgs &a, int d_dtype, int bias_dtype, hipStream_t st);

}  // namespace ac4k
