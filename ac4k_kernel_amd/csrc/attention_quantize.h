// Front ends of the two attention forwards: quantization of bf16 Q, K and V into a workspace.
#pragma once

#include "ac4k_common.h"

namespace ac4k {

struct AttnOperand {
  const uint16_t *p;  // bf16 [B, N, H, D] or [B, H, N, D], head dim contiguous
  int64_t s_b, s_h, s_n;
};

constexpr int AQ_Q_BLOCK = 64, AQ_K_BLOCK = 128;  // tokens per int8 scale

struct AttnQuantArgs {
  AttnOperand q, k, v;
  int B, H, Nq, Nkv, D, Dv;
  float v_smax;
  // filled by attn_quant_plan
  int nsplit, span;
  int waves;    // of a workgroup of the statistics
  int classes;  // 0, or: the tiles take the statistics themselves, a span as so many interleaved sums
  float inv_nkv;
  // filled by attn_quant_layout: the operands of ac4k_mha_int8_x_fp8_fwd and the partial results, all in the workspace
  int Dp, Dvp, nqb, nkb, nvb;
  int64_t Nkv16;
  int8_t *q8, *k8;
  uint8_t *v8;
  float *q_sf, *k_sf, *v_sf, *ksum;
  uint32_t *vmax;
};

int64_t attn_quant_layout(AttnQuantArgs &a, void *ws);  // -> bytes of the workspace (ws may be null: size only)
void attn_quant_plan(AttnQuantArgs &a);
void launch_attn_quant(const AttnQuantArgs &a, hipStream_t st);

constexpr int AQ_MAX_PARTS = 256;  // workgroups per tensor of the maximum kernel

struct AttnNvfp4Args {
  AttnOperand q, k, v;  // dense
  int B, H, Nq, Nkv, D, Dv;
  float max_scale;
  // filled by attn_nvfp4_layout: the operands of ac4k_mha_nvfp4_fwd and the partial maxima, all in the workspace
  int Dp, Dvp, Nqp, Nkvp, Nkv64, nqt, nkt, nvt;
  uint8_t *q4, *k4, *v4, *q_sf, *k_sf, *v_sf;
  float *gs;             // global scales of Q, K, V, four bytes apart
  uint32_t *parts;       // [3][AQ_MAX_PARTS]
  int nparts[3];
};

int64_t attn_nvfp4_layout(AttnNvfp4Args &a, void *ws);
void launch_attn_nvfp4(const AttnNvfp4Args &a, hipStream_t st);

// int8 block scale = max|x| / 127 of a block of bf16 values, q = int8(trunc(x / scale)).
// One correction step on x * (1 / scale) gives the correctly rounded quotient: residual by fma, times the correctly rounded
// reciprocal (Markstein's division step).  For bf16 x with |x| <= max and scale = max / 127 it equals the IEEE division
// for every significand pair and exponent distance - all 1 024 320 combinations were compared - as long as nothing
// underflows; blocks with a maximum below 2^-90 divide.  Three vector instructions instead of about ten per element.
struct Int8BlockScale {
  float scale, inv;
  bool divide;
  __device__ __forceinline__ explicit Int8BlockScale(uint32_t absmax_bits) {
    const float m = bf16_bits_to_f32(absmax_bits);
    scale = m / 127.0f;
    inv = scale != 0.0f ? 1.0f / scale : 0.0f;
    divide = m < 0x1p-90f;
  }
  __device__ __forceinline__ uint32_t quantize4(float a, float b, float c, float d) const {
    const float x[4] = {a, b, c, d};
    uint32_t w = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float q;
      if (divide) {  // (uniform over the block)
        q = scale != 0.0f ? x[e] / scale : 0.0f;
      } else {
        const float q0 = x[e] * inv;
        q = __builtin_fmaf(__builtin_fmaf(-q0, scale, x[e]), inv, q0);
      }
      w |= ((uint32_t)(int)q & 0xffu) << (8 * e);  // toward zero; |q| <= 127 up to rounding
    }
    return w;
  }
  __device__ __forceinline__ uint2 quantize8(uint4 v) const {
    return make_uint2(quantize4(bf16_lo(v.x), bf16_hi(v.x), bf16_lo(v.y), bf16_hi(v.y)),
                      quantize4(bf16_lo(v.z), bf16_hi(v.z), bf16_lo(v.w), bf16_hi(v.w)));
  }
};

}  // namespace ac4k
