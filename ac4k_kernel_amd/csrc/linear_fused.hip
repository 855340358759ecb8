// Decode-sized linear on a bf16 activation that is small enough for every workgroup to quantize it itself: one launch where
// quantize + linear are two, the second of which waits for the first; and the same kernel on an activation that is quantized already.
#include "linear_common.h"

namespace ac4k {

// A workgroup takes 16 weight rows and all of K, as linear_nvfp4_rows16_kernel does, with its first weights under way while it
// reads the whole activation (from the L2, all but the first time), takes its maximum and quantizes it - a thread one or two 16-blocks,
// by the quantizers' own steps, so the operands are theirs bit for bit.  The activation stays in LDS as the fp16 operands of
// the MFMAs and is not decoded again for every workgroup's weights.  Workgroup 0 stores the packed activation for the caller.
// Bound by the weights from memory (1 x 28672 x 8192: 140.4 MiB read for 126.0 in 31 us, 4.7 TB/s); small ones by the launch.
// Two launches -> one, us in a graph, weights from HBM: 1 x 4096 x 4096 8.1 -> 5.9, 1 x 14336 x 4096 13.9 -> 11.5, 1 x 4096 x 14336 14.2 -> 11.3, 4 x 4096 x 4096 8.5 -> 6.7, 16 x 4096 x 1024 6.2 -> 4.6,
// 1 x 1024 x 2048 5.9 -> 4.0; called one after the other 1 x 4096 x 4096 22.2 -> 19.4 (host time), 1 x 28672 x 8192 33.0 -> 31.4.
// DEPTH steps of weights in flight per wave: four, and six for K above 4096 on 16384 rows and more, several rounds of workgroups.  It is
// K = 8192 and 16384 that need them (rows a power of two apart meet on few memory channels, and a step takes longer to come; us in a graph,
// four / six): 1 x 28672 x 8192 33.1 / 31.0, 1 x 20480 x 8192 25.5 / 24.0, 2 x 16384 x 8192 23.5 / 22.0, 1 x 16384 x 16384 35.3 / 34.6.  Other K do
// not mind (1 x 28672 x 5120 22.8 / 22.7, 1 x 20480 x 12288 32.3 / 32.9, 3 x 28672 x 5120 25.1 / 24.6), short ones neither (1 x 28672 x 4096 19.3 /
// 19.4), and fewer rows lose as often as they gain (1 x 8192 x 12288 15.1 / 16.2, 1 x 8192 x 5120 9.1 / 9.4, 1 x 14336 x 8192 20.5 / 19.1).
constexpr int FU_THREADS = 64 * R16_WAVES;
constexpr int FU_BLOCKS = (int)(FUSED_ELEMS / 16 / FU_THREADS);  // 16-blocks of a thread
constexpr int FU_PAD = 8;  // elements between the rows in LDS: rows start on different banks

// PACKED: X_q, X_sf and X_gs hold the activation, quantized before; M <= 16.
template <int D_DT, int BIAS_DT, int MT, int DEPTH, bool PACKED>
__global__ __launch_bounds__(FU_THREADS, 2) void linear_nvfp4_fused_rows16_kernel(FusedArgs a) {
  __shared__ __attribute__((aligned(16))) _Float16 xs[FUSED_ELEMS + 16 * MT * FU_PAD];
  __shared__ float4 part[R16_WAVES][MT][64];
  __shared__ float lut[128];
  __shared__ uint32_t red[R16_WAVES];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r = lane & 15, g = lane >> 4;
  const int K = (int)a.K, M = (int)a.M, pitch = K + FU_PAD;
  const int64_t n0 = (int64_t)blockIdx.x * R16_ROWS, kb = a.K >> 1;
  const int nst = K / R16_STEP, cnt = (nst - wave + R16_WAVES - 1) / R16_WAVES;  // steps of this wave; none where K is short
  const int wr = n0 + r < a.N ? r : (int)(a.N - 1 - n0);  // rows past N read the last row; their outputs are never stored
  const uint8_t *const w_src = uniform_ptr(a.B + n0 * kb), *const ws_src = uniform_ptr(reinterpret_cast<const uint8_t *>(a.B_sf) + n0 * 4);
  const uint32_t w_lane = (uint32_t)(wr * kb + g * 16), ws_lane = (uint32_t)((g >> 1) * a.Np * 4 + wr * 4 + (g & 1) * 2);
  struct Step {
    uint4 w;
    uint32_t ws;
  };
  auto load = [&](Step &st, int t) {
    const int s = wave + t * R16_WAVES;
    st.w = *reinterpret_cast<const uint4 *>(w_src + (int64_t)s * (R16_STEP / 2) + w_lane);
    st.ws = *reinterpret_cast<const uint16_t *>(ws_src + (int64_t)(2 * s) * a.Np * 4 + ws_lane);
  };

  // the activation first: what follows waits for it
  const int blocks = M * (K / 16);
  Step ring[DEPTH];
  auto first_steps = [&] {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      if (d < cnt) load(ring[d], d);
  };
  auto keep = [&](int row, int kblk, uint32_t p0, uint32_t p1, uint32_t code) {
    const f16x2 sc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(code, 1.0f, false);
    f16x8 *const x = reinterpret_cast<f16x8 *>(xs + row * pitch + kblk * 16);
    x[0] = decode_dword<false>(p0, sc), x[1] = decode_dword<false>(p1, sc);
  };
  float gs;
  if constexpr (PACKED) {
    uint2 v[FU_BLOCKS];
    uint32_t code[FU_BLOCKS];
    gs = *a.X_gs;
#pragma unroll
    for (int i = 0; i < FU_BLOCKS; ++i) {
      const int b = tid + i * FU_THREADS;
      v[i] = make_uint2(0, 0), code[i] = 0;
      if (b >= blocks) continue;
      const int row = b / (K / 16), kblk = b - row * (K / 16);
      v[i] = reinterpret_cast<const uint2 *>(a.X_q)[b], code[i] = a.X_sf[((int64_t)(kblk >> 2) * a.Mp + row) * 4 + (kblk & 3)];
    }
    first_steps();
#pragma unroll
    for (int i = 0; i < FU_BLOCKS; ++i) {
      const int b = tid + i * FU_THREADS, row = b / (K / 16);
      if (b < blocks) keep(row, b - row * (K / 16), v[i].x, v[i].y, code[i]);
    }
  } else {
    uint4 v[FU_BLOCKS][2];
#pragma unroll
    for (int i = 0; i < FU_BLOCKS; ++i) {
      const int b = tid + i * FU_THREADS;
      v[i][0] = v[i][1] = make_uint4(0, 0, 0, 0);
      if (b < blocks) v[i][0] = reinterpret_cast<const uint4 *>(a.X)[2 * b], v[i][1] = reinterpret_cast<const uint4 *>(a.X)[2 * b + 1];
    }
    first_steps();
    uint32_t bm[FU_BLOCKS], m = 0;
#pragma unroll
    for (int i = 0; i < FU_BLOCKS; ++i) {
      bm[i] = umax32(absmax_bf16x8(v[i][0]), absmax_bf16x8(v[i][1]));
      m = umax32(m, bm[i]);
    }
    m = group_umax<64>(m);
    if (lane == 0) red[wave] = m;
    load_rcp_table(lut);  // (ends with a barrier)
    gs = bf16_bits_to_f32(group_umax<8>(red[lane & 7])) / 2688.0f;
    const float alpha = 1.0f / gs;
#pragma unroll
    for (int i = 0; i < FU_BLOCKS; ++i) {
      const int b = tid + i * FU_THREADS;
      if (b >= blocks) break;
      uint32_t code;
      const float o = nvfp4_block_scale(bf16_bits_to_f32(bm[i]), alpha, lut, code);
      const uint32_t p0 = nvfp4_pack8(v[i][0], o), p1 = nvfp4_pack8(v[i][1], o);
      const int row = b / (K / 16), kblk = b - row * (K / 16);
      keep(row, kblk, p0, p1, code);
      if (blockIdx.x == 0) {
        reinterpret_cast<uint2 *>(a.X_q)[b] = make_uint2(p0, p1);
        a.X_sf[((int64_t)(kblk >> 2) * a.Mp + row) * 4 + (kblk & 3)] = (uint8_t)code;
      }
    }
    if (blockIdx.x == 0) {
      if (tid == 0) *a.X_gs = gs;
      const int pad = (int)a.Mp - M;  // rows whose scales are zero
      for (int i = tid; i < K / 64 * pad; i += FU_THREADS) reinterpret_cast<uint32_t *>(a.X_sf)[(int64_t)(i / pad) * a.Mp + M + i % pad] = 0u;
    }
  }
  __syncthreads();

  int x_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) x_row[i] = (i * 16 + r < M ? i * 16 + r : M - 1) * pitch + g * 32;  // rows past M read the last one
  f32x4 acc[MT][2];  // two independent accumulation chains
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i][0] = acc[i][1] = (f32x4)(0.0f);
  auto multiply = [&](const Step &st, int t) {
    const f16x2 wsc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(st.ws, 1.0f, false);
    const f16x8 w[4] = {decode_dword<false>(st.w.x, wsc), decode_dword<false>(st.w.y, wsc), decode_dword<true>(st.w.z, wsc),
                        decode_dword<true>(st.w.w, wsc)};
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const f16x8 *const x = reinterpret_cast<const f16x8 *>(xs + x_row[i] + (wave + t * R16_WAVES) * R16_STEP);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j & 1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[j], x[j], acc[i][j & 1], 0, 0, 0);
    }
  };
  int t = 0;
  for (; t + DEPTH < cnt; t += DEPTH) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      multiply(ring[d], t + d);
      if (t + d + DEPTH < cnt) load(ring[d], t + d + DEPTH);
    }
  }
#pragma unroll
  for (int d = 0; d < DEPTH; ++d)
    if (t + d < cnt) multiply(ring[d], t + d);
  rows16_finish<D_DT, BIAS_DT, MT>(acc, part, a.D, a.bias, gs * (*a.B_gs), a.M, a.N, n0);
}

template <int D_DT, int BIAS_DT, bool PACKED>
static int launch(const FusedArgs &a, hipStream_t st) {
  const bool deep = a.K > 4096 && a.N >= 16384;  // (K > 4096: M <= 3)
  void (*kern)(FusedArgs) = deep ? linear_nvfp4_fused_rows16_kernel<D_DT, BIAS_DT, 1, 6, PACKED> : linear_nvfp4_fused_rows16_kernel<D_DT, BIAS_DT, 1, 4, PACKED>;
  if constexpr (!PACKED)
    if (a.M > 16) kern = linear_nvfp4_fused_rows16_kernel<D_DT, BIAS_DT, 2, 4, PACKED>;
  hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(a.N, R16_ROWS)), dim3(FU_THREADS), 0, st, a);
  return 0;
}

template <int D_DT, bool PACKED>
static int launch_bias(const FusedArgs &a, int bias_dtype, hipStream_t st) {
  if (!a.bias) return launch<D_DT, BIAS_NONE, PACKED>(a, st);
  switch (bias_dtype) {
    case AC4K_DTYPE_BF16: return launch<D_DT, AC4K_DTYPE_BF16, PACKED>(a, st);
    case AC4K_DTYPE_FP16: return launch<D_DT, AC4K_DTYPE_FP16, PACKED>(a, st);
    case AC4K_DTYPE_FP32: return launch<D_DT, AC4K_DTYPE_FP32, PACKED>(a, st);
  }
  return set_error("bias must be bfloat16, half or float (dtype tag %d)", bias_dtype);
}

template <bool PACKED>
static int launch_dtype(const FusedArgs &a, int d_dtype, int bias_dtype, hipStream_t st) {
  switch (d_dtype) {
    case AC4K_DTYPE_BF16: return launch_bias<AC4K_DTYPE_BF16, PACKED>(a, bias_dtype, st);
    case AC4K_DTYPE_FP16: return launch_bias<AC4K_DTYPE_FP16, PACKED>(a, bias_dtype, st);
    case AC4K_DTYPE_FP32: return launch_bias<AC4K_DTYPE_FP32, PACKED>(a, bias_dtype, st);
  }
  return set_error("d must be bfloat16, half or float (dtype tag %d)", d_dtype);
}

int launch_fused_rows16(const FusedArgs &a, int d_dtype, int bias_dtype, hipStream_t st) {
  return a.X ? launch_dtype<false>(a, d_dtype, bias_dtype, st) : launch_dtype<true>(a, d_dtype, bias_dtype, st);
}

}  // namespace ac4k
