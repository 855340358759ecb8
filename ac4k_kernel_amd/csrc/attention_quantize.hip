// The quantizers in front of the INT8 x FP8 attention forward as two launches, for the whole-attention entry point
// (python/ac4k_kernel/ops/attention.py:137-190: K minus its token mean, per-token-block int8 of Q and K, per-channel
// e4m3 of V with the 16-group swizzle).  Operator by operator the same work is nine launches - mean, subtraction, two
// block quantizers, and fill / maxima / quantize / finalize for V - and K crosses memory four times:
//   1. attn_column_stats_kernel     per (head, channel): sum of K and maximum of |V| over a span of tokens, one partial
//                                   result per span (no atomics, so a call gives the same bits every time)
//   2. attn_quantize_int8_fp8_kernel  every workgroup adds up the partials of its own channels (a few KB from L2) and
//                                   quantizes one tile of V, K or Q
// and as one for short heads, whose tiles take the statistics themselves (aq_own_faster).
// Both are bound by HBM: 2 (K + V) bytes read in the first, 2 (Q + K + V) read and half of that written in the second.
// MI355X, quantizers alone: B 1, N 16384, H 40, D 128 (BNHD) 350 -> 208 us = 84 (4.0 TB/s) + 124 (6.1 TB/s); a whole
// attention of 777 queries on 257 keys, B 2, H 12, D 64: 64 -> 21 us, three launches instead of nine, 19 with two.  The operands are those
// of the separate calls bit for bit, except that a channel mean of K summed in another order may round to the other bf16.
#include "attention_quantize.h"
#include "quantize_nvfp4.h"

namespace ac4k {

namespace {

constexpr int AQ_MAX_SPLITS = 32; // token spans: every tile of the second kernel reads one partial row per span
constexpr int AQ_MIN_SPAN = 32;
constexpr int AQ_STAT_WAVES = 16;  // most waves of a workgroup of the first kernel
constexpr int AQ_STAT_LOADS = 8;   // loads in flight per lane there

// Lanes that share one row of a head: eight channels per lane.  The last lane of a head dim that is no multiple of
// eight is moved back to end at it; channels that two lanes share are computed twice, with the same result.
__device__ __forceinline__ int aq_lane_shift(int D) { return D > 64 ? 4 : 3; }
__device__ __forceinline__ int aq_channel(int c, int D) { return c * 8 + 8 <= D ? c * 8 : D - 8; }

__device__ __forceinline__ uint4 aq_load(const uint16_t *p) {
  const u32x4 v = *reinterpret_cast<const u32x4_elem *>(p);
  return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint4 aq_load_stream(const uint16_t *p) {
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_elem *>(p));
  return make_uint4(v.x, v.y, v.z, v.w);
}

// ---- 1. sums of K, maxima of |V| -------------------------------------------------------------------------------
// A wave instruction reads 1 KB: the rows of neighbouring heads of one token where these are neighbours in memory
// (BNHD), rows of neighbouring tokens otherwise (BHND).
template <bool ABSMAX>
__device__ __forceinline__ void aq_column_stats(const AttnQuantArgs &a, const AttnOperand &t, int N, int D, int Dp, void *part,
                                                uint32_t (*red)[64][8]) {
  const int W = blockDim.x >> 6;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ls = aq_lane_shift(D), lpr = 1 << ls, G = 64 >> ls;
  const bool heads_adjacent = t.s_h < t.s_n && a.H > 1;
  const int heads = heads_adjacent ? G : 1, HG = (a.H + heads - 1) / heads;
  const int unit = blockIdx.x;
  if (unit >= a.nsplit * a.B * HG) return;  // (whole workgroup)
  const int hg = unit % HG, b = (unit / HG) % a.B, split = unit / (HG * a.B);
  const int g = lane >> ls, c = lane & (lpr - 1);
  const int head = heads_adjacent ? hg * G + g : hg;
  const bool live = head < a.H && c * 8 < D;
  const int c0 = aq_channel(live ? c : 0, D);
  const uint16_t *src = t.p + b * t.s_b + (live ? head : 0) * t.s_h + c0;
  const int beg = split * a.span, end = beg + a.span < N ? beg + a.span : N;
  const int step = heads_adjacent ? W : W * G;
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  uint32_t m[4] = {0, 0, 0, 0};
  constexpr int U = AQ_STAT_LOADS;
  for (int n = beg + (heads_adjacent ? wave : wave * G + g); n < end; n += U * step) {
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      v[u] = make_uint4(0, 0, 0, 0);
      if (live && n + u * step < end) v[u] = aq_load(src + (int64_t)(n + u * step) * t.s_n);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (ABSMAX) {
          m[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, m[i]), __builtin_bit_cast(u16x2, w[i] & 0x7fff7fffu)));
        } else {
          s[2 * i] += bf16_lo(w[i]);
          s[2 * i + 1] += bf16_hi(w[i]);
        }
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    red[wave][lane][2 * i] = ABSMAX ? m[i] & 0xffffu : __float_as_uint(s[2 * i]);
    red[wave][lane][2 * i + 1] = ABSMAX ? m[i] >> 16 : __float_as_uint(s[2 * i + 1]);
  }
  __syncthreads();
  const int groups = heads_adjacent ? 1 : G;  // lane groups of a wave that hold the same head
  for (int i = tid; i < heads * lpr * 8; i += 64 * W) {
    const int l = i >> 3, e = i & 7, oc = l & (lpr - 1), oh = heads_adjacent ? hg * G + (l >> ls) : hg;
    float sum = 0.f;
    uint32_t mx = 0;
    for (int w = 0; w < W; ++w)
      for (int k = 0; k < groups; ++k) {
        const uint32_t x = red[w][l + k * lpr][e];
        if (ABSMAX) mx = umax32(mx, x);
        else sum += __uint_as_float(x);
      }
    if (oh < a.H && oc * 8 < D) {
      const int64_t at = ((int64_t)split * a.B * a.H + b * a.H + oh) * Dp + aq_channel(oc, D) + e;
      if (ABSMAX) static_cast<uint32_t *>(part)[at] = mx;
      else static_cast<float *>(part)[at] = sum;
    }
  }
}

// MOST: waves that the LDS of a workgroup holds
template <int MOST>
__global__ __launch_bounds__(64 * MOST) void attn_column_stats_kernel(AttnQuantArgs a) {
  __shared__ uint32_t red[MOST][64][8];
  if (blockIdx.y == 0) aq_column_stats<false>(a, a.k, a.Nkv, a.D, a.Dp, a.ksum, red);
  else aq_column_stats<true>(a, a.v, a.Nkv, a.Dv, a.Dvp, a.vmax, red);
}

// workgroup index -> tile: the dim that is nearer in memory runs fastest
__device__ __forceinline__ void aq_tile(const AttnOperand &t, uint32_t H, uint32_t nblk, uint32_t idx, int &b, int &head, int &blk) {
  const uint32_t inner = t.s_h < t.s_n ? H : nblk, i = idx % inner, o = idx / inner;
  if (t.s_h < t.s_n) {
    head = i;
    blk = o % nblk;
    b = o / nblk;
  } else {
    blk = i;
    head = o % H;
    b = o / H;
  }
}

// ---- 2. the tiles ----------------------------------------------------------------------------------------------
// The partial results of a head's channels put together in the order of the spans, a channel per thread: channel[i] = the result of
// add(a, b) over all spans.  Every lane of a tile needs eight of them and used to fetch these from all spans by itself, one span after
// the other, up to 32 waits for the L2.  Whole calls, us, before -> after: 600 queries on 16000 keys of 12 heads 190 -> 174, 2048 x 8 x 100 52.5 -> 46.7,
// 1024 x 40 x 128 56.4 -> 52.0, 16384 x 40 x 128 3336 -> 3300, 2 x 2048 on 512 keys, 12 x 64, 34.7 -> 32.0; sixteen spans in flight the same; eight
// in every lane's registers cost a wave per SIMD (16384 queries on 77 keys 137 -> 145).
constexpr int AQ_PART_LOADS = 8;  // spans in flight
template <typename Add>
__device__ __forceinline__ void aq_join_spans(const uint32_t *part, int D, int nsplit, int64_t pitch, uint32_t *channel, Add add) {
  const int tid = threadIdx.x;
  if (tid < D) {
    uint32_t sum = 0;
    for (int s = 0; s < nsplit; s += AQ_PART_LOADS) {
      uint32_t x[AQ_PART_LOADS];
#pragma unroll
      for (int u = 0; u < AQ_PART_LOADS; ++u) x[u] = s + u < nsplit ? part[(s + u) * pitch + tid] : 0u;
#pragma unroll
      for (int u = 0; u < AQ_PART_LOADS; ++u)
        if (s + u < nsplit) sum = add(sum, x[u]);
    }
    channel[tid] = sum;
  }
  __syncthreads();
}

// The statistics of a short head by its tiles themselves, with no launch in front.  The sums of K are taken in the order of
// aq_column_stats, so they have its bits: a span is a.classes interleaved sums there (its waves, times the tokens that a wave reads at
// once), and `part` holds those of all spans.  Bound by the waits for the loads.
// PAIRS sums of a lane at a time, ROWS tokens of each in flight.
template <int PAIRS, int ROWS>
__device__ __forceinline__ void aq_own_partial_sums(const AttnQuantArgs &a, int b, int head, float *part) {
  const int tid = threadIdx.x, ls = aq_lane_shift(a.D), c = tid & ((1 << ls) - 1), slots = 256 >> ls, pairs = a.nsplit * a.classes;
  if (c * 8 >= a.D) return;
  const int c0 = aq_channel(c, a.D), step = a.classes;
  const uint16_t *src = a.k.p + b * a.k.s_b + head * a.k.s_h + c0;
  for (int p = tid >> ls; p < pairs; p += PAIRS * slots) {
    int n[PAIRS], end[PAIRS];
    float s[PAIRS][8] = {};
#pragma unroll
    for (int q = 0; q < PAIRS; ++q) {
      const int split = (p + q * slots) / step, beg = split * a.span, last = beg + a.span < a.Nkv ? beg + a.span : a.Nkv;
      n[q] = beg + p + q * slots - split * step;
      end[q] = p + q * slots < pairs ? last : 0;
    }
    for (int i = 0; i < a.span; i += ROWS * step) {
      uint4 v[PAIRS][ROWS];
#pragma unroll
      for (int q = 0; q < PAIRS; ++q)
#pragma unroll
        for (int u = 0; u < ROWS; ++u) {
          v[q][u] = make_uint4(0, 0, 0, 0);
          const int k = n[q] + i + u * step;
          if (k < end[q]) v[q][u] = aq_load(src + (int64_t)k * a.k.s_n);
        }
#pragma unroll
      for (int q = 0; q < PAIRS; ++q)
#pragma unroll
        for (int u = 0; u < ROWS; ++u) {
          const uint32_t w[4] = {v[q][u].x, v[q][u].y, v[q][u].z, v[q][u].w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            s[q][2 * e] += bf16_lo(w[e]);
            s[q][2 * e + 1] += bf16_hi(w[e]);
          }
        }
    }
#pragma unroll
    for (int q = 0; q < PAIRS; ++q)
      if (p + q * slots < pairs)
#pragma unroll
        for (int e = 0; e < 8; ++e) part[(p + q * slots) * a.D + c0 + e] = s[q][e];
  }
}
__device__ __forceinline__ void aq_own_sums(const AttnQuantArgs &a, int b, int head, float *part, uint32_t *channel) {
  if (a.classes == 1) aq_own_partial_sums<1, 8>(a, b, head, part);
  else aq_own_partial_sums<2, 4>(a, b, head, part);
  __syncthreads();
  const int tid = threadIdx.x;
  if (tid < a.D) {
    float all = 0.0f;
    for (int split = 0; split < a.nsplit; ++split) {
      float sum = 0.0f;
#pragma unroll 8
      for (int k = 0; k < a.classes; ++k) sum += part[(split * a.classes + k) * a.D + tid];
      all += sum;
    }
    channel[tid] = __float_as_uint(all);
  }
  __syncthreads();
}

// `BLOCK` tokens of one head to int8 with one scale; MEAN: minus the token mean of their channel, both rounded to
// bf16 as the subtraction of two bf16 tensors rounds them.
template <int BLOCK, bool MEAN, bool OWN>
__device__ __forceinline__ void aq_int8_tile(const AttnQuantArgs &a, const AttnOperand &t, int N, int nb, int8_t *y,
                                             float *scale, int b, int head, int blk, uint32_t *wmax, uint32_t *channel, float *part) {
  const int tid = threadIdx.x;
  const int ls = aq_lane_shift(a.D), c = tid & ((1 << ls) - 1), r0 = tid >> ls, rstep = 256 >> ls;
  constexpr int NV = BLOCK / 16;  // vectors per thread with 16 lanes per row (half of them with eight)
  const bool live = c * 8 < a.D;
  const int c0 = aq_channel(live ? c : 0, a.D);
  const int n0 = blk * BLOCK, rows = N - n0 < BLOCK ? N - n0 : BLOCK;
  const int64_t bh = (int64_t)b * a.H + head;
  const uint16_t *src = t.p + b * t.s_b + head * t.s_h + (int64_t)n0 * t.s_n + c0;
  uint4 v[NV];
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int r = r0 + j * rstep;
    v[j] = make_uint4(0, 0, 0, 0);
    if (live && r < rows) v[j] = aq_load_stream(src + r * t.s_n);
  }
  if (MEAN) {
    if constexpr (OWN) aq_own_sums(a, b, head, part, channel);
    else aq_join_spans(reinterpret_cast<const uint32_t *>(a.ksum + bh * a.Dp), a.D, a.nsplit, (int64_t)a.B * a.H * a.Dp, channel,
                  [](uint32_t sum, uint32_t x) { return __float_as_uint(__uint_as_float(sum) + __uint_as_float(x)); });
    float mean[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) mean[e] = (float)(__bf16)(__uint_as_float(channel[c0 + e]) * a.inv_nkv);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      if (!(live && r0 + j * rstep < rows)) continue;  // rows past the end stay zero
      uint32_t w[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint16_t lo = __builtin_bit_cast(uint16_t, (__bf16)(bf16_lo(w[i]) - mean[2 * i]));
        const uint16_t hi = __builtin_bit_cast(uint16_t, (__bf16)(bf16_hi(w[i]) - mean[2 * i + 1]));
        w[i] = lo | ((uint32_t)hi << 16);
      }
      v[j] = make_uint4(w[0], w[1], w[2], w[3]);
    }
  }
  uint32_t mx = 0;
#pragma unroll
  for (int j = 0; j < NV; ++j) mx = umax32(mx, absmax_bf16x8(v[j]));
  mx = group_umax<64>(mx);
  if ((tid & 63) == 0) wmax[tid >> 6] = mx;
  __syncthreads();
  mx = umax32(umax32(wmax[0], wmax[1]), umax32(wmax[2], wmax[3]));
  const Int8BlockScale sc(mx);
  if (tid == 0) scale[bh * nb + blk] = sc.scale;
  int8_t *dst = y + (bh * N + n0) * a.Dp;
#pragma unroll
  for (int j = 0; j < NV; ++j) {
    const int r = r0 + j * rstep;
    if (live && r < rows) st_elem_u2(dst + r * a.Dp + c0, sc.quantize8(v[j]));
  }
  if (a.Dp != a.D) {  // pad columns
    const int pad = a.Dp - a.D;
    for (int i = tid; i < rows * pad; i += 256) dst[(i / pad) * a.Dp + a.D + i % pad] = 0;
  }
}

// 64 kv positions per wave, all channels of one head, to e4m3 along kv (the cross-major layout of the quantizers: a lane
// holds eight channels of 16 stored positions)
template <bool OWN>
__device__ __forceinline__ void aq_fp8_tile(const AttnQuantArgs &a, int b, int head, int blk, uint32_t *channel, uint32_t *part) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, kb = lane & 3, rg = lane >> 2;
  const int64_t bh = (int64_t)b * a.H + head;
  const int k0 = (blk * 4 + wave) * 64 + kb * 16;
  const bool live = rg * 8 < a.Dv;
  const int c0 = aq_channel(live ? rg : 0, a.Dv);
  const uint16_t *src = a.v.p + b * a.v.s_b + head * a.v.s_h + c0;
  uint4 v[16];
  u16x2 top[4] = {};
  auto load = [&](int k1) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int k = k1 + ((i & 3) >> 1) * 8 + (i >> 2) * 2 + (i & 1);  // the 16-group swizzle
      v[i] = make_uint4(0, 0, 0, 0);
      if (live && k < a.Nkv) v[i] = aq_load(src + (int64_t)k * a.v.s_n);
    }
    if constexpr (OWN) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const uint32_t w[4] = {v[i].x, v[i].y, v[i].z, v[i].w};
#pragma unroll
        for (int j = 0; j < 4; ++j) top[j] = __builtin_elementwise_max(top[j], __builtin_bit_cast(u16x2, w[j] & 0x7fff7fffu));
      }
    }
  };
  if constexpr (OWN)
    for (int other = 0; other < a.nvb; ++other)
      if (other != blk) load((other * 4 + wave) * 64 + kb * 16);
  load(k0);
  if constexpr (OWN) {  // maxima of the whole head: over the four lanes of a channel, then over the waves
#pragma unroll
    for (int j = 0; j < 4; ++j) {
#pragma unroll
      for (int x = 1; x < 4; x *= 2)
        top[j] = __builtin_elementwise_max(top[j], __builtin_bit_cast(u16x2, __shfl_xor((int)__builtin_bit_cast(uint32_t, top[j]), x)));
      if (live && kb == 0) part[wave * 128 + c0 + 2 * j] = top[j].x, part[wave * 128 + c0 + 2 * j + 1] = top[j].y;
    }
    __syncthreads();
    if (tid < a.Dv) channel[tid] = umax32(umax32(part[tid], part[128 + tid]), umax32(part[256 + tid], part[384 + tid]));
    __syncthreads();
  } else aq_join_spans(a.vmax + bh * a.Dvp, a.Dv, a.nsplit, (int64_t)a.B * a.H * a.Dvp, channel, [](uint32_t m, uint32_t x) { return umax32(m, x); });
  uint32_t mx[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) mx[e] = channel[c0 + e];
  if (blk == 0 && wave == 0 && kb == 0) {  // the scales of this head
    float *sf = a.v_sf + bh * a.Dvp;
    if (live)
#pragma unroll
      for (int e = 0; e < 8; ++e) sf[c0 + e] = bf16_bits_to_f32(mx[e]) / a.v_smax;
    if (rg == 0)
      for (int d = a.Dv; d < a.Dvp; ++d) sf[d] = 0.0f / a.v_smax;
  }
  if (!live || k0 >= a.Nkv16) return;
  uint8_t *dst = a.v8 + (bh * a.Dv + c0) * a.Nkv16 + k0;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float amax = bf16_bits_to_f32(mx[e]), recp = a.v_smax / amax;
    float f[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const uint32_t w = (e >> 1) == 0 ? v[i].x : (e >> 1) == 1 ? v[i].y : (e >> 1) == 2 ? v[i].z : v[i].w;
      f[i] = ((e & 1) ? bf16_hi(w) : bf16_lo(w)) * recp;
    }
    uint4 o = make_uint4(f32x4_to_e4m3x4(f[0], f[1], f[2], f[3]), f32x4_to_e4m3x4(f[4], f[5], f[6], f[7]),
                         f32x4_to_e4m3x4(f[8], f[9], f[10], f[11]), f32x4_to_e4m3x4(f[12], f[13], f[14], f[15]));
    if (amax == 0.0f) o = make_uint4(0x7f7f7f7fu, 0x7f7f7f7fu, 0x7f7f7f7fu, 0x7f7f7f7fu);  // 0 * inf
    *reinterpret_cast<uint4 *>(dst + (int64_t)e * a.Nkv16) = o;
  }
}

template <bool OWN>
__global__ __launch_bounds__(256) void attn_quantize_int8_fp8_kernel(AttnQuantArgs a) {
  __shared__ uint32_t wmax[4], channel[128];
  extern __shared__ __attribute__((aligned(16))) float aq_part[];  // OWN: aq_own_bytes
  uint32_t idx = blockIdx.x;
  const uint32_t BH = a.B * a.H;
  int b, head, blk;
  const uint32_t nv = BH * a.nvb, nk = BH * a.nkb;
  if (idx < nv) {
    aq_tile(a.v, a.H, a.nvb, idx, b, head, blk);
    aq_fp8_tile<OWN>(a, b, head, blk, channel, reinterpret_cast<uint32_t *>(aq_part));
  } else if (idx < nv + nk) {
    idx -= nv;
    aq_tile(a.k, a.H, a.nkb, idx, b, head, blk);
    aq_int8_tile<AQ_K_BLOCK, true, OWN>(a, a.k, a.Nkv, a.nkb, a.k8, a.k_sf, b, head, blk, wmax, channel, aq_part);
  } else {
    idx -= nv + nk;
    aq_tile(a.q, a.H, a.nqb, idx, b, head, blk);
    aq_int8_tile<AQ_Q_BLOCK, false, OWN>(a, a.q, a.Nq, a.nqb, a.q8, a.q_sf, b, head, blk, wmax, channel, aq_part);
  }
}

// ---- NVFP4 ------------------------------------------------------------------------------------------------------
// (python/ac4k_kernel/ops/attention.py:100-133: three quantize calls) as two launches instead of up to nine: maxima of Q, K
// and V as one partial result per workgroup, then tiles of all three, every workgroup taking the global scale of its
// tensor from the partial results.  MI355X, B 1, N 4096, H 40, D 128 (BHND):
// 73 -> 57 us (25 + 31: 5.0 and 5.2 TB/s) with bit-identical operands, the whole attention 440 -> 431 us.
__global__ __launch_bounds__(512) void attn_nvfp4_absmax_kernel(AttnNvfp4Args a) {
  const int t = blockIdx.y;
  if ((int)blockIdx.x >= a.nparts[t]) return;
  const uint16_t *x = t == 0 ? a.q.p : t == 1 ? a.k.p : a.v.p;
  const int64_t n = (int64_t)a.B * a.H * (t == 0 ? a.Nq : a.Nkv) * (t == 2 ? a.Dv : a.D), nvec = n / 8;
  constexpr int U = 8;  // loads in flight per lane
  const int64_t span = align_up(ceil_div(nvec, (int64_t)a.nparts[t]), 512);
  const int64_t beg = blockIdx.x * span, end = beg + span < nvec ? beg + span : nvec;
  uint32_t m = 0;
  for (int64_t i = beg + threadIdx.x; i < end; i += U * 512) {
    uint4 v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      v[u] = make_uint4(0, 0, 0, 0);
      if (i + u * 512 < end) v[u] = aq_load(x + (i + u * 512) * 8);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) m = umax32(m, absmax_bf16x8(v[u]));
  }
  if (blockIdx.x == 0 && (int64_t)threadIdx.x < n - nvec * 8) m = umax32(m, x[nvec * 8 + threadIdx.x] & 0x7fffu);
  m = group_umax<64>(m);
  __shared__ uint32_t red[8];
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 8; ++w) m = umax32(m, red[w]);
    a.parts[t * AQ_MAX_PARTS + blockIdx.x] = m;
  }
}

// 128 tokens of one head, head dim contiguous: the row-major layout of the quantizers (a lane owns eight elements, a lane
// pair a block, eight lanes a 64-chunk)
__device__ __forceinline__ void aq_nvfp4_tile(const AttnNvfp4Args &a, const AttnOperand &t, int N, int Np, uint8_t *out, uint8_t *sf,
                                              int b, int head, int blk, float alpha, const float *lut) {
  const int tid = threadIdx.x, ls = a.Dp > 64 ? 4 : 3, c = tid & ((1 << ls) - 1), r0 = tid >> ls, rstep = 256 >> ls;
  const int64_t bh = (int64_t)b * a.H + head;
  const uint16_t *src = t.p + b * t.s_b + head * t.s_h + (int64_t)blk * 128 * t.s_n;
  const int rows = N - blk * 128 < 128 ? N - blk * 128 : 128, rows_sf = Np - blk * 128 < 128 ? Np - blk * 128 : 128;
  uint4 v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int r = r0 + j * rstep;
    v[j] = make_uint4(0, 0, 0, 0);
    if (r < rows && c * 8 < a.D) v[j] = ld_row_u4(src + r * t.s_n, c * 8, a.D);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const int r = r0 + j * rstep;
    if (r >= 128) break;
    v[j] = row_tail_u4(v[j], c * 8, a.D);
    uint32_t m = absmax_bf16x8(v[j]), code;
    m = umax32(m, dpp_u32<DPP_QUAD_XOR1>(m));
    const float o = nvfp4_block_scale(bf16_bits_to_f32(m), alpha, lut, code);
    if (r >= rows) code = 0;  // pad rows carry zero scales
    const uint32_t packed = nvfp4_pack8(v[j], o);
    const uint32_t sfw = code | (dpp_u32<DPP_ROW_SHL(2)>(code) << 8) | (dpp_u32<DPP_ROW_SHL(4)>(code) << 16) |
                         (dpp_u32<DPP_ROW_SHL(6)>(code) << 24);
    if (r < rows) *reinterpret_cast<uint32_t *>(out + (bh * N + blk * 128 + r) * (a.Dp / 2) + c * 4) = packed;
    if ((c & 7) == 0 && r < rows_sf)
      reinterpret_cast<uint32_t *>(sf)[(bh * (a.Dp / 64) + (c >> 3)) * Np + blk * 128 + r] = sfw;
  }
}

__global__ __launch_bounds__(256) void attn_nvfp4_quantize_kernel(AttnNvfp4Args a) {
  __shared__ float lut[128];
  __shared__ uint32_t red[4];
  uint32_t idx = blockIdx.x;
  const uint32_t BH = a.B * a.H, nv = BH * a.nvt, nk = BH * a.nkt;
  const int t = idx < nv ? 2 : idx < nv + nk ? 1 : 0;
  idx -= t == 2 ? 0 : t == 1 ? nv : nv + nk;
  uint32_t m = (int)threadIdx.x < a.nparts[t] ? a.parts[t * AQ_MAX_PARTS + threadIdx.x] : 0u;
  m = group_umax<64>(m);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  load_rcp_table(lut);  // (ends with a barrier)
  m = umax32(umax32(red[0], red[1]), umax32(red[2], red[3]));
  const float gs = bf16_bits_to_f32(m) / a.max_scale, alpha = 1.0f / gs;
  if (idx == 0 && threadIdx.x == 0) a.gs[t] = gs;
  const AttnOperand &op = t == 2 ? a.v : t == 1 ? a.k : a.q;
  const uint32_t nblk = t == 2 ? a.nvt : t == 1 ? a.nkt : a.nqt;
  int b, head, blk;
  aq_tile(op, a.H, nblk, idx, b, head, blk);
  if (t == 2) {
    const int lane = threadIdx.x & 63, cc = blk * 4 + (threadIdx.x >> 6), group0 = (lane >> 2) * 8;
    if (cc * 64 >= a.Nkv64 || group0 >= a.Dvp) return;
    const int64_t bh = (int64_t)b * a.H + head;
    nvfp4_crossmajor_lane<true>(a.v4 + bh * a.Dv * (a.Nkv64 / 2), reinterpret_cast<uint32_t *>(a.v_sf) + (bh * (a.Nkv64 / 64) + cc) * a.Dvp,
                                op.p + b * op.s_b + head * op.s_h, op.s_n, a.Dv, a.Nkv, a.Nkv64, cc, group0, lane & 3, alpha, lut);
  } else if (t == 1) {
    aq_nvfp4_tile(a, op, a.Nkv, a.Nkvp, a.k4, a.k_sf, b, head, blk, alpha, lut);
  } else {
    aq_nvfp4_tile(a, op, a.Nq, a.Nqp, a.q4, a.q_sf, b, head, blk, alpha, lut);
  }
}

int64_t take(int64_t &at, int64_t bytes) {
  const int64_t p = at;
  at += align_up(bytes, 256);
  return p;
}

}  // namespace

// Token spans of the first kernel: enough workgroups to have the whole GPU loading, at least 32 tokens each, and at most
// 32 spans, because every tile of the second kernel reads one partial row per span.  `groups`: groups of heads that a
// workgroup takes, K and V together.
static int64_t aq_spans(int64_t groups, int64_t Nkv) {
  int64_t n = ceil_div(512, groups);
  if (n > AQ_MAX_SPLITS) n = AQ_MAX_SPLITS;
  return n < ceil_div(Nkv, AQ_MIN_SPAN) ? n : ceil_div(Nkv, AQ_MIN_SPAN);
}
static int aq_heads_per_wave(int D) { return D > 64 ? 4 : 8; }  // where the rows of neighbouring heads are adjacent
static bool aq_heads_adjacent(const AttnQuantArgs &a, const AttnOperand &t) { return t.s_h < t.s_n && a.H > 1; }

// workgroups of the statistics of one operand
static int64_t aq_stat_units(const AttnQuantArgs &a, const AttnOperand &t, int D) {
  return (int64_t)a.nsplit * a.B * ceil_div(a.H, aq_heads_adjacent(a, t) ? aq_heads_per_wave(D) : 1);
}
// LDS of a tile that takes the statistics itself: the sums of K, or the maxima of V of four waves
static int aq_own_bytes(const AttnQuantArgs &a, int classes) {
  const int sums = a.nsplit * classes * a.D * 4;
  return sums > 2048 ? sums : 2048;
}

// Whether the tiles of short heads take the statistics themselves (the operands have the same bits either way).  That takes a launch
// and its 4 us away and adds, in every tile of K, waits for eight loads a lane and the joining of the sums; heads of more than
// 512 keys would be read by too many tiles.  `rounds` is the score that the timings below were sorted by: the waits of one sum of a lane with eight
// tokens in flight.  That is what one class runs; several run two sums of four tokens, and wait two times where it says three, three where it says five.
// Sums of up to 24 KB in LDS stay in front of the line.  Whole calls of 777 queries, us, two launches -> one: BNHD 4 heads of 32 keys, D = 64, 13.7 -> 10.5, 2 x 12
// of 257 21.0 -> 19.1, 2 x 40 of 128, D = 128, 31.3 -> 28.3; BHND 12 heads of 512, D = 64, 22.4 -> 19.5, 2 x 40 of 77 25.9 -> 21.6.  Behind the line: BNHD
// 4 heads of 257, D = 128 (a score of five) 19.1 -> 19.0, of 400 20.5 -> 22.1; BHND 2 x 12 heads of 700, D = 64, 29.8 -> 31.9.
// Grids of many tiles pay for the registers of this kernel (112 against 91) in waves, heads of more than one tile for what the tiles read again:
// `pays`, in us, fitted to 611 calls of 16 to 512 keys, 1 to 4096 heads and 20 to 16000 queries (3 us rms), against 3.25 that the launch takes, less
// a margin of 1.5 for what the fit errs.  2048 heads of 264, D = 40, 239 -> 272, 768 of 318 109 -> 121, 512 of 338, D = 64, 73 -> 79, 512 of 34 with 5510
// queries each, D = 32, 342 -> 355: of the 611 36 were 1 to 14 % slower, none of the 537 that are in front of this line.  Few large tiles
// gain: 3072 of 128, D = 128, 186 -> 164.
static bool aq_own_faster(const AttnQuantArgs &a, int classes) {
  const int slots = 256 >> (a.D > 64 ? 4 : 3);  // sums that a tile takes at a time
  const int64_t rounds = ceil_div(a.nsplit * classes, slots) * ceil_div(ceil_div(a.span, classes), 8), heads = (int64_t)a.B * a.H;
  const double keys_mb = 1e-6 * (double)(heads * a.Nkv * (a.D > 64 ? 256 : 128));  // K as the lanes read it
  const double pays = (double)heads * (0.23e-3 * a.nqb + 1.9e-3 * a.nkb) + (0.25 * (a.nvb - 1) - 0.164) * keys_mb;
  return a.Nkv <= 512 && rounds <= (classes == 1 ? 6 : 3) && heads <= (a.D > 64 ? 4096 : 2048) && pays < 1.75;
}

void attn_quant_plan(AttnQuantArgs &a) {  // (after attn_quant_layout)
  const bool k_adjacent = aq_heads_adjacent(a, a.k);
  const int64_t groups = 2 * (int64_t)a.B * ceil_div(a.H, k_adjacent ? aq_heads_per_wave(a.D) : 1);
  a.span = (int)ceil_div(a.Nkv, aq_spans(groups, a.Nkv));
  a.nsplit = (int)ceil_div(a.Nkv, a.span);
  a.inv_nkv = 1.0f / (float)a.Nkv;
  // Sixteen waves a workgroup where a span lasts them for several rounds of loads: with about two workgroups per CU (more
  // would be more spans) the loads in flight are what the pass lives on, 116 us with 4 waves, 95 with 8, 83 with 16 for
  // K and V of 16384 x 40 x 128.  Short spans: eight (one round, 4.9 against 5.6 us at 257 x 12 x 64).
  // More workgroups than the GPU holds at once, neighbouring tokens in a wave: no more waves than one round of loads needs, so
  // that the sums of a wave meet fewer others and more workgroups are there (BHND, us with eight waves and now: 1024 x 8 windows
  // of 49 tokens, D = 32, 80 and 17; 256 x 12 of 64, D = 64, 32 and 11; 128 x 16 of 100, D = 128, 23 and 18).
  a.waves = a.span > 256 ? AQ_STAT_WAVES : 8;
  if (a.span <= 256 && aq_stat_units(a, a.k, a.D) + aq_stat_units(a, a.v, a.Dv) > 1024 && !k_adjacent && !aq_heads_adjacent(a, a.v)) {
    const int rows = AQ_STAT_LOADS * aq_heads_per_wave(a.D > a.Dv ? a.D : a.Dv);
    for (a.waves = 1; a.waves * rows < a.span; a.waves *= 2) {}
  }
  // classes of one token each are one sum in the order of the tokens
  int classes = a.waves * (k_adjacent ? 1 : aq_heads_per_wave(a.D));
  if (classes >= a.span) classes = 1;
  a.classes = aq_own_faster(a, classes) ? classes : 0;
}

int64_t attn_quant_layout(AttnQuantArgs &a, void *ws) {
  const int64_t BH = (int64_t)a.B * a.H;
  a.Dp = (int)align_up(a.D, 16), a.Dvp = (int)align_up(a.Dv, 16), a.Nkv16 = align_up(a.Nkv, 16);
  a.nqb = (int)ceil_div(a.Nq, AQ_Q_BLOCK), a.nkb = (int)ceil_div(a.Nkv, AQ_K_BLOCK), a.nvb = (int)ceil_div(a.Nkv, 256);
  uint8_t *w = static_cast<uint8_t *>(ws);
  int64_t at = 0;
  a.q8 = reinterpret_cast<int8_t *>(w + take(at, BH * a.Nq * a.Dp));
  a.k8 = reinterpret_cast<int8_t *>(w + take(at, BH * a.Nkv * a.Dp));
  a.v8 = w + take(at, BH * a.Dv * a.Nkv16);
  a.q_sf = reinterpret_cast<float *>(w + take(at, BH * a.nqb * 4));
  a.k_sf = reinterpret_cast<float *>(w + take(at, BH * a.nkb * 4));
  a.v_sf = reinterpret_cast<float *>(w + take(at, BH * a.Dvp * 4));
  // the plan has at most the spans of the fewest groups, so that the size does not depend on the strides: one where there
  // are many heads (4096 x 12 heads of 64 tokens, D = 64: 25 MB in all)
  const int64_t most = aq_spans(2 * (int64_t)a.B * ceil_div(a.H, aq_heads_per_wave(a.D)), a.Nkv);
  a.ksum = reinterpret_cast<float *>(w + take(at, most * BH * a.Dp * 4));
  a.vmax = reinterpret_cast<uint32_t *>(w + take(at, most * BH * a.Dvp * 4));
  return at;
}

void launch_attn_quant(const AttnQuantArgs &a, hipStream_t st) {
  const dim3 tiles((unsigned)((int64_t)a.B * a.H * (a.nvb + a.nkb + a.nqb)));
  if (a.classes > 0) {
    hipLaunchKernelGGL(attn_quantize_int8_fp8_kernel<true>, tiles, dim3(256), aq_own_bytes(a, a.classes), st, a);
    return;
  }
  const int64_t uk = aq_stat_units(a, a.k, a.D), uv = aq_stat_units(a, a.v, a.Dv);
  // (less LDS, more workgroups; the LDS sized by the launch instead cost the kernel of long spans 0.1 us)
  hipLaunchKernelGGL(a.waves <= 4 ? attn_column_stats_kernel<4> : attn_column_stats_kernel<AQ_STAT_WAVES>,
                     dim3((unsigned)(uk > uv ? uk : uv), 2), dim3(64 * a.waves), 0, st, a);
  hipLaunchKernelGGL(attn_quantize_int8_fp8_kernel<false>, tiles, dim3(256), 0, st, a);
}

int64_t attn_nvfp4_layout(AttnNvfp4Args &a, void *ws) {
  const int64_t BH = (int64_t)a.B * a.H;
  a.Dp = (int)align_up(a.D, 64), a.Dvp = (int)align_up(a.Dv, 16), a.Nqp = (int)align_up(a.Nq, 16), a.Nkvp = (int)align_up(a.Nkv, 16);
  a.Nkv64 = (int)align_up(a.Nkv, 64);
  a.nqt = (int)ceil_div(a.Nqp, 128), a.nkt = (int)ceil_div(a.Nkvp, 128), a.nvt = (int)ceil_div(a.Nkv64, 256);
  const int64_t n[3] = {BH * a.Nq * a.D, BH * a.Nkv * a.D, BH * a.Nkv * a.Dv};
  // a part of 32 KB and more: half of what a workgroup has in flight (512 lanes, eight loads), so that smaller tensors spread wider
  for (int t = 0; t < 3; ++t) {
    const int64_t parts = ceil_div(n[t], 512 * 8 * 4);
    a.nparts[t] = (int)(parts < 1 ? 1 : parts < AQ_MAX_PARTS ? parts : AQ_MAX_PARTS);
  }
  uint8_t *w = static_cast<uint8_t *>(ws);
  int64_t at = 0;
  a.q4 = w + take(at, BH * a.Nq * a.Dp / 2);
  a.k4 = w + take(at, BH * a.Nkv * a.Dp / 2);
  a.v4 = w + take(at, BH * a.Dv * (int64_t)a.Nkv64 / 2);
  a.q_sf = w + take(at, BH * a.Dp / 16 * a.Nqp);
  a.k_sf = w + take(at, BH * a.Dp / 16 * a.Nkvp);
  a.v_sf = w + take(at, BH * (a.Nkv64 / 16) * a.Dvp);
  a.gs = reinterpret_cast<float *>(w + take(at, 16));
  a.parts = reinterpret_cast<uint32_t *>(w + take(at, 3 * AQ_MAX_PARTS * 4));
  return at;
}

void launch_attn_nvfp4(const AttnNvfp4Args &a, hipStream_t st) {
  int most = a.nparts[0] > a.nparts[1] ? a.nparts[0] : a.nparts[1];
  if (a.nparts[2] > most) most = a.nparts[2];
  hipLaunchKernelGGL(attn_nvfp4_absmax_kernel, dim3(most, 3), dim3(512), 0, st, a);
  hipLaunchKernelGGL(attn_nvfp4_quantize_kernel, dim3((unsigned)((int64_t)a.B * a.H * (a.nvt + a.nkt + a.nqt))), dim3(256), 0, st, a);
}

}  // namespace ac4k
