// NVFP4 dot-scale linear for gfx950:  D = (A . B^T) * (gsA*gsB) + bias.
//
// Math contract of the reference kernel (lib/cuda/sm120/linear_nvfp4.cu:337-751, block-scaled
// MMA in lib/cuda/sm120/mma.cuh:13-56): every product e2m1*e2m1 is weighted by the two E4M3
// block scales of its 16-block, accumulated in fp32, then scaled by gsA*gsB, bias added,
// and rounded to the output type (:586-633).
//
// gfx950's scaled MFMA takes power-of-two scales per 32 elements, not E4M3 per 16, so the
// packed tiles are decoded on the fly: v_cvt_scalef32_pk_f16_fp4 expands two nibbles to two
// fp16 values and one v_pk_mul_f16 applies the E4M3 block scale.  e2m1 * e4m3 has at most
// 6 significant bits and lies in [2^-10, 2688], so the fp16 product is exact; the MFMA
// (v_mfma_f32_32x32x16_f16, same rate as bf16) accumulates in fp32.
#include <stdlib.h>
#include <string.h>

#include <atomic>
#include <mutex>
#include <type_traits>

#include "linear_common.h"

namespace ac4k {

struct LinearArgs {
  void *D;
  const uint8_t *A, *B;
  const uint32_t *A_sf, *B_sf;  // one dword per (64-chunk, row): sf_u32[chunk * rows_padded + row]
  const float *A_gs, *B_gs;
  const void *bias;
  int64_t M, N, K, Mp, Np;
  int prepacked = 0;  // B points at a weight image (W_BLOCK_BYTES blocks, see below) and B_sf is unused
};

// --- pre-packed weight image -----------------------------------------------------
// Static weights can be re-laid once into the order the kernels fetch them: one block per
// (128 rows, 128 k), blocks of a 128-row band consecutive along k, bands consecutive along n (N is
// padded with zero rows to a whole band).  A block is the LDS stage picture of those rows: 128 rows x
// 64 packed bytes with the 16-byte piece p of row r at position p ^ ((r >> 1) & 3), followed by the
// scale dwords [2 chunks][128 rows].  Every LDS-DMA transfer of a stage then reads one contiguous
// kilobyte, and a stage of the decode-sized kernel (256 k) is one contiguous run of two blocks.
constexpr int W_BLOCK_ROWS = 128, W_BLOCK_K = 128;
constexpr int W_BLOCK_DATA = W_BLOCK_ROWS * W_BLOCK_K / 2;            // 8192
constexpr int W_BLOCK_BYTES = W_BLOCK_DATA + 2 * W_BLOCK_ROWS * 4;    // 9216

// --- decode -------------------------------------------------------------------
// E4M3 scale byte -> fp16x2 pattern worth scale * 2^-8 in both halves (exponent bias 7 vs 15;
// E4M3 subnormals land on fp16 subnormals with the same ratio).  The scale bytes are read as
// the signed float8_e4m3fn their tensor type says, by every linear kernel (the quantizers only
// produce non-negative scales).
__device__ __forceinline__ f16x2 scale_pattern(uint32_t byte) {
  return __builtin_bit_cast(f16x2, (byte & 0x7fu) * 0x00800080u + (byte & 0x80u) * 0x01000100u);
}

// eight nibbles of `w` times the block scale -> eight fp16 (exact); the converter multiplies
// by 2^8 to undo the 2^-8 carried by the scale pattern.
__device__ __forceinline__ void decode8(uint32_t w, f16x2 sp, f16x2 (&h)[4]) {
  h[0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 0) * sp;
  h[1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 1) * sp;
  h[2] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 2) * sp;
  h[3] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 256.0f, 3) * sp;
}

// --- workgroup -> output tile ---------------------------------------------------
// Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  Workgroup `pid` is first
// renumbered so that every XCD owns one contiguous run of the tile sequence, and the sequence walks
// the tiles in bands of GROUP_M tile-rows, column by column inside a band: the workgroups resident
// on one XCD at a time then cover a compact GROUP_M x (CUs / GROUP_M) patch and share its operand
// panels through that L2.
// (32 bits: a grid has fewer than 2^32 workgroups.  The quotients of 64 bits that were here, and of the range below where there is only one, took every
// workgroup a third of a microsecond: 300 x 1024 x 256 5.23 -> 4.83 us, 2898 x 600 x 256 5.83 -> 5.46.)
struct TileCoord {
  uint32_t m, n;
};
template <int GROUP_M>
__device__ __forceinline__ TileCoord tile_of_workgroup(uint32_t pid, uint32_t tiles_m, uint32_t tiles_n) {
  const uint32_t ntiles = tiles_m * tiles_n;
  const uint32_t per = ntiles / 8, rem = ntiles % 8;
  const uint32_t xcd = pid % 8, idx = pid / 8;
  pid = xcd * per + (xcd < rem ? xcd : rem) + idx;
  const uint32_t band = pid / (GROUP_M * tiles_n), in_band = pid - band * (GROUP_M * tiles_n);
  const uint32_t first_m = band * GROUP_M;
  const uint32_t rows = (tiles_m - first_m) < GROUP_M ? (tiles_m - first_m) : GROUP_M;
  const uint32_t col = in_band / rows;
  return {first_m + in_band - col * rows, col};
}
// stages [first, first + count) of K range `range` of `ranges`; in scalar registers, said plainly: the compiler otherwise takes the
// quotients, and with them the loop and the addresses, to the lanes
struct StageRange {
  int first, count;
};
__device__ __forceinline__ StageRange stage_range(int stages, uint32_t range, int ranges) {
  if (ranges == 1) return {0, stages};
  const int first = __builtin_amdgcn_readfirstlane((int)((int64_t)stages * range / ranges));
  return {first, __builtin_amdgcn_readfirstlane((int)((int64_t)stages * (range + 1) / ranges)) - first};
}

// ===========================================================================
// 128x128x64 tile kernel, 4 waves (2x2), each wave 64x64 = 2x2 MFMA 32x32x16 tiles.
// LDS holds the decoded fp16 tiles: row pitch 128 B (64 k), 16-byte chunk index XORed with
// LDS_SWZ(row) so that both the decode stores and the MFMA fragment loads are conflict-free.
// ===========================================================================
constexpr int T_BM = 128, T_BN = 128, T_BK = 64;
#define LDS_SWZ(row) ((row) & 7)

struct PackedRegs {
  uint2 d[2];    // two 16-blocks (8 bytes each) of this thread's row
  uint32_t sf;   // scale bytes of the two blocks in bits 0..7 and 8..15
};

__device__ __forceinline__ PackedRegs load_packed(const uint8_t *base, const uint32_t *sf, int64_t rows,
                                                  int64_t rows_p, int64_t K, int64_t row, int64_t k0,
                                                  int half) {
  PackedRegs r;
  r.d[0] = r.d[1] = make_uint2(0, 0);
  r.sf = 0;
  if (row < rows_p) {
    uint32_t w = sf[(k0 >> 6) * rows_p + row] >> (16 * half);
    const uint8_t *p = base + row * (K >> 1) + (k0 >> 1) + half * 16;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      if (row < rows && k0 + half * 32 + b * 16 < K) {
        r.d[b] = *reinterpret_cast<const uint2 *>(p + b * 8);
        r.sf |= ((w >> (8 * b)) & 0xffu) << (8 * b);
      }
    }
  }
  return r;
}

__device__ __forceinline__ void decode_to_lds(_Float16 *tile, int row, int half, const PackedRegs &r) {
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    f16x2 sp = scale_pattern(r.sf >> (8 * b));
    f16x2 lo[4], hi[4];
    decode8(r.d[b].x, sp, lo);
    decode8(r.d[b].y, sp, hi);
    const int c0 = half * 4 + b * 2;  // logical 16-byte chunk of elements [c0*8, c0*8+8)
    uint4 v0 = make_uint4(__builtin_bit_cast(uint32_t, lo[0]), __builtin_bit_cast(uint32_t, lo[1]),
                          __builtin_bit_cast(uint32_t, lo[2]), __builtin_bit_cast(uint32_t, lo[3]));
    uint4 v1 = make_uint4(__builtin_bit_cast(uint32_t, hi[0]), __builtin_bit_cast(uint32_t, hi[1]),
                          __builtin_bit_cast(uint32_t, hi[2]), __builtin_bit_cast(uint32_t, hi[3]));
    *reinterpret_cast<uint4 *>(tile + row * 64 + ((c0 ^ LDS_SWZ(row)) << 3)) = v0;
    *reinterpret_cast<uint4 *>(tile + row * 64 + (((c0 + 1) ^ LDS_SWZ(row)) << 3)) = v1;
  }
}

__device__ __forceinline__ f16x8 lds_frag(const _Float16 *tile, int row, int chunk) {
  return *reinterpret_cast<const f16x8 *>(tile + row * 64 + ((chunk ^ LDS_SWZ(row)) << 3));
}

template <int D_DT, int BIAS_DT>
__global__ __launch_bounds__(256) void linear_nvfp4_tile128_kernel(LinearArgs a) {
  __shared__ __attribute__((aligned(16))) _Float16 sA[T_BM * T_BK];
  __shared__ __attribute__((aligned(16))) _Float16 sB[T_BN * T_BK];

  const TileCoord tc = tile_of_workgroup<8>(blockIdx.x, ceil_div(a.M, T_BM), ceil_div(a.N, T_BN));
  const int64_t tm = tc.m, tn = tc.n;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int ld_row = tid >> 1, ld_half = tid & 1;
  const int64_t arow = tm * T_BM + ld_row, brow = tn * T_BN + ld_row;

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  const int64_t nk = ceil_div(a.K, T_BK);
  PackedRegs ra = load_packed(a.A, a.A_sf, a.M, a.Mp, a.K, arow, 0, ld_half);
  PackedRegs rb = load_packed(a.B, a.B_sf, a.N, a.Np, a.K, brow, 0, ld_half);
  for (int64_t kt = 0; kt < nk; ++kt) {
    decode_to_lds(sA, ld_row, ld_half, ra);
    decode_to_lds(sB, ld_row, ld_half, rb);
    __syncthreads();
    if (kt + 1 < nk) {  // prefetch the next packed slices while the MFMAs run
      ra = load_packed(a.A, a.A_sf, a.M, a.Mp, a.K, arow, (kt + 1) * T_BK, ld_half);
      rb = load_packed(a.B, a.B_sf, a.N, a.Np, a.K, brow, (kt + 1) * T_BK, ld_half);
    }
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int chunk = ks * 2 + (lane >> 5);
      f16x8 fa[2], fb[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[i] = lds_frag(sA, wm * 64 + i * 32 + (lane & 31), chunk);
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[j] = lds_frag(sB, wn * 64 + j * 32 + (lane & 31), chunk);
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }

  // epilogue: * (gsA*gsB), + bias, round, store (linear_nvfp4.cu:586-633)
  const float scale = (*a.A_gs) * (*a.B_gs);
  using DE = Elem<D_DT>;
  typename DE::T *D = static_cast<typename DE::T *>(a.D);
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int64_t n = tn * T_BN + wn * 64 + j * 32 + (lane & 31);
    float bv = 0.0f;
    if constexpr (BIAS_DT != BIAS_NONE) {
      if (n < a.N) bv = Elem<BIAS_DT>::load(a.bias, n);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int64_t m = tm * T_BM + wm * 64 + i * 32 + (e >> 2) * 8 + (lane >> 5) * 4 + (e & 3);
        if (m < a.M && n < a.N) {
          float v = acc[i][j][e] * scale;
          if constexpr (BIAS_DT != BIAS_NONE) v += bv;
          D[m * a.N + n] = DE::cvt(v);
        }
      }
    }
  }
}

// ===========================================================================
// (64 MI) x (64 NJ) tile, packed operands in LDS, decode after the fragment load.
//
// The packed A/B slices and their scale dwords go from global memory straight into LDS with
// LDS-DMA loads (global_load_lds: no VGPR staging, no LDS store instruction), PS stages of
// 128 k each.  A wave (4 waves, 2x2, (32 MI) x (32 NJ) each) reads for every 32-row fragment ONE
// 16-byte word per lane per 64-chunk: lane (row r, half h) owns elements [32h, 32h+32) of the
// chunk; dword s of that word feeds MFMA sub-step s.  The same k-slot assignment is used for A
// and B, so the permutation of k inside a chunk cancels in the dot product.  Decode per dword:
// 4 x v_cvt_scalef32_pk_f16_fp4 + 4 x v_pk_mul_f16 by the block scale (E4M3 -> fp16 with
// v_cvt_scalef32_pk_f16_fp8, splat through op_sel); the decode of a sub-step is interleaved with
// the MFMAs of the previous one (TileWave below).
// KW == 1: the waves multiply a quarter of the tile each, over all of a stage, with one workgroup barrier per 128 k, placed in the
// middle of the step so that the next stage is readable before the current one ends.  KW == 2, for the tiles of up to 256 x 128: two waves
// multiply one half of the tile each over one 64-chunk of a stage and two over the other, and meet at the end through LDS: 4 decode
// instructions per MFMA instead of 6 for 256 x 128 and 128 x 256, 4.7 instead of 6.7 for 192 x 128, 6 instead of 8 for 128 x 128.
// Bound by instruction issue of a single wave per SIMD and, where the whole GPU is busy for long, by power.  Cycles per MFMA and wave, with
// KW == 1, the decoding pinned between the MFMAs and the scales fetched a dword per lane / now: 256 x 256 41.2 / 35.2, 256 x 128 51 / 39,
// 192 x 128 58 / 44, 128 x 128 70 / 51.  Back to back, us: 1024 x 4096 x 4096 38.3 / 32.8, 1001 x 5003 x 2880 35.7 / 33.6, 2048 x 4096 x 4096
// 58.2 / 53.8, 2048 x 14336 x 4096 183.8 / 175.5, 75600 x 5120 x 5120 2776 / 2673 (the clock comes down by half of what the loop gains).  256 x 128
// and 128 x 256 tiles run KW == 2 on long ranges only (PAIR_STAGES), for the exchange.
// Split-K: blockIdx.y selects a contiguous range of stages; with more than one range the
// accumulators go to an fp32 partial buffer and a second kernel adds the ranges.
// Requires K % 64 == 0, K >= 128 and 16-byte aligned operands.  EARLY: K % 128 == 64.  The stages start one
// chunk early, at k = -64, so that only stage 0 is special and the loop is not: the prologue fetches k-chunk 0
// into both halves of it and clears the scales of the first half.  (1001 x 5003 x 2880, fp32 out: 75 -> 45 us, the
// 128x128 kernel against this one; 300 x 4096 x 4160: 93 -> 28.)  A variant of its own: decided at run time, the longer
// prologue cost the 128 x 128 tiles of every other K 0.2 to 0.4 us (kernel alone, 160 x 2000 x 8192 in eight K ranges:
// 18.1 us, 17.3 without; 256 x 4096 x 4096 in four 20.7 and 19.8).
// ===========================================================================
constexpr int P_BK = 128;     // k per stage (two 64-chunks)
constexpr int P_ROW = 64;     // packed bytes per row per stage: [chunk][half] x 16 B

template <int BM, int BN, int PS>
struct PLayout {               // byte offsets inside one LDS stage; PS stages
  static constexpr int OFF_B = BM * P_ROW;                 // B rows follow the A rows
  static constexpr int OFF_SFA = OFF_B + BN * P_ROW;       // scale dwords: [chunk][BM rows]
  static constexpr int NSA = (BM + 127) / 128, NSB = (BN + 127) / 128;  // kilobytes, and transfers, of scales
  static constexpr int OFF_SFB = OFF_SFA + NSA * 1024;     // [chunk][BN rows]
  static constexpr int STAGE_BYTES = OFF_SFB + NSB * 1024;
  static_assert(NSA + NSB <= 4, "a scale transfer per wave");
  static constexpr int LDS_BYTES = PS * STAGE_BYTES;
  static_assert(LDS_BYTES <= 160 * 1024, "stages must fit in the CU's LDS");
};

// two of the eight values of a dword of nibbles, without their scale; q (0..3) is a constant after unrolling
__device__ __forceinline__ f16x2 decode_pair(uint32_t w, int q) {
  if (q == 0) return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0);
  if (q == 1) return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1);
  if (q == 2) return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2);
  return __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3);
}

// f(i) for the share of COUNT things that belongs behind the m-th of OF instructions (a loop of a known length, so that it unrolls
// before the one over m does)
template <int COUNT, int OF, typename F>
__device__ __forceinline__ void deal(int m, F &&f) {
#pragma unroll
  for (int x = 0; x < (COUNT + OF - 1) / OF; ++x) {
    const int i = COUNT * m / OF + x;
    if (i < COUNT * (m + 1) / OF) f(i);
  }
}

// What a wave of the tile kernels holds: packed fragments of a 64-chunk, 32 rows each, WI of A first, then WJ of B, in two sets (one
// multiplied while the other arrives), and the sums of WI x WJ blocks.  Lane (row r, half h) of a fragment has elements
// [32 h, 32 h + 32) of the chunk; dword s of them belongs to sub-step s, 16 k.
//
// The loop bodies are written out in the order in which they issue.  A wave is alone on its SIMD and issues an instruction of any kind
// every 5 cycles; an MFMA takes 8.6 of these and keeps the matrix core busy for 32.  Up to four or five instructions behind every
// MFMA are free, and what stands in a clump leaves the matrix core idle, so everything is dealt out evenly: the decoding,
// the LDS reads and the transfers.  (Left to the compiler, with only the decoding pinned between the MFMAs: 41.2 cycles an MFMA in
// 256 x 256 tiles, 36.4 so, 35.2 with the scales in 16-byte transfers.)
template <int WI, int WJ>
struct TileWave {
  static constexpr int NF = WI + WJ, NM = WI * WJ;
  uint4 packed[2][NF];
  uint32_t sf[2][NF];    // the scale bytes of the lane's two blocks
  f16x2 scale[2][NF];    // the same as fp16
  u32x4 decoded[2][NF];  // operands of a sub-step, double buffered
  f32x16 acc[WI][WJ];

  // item i of decoding sub-step s of set `set` into buffer d: two values of fragment i / 4.  wfac: power of two on the scales of B
  __device__ __forceinline__ void decode_item(int d, int set, int s, int i, float wfac = 1.0f) {
    const int f = i >> 2, q = i & 3;
    if (s == 0 && q == 0) scale[set][f] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(sf[set][f], f < WI ? 1.0f : wfac, false);
    const f16x2 sc = s < 2 ? (f16x2){scale[set][f].x, scale[set][f].x} : (f16x2){scale[set][f].y, scale[set][f].y};
    const uint4 &v = packed[set][f];
    decoded[d][f][q] = __builtin_bit_cast(uint32_t, decode_pair(s == 0 ? v.x : s == 1 ? v.y : s == 2 ? v.z : v.w, q) * sc);
  }
  // One sub-step: the MFMAs on buffer d, under them the decoding of sub-step s of set `set` into the other buffer, and extra(m) behind MFMA m
  template <typename F>
  __device__ __forceinline__ void substep(int d, int set, int s, F &&extra, float wfac = 1.0f) {
#pragma unroll
    for (int m = 0; m < NM; ++m) {
      // boustrophedon order: every MFMA shares one operand with the one before it (measured 0.6 %
      // faster than row by row on the power-limited 8192^3 problem: less operand switching)
      const int i = m / WJ, j = (i & 1) ? WJ - 1 - m % WJ : m % WJ;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, decoded[d][WI + j]), __builtin_bit_cast(f16x8, decoded[d][i]),
                                                         acc[i][j], 0, 0, 0);  // D^T block
      deal<4 * NF, NM>(m, [&](int e) { decode_item(1 - d, set, s, e, wfac); });
      extra(m);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < WI; ++i)
#pragma unroll
      for (int j = 0; j < WJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  }
};

// Build with -DAC4K_LINEAR_TIMELINE (`build.py --timeline`) to record per workgroup the 100 MHz clock at
// kernel entry, loop entry, loop exit and kernel exit plus the shader cycles spent in the loop of the
// tile kernel and of the K-split-waves kernel; ac4k_debug_linear_timeline copies the stamps out
// (a profiling aid; not compiled into the library).
#ifdef AC4K_LINEAR_TIMELINE
__device__ uint64_t g_linear_timeline[8192][6];
#define AC4K_LTL(i, v)                                                     \
  do {                                                                     \
    if (threadIdx.x == 0 && blockIdx.x + gridDim.x * blockIdx.y < 8192)      \
      g_linear_timeline[blockIdx.x + gridDim.x * blockIdx.y][i] = (v);        \
  } while (0)
#else
#define AC4K_LTL(i, v)
#endif

struct SplitK {
  float *partial;  // [splits][M][N] fp32, or null: convert and store to D
  int splits;
};

// the first `cols` elements of S bytes (at least one) of a 16-byte piece, to any element
template <int S>
__device__ __forceinline__ void store_piece(char *dst, const u32x4 &v, int cols) {
  if (cols >= 16 / S) {
    *reinterpret_cast<u32x4_elem *>(dst) = v;
    return;
  }
  const int dwords = cols * S / 4;  // whole ones
  if (dwords & 2) *reinterpret_cast<u32x2_elem *>(dst) = (u32x2){v.x, v.y};
  if (dwords & 1) *reinterpret_cast<u32_elem *>(dst + (dwords & 2) * 4) = dwords & 2 ? v.z : v.x;
  if constexpr (S == 2)
    if (cols & 1) *reinterpret_cast<uint16_t *>(dst + dwords * 4) = (uint16_t)(dwords & 2 ? dwords & 1 ? v.w : v.z : dwords & 1 ? v.y : v.x);
}

// Epilogue of the packed-LDS tile kernel: the accumulators of one wave, (32*MI) x (32*NJ) outputs, to
// `out` (row stride N).  acc[i][j] holds the TRANSPOSED 32x32 block (the MFMAs are issued with the
// operands swapped): lane l, element e <-> n = j*32 + (e>>2)*8 + (l>>5)*4 + (e&3), m = i*32 + (l&31),
// i.e. four consecutive n per lane.  RAW stores the fp32 sums as they are (split-K partials);
// otherwise out = cvt(acc * scale + bias).  Outputs are staged through LDS (`lds`, free at this
// point), one wave-private block of RP rows at a time, so that every lane stores 16 bytes and a
// wave store covers whole row segments; the bias of the tile's columns sits behind the staging
// blocks as fp32.  Callers have passed a workgroup barrier after their last read of `lds`.
template <int OUT_DT, int BIAS_DT, bool RAW, int MI, int NJ, int LDS_BYTES>
__device__ __forceinline__ void store_tile(const f32x16 (&acc)[MI][NJ], char *lds, void *out, const void *bias,
                                           float scale, int64_t M, int64_t N, int64_t m0, int64_t n0,
                                           int64_t tile_n0) {
  using DE = Elem<OUT_DT>;
  using DT = typename DE::T;
  DT *Dp = static_cast<DT *>(out);
  constexpr int S = sizeof(DT);
  constexpr int WN = 32 * NJ;               // columns per wave
  constexpr int RP = S == 2 && MI % 2 == 0 ? 64 : 32;  // rows per staging pass
  constexpr int PITCH = WN * S + 16;        // bytes per staged row, 16 bytes of padding
  constexpr int STG_BYTES = 4 * RP * PITCH;
  static_assert(STG_BYTES + 2 * WN * 4 <= LDS_BYTES, "epilogue staging and bias must fit in LDS");
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, half = lane >> 5, wn = wave & 1;
  const float *bias_s = reinterpret_cast<const float *>(lds + STG_BYTES) + wn * WN + half * 4;
  if constexpr (BIAS_DT != BIAS_NONE) {
    if (tid < 2 * WN) {
      const int64_t n = tile_n0 + tid;
      reinterpret_cast<float *>(lds + STG_BYTES)[tid] = n < N ? Elem<BIAS_DT>::load(bias, n) : 0.0f;
    }
    __syncthreads();
  }
  // the four outputs acc[i][j][4g .. 4g+3] of a lane, scaled, plus their bias b
  // The 256x256 tile keeps its 256 sums per lane in accumulation registers.  Left alone, the compiler
  // moves all of them to ordinary registers at the top of the epilogue and spills what does not fit;
  // reading them with a volatile move keeps each read inside the pass that stages the value.
  auto sum_of = [&](int i, int j, int e) {
    if constexpr (MI * NJ == 16) {
      float v;
      asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc[i][j][e]));
      return v;
    } else {
      return acc[i][j][e];
    }
  };
  auto value4 = [&](int i, int j, int g, const float4 &b) {
    float4 v = make_float4(sum_of(i, j, 4 * g), sum_of(i, j, 4 * g + 1), sum_of(i, j, 4 * g + 2), sum_of(i, j, 4 * g + 3));
    if constexpr (!RAW) {
      v.x *= scale; v.y *= scale; v.z *= scale; v.w *= scale;
    }
    if constexpr (BIAS_DT != BIAS_NONE) {
      v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
    }
    return v;
  };
  // bias of column block j: four 16-byte LDS reads in one go (one wait), kept for the rows of a pass
  auto bias_of = [&](int j, float4 (&b)[4]) {
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      b[g] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
      if constexpr (BIAS_DT != BIAS_NONE) b[g] = *reinterpret_cast<const float4 *>(bias_s + j * 32 + g * 8);
    }
  };
  // Rows that start on any element leave in 16-byte stores like aligned ones; the last, partial piece of a row in up to three
  // smaller ones (element by element before, in a loop: fp32 1001 x 5003 x 2880 46.4 -> 40.9 us, bf16 4000 x 5003 x 2880 144 -> 133,
  // N = 5008 129)
  char *stg = lds + wave * (RP * PITCH);
  constexpr int CPR = WN * S / 16;   // 16-byte pieces per staged row
  constexpr int RS = 64 / CPR;       // rows covered by one wave store
  const int lrow = lane / CPR, lq = lane % CPR;
  const int64_t row_bytes = N * S;
  const uint32_t lane_off = (uint32_t)(lrow * row_bytes) + lq * 16;
  char *out0 = reinterpret_cast<char *>(Dp) + (m0 * N + n0) * S;  // wave-uniform
  const bool interior = m0 + 32 * MI <= M && n0 + WN <= N;
  const bool whole = N % (16 / S) == 0 || n0 + WN <= N;  // no piece is cut: rows past M and pieces past N are left out
  const int64_t cl = N - n0 - lq * (16 / S);
  const int cols_left = cl > 16 / S ? 16 / S : (int)cl;  // columns of this lane's piece inside the matrix
  const int64_t rl = M - m0 - lrow;
  const int rows_left = rl > 32 * MI ? 32 * MI : (int)rl;  // rows of the block below this lane's first one
#pragma unroll
  for (int p = 0; p < 32 * MI / RP; ++p) {
    asm volatile("" ::: "memory");  // keeps the bias reads of one pass from being merged with the next one's
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      float4 b[4];
      bias_of(j, b);
#pragma unroll
      for (int ii = 0; ii < RP / 32; ++ii) {
        const int i = p * (RP / 32) + ii;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 v = value4(i, j, g, b[g]);
          char *dst = stg + (ii * 32 + (lane & 31)) * PITCH + (j * 32 + g * 8 + half * 4) * S;
          if constexpr (S == 2) *reinterpret_cast<uint2 *>(dst) = make_uint2(DE::cvt2(v.x, v.y), DE::cvt2(v.z, v.w));
          else *reinterpret_cast<float4 *>(dst) = v;
        }
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the staging block is private to the wave
    // pass `it` stores rows it*RS .. it*RS+RS-1 of the block: a wave-uniform base that advances by
    // RS rows, plus a fixed 32-bit lane offset; the bounds checks are per lane only on edge tiles
    const char *src = stg + lrow * PITCH + lq * 16;
    char *rowp = out0 + (int64_t)p * RP * row_bytes;
    if (interior) {
#pragma unroll
      for (int it = 0; it < RP / RS; ++it)
        *reinterpret_cast<u32x4_elem *>(rowp + it * RS * row_bytes + lane_off) = *reinterpret_cast<const u32x4 *>(src + it * RS * PITCH);
    } else if (whole) {
#pragma unroll
      for (int it = 0; it < RP / RS; ++it) {
        const u32x4 v = *reinterpret_cast<const u32x4 *>(src + it * RS * PITCH);
        if (cols_left > 0 && p * RP + it * RS < rows_left) *reinterpret_cast<u32x4_elem *>(rowp + it * RS * row_bytes + lane_off) = v;
      }
    } else {
      // (unrolled by four for the small tiles: with all of it 128 x 128 tiles ran 2 % longer, also where no piece is cut - 256 x 4096 x 4096
      // 34.7 -> 33.7 us, 34.3 before there were pieces -; the larger ones lose 0.5 % by it)
      constexpr int CUT = MI * NJ <= 4 ? 4 : RP / RS;
#pragma unroll CUT
      for (int it = 0; it < RP / RS; ++it) {
        const u32x4 v = *reinterpret_cast<const u32x4 *>(src + it * RS * PITCH);
        if (cols_left > 0 && p * RP + it * RS < rows_left) store_piece<S>(rowp + it * RS * row_bytes + lane_off, v, cols_left);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  }
}

// MI = 32-row fragments that a wave stores along M: 4 (BM = 256), 3 (BM = 192) or 2 (BM = 128);
// NJ = 32-column fragments that a wave stores along N: 4 (BN = 256), 2 (BN = 128) or 1 (BN = 64);
// KW = waves that share the K of a stage; with two of them a wave multiplies twice as many fragments along one side (WI x WJ);
// PS = LDS stages: PS - 1 k-steps (KW == 2: PS) are in flight ahead of the one being multiplied, which a small
// tile needs because its k-step is much shorter than the memory latency.
template <int D_DT, int BIAS_DT, int MI, int NJ, int PS, int KW, bool EARLY>
__global__ __launch_bounds__(256, 1) void linear_nvfp4_tile256p_kernel(LinearArgs a, SplitK sk) {
  extern __shared__ __attribute__((aligned(16))) char plds[];
  AC4K_LTL(0, wall_clock64());
  constexpr int BM = 64 * MI, BN = 64 * NJ;  // two waves along M, two along N
  using PL = PLayout<BM, BN, PS>;
  constexpr int NDA = BM / 4 / 16;         // 16-row A transfers per wave per stage
  constexpr int NDB = BN / 4 / 16;         // 16-row B transfers per wave per stage
  constexpr int NPIECES = NDA + NDB + 1;   // and one of scales

  const TileCoord tc = tile_of_workgroup<4>(blockIdx.x, (uint32_t)ceil_div(a.M, BM), (uint32_t)ceil_div(a.N, BN));
  const int64_t tm = (uint32_t)__builtin_amdgcn_readfirstlane((int)tc.m), tn = (uint32_t)__builtin_amdgcn_readfirstlane((int)tc.n);

  // KW == 2: the pair of waves (WI > MI: 0 and 2, 1 and 3; WJ > NJ: 0 and 1, 2 and 3) multiplies the blocks of both
  constexpr bool PAIR_M = KW == 2 && MI < NJ, PAIR_N = KW == 2 && !PAIR_M;
  constexpr int WI = PAIR_M ? 2 * MI : MI, WJ = PAIR_N ? 2 * NJ : NJ;  // fragments that a wave multiplies
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = PAIR_M ? 0 : wave >> 1, wn = PAIR_N ? 0 : wave & 1;
  const int half = lane >> 5;
  // this workgroup's range of 128-k stages; `early`: bytes by which they start in front of the row
  const int nkt_all = (int)(EARLY ? ceil_div(a.K, P_BK) : a.K / P_BK);
  constexpr int early = EARLY ? 32 : 0;
  const StageRange range = stage_range(nkt_all, blockIdx.y, sk.splits);
  const int kt0 = range.first, nkt = range.count;

  // LDS-DMA.  One transfer moves 16 rows x 64 B: the four lanes 4r .. 4r+3 read the four 16-byte
  // pieces of row r (one 64-byte sector) and land at LDS base + 16*l, i.e. row-major 64-byte rows.
  // Piece p of row r sits at position p ^ ((r >> 1) & 3) of its row: a fragment read takes one piece
  // of each of 32 rows, and unswizzled those addresses fall on a quarter of the LDS banks (an
  // eight-way conflict on every ds_read_b128).  The 32-bit lane offset is loop invariant and the
  // 64-bit part is a scalar base that advances by 64 bytes per stage.
  const int dma_piece = (lane & 3) ^ ((lane >> 3) & 3);  // tile rows of a transfer start at a multiple of 16
  const int swave = __builtin_amdgcn_readfirstlane(wave);
  const int64_t kb = a.K >> 1;
  uint32_t offA[NDA], offB[NDB];
#pragma unroll
  for (int q = 0; q < NDA; ++q) {
    int64_t ra = (swave * NDA + q) * 16 + (lane >> 2);
    ra = tm * BM + ra < a.M ? ra : a.M - 1 - tm * BM;  // rows past the matrix read the last valid row
    offA[q] = (uint32_t)(ra * kb + dma_piece * 16);
  }
  // weight image: a transfer's 16 rows are one contiguous kilobyte of a block (the swizzle is part of
  // the image); bands past the last one read the last band, whose outputs are never stored
  const int64_t w_band_bytes = (int64_t)nkt_all * W_BLOCK_BYTES, w_last_band = (a.N - 1) / W_BLOCK_ROWS;
  auto w_band_of = [&](int64_t row, int64_t &within) {
    int64_t band = row / W_BLOCK_ROWS;
    within = row % W_BLOCK_ROWS;
    return band < w_last_band ? band : w_last_band;
  };
#pragma unroll
  for (int q = 0; q < NDB; ++q) {
    if (a.prepacked) {
      int64_t within;
      const int64_t band = w_band_of(tn * BN + (swave * NDB + q) * 16, within);
      offB[q] = (uint32_t)(band * w_band_bytes + within * P_ROW + lane * 16);
    } else {
      int64_t rb = (swave * NDB + q) * 16 + (lane >> 2);
      rb = tn * BN + rb < a.N ? rb : a.N - 1 - tn * BN;
      offB[q] = (uint32_t)(rb * kb + dma_piece * 16);
    }
  }
  const int64_t strideB = a.prepacked ? W_BLOCK_BYTES : P_ROW;  // bytes per stage along k
  const uint8_t *baseA = uniform_ptr(a.A + tm * BM * kb + (int64_t)kt0 * P_ROW - early);
  const uint8_t *baseB = uniform_ptr(a.prepacked ? a.B + (int64_t)kt0 * W_BLOCK_BYTES : a.B + tn * BN * kb + (int64_t)kt0 * P_ROW - early);
  // scales: a transfer is 256 dwords of the [chunk][row] picture of an operand, a lane four rows of a chunk (16 bytes; the address is on
  // four).  Waves 0 .. NSA - 1 move those of A, the others those of B; a wave past the last transfer repeats the last one, and so do
  // lanes past the picture's end with rows of its last chunk, into the rest of the kilobyte.  (A dword per lane, up to four transfers a wave, cost
  // the loop of 192 x 128 tiles 377 of its 2420 cycles a stage.)
  uint32_t offS, ldsS;
  const uint8_t *baseS;
  int64_t strideS;
  bool firstS;  // this lane's rows belong to the first chunk of a stage
  {
    const int t = swave < PL::NSA + PL::NSB ? swave : PL::NSA + PL::NSB - 1;
    const bool isB = t >= PL::NSA;
    const int tt = isB ? t - PL::NSA : t, rows_t = isB ? BN : BM;
    const int at = tt * 256 + lane * 4, c = at >= rows_t ? 1 : 0;
    const int loc = at < 2 * rows_t ? at - c * rows_t : 0;
    const int64_t rows = isB ? a.Np : a.Mp, first = isB ? tn * BN : tm * BM;
    firstS = c == 0;
    if (isB && a.prepacked) {  // the scale dwords follow the packed rows of the block
      int64_t within;
      const int64_t band = w_band_of(first + loc, within);
      offS = (uint32_t)(band * w_band_bytes + W_BLOCK_DATA + c * (W_BLOCK_ROWS * 4) + within * 4);
      strideS = W_BLOCK_BYTES;
      baseS = uniform_ptr(a.B + (int64_t)kt0 * W_BLOCK_BYTES);
    } else {
      const int64_t row = first + loc + 4 <= rows ? loc : rows - 4 - first;  // (rows are padded to 16)
      offS = (uint32_t)((c * rows + row) * 4);
      strideS = 2 * rows * 4;  // two planes (chunks) per stage
      baseS = uniform_ptr(reinterpret_cast<const uint8_t *>(isB ? a.B_sf : a.A_sf) + (first - (EARLY ? rows : 0)) * 4 + kt0 * strideS);
    }
    strideS = (int64_t)uniform_ptr((const void *)strideS);
    ldsS = (uint32_t)__builtin_amdgcn_readfirstlane((isB ? PL::OFF_SFB : PL::OFF_SFA) + tt * 1024);
  }
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)plds;
  // LDS destinations of this wave's transfers inside a stage (wave-uniform, loop invariant)
  uint32_t ldsA[NDA], ldsB[NDB];
#pragma unroll
  for (int q = 0; q < NDA; ++q) ldsA[q] = (uint32_t)__builtin_amdgcn_readfirstlane((swave * NDA + q) * 1024);
#pragma unroll
  for (int q = 0; q < NDB; ++q) ldsB[q] = (uint32_t)__builtin_amdgcn_readfirstlane(PL::OFF_B + (swave * NDB + q) * 1024);
  // Source pointers of the k-step being fetched.  They advance by one step per iteration and stop
  // at the last step of the range: fetches past the end re-read the last slice into a stage buffer
  // nobody reads again, which keeps the main loop free of branches.
  struct Src {
    const uint8_t *a, *b, *s;
  };
  auto src_at = [&](int kt) {
    Src p;
    p.a = baseA + (int64_t)kt * P_ROW;
    p.b = baseB + (int64_t)kt * strideB;
    p.s = baseS + kt * strideS;
    return p;
  };
  auto issue_piece = [&](uint32_t stage_lds, const Src &p, int q) {
    if (q < NDA) {
      dma16(p.a, offA[q], stage_lds, ldsA[q]);
    } else if (q < NDA + NDB) {
      dma16(p.b, offB[q - NDA], stage_lds, ldsB[q - NDA]);
    } else {
      dma16(p.s, offS, stage_lds, ldsS);
    }
  };
  auto issue_stage = [&](uint32_t stage_lds, const Src &p) {
#pragma unroll
    for (int q = 0; q < NPIECES; ++q) issue_piece(stage_lds, p, q);
  };
  TileWave<WI, WJ> w;
  w.clear();

  // fragment addresses inside a stage (bytes)
  // (a lane's rows differ by multiples of 32, so the swizzle term of its row is (lane >> 1) & 3 for all of them)
  const int fa_off = (wm * (32 * MI) + (lane & 31)) * P_ROW;
  const int fb_off = PL::OFF_B + (wn * (32 * NJ) + (lane & 31)) * P_ROW;
  const int piece_off[2] = {((0 + half) ^ ((lane >> 1) & 3)) * 16, ((2 + half) ^ ((lane >> 1) & 3)) * 16};  // chunk 0, chunk 1
  // KW == 2: the chunk of every stage that this wave multiplies; its first MI x NJ fragments are the ones that it will keep, behind
  // them those of the other wave of the pair, so that no register is chosen at run time
  const int kw = PAIR_M ? swave >> 1 : swave & 1;
  auto row_a = [&](int i) { return 32 * (PAIR_M ? (i < MI ? kw * MI : (1 - kw) * MI) + i % MI : i); };
  auto row_b = [&](int j) { return 32 * (PAIR_N ? (j < NJ ? kw * NJ : (1 - kw) * NJ) + j % NJ : j); };
  // a lane needs the two scale bytes of its half of the chunk: blocks 2*half, 2*half+1
  const int sa_off = PL::OFF_SFA + (wm * (32 * MI) + (lane & 31)) * 4 + half * 2;
  const int sb_off = PL::OFF_SFB + (wn * (32 * NJ) + (lane & 31)) * 4 + half * 2;

  // read r of a chunk into set `set` (by chunk parity, KW == 2 by stage parity): the packed fragments, then the scale bytes
  constexpr int NF = WI + WJ, NM = WI * WJ;
  auto load_item = [&](uint32_t stage_off, int c, int set, int r) {
    const char *st = plds + stage_off;
    const int f = r % NF;
    if (r < NF) {
      const int piece = KW == 2 ? (kw ? piece_off[1] : piece_off[0]) : piece_off[c];
      w.packed[set][f] = *reinterpret_cast<const uint4 *>(st + piece + (f < WI ? fa_off + row_a(f) * P_ROW : fb_off + row_b(f - WI) * P_ROW));
    } else {
      w.sf[set][f] = *reinterpret_cast<const uint16_t *>(st + (f < WI ? sa_off + c * (BM * 4) + row_a(f) * 4 : sb_off + c * (BN * 4) + row_b(f - WI) * 4));
    }
  };

  // prologue: stages 0 .. PS-2 (KW == 2: PS-1) in flight (past the last k-step: the last one again), stage 0
  // visible, the wave's first fragments and first decode
  constexpr int AHEAD = KW == 2 ? PS : PS - 1;
  static_assert(PS >= 3 && (AHEAD - 1) * NPIECES <= 63, "the wait counts below must fit the 6-bit counter");
  const int last = nkt - 1;
  // the stage that fetches past the end repeat: never the short one, whose first half lies in front of the rows
  // (a range of one stage then repeats the stage behind it, which exists: K >= 192)
  const bool short0 = EARLY && kt0 == 0;
  const int again = short0 && last == 0 ? 1 : last;
  {  // stage 0; a short one takes k-chunk 0 into both halves, by its addresses
    Src p = src_at(0);
    const uint32_t shift = short0 && dma_piece < 2 ? 32u : 0u;
#pragma unroll
    for (int q = 0; q < NDA; ++q) dma16(p.a, offA[q] + shift, lds_base, ldsA[q]);
#pragma unroll
    for (int q = 0; q < NDB; ++q) dma16(p.b, offB[q] + shift, lds_base, ldsB[q]);
    dma16(p.s, offS + (short0 && firstS ? (uint32_t)(strideS / 2) : 0), lds_base, ldsS);
  }
  // A range shorter than the ring is fetched as it is and waited for as a whole: its repeats would be most of a short prologue
  // (10650 x 512 x 384 11.4 -> 10.9 us).
  const bool brief = nkt < AHEAD;
#pragma unroll
  for (int d = 1; d < AHEAD; ++d)
    if (!brief || d < nkt) issue_stage(lds_base + d * PL::STAGE_BYTES, src_at(d < last ? d : again));
  if (brief) wait_vmcnt<0>();
  else wait_vmcnt<(AHEAD - 1) * NPIECES>();  // everything of stage 0 has landed, later stages may be in flight
  __syncthreads();
#pragma unroll
  for (int r = 0; r < 2 * NF; ++r) load_item(0, KW == 2 ? kw : 0, 0, r);
  if (short0 && (KW == 1 || kw == 0)) {
#pragma unroll
    for (int f = 0; f < NF; ++f) w.sf[0][f] = 0;
  }
#pragma unroll
  for (int e = 0; e < 4 * NF; ++e) w.decode_item(0, 0, 0, e);
  if constexpr (KW == 2) {  // stage 1 landed, and everybody's fragments of stage 0 in registers
    wait_vmcnt<(AHEAD - 2) * NPIECES>();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __syncthreads();
  }

  // loop-carried, wave-uniform: LDS offsets of the stages holding k-steps kt, kt+1 and of the one
  // being filled with kt+AHEAD (a ring of PS), and the source pointers of k-step min(kt+AHEAD, last)
  uint32_t st_cur = 0, st_nxt = PL::STAGE_BYTES, st_dma = (PS - 1) * PL::STAGE_BYTES;
  auto ring_next = [](uint32_t o) { return o + PL::STAGE_BYTES == (uint32_t)PL::LDS_BYTES ? 0u : o + PL::STAGE_BYTES; };
  Src src = src_at(last < AHEAD ? again : AHEAD);
  auto advance = [&](int kt) {  // the sources, unless they already sit on the last k-step
    const bool adv = kt + AHEAD < last;
    src.a += adv ? P_ROW : 0;
    src.b += adv ? strideB : 0;
    src.s += adv ? strideS : 0;
  };
#ifdef AC4K_LINEAR_TIMELINE
  const uint64_t tl_c0 = __builtin_readcyclecounter();
#endif
  AC4K_LTL(1, wall_clock64());
  // KW == 2: a step multiplies chunk kw of stage kt out of registers (set kt & 1) while that of stage kt+1, which landed before
  // the last barrier, travels to the other set, and stage kt+PS to the ring slot of stage kt
  auto pair_step = [&](int kt, int cur) {
    const uint32_t dma_lds = lds_base + st_cur;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      w.substep(s & 1, s < 3 ? cur : 1 - cur, (s + 1) & 3, [&](int m) {
        if (s < 3) deal<2 * NF, 3 * NM>(s * NM + m, [&](int r) { load_item(st_nxt, kw, 1 - cur, r); });  // past the end this reads a stale stage; the result is never used
        deal<NPIECES, 4 * NM>(s * NM + m, [&](int q) { issue_piece(dma_lds, src, q); });
      });
    wait_vmcnt<(PS - 2) * NPIECES>();                   // own transfers of stage kt+2 have landed
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and the fragments of stage kt+1 are in registers
    __syncthreads();
    st_cur = st_nxt;
    st_nxt = ring_next(st_nxt);
    advance(kt);
  };
  if constexpr (KW == 2) {  // (nkt >= 1: splits <= stages)
    int kt = 0;
    do {
      pair_step(kt, 0);
      if (kt + 1 < nkt) pair_step(kt + 1, 1);
      kt += 2;
    } while (kt < nkt);
  }
  for (int kt = 0; KW == 1 && kt < nkt; ++kt) {
    // chunk 0: sub-steps 0..3 (fragments of chunk 1 are fetched meanwhile)
#pragma unroll
    for (int s = 0; s < 4; ++s)
      w.substep(s & 1, s < 3 ? 0 : 1, (s + 1) & 3, [&](int m) {
        if (s < 3) deal<2 * NF, 3 * NM>(s * NM + m, [&](int r) { load_item(st_cur, 1, 1, r); });
      });
    // stage kt+1 must be complete (own DMA done, then everybody's; stages kt+2 .. kt+PS-2 may still
    // be in flight); stage kt-1 is free after this
    wait_vmcnt<(PS - 3) * NPIECES>();
    __syncthreads();
    // chunk 1: sub-steps 4..7 (chunk 0 of the next stage is fetched meanwhile); the DMA of stage
    // kt+PS-1 is spread over these sub-steps
    const uint32_t dma_lds = lds_base + st_dma;
#pragma unroll
    for (int s = 0; s < 4; ++s)
      w.substep(s & 1, s < 3 ? 1 : 0, (s + 1) & 3, [&](int m) {
        if (s < 3) deal<2 * NF, 3 * NM>(s * NM + m, [&](int r) { load_item(st_nxt, 0, 0, r); });  // past the end this reads a stale stage; the result is never used
        deal<NPIECES, 4 * NM>(s * NM + m, [&](int q) { issue_piece(dma_lds, src, q); });
      });
    st_cur = st_nxt;
    st_nxt = ring_next(st_nxt);
    st_dma = ring_next(st_dma);
    advance(kt);
  }
  AC4K_LTL(2, wall_clock64());
#ifdef AC4K_LINEAR_TIMELINE
  AC4K_LTL(4, __builtin_readcyclecounter() - tl_c0);
  {
    uint32_t xcc, hwid;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hwid));
    AC4K_LTL(5, (xcc & 0xf) | (hwid << 8));
  }
#endif

  // ---- epilogue.  The MFMAs were issued with the operands swapped, so acc[i][j] holds the
  // TRANSPOSED 32x32 block: lane l, element e <-> n = j*32 + (e>>2)*8 + (l>>5)*4 + (e&3),
  // m = i*32 + (l&31): four consecutive n per lane.
  const int64_t m0 = tm * BM + (swave >> 1) * (32 * MI), n0 = tn * BN + (swave & 1) * (32 * NJ);
  // the last iterations' LDS-DMA fetches (into a stage nobody reads) must have landed before the
  // stages are reused, and every wave must be done reading them
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  auto store = [&](const f32x16 (&sums)[MI][NJ]) {
    if (sk.partial) {  // split-K: raw fp32 sums of this K range; the reduce kernel scales and converts
      store_tile<AC4K_DTYPE_FP32, BIAS_NONE, true, MI, NJ, PL::LDS_BYTES>(
          sums, plds, sk.partial + (int64_t)blockIdx.y * a.M * a.N, nullptr, 1.0f, a.M, a.N, m0, n0, tn * BN);
    } else {
      store_tile<D_DT, BIAS_DT, false, MI, NJ, PL::LDS_BYTES>(sums, plds, a.D, a.bias, (*a.A_gs) * (*a.B_gs), a.M, a.N,
                                                             m0, n0, tn * BN);
    }
  };
  const auto &acc = w.acc;
  if constexpr (KW == 1) {
    store(acc);
  } else {
    // the waves of a pair exchange halves of their blocks and add them: wave (wm, wn) of the 2 x 2 grid keeps its own
    static_assert(4 * MI * NJ * 4096 <= PL::LDS_BYTES, "the exchanged halves must fit in LDS");
    float4 *xch = reinterpret_cast<float4 *>(plds) + lane;
    auto xch_at = [&](int w, int i, int j, int g) { return xch + ((w * MI * NJ + i * NJ + j) * 4 + g) * 64; };
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x16 &o = acc[PAIR_M ? MI + i : i][PAIR_N ? NJ + j : j];
          *xch_at(swave ^ (PAIR_M ? 2 : 1), i, j, g) = make_float4(o[4 * g], o[4 * g + 1], o[4 * g + 2], o[4 * g + 3]);
        }
    __syncthreads();
    f32x16 sums[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const float4 t = *xch_at(swave, i, j, g);
          sums[i][j][4 * g] = acc[i][j][4 * g] + t.x;
          sums[i][j][4 * g + 1] = acc[i][j][4 * g + 1] + t.y;
          sums[i][j][4 * g + 2] = acc[i][j][4 * g + 2] + t.z;
          sums[i][j][4 * g + 3] = acc[i][j][4 * g + 3] + t.w;
        }
    __syncthreads();  // what follows lies over the halves
    store(sums);
  }
  AC4K_LTL(3, wall_clock64());
}

// Raises a kernel's dynamic LDS limit once per (kernel instantiation, device): the attribute belongs
// to the device the call is made on.
template <typename Kernel>
static int allow_dynamic_lds(Kernel *kern, std::atomic<uint32_t> &done_mask, int bytes) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  const uint32_t bit = 1u << (dev & 31);
  if (done_mask.load(std::memory_order_relaxed) & bit) return 0;
  hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return set_error("hipFuncSetAttribute(LDS=%d): %s", bytes, hipGetErrorString(e));
  done_mask.fetch_or(bit, std::memory_order_relaxed);
  return 0;
}

// LDS stages per tile shape: enough k-steps in flight to cover the memory latency
constexpr int tile_stages(int mi, int nj, int kw) { return mi * nj >= 16 ? 3 : mi * nj > 8 ? 4 : mi * nj == 8 ? 3 + kw : mi * nj >= 4 ? 6 : 8; }

template <int D_DT, int BIAS_DT, int MI, int NJ, int KW>
static int launch_tile_kw(const LinearArgs &a, const SplitK &sk, hipStream_t st) {
  constexpr int PS = tile_stages(MI, NJ, KW);
  const bool early = a.K % P_BK != 0;
  auto *kern = early ? linear_nvfp4_tile256p_kernel<D_DT, BIAS_DT, MI, NJ, PS, KW, true> : linear_nvfp4_tile256p_kernel<D_DT, BIAS_DT, MI, NJ, PS, KW, false>;
  using PL = PLayout<64 * MI, 64 * NJ, PS>;
  static std::atomic<uint32_t> lds_ok[2];
  if (int rc = allow_dynamic_lds(kern, lds_ok[early], PL::LDS_BYTES)) return rc;
  const int64_t ntiles = ceil_div(a.M, 64 * MI) * ceil_div(a.N, 64 * NJ);
  hipLaunchKernelGGL(kern, dim3((unsigned)ntiles, (unsigned)sk.splits), dim3(256), PL::LDS_BYTES, st, a, sk);
  return 0;
}

// 256 x 128 and 128 x 256 tiles multiply in pairs of waves from this length of a range on: the exchange of halves costs them 1.4 us a round, a
// stage 0.08 less in pairs.  us, back to back, every wave by itself / pairs (and the loops before, which had no pairs): 8155 x 2056 x 256
// 24.9 / 28.5 (27.3), x 512 31.7 / 36.7 (34.8), x 1024 47.4 / 50.0 (50.9), x 1792 74.3 / 74.4 (78.6), x 2304 88.9 / 87.7 (94.4); 473 x 11008 x 256
// 9.3 / 10.4 (10.2), x 1792 23.6 / 23.9 (25.6), x 2304 28.6 / 28.2 (30.8).  The smaller tiles exchange half as much, and in
// pairs they are faster than their loops before at any length.
constexpr int PAIR_STAGES = 15;
template <int D_DT, int BIAS_DT, int MI, int NJ>
static int launch_tile_p(const LinearArgs &a, const SplitK &sk, hipStream_t st) {
  if constexpr (MI * NJ == 8)
    if (ceil_div(ceil_div(a.K, P_BK), sk.splits) < PAIR_STAGES) return launch_tile_kw<D_DT, BIAS_DT, MI, NJ, 1>(a, sk, st);
  return launch_tile_kw<D_DT, BIAS_DT, MI, NJ, MI * NJ <= 8 ? 2 : 1>(a, sk, st);
}

// Tile shape and K split of the packed-LDS kernel for one problem.
struct TilePlan {
  int mi, nj;              // tile = (64 mi) x (64 nj)
  int splits;              // K ranges per tile; > 1 needs `partial_bytes` of fp32 scratch
  int64_t partial_bytes;
};

// Tuning overrides (ac4k_set_linear_tuning): a forced tile plan packed as mi | nj << 8 | splits << 16
// (0 = the cost model decides) and a forced K slice of the decode-sized kernel (0 = automatic).
static std::atomic<uint32_t> g_forced_tile_plan{0};
static std::atomic<int> g_forced_skinny_ks{0};
static bool forced_tile_plan(int64_t M, int64_t N, int64_t K, TilePlan &p) {
  const uint32_t f = g_forced_tile_plan.load(std::memory_order_relaxed);
  const int64_t sp = f >> 16;
  p = TilePlan{(int)(f & 0xff), (int)((f >> 8) & 0xff), (int)sp, sp > 1 ? sp * M * N * 4 : 0};
  return f != 0 && sp <= ceil_div(K, P_BK);
}

// What both estimates below use for every number of K ranges that they weigh: `most` of them, each two stages long at least (beyond
// 32 the sums cost more than any of the measured shapes gained).
struct SplitCosts {
  double len[33], sums_us[33];  // stages of a range; the partial sums written and read and the second launch
  int most;
};
static SplitCosts split_costs(int64_t M, int64_t N, int stages, double bytes_per_us, double launch_us, int most) {
  SplitCosts c;
  c.most = stages / 2 < most ? stages / 2 : most;
  if (c.most < 1) c.most = 1;
  c.len[1] = stages, c.sums_us[1] = 0.0;
  const double sum_us = (double)M * (double)N * 8.0 / bytes_per_us;
  for (int sp = 2; sp <= c.most; ++sp) c.len[sp] = (double)((stages + sp - 1) / sp), c.sums_us[sp] = sp * sum_us + launch_us;
  return c;
}

// Scratch that the entry points ask for, for the tile kernel's partial sums; 0: they take none (and ac4k_linear_nvfp4_skinny not
// the shape).  Callers keep these sizes, so they stay what this estimate has always given, although the plan comes from the
// measured costs below and fits into them.
static int64_t tile_scratch_bytes(int64_t M, int64_t N, int64_t K) {
  TilePlan forced;
  if (forced_tile_plan(M, N, K, forced)) return forced.partial_bytes;
  const int stages = (int)ceil_div(K, P_BK);
  if (ceil_div(M, M <= 128 ? 128 : 256) * ceil_div(N, 256) >= 192) return 0;
  const SplitCosts c = split_costs(M, N, stages, 4.5e6, 2.5, 32);
  double best_t = 0.0;
  int64_t best = 0;
  for (int mi = 2; mi <= 4; mi += 2) {
    if (mi == 4 && M <= 128) continue;
    for (int nj = 4; nj >= 1; nj >>= 1) {
      if (mi == 4 && nj == 1) continue;
      if (nj < 4 && N < 64 * nj * 2) continue;
      const int nm = mi * nj, nv = 8 * (mi + nj);
      const double stage_us = (8.0 * (14.0 * nm + 5.0 * nv) + 400.0) / 2100.0;
      const double fixed_us = 5.0 + 0.1 * nm;
      const int tiles = (int)(ceil_div(M, 64 * mi) * ceil_div(N, 64 * nj));
      const double least = fixed_us + 0.999 * tiles * stages / 256.0 * stage_us;  // without the partial sums
      for (int sp = 1; sp <= c.most; ++sp) {
        if (best && least + c.sums_us[sp] >= best_t) break;  // nor will more ranges be faster
        const double t = (double)((tiles * sp + 255) / 256) * c.len[sp] * stage_us + fixed_us + c.sums_us[sp];
        if (best == 0 || t < best_t) best_t = t, best = sp;
      }
    }
  }
  return best > 1 ? best * M * N * 4 : 0;
}

// Picks the tile and the K split by measured costs in microseconds on 256 CUs, with at most `scratch` bytes of partial sums:
// rounds of 256 workgroups, stages per range times the time of a 128-k stage of that tile, a prologue and epilogue per round
// and for more than one range the partial sums and the second launch.  A stage takes `stage` as long as up to three fifths of the
// CUs have work and grows with their share from there to stage + 0.4 power, as the clock comes down.  A round beyond the first takes `round`.
// Fitted to 1000 random shapes of
// M = 129 to 12000, N = 256 to 28672, K = 256 to 14336 with every tile and up to 32 ranges that fit the scratch and to 200 of K up to 2048 and M up
// to 75600, and checked on 431 and 130 more: on average 0.3 and 0.1 % slower than the fastest of these plans, 24 of the 431 by 2 to 10 % (few tiles in many
// ranges).  (The costs of the loops before, with what pairs of waves now multiply together decoded by each of them: 0.8 %, 60 by 2 to
// 12 %; one time of a round for all tiles took 256 x 128, whose rounds ended with the exchange of halves, on many rows of short K: 56744 x 384 x 384
// 33.1 us, 256 x 256 30.2.)  The fit had the exchange in the short ranges of 256 x 128 and 128 x 256, too, which run without it: its time is taken out of the
// rounds beyond the first (74018 x 320 x 384 43.5 -> 36.7, 300 shapes of more than one round 0.2 % less time on average, 10 of them 1 to 2.5 % more and 32
// 1 to 7 % less; out of the first round, too, they were chosen where the small tiles are faster than their estimate: 171 x 8409 x 192 7.0 -> 8.8).
// It had no K of one stage; a round of 256 x 256 takes longer there: 71074 x 256 x 128 20.8 -> 17.0 us, and 260 shapes of K = 128 to 256 and more than
// one round 2.3 % less time on average, one of them 2 % more.  The sweeps held up to four rounds of workgroups and 32 ranges, and so does the plan.
// The tiles of 192 rows are what fills a round where 128 or 256 rows leave CUs idle (us, best of the other tiles / with
// them, loops before these): 4096 x 5120 x 5120 197.5 / 180.9, 7000 x 5120 x 5120 328.4 / 284.6, 6000 x 4096 x 4096 171.5 / 157.6, 300 x 14336 x 4096 50.9 / 45.3.
struct TileCost {
  int mi, nj;
  double stage, power, fixed, round;
};
constexpr TileCost TILE_COSTS[] = {{4, 4, 2.209, 2.092, 8.603, 4.001}, {3, 4, 1.652, 1.604, 8.664, 5.286}, {4, 2, 1.328, 0.823, 7.567, 5.041},
                                   {2, 4, 1.254, 0.952, 7.927, 4.367}, {3, 2, 1.062, 0.522, 7.758, 5.014}, {2, 2, 0.781, 0.281, 7.945, 4.549},
                                   {2, 1, 0.519, 0.139, 5.454, 4.77}};
static TilePlan tile_plan(int64_t M, int64_t N, int64_t K, int64_t scratch) {
  TilePlan best{};
  if (forced_tile_plan(M, N, K, best) && best.partial_bytes <= scratch) return best;
  constexpr double SPLIT_US = 3.41, PARTIAL_BYTES_PER_US = 7.8e6;  // (8 bytes of a sum: written and read)
  const int stages = (int)ceil_div(K, P_BK);
  const int64_t sums_bytes = M * N * 4;
  const SplitCosts s = split_costs(M, N, stages, PARTIAL_BYTES_PER_US, SPLIT_US, scratch / sums_bytes < 32 ? (int)(scratch / sums_bytes) : 32);
  double best_t = 0.0;
  best.splits = 0;
  for (const TileCost &c : TILE_COSTS) {
    if (c.mi > 2 && M <= 128) continue;
    if (c.nj < 4 && N < 64 * c.nj * 2) continue;
    const int64_t tiles = ceil_div(M, 64 * c.mi) * ceil_div(N, 64 * c.nj);
    const double least = c.fixed + 0.999 * (double)tiles * stages / 256.0 * c.stage;  // without the partial sums
    for (int sp = 1; sp <= s.most && (sp == 1 || tiles * sp <= 1024); ++sp) {
      if (best.splits && least + s.sums_us[sp] >= best_t) break;  // nor will more ranges be faster
      const double len = s.len[sp];
      const int64_t full = tiles * sp / 256, tail = tiles * sp % 256;
      double round = c.round;
      if (c.mi * c.nj == 8 && len < PAIR_STAGES) round -= 1.4 - 0.08 * len;  // no exchange
      if (c.mi * c.nj == 16 && len < 2.0) round += 1.5;                      // one stage is over before the stores of the round in front
      double t = c.fixed - round + (double)full * (len * (c.stage + 0.4 * c.power) + round) + s.sums_us[sp];
      if (tail) t += len * (c.stage + (tail > 153 ? ((double)tail / 256.0 - 0.6) * c.power : 0.0)) + round;
      if (best.splits == 0 || t < best_t) {
        best_t = t;
        best = TilePlan{c.mi, c.nj, sp, sp > 1 ? sp * sums_bytes : 0};
      }
    }
  }
  return best;
}

template <int D_DT, int BIAS_DT>
static int launch_tile_plan(const LinearArgs &a, const TilePlan &p, const SplitK &sk, hipStream_t st) {
  if (p.mi == 4) return p.nj == 4 ? launch_tile_p<D_DT, BIAS_DT, 4, 4>(a, sk, st) : launch_tile_p<D_DT, BIAS_DT, 4, 2>(a, sk, st);
  if (p.mi == 3) return p.nj == 4 ? launch_tile_p<D_DT, BIAS_DT, 3, 4>(a, sk, st) : launch_tile_p<D_DT, BIAS_DT, 3, 2>(a, sk, st);
  if (p.nj == 4) return launch_tile_p<D_DT, BIAS_DT, 2, 4>(a, sk, st);
  return p.nj == 2 ? launch_tile_p<D_DT, BIAS_DT, 2, 2>(a, sk, st) : launch_tile_p<D_DT, BIAS_DT, 2, 1>(a, sk, st);
}

// the packed-LDS kernel with the tile that suits the shape; no split-K (one K range, output to D)
template <int D_DT, int BIAS_DT>
static int launch_tile256p(const LinearArgs &a, hipStream_t st) {
  const SplitK one{nullptr, 1};
  return launch_tile_plan<D_DT, BIAS_DT>(a, tile_plan(a.M, a.N, a.K, 0), one, st);
}

// ===========================================================================
// Mid-sized M (33 .. 128): every weight byte is used by at most four 32-row activation fragments, so
// the problem is bound by streaming the weights and by decode instructions, not by the MFMA rate, and
// there are too few 256-wide tiles to fill the GPU.  Tile (32 MI) x (32 NJ) with ALL of M in one tile
// (MI = 4, NJ = 2: 128 x 64) and the four waves of the workgroup splitting K, not the tile: a stage is
// 256 k = four 64-chunks, wave w multiplies the whole tile over chunk w.  Every packed fragment of the
// stage is then decoded exactly once per workgroup (the 2 x 2 wave grid of the tile kernel decodes each
// one twice): (MI + NJ) * 8 decode instructions per MI * NJ MFMAs, 6 per MFMA for 128 x 64, with one
// wave per SIMD.  Packed rows and scale dwords of a stage travel by LDS-DMA into a ring (128-byte rows,
// 16-byte pieces at position piece ^ (row & 7), scales as [chunk][row] dwords); one workgroup barrier
// per stage.  The four k parts of the tile meet through LDS at the end: wave w receives the sums of a
// quarter of the tile from the other three, adds them in wave order, and stores its quarter
// (times gsA * gsB, plus bias), or the raw fp32 sums of this K range when K is split over workgroups.
// Requires K % 64 == 0, K >= 256 and 16-byte aligned operands and scale tensors.  The last stage of any other K
// starts early enough to be whole, and the chunks of it that the stage before holds too count as zero.
// (100 x 5003 x 2880: 66 -> 20 us, the 128x128 kernel against this one.)
// ===========================================================================
// Kernels with stages of four chunks.  TAIL: K is no multiple of 256 (a variant of its own: the few scalar instructions
// a stage that it needs cost the other K 2 % in the K-split-waves kernel and 5 % in the LDS-ring kernels).  Of `nch` >= 4
// chunks the last stage takes the last four; chunk c of it counts for nothing when the stage before holds it too:
// `weight_factor` multiplies the weight scales, by 1 or by so little that the fp16 scale rounds to zero (the scale
// conversion takes a power of two at no cost).  `offset` is where a stage starts, from the row's first chunk (TAIL) or
// from the first one of the workgroup's range.
template <bool TAIL>
struct StageWalk {
  int s0, nch;  // first stage of the range, chunks in the row
  // what a source advances by, given its bytes per chunk: a chunk (TAIL) or a whole stage
  template <typename T>
  static __device__ __forceinline__ constexpr T step(T per_chunk) { return TAIL ? per_chunk : 4 * per_chunk; }
  __device__ __forceinline__ int chunk(int st) const { return 4 * (s0 + st) < nch - 4 ? 4 * (s0 + st) : nch - 4; }
  template <typename T>
  __device__ __forceinline__ int64_t offset(int st, T step) const { return (TAIL ? chunk(st) : st) * (int64_t)step; }
  template <typename T>
  __device__ __forceinline__ int64_t start(T step) const { return TAIL ? 0 : s0 * (int64_t)step; }
  __device__ __forceinline__ float weight_factor(int st, int c) const {
    if constexpr (TAIL) return 4 * (s0 + st) - chunk(st) > c ? 0x1p-60f : 1.0f;
    else return 1.0f;
  }
};

constexpr int KW_BK = 256;          // k per stage
constexpr int KW_ROW = KW_BK / 2;   // packed bytes per row per stage

template <int MI, int NJ>
struct KWLayout {
  static constexpr int BM = 32 * MI, BN = 32 * NJ;
  static_assert(BM % 64 == 0 && BN % 64 == 0, "a scale transfer covers 64-row blocks");
  static constexpr int OFF_W = 0;                         // BN weight rows, then BM activation rows
  static constexpr int OFF_A = BN * KW_ROW;
  static constexpr int OFF_SFW = OFF_A + BM * KW_ROW;     // scale dwords [4 chunks][BN rows]
  static constexpr int OFF_SFA = OFF_SFW + 4 * BN * 4;    // [4 chunks][BM rows]
  static constexpr int STAGE_BYTES = OFF_SFA + 4 * BM * 4;
  static constexpr int PS = (160 * 1024) / STAGE_BYTES < 8 ? (160 * 1024) / STAGE_BYTES : 8;  // ring slots
  static constexpr int LDS_BYTES = PS * STAGE_BYTES;
  static constexpr int NRW = BN / 8 / 4, NRA = BM / 8 / 4, NROW = NRW + NRA;  // 8-row transfers per wave per stage
  static constexpr int NSCW = BN / 64, NSCA = BM / 64;    // scale transfers per stage (1 KB each)
  static constexpr int NPIECES = NROW + 1;                // every wave issues the same count
  static constexpr int PPW = MI * NJ / 4;                 // 32 x 32 output blocks a wave finishes
  static_assert((BM + BN) % 32 == 0 && NSCW + NSCA <= 4 && MI * NJ % 4 == 0, "transfers are dealt evenly to four waves");
  static_assert(PS >= 3 && (PS - 2) * NPIECES <= 63, "the wait counts must fit the 6-bit counter");
  static_assert(LDS_BYTES >= 16 * PPW * 4096, "the ring doubles as the exchange buffer of the four k parts");
};

template <int D_DT, int BIAS_DT, int MI, int NJ, bool TAIL>
__global__ __launch_bounds__(256, 1) void linear_nvfp4_ksplit_kernel(LinearArgs a, SplitK sk) {
  using L = KWLayout<MI, NJ>;
  constexpr int BM = L::BM, BN = L::BN, PS = L::PS, NP = L::NPIECES;
  extern __shared__ __attribute__((aligned(16))) char kwlds[];
  AC4K_LTL(0, wall_clock64());
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, r32 = lane & 31;
  const int swave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t tiles_n = (uint32_t)ceil_div(a.N, BN), row_of_tiles = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x / tiles_n));
  const int64_t m0 = (int64_t)row_of_tiles * BM, n0 = (int64_t)(blockIdx.x - row_of_tiles * tiles_n) * BN;
  const int nst_all = (int)ceil_div(a.K, KW_BK);
  const StageRange range = stage_range(nst_all, blockIdx.y, sk.splits);
  const int s0 = range.first, nst = range.count;  // >= 1: splits <= stages
  const StageWalk<TAIL> walk{s0, (int)(a.K >> 6)};
  const int64_t kb = a.K >> 1;
  // workgroup b starts at stage b % nst of its range and wraps around, so that the workgroups of a
  // launch do not all ask for the same column of their rows at the same time (memory channels)
  const int rot = (int)(blockIdx.x % (unsigned)nst);
  const int last = nst - 1;
  auto stage_of = [&](int step) {
    const int p = (step < last ? step : last) + rot;
    return p >= nst ? p - nst : p;
  };

  // --- this wave's transfers of a stage
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)kwlds;
  // rows: a transfer moves eight rows of the stage, lane l the piece of row l / 8 that belongs at position l % 8; every wave as many of
  // the weights (the first NRW) as of the activation
  // On a weight image (a.prepacked) a stage is two blocks of the row's 128-row band, 64 bytes of the row in
  // each, pieces at p ^ ((row >> 1) & 3), and the four chunk planes of scale dwords sit behind the blocks' data.
  const int64_t img_band_bytes = (a.K / W_BLOCK_K) * (int64_t)W_BLOCK_BYTES;
  uint32_t offR[L::NROW], ldsR[L::NROW];
#pragma unroll
  for (int q = 0; q < L::NROW; ++q) {
    const bool isW = q < L::NRW;
    const int t = isW ? swave * L::NRW + q : swave * L::NRA + q - L::NRW;
    const int loc = t * 8 + (lane >> 3);
    const int pp = (lane & 7) ^ (loc & 7);  // the piece of the stage row that belongs at this lane's position
    if (isW && a.prepacked) {
      const int64_t wrow = n0 + loc;  // rows past N exist in the image (zeros)
      const int64_t band = wrow / W_BLOCK_ROWS, within = wrow % W_BLOCK_ROWS;
      offR[q] = (uint32_t)(band * img_band_bytes + (pp >> 2) * W_BLOCK_BYTES + within * 64 + (((pp & 3) ^ ((within >> 1) & 3)) * 16));
    } else {
      const int64_t rows = isW ? a.N : a.M, first = isW ? n0 : m0;
      const int64_t row = first + loc < rows ? loc : rows - 1 - first;  // rows past the matrix read its last row
      offR[q] = (uint32_t)(row * kb + pp * 16);
    }
    ldsR[q] = (uint32_t)__builtin_amdgcn_readfirstlane((isW ? L::OFF_W : L::OFF_A) + t * 1024);
  }
  // bytes per step of the walk along k
  const int strideW = __builtin_amdgcn_readfirstlane(walk.step(a.prepacked ? W_BLOCK_BYTES / 2 : KW_ROW / 4)), strideA = walk.step(KW_ROW / 4);
  const uint8_t *srcW = uniform_ptr((a.prepacked ? a.B : a.B + n0 * kb) + walk.start(strideW));
  const uint8_t *srcA = uniform_ptr(a.A + m0 * kb + walk.start(strideA));
  // scales: one transfer is 256 dwords of the [chunk][row] picture, a lane the four dwords of rows
  // 4 g .. 4 g + 3 of one chunk (16 bytes of the scale tensor).  Transfers 0 .. NSCW - 1 are the weights',
  // the others the activation's; a wave past the last transfer repeats the last one.
  uint32_t offS, ldsS;
  const uint8_t *srcS;
  int64_t strideS;
  {
    const int t = swave < L::NSCW + L::NSCA ? swave : L::NSCW + L::NSCA - 1;
    const bool isW = t < L::NSCW;
    const int tt = isW ? t : t - L::NSCW;
    const int bx = isW ? BN : BM;                         // rows of the operand's tile
    const int cpt = 256 / bx;                             // chunks per transfer (4 or 2)
    const int chunk = tt * cpt + lane / (bx / 4), grp = lane % (bx / 4);
    const int64_t rows_p = isW ? a.Np : a.Mp, first = isW ? n0 : m0;
    int64_t row = first + 4 * grp;
    if (isW && a.prepacked) {
      const int64_t band = row / W_BLOCK_ROWS, within = row % W_BLOCK_ROWS;
      offS = (uint32_t)(band * img_band_bytes + (chunk >> 1) * W_BLOCK_BYTES + W_BLOCK_DATA + (chunk & 1) * (W_BLOCK_ROWS * 4) + within * 4);
      strideS = walk.step(W_BLOCK_BYTES / 2);
      srcS = uniform_ptr(a.B + walk.start(strideS));
    } else {
      row = row + 4 <= rows_p ? row : rows_p - 4;         // groups past the padded rows read the last group
      offS = (uint32_t)((chunk * rows_p + row) * 4);
      strideS = walk.step(rows_p * 4);                    // chunk planes
      srcS = uniform_ptr(reinterpret_cast<const uint8_t *>(isW ? a.B_sf : a.A_sf) + walk.start(strideS));
    }
    ldsS = (uint32_t)__builtin_amdgcn_readfirstlane((isW ? L::OFF_SFW : L::OFF_SFA) + tt * 1024);
  }
  // Transfer q of this wave's NPIECES for stage `st` into the ring slot at `base`.  Past the end of the range
  // the loop keeps issuing, so that it stays free of branches and its wait counts stay fixed: those transfers
  // read the last stage again (cache hits) into slots nobody reads any more.
  // (`st` counts from the start of the range; a weight image has K % 128 == 0, so its stages start at whole blocks)
  struct Src {
    const uint8_t *w, *a, *s;
  };
  auto src_at = [&](int st) { return Src{srcW + walk.offset(st, strideW), srcA + walk.offset(st, strideA), srcS + walk.offset(st, strideS)}; };
  auto issue_piece = [&](uint32_t base, const Src &p, int q) {
    if (q < L::NROW) dma16(q < L::NRW ? p.w : p.a, offR[q], base, ldsR[q]);
    else dma16(p.s, offS, base, ldsS);
  };

  // --- this wave's fragments of a stage: chunk swave; lane (r32, half) holds elements [32 half, 32 half + 32)
  // of the chunk of one row per fragment (16 packed bytes) and the two block scales that go with them
  TileWave<MI, NJ> w;
  w.clear();
  const int piece = swave * 2 + half;
  const int f_off = r32 * KW_ROW + ((piece ^ (r32 & 7)) * 16);  // rows 32 apart share the swizzle term
  const int ws_off = L::OFF_SFW + (swave * BN + r32) * 4 + half * 2;
  const int xs_off = L::OFF_SFA + (swave * BM + r32) * 4 + half * 2;
  constexpr int NF = MI + NJ, NM = MI * NJ;
  auto load_item = [&](uint32_t stage_off, int set, int r) {  // as in the tile kernel
    const char *st = kwlds + stage_off;
    const int f = r % NF;
    if (r < NF) w.packed[set][f] = *reinterpret_cast<const uint4 *>(st + (f < MI ? L::OFF_A + f * 32 * KW_ROW : L::OFF_W + (f - MI) * 32 * KW_ROW) + f_off);
    else w.sf[set][f] = *reinterpret_cast<const uint16_t *>(st + (f < MI ? xs_off + f * 128 : ws_off + (f - MI) * 128));
  };

  // prologue: the first PS stages in flight, stage 0 landed and its fragments in registers (every wave's,
  // before slot 0 is refilled), then stage 1 landed
#pragma unroll
  for (int d = 0; d < PS; ++d) {
    const Src p = src_at(stage_of(d));
#pragma unroll
    for (int q = 0; q < NP; ++q) issue_piece(lds_base + d * L::STAGE_BYTES, p, q);
  }
  wait_vmcnt<(PS - 1) * NP>();
  __syncthreads();
  float wfac = walk.weight_factor(stage_of(0), swave);  // of the stage whose fragments were read last
#pragma unroll
  for (int r = 0; r < 2 * NF; ++r) load_item(0, 0, r);
#pragma unroll
  for (int e = 0; e < 4 * NF; ++e) w.decode_item(0, 0, 0, e, wfac);
  wait_vmcnt<(PS - 2) * NP>();
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __syncthreads();

  uint32_t st_cur = 0, st_nxt = L::STAGE_BYTES;  // LDS offsets of the stages at hand and next
#ifdef AC4K_LINEAR_TIMELINE
  const uint64_t tl_c0 = __builtin_readcyclecounter();
#endif
  AC4K_LTL(1, wall_clock64());
  // one stage: set `cur` holds its fragments, the other receives those of the next one
  auto stage_step = [&](int s, int cur) {
    // The slot of this stage is free (every wave had its fragments in registers before the previous
    // barrier): stage s + PS goes there.
    const uint32_t base_new = lds_base + st_cur;
    const Src src = src_at(stage_of(s + PS));
    wfac = walk.weight_factor(stage_of(s + 1), swave);
    // fragments of the next stage (it landed before the previous barrier) travel from LDS while this
    // one is decoded and multiplied (past the range: a stage nobody uses)
#pragma unroll
    for (int sub = 0; sub < 4; ++sub)
      w.substep(sub & 1, sub < 3 ? cur : 1 - cur, (sub + 1) & 3, [&](int m) {
        if (sub < 3) deal<2 * NF, 3 * NM>(sub * NM + m, [&](int r) { load_item(st_nxt, 1 - cur, r); });
        deal<NP, 4 * NM>(sub * NM + m, [&](int q) { issue_piece(base_new, src, q); });
      }, wfac);
    wait_vmcnt<(PS - 2) * NP>();                        // own transfers of stage s + 2 have landed
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and the fragments of stage s + 1 are in registers
    __syncthreads();
    st_cur = st_nxt;
    st_nxt = st_nxt + L::STAGE_BYTES == (uint32_t)L::LDS_BYTES ? 0 : st_nxt + L::STAGE_BYTES;
  };
  {
    int s = 0;
    do {  // (nst >= 1)
      stage_step(s, 0);
      if (s + 1 < nst) stage_step(s + 1, 1);
      s += 2;
    } while (s < nst);
  }
  AC4K_LTL(2, wall_clock64());
#ifdef AC4K_LINEAR_TIMELINE
  AC4K_LTL(4, __builtin_readcyclecounter() - tl_c0);
#endif
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS-DMA may land after this point: the ring is reused
  __syncthreads();

  // --- the four k parts meet: wave d finishes blocks p = d * PPW + q (i = p / NJ, j = p % NJ).
  // acc[i][j]: lane l, element e <-> m = 32 i + (l & 31), n = 32 j + (e >> 2) * 8 + (l >> 5) * 4 + (e & 3)
  constexpr int PPW = L::PPW;
  const auto &acc = w.acc;
  float4 *xch = reinterpret_cast<float4 *>(kwlds);
  auto xch_at = [&](int d, int src, int q, int g) { return xch + ((((d * 4 + src) * PPW + q) * 4 + g) * 64 + lane); };
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    if (d == swave) continue;
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
      const int p = d * PPW + q, i = p / NJ, j = p % NJ;
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *xch_at(d, swave, q, g) = make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
    }
  }
  __syncthreads();
  const float scale = sk.partial ? 1.0f : (*a.A_gs) * (*a.B_gs);
  using DE = Elem<D_DT>;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    if (d != swave) continue;
#pragma unroll
    for (int q = 0; q < PPW; ++q) {
      const int p = d * PPW + q, i = p / NJ, j = p % NJ;
      const int64_t m = m0 + 32 * i + r32;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
        for (int src = 0; src < 4; ++src) {  // always in wave order
          const float4 t = src == d ? make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3])
                                    : *xch_at(d, src, q, g);
          if (src == 0) sum = t;
          else { sum.x += t.x; sum.y += t.y; sum.z += t.z; sum.w += t.w; }
        }
        const int64_t n = n0 + 32 * j + g * 8 + half * 4;
        if (m >= a.M || n >= a.N) continue;
        if (sk.partial) {  // raw fp32 sums of this K range; the reduce kernel scales and converts
          float *pp = sk.partial + ((int64_t)blockIdx.y * a.M + m) * a.N + n;
          if (n + 3 < a.N) *reinterpret_cast<f32x4_elem *>(pp) = (f32x4){sum.x, sum.y, sum.z, sum.w};
          else {
            const float v[4] = {sum.x, sum.y, sum.z, sum.w};
#pragma unroll
            for (int c = 0; c < 4; ++c)
              if (n + c < a.N) pp[c] = v[c];
          }
          continue;
        }
        float v[4] = {sum.x * scale, sum.y * scale, sum.z * scale, sum.w * scale};
        if constexpr (BIAS_DT != BIAS_NONE) {
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] += n + c < a.N ? Elem<BIAS_DT>::load(a.bias, n + c) : 0.0f;
        }
        typename DE::T *dst = static_cast<typename DE::T *>(a.D) + m * a.N + n;
        if (n + 3 < a.N) {  // to any element: 128 x 5003 x 4096 bf16 23.1 -> 19.8 us, element by element before
          if constexpr (sizeof(typename DE::T) == 2)
            *reinterpret_cast<u32x2_elem *>(dst) = (u32x2){DE::cvt2(v[0], v[1]), DE::cvt2(v[2], v[3])};
          else
            *reinterpret_cast<f32x4_elem *>(dst) = (f32x4){v[0], v[1], v[2], v[3]};
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (n + c < a.N) dst[c] = DE::cvt(v[c]);
        }
      }
    }
  }
  AC4K_LTL(3, wall_clock64());
}

template <int D_DT, int BIAS_DT, int MI, int NJ>
static int launch_ksplit_t(const LinearArgs &a, const SplitK &sk, hipStream_t st) {
  using L = KWLayout<MI, NJ>;
  const bool tail = a.K % KW_BK != 0;
  auto *kern = tail ? linear_nvfp4_ksplit_kernel<D_DT, BIAS_DT, MI, NJ, true> : linear_nvfp4_ksplit_kernel<D_DT, BIAS_DT, MI, NJ, false>;
  static std::atomic<uint32_t> lds_ok[2];
  if (int rc = allow_dynamic_lds(kern, lds_ok[tail], L::LDS_BYTES)) return rc;
  const int64_t ntiles = ceil_div(a.M, L::BM) * ceil_div(a.N, L::BN);
  hipLaunchKernelGGL(kern, dim3((unsigned)ntiles, (unsigned)sk.splits), dim3(256), L::LDS_BYTES, st, a, sk);
  return 0;
}

// Tile and K split of the K-split-waves kernel.
struct KsplitPlan {
  int mi, nj;
  int splits;              // K ranges per tile; > 1 needs `partial_bytes` of fp32 scratch
  int64_t partial_bytes;
};

// shapes the K-split-waves kernel takes (its pointer conditions are in ksplit_aligned)
static bool ksplit_shape(int64_t M, int64_t N, int64_t K) {
  return M > 32 && M <= 128 && N >= 64 && K >= KW_BK && K % 64 == 0 && (K >> 1) * 128 < (1ll << 31) && N < (1ll << 27) &&
         g_forced_tile_plan.load(std::memory_order_relaxed) == 0;
}
static bool ksplit_aligned(const LinearArgs &a) {
  return (((uintptr_t)a.A | (uintptr_t)a.B | (uintptr_t)a.A_sf | (uintptr_t)a.B_sf) & 15) == 0;
}

// All of M in one tile: 128 x 64 above 64 rows, 64 x 64 below (64 x 128 when even those fill the GPU).
// Fewer than 192 tiles: as many K ranges as make about 256 workgroups, each at least two stages long.
static KsplitPlan ksplit_plan(int64_t M, int64_t N, int64_t K, bool allow_split) {
  KsplitPlan p{M <= 64 ? 2 : 4, 2, 1, 0};
  if (M <= 64 && ceil_div(N, 128) >= 192) p.nj = 4;
  const int64_t tiles = ceil_div(M, 32 * p.mi) * ceil_div(N, 32 * p.nj), stages = ceil_div(K, KW_BK);
  int64_t splits = 1;
  if (allow_split) {
    if (const int f = g_forced_skinny_ks.load(std::memory_order_relaxed)) {  // forced length of a K range
      splits = K / f;
    } else if (tiles < 192) {
      splits = 256 / tiles;
      if (splits > stages / 2) splits = stages / 2;
      if (splits > 32) splits = 32;
    }
    if (splits < 1) splits = 1;
    if (splits > stages) splits = stages;
  }
  p.splits = (int)splits;
  p.partial_bytes = splits > 1 ? splits * M * N * 4 : 0;
  return p;
}

template <int D_DT, int BIAS_DT>
static int launch_ksplit(const LinearArgs &a, const KsplitPlan &p, const SplitK &sk, hipStream_t st) {
  if (p.mi == 4) return launch_ksplit_t<D_DT, BIAS_DT, 4, 2>(a, sk, st);
  return p.nj == 4 ? launch_ksplit_t<D_DT, BIAS_DT, 2, 4>(a, sk, st) : launch_ksplit_t<D_DT, BIAS_DT, 2, 2>(a, sk, st);
}

// ===========================================================================
// Decode-sized linear (1 <= M <= 32): bound by streaming the weights once.  Two kernels; this one
// streams the weights into registers, linear_nvfp4_stream_kernel below through an LDS ring, and
// skinny_plan chooses between them by shape.
//
// A workgroup (4 waves) owns 128 weight rows and one K-slice; every wave one 32-row tile.  It
// first decodes its slice of the packed activation to fp16 (exact, without the global scale)
// into LDS, shared by the four waves (with more than 16 activation rows, 512 k at a time, so that
// the LDS footprint stays at 33 KB).  Lane (row r, half h) streams 64 contiguous bytes of its weight row per 256-k step
// (elements [128h, 128h+128) of the step) and decodes them dword by dword into MFMA operands; the
// MFMA is issued as D^T = W . Ahat^T so a lane ends up with 4 consecutive n for one m.  K-slices of one row
// group meet through fp32 partial tiles in a caller-provided workspace; a small second kernel
// adds them in slice order (deterministic), applies gsA*gsB and the bias, converts and stores.
// (A last-arriver reduction inside the kernel needs device-scope fences, which write back the
// XCD's L2 and cost far more than the second launch.)
// Requires K % 256 == 0 and 16-byte aligned weights.
// ===========================================================================
struct SkinnyArgs {
  void *D;
  const uint8_t *Aq;         // packed activation [M, K/2] and its scale bytes [K/64, Mp, 4]
  const uint8_t *A_sf;
  int64_t Mp;
  const uint8_t *B;
  const uint32_t *B_sf;
  const float *A_gs, *B_gs;
  const void *bias;
  float *partial;      // [splitK][M][N]
  int64_t M, N, K, Np;
  int ks_len, split_k;
  int prepacked = 0;  // B is a weight image (LDS-ring kernel, 16-row workgroups), B_sf unused
};

constexpr int SK_ROWS = 128;   // weight rows per workgroup
constexpr int SK_STEP = 256;   // k per step

// MAX_IT: 16-byte activation vectors a lane may have to fetch (M * 32 / 256 rounded up): 1 for M <= 8, 2 for
// M <= 16, 4 for M <= 32.  With one accumulator tile (the MFMAs of a lane then queue behind each other, which a
// kernel that waits for memory does not notice) the two smaller variants fit four workgroups on a CU.
template <int D_DT, int BIAS_DT, int MAX_IT>
__global__ __launch_bounds__(256, MAX_IT <= 2 ? 4 : 3) void linear_nvfp4_skinny_kernel(SkinnyArgs a) {
  extern __shared__ __attribute__((aligned(16))) char slds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, h = lane >> 5;
  // K-slice is the fast grid index: workgroups that run together then read neighbouring pieces of the
  // same rows (all HBM channels), not the same 512-byte column of different rows (a few channels)
  const int ksl = blockIdx.x;
  const int64_t ng = blockIdx.y, n0 = ng * SK_ROWS + wave * 32;
  const int64_t kbeg = (int64_t)ksl * a.ks_len;
  const int nsteps = a.ks_len / SK_STEP;  // 1..4
  // With more than 16 activation rows a 1024-k slice goes through LDS in two halves of 512 k, which
  // keeps the slice at 33 KB and three workgroups on a CU.
  const bool halves = a.M > 16 && nsteps == 4;
  const int lds_k = halves ? 512 : a.ks_len;  // k positions held in LDS at a time
  const int pitch = lds_k * 2 + 16;       // LDS row pitch in bytes (16 bytes of padding: no bank conflicts)

  // activation slice -> LDS as its exact fp16 dequantization (without the global scale).  A thread
  // takes 32 elements (16 packed bytes, two 16-blocks) at a time; every load of the slice is issued
  // before the first decode, so the slice costs one memory latency whatever M is.
  // (the activation loads go out before the weight stream: the memory counter is in order, so loads
  // issued behind the stream could only be waited for together with all of it)
  const int vec_per_row = a.ks_len / 32;
  const int total = (int)a.M * vec_per_row;
  uint4 aw[MAX_IT];
  uint32_t ac[MAX_IT];
#pragma unroll
  for (int it = 0; it < MAX_IT; ++it) {
    const int i = it * 256 + tid;
    if (i < total) {
      const int m = i / vec_per_row, v = i % vec_per_row;
      const int64_t k = kbeg + v * 32;
      aw[it] = *reinterpret_cast<const uint4 *>(a.Aq + (int64_t)m * (a.K >> 1) + (k >> 1));
      // scale bytes of blocks (k/16) % 4 and the next one: k % 32 == 0, so an aligned pair
      ac[it] = *reinterpret_cast<const uint16_t *>(a.A_sf + (((k >> 6) * a.Mp + m) << 2) + ((k >> 4) & 3));
    }
  }
  // weight stream of this lane: all steps of the slice are requested up front
  int64_t wrow = n0 + r;
  wrow = wrow < a.N ? wrow : a.N - 1;  // rows past N feed outputs that are never stored
  const uint8_t *wp = a.B + wrow * (a.K >> 1) + (kbeg >> 1) + h * 64;
  const uint32_t *sp = a.B_sf + ((kbeg >> 6) + 2 * h) * a.Np + wrow;
  uint4 W[4][4];
  uint32_t S[4][2];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t < nsteps) {
#pragma unroll
      for (int q = 0; q < 4; ++q) W[t][q] = *reinterpret_cast<const uint4 *>(wp + t * 128 + q * 16);  // cached: the four words share a line
      S[t][0] = sp[(int64_t)(t * 4) * a.Np];
      S[t][1] = sp[(int64_t)(t * 4 + 1) * a.Np];
    }
  }
  // decode of the activation slice (or of its half `part`), in the shadow of the weight loads
  auto decode_activation = [&](int part) {
#pragma unroll
    for (int it = 0; it < MAX_IT; ++it) {
      const int i = it * 256 + tid;
      if (i < total) {
        const int m = i / vec_per_row, v = i % vec_per_row;
        if (halves && (v >> 4) != part) continue;
        const f16x2 sc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(ac[it], 1.0f, false);
        f16x8 *dst = reinterpret_cast<f16x8 *>(slds + m * pitch + (halves ? v & 15 : v) * 64);
        dst[0] = decode_dword<false>(aw[it].x, sc);
        dst[1] = decode_dword<false>(aw[it].y, sc);
        dst[2] = decode_dword<true>(aw[it].z, sc);
        dst[3] = decode_dword<true>(aw[it].w, sc);
      }
    }
  };
  decode_activation(0);
  __syncthreads();

  f32x16 acc0;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc0[e] = 0.0f;
  const int am = r < (int)a.M ? r : (int)a.M - 1;  // lanes past M read a valid row; their outputs are dropped
  const char *arow = slds + am * pitch + h * 256;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    if (t == 2 && halves) {  // second half of the slice replaces the first in LDS
      __syncthreads();
      decode_activation(1);
      __syncthreads();
    }
    if (t < nsteps) {
      f16x2 sc[2][2];  // [chunk][block pair] -> scales of blocks (0,1) and (2,3) of each 64-chunk
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        sc[c][0] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(S[t][c], 1.0f, false);
        sc[c][1] = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(S[t][c], 1.0f, true);
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {       // 16-byte word q: elements [32q, 32q+32) of the lane's 128
        const uint32_t w[4] = {W[t][q].x, W[t][q].y, W[t][q].z, W[t][q].w};
#pragma unroll
        for (int d = 0; d < 4; ++d) {     // dword d: elements [32q + 8d, +8): block (4q + d) / 2 of the lane
          const int blk = (4 * q + d) >> 1;   // 0..7: chunk blk/4, block blk%4
          const f16x2 pair = sc[blk >> 2][(blk & 3) >> 1];
          f16x8 wdec = (blk & 1) ? decode_dword<true>(w[d], pair) : decode_dword<false>(w[d], pair);
          const f16x8 afrag = *reinterpret_cast<const f16x8 *>(arow + (halves ? t & 1 : t) * 512 + (q * 4 + d) * 16);
          acc0 = __builtin_amdgcn_mfma_f32_32x32x16_f16(wdec, afrag, acc0, 0, 0, 0);
        }
      }
    }
  }

  // acc0: lane <-> m = r, element e <-> n = n0 + (e>>2)*8 + h*4 + (e&3): 4 consecutive n per group
  const int m = r;
  if (m >= (int)a.M) return;
  if (a.split_k > 1) {  // fp32 partial tile of this K-slice; skinny_reduce_kernel adds the slices
    float *pp = a.partial + ((int64_t)ksl * a.M + m) * a.N;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int64_t n = n0 + g * 8 + h * 4;
      if (n + 3 < a.N && (a.N & 3) == 0) {
        *reinterpret_cast<float4 *>(pp + n) = make_float4(acc0[4 * g], acc0[4 * g + 1], acc0[4 * g + 2], acc0[4 * g + 3]);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (n + q < a.N) pp[n + q] = acc0[4 * g + q];
      }
    }
    return;
  }
  using DE = Elem<D_DT>;
  typename DE::T *Dp = static_cast<typename DE::T *>(a.D);
  const float scale = (*a.A_gs) * (*a.B_gs);
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    const int64_t n = n0 + (e >> 2) * 8 + h * 4 + (e & 3);
    if (n < a.N) {
      float v = acc0[e] * scale;
      if constexpr (BIAS_DT != BIAS_NONE) v += Elem<BIAS_DT>::load(a.bias, n);
      Dp[(int64_t)m * a.N + n] = DE::cvt(v);
    }
  }
}

// D[m, n] = cvt( (sum over K-slices of partial[s][m][n]) * gsA*gsB + bias[n] ), slices added in order.
// V outputs per thread (V = 4: 16-byte loads; needs N % 4 == 0); the loads of eight slices are in
// flight together, the additions stay in slice order.
template <int D_DT, int BIAS_DT, int V>
__global__ __launch_bounds__(256) void skinny_reduce_kernel(SkinnyArgs a) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * V;
  const int64_t total = a.M * a.N;
  if (i >= total) return;
  float v[V];
#pragma unroll
  for (int q = 0; q < V; ++q) v[q] = 0.0f;
  const float *p = a.partial + i;
  int sidx = 0;
  for (; sidx + 8 <= a.split_k; sidx += 8) {
    float t[8][V];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      if constexpr (V == 4) {
        const float4 f = *reinterpret_cast<const float4 *>(p + (int64_t)(sidx + u) * total);
        t[u][0] = f.x; t[u][1] = f.y; t[u][2] = f.z; t[u][3] = f.w;
      } else {
        t[u][0] = p[(int64_t)(sidx + u) * total];
      }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int q = 0; q < V; ++q) v[q] += t[u][q];
  }
  for (; sidx < a.split_k; ++sidx) {
    if constexpr (V == 4) {
      const float4 f = *reinterpret_cast<const float4 *>(p + (int64_t)sidx * total);
      v[0] += f.x; v[1] += f.y; v[2] += f.z; v[3] += f.w;
    } else {
      v[0] += p[(int64_t)sidx * total];
    }
  }
  const float scale = (*a.A_gs) * (*a.B_gs);
  using DE = Elem<D_DT>;
  typename DE::T *D = static_cast<typename DE::T *>(a.D);
  const int64_t n = i % a.N;  // V consecutive outputs share a row (N % V == 0)
#pragma unroll
  for (int q = 0; q < V; ++q) {
    v[q] *= scale;
    if constexpr (BIAS_DT != BIAS_NONE) v[q] += Elem<BIAS_DT>::load(a.bias, n + q);
  }
  if constexpr (V == 4 && sizeof(typename DE::T) == 2) {
    *reinterpret_cast<uint2 *>(D + i) = make_uint2(DE::cvt2(v[0], v[1]), DE::cvt2(v[2], v[3]));
  } else if constexpr (V == 4) {
    *reinterpret_cast<float4 *>(D + i) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    D[i] = DE::cvt(v[0]);
  }
}

template <int D_DT, int BIAS_DT>
static void launch_reduce(const SkinnyArgs &a, hipStream_t st) {
  const int64_t total = a.M * a.N;
  const bool v4 = a.N % 4 == 0 && ((uintptr_t)a.D & 15) == 0 && ((uintptr_t)a.partial & 15) == 0;
  if (v4)
    hipLaunchKernelGGL((skinny_reduce_kernel<D_DT, BIAS_DT, 4>), dim3((unsigned)ceil_div(total / 4, 256)), dim3(256), 0, st, a);
  else
    hipLaunchKernelGGL((skinny_reduce_kernel<D_DT, BIAS_DT, 1>), dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, st, a);
}

// ===========================================================================
// Decode-sized linear (1 <= M <= 32, K % 64 == 0, K >= 256): the weights are streamed once, through LDS.
// (The last stage of a K that is no multiple of 256 is treated as in the K-split-waves kernel: 1 x 28672 x 8320
// 177 -> 36 us, 16 x 4096 x 14400 307 -> 18 us, the 128x128 kernel against these.)
//
// A workgroup (8 waves) owns 128 weight rows and a contiguous range of 256-k stages.  Weights, weight
// scales, the packed activation rows and their scales go from global memory straight into an LDS ring
// of six or seven stages with LDS-DMA loads: lane l of a transfer fetches piece l % 8 of row l / 8, so eight
// lanes read one 128-byte run of a row, and every request is a full 64-byte line.  (With loads into
// registers in the MFMA operand layout every lane reads from a different row: four times the address
// work per byte, and the partial sums of a K split on top; the same pattern with 16 bytes per lane, as a
// wave's fragment of one stage would need, measured 2 TB/s.)  Wave (wn, kh) = (wave % 4, wave / 4) takes
// weight rows 32 wn .. 32 wn + 31 and the 64-chunks 2 kh, 2 kh + 1 of every stage: its packed
// fragments of the NEXT stage travel from LDS to registers while it decodes the current ones in
// registers (weights and activation alike: 4 converts + 4 packed multiplies per 8 elements) and
// issues D^T += W . Xhat^T with v_mfma_f32_32x32x16_f16, so a lane ends up with four consecutive n for
// one m.  One workgroup barrier per stage: a stage costs about 0.45 us of barrier, transfer issue and
// waits whatever its size, which is why it is 256 k long (128-k stages: 40 us on N = 28672, K = 8192).
// The two k halves meet through LDS at the end, always added in the same order.  Activation rows past
// M read row M - 1 and feed outputs that are never stored.  With one K range per tile the epilogue
// applies gsA*gsB and the bias and stores D; with several (too few tiles to fill the GPU) the fp32
// sums go to the caller's workspace and skinny_reduce_kernel adds the ranges in order.
// ===========================================================================
constexpr int ST_BN = 128;        // weight rows per workgroup
constexpr int ST_THREADS = 512;
constexpr int ST_BK = 256;        // k per stage (four 64-chunks)
constexpr int ST_ROW = ST_BK / 2; // packed bytes per row per stage
constexpr int ST_NPIECES = 4;     // LDS-DMA instructions per wave per stage (three from a weight image)
// A stage: the weight rows, their scale dwords [chunk][128 rows], MR packed activation rows and their scale
// dwords [chunk][MR rows].  MR is 32, or 16 when M <= 16: the smaller stage leaves room for a seventh one
// in the ring, i.e. one more stage of weights in flight.
constexpr int ST_OFF_B = 0;
constexpr int ST_OFF_SFB = ST_OFF_B + ST_BN * ST_ROW;
constexpr int ST_OFF_A = ST_OFF_SFB + 4 * ST_BN * 4;  // 18432
__host__ __device__ constexpr int st_off_sfa(int mr) { return ST_OFF_A + mr * ST_ROW; }
__host__ __device__ constexpr int st_stage_bytes(int mr) { return st_off_sfa(mr) + 4 * mr * 4; }
__host__ __device__ constexpr int st_stages(int mr) { return mr == 32 ? 6 : 7; }
__host__ __device__ constexpr int st_lds_bytes(int mr) { return st_stages(mr) * st_stage_bytes(mr); }
static_assert(st_lds_bytes(32) <= 160 * 1024 && st_lds_bytes(16) <= 160 * 1024, "the ring must fit in the CU's LDS");
static_assert((st_stages(16) - 3) * ST_NPIECES <= 63, "the wait counts must fit the 6-bit counter");
static_assert(st_lds_bytes(16) >= 4 * 64 * 16 * 4, "the ring doubles as the exchange buffer of the two k halves");
// From a weight image (PRE) the weights and weight scales of a stage are ONE contiguous run of two blocks,
// copied as it lies to the head of the LDS stage by 18 one-kilobyte transfers; with the transfers of the
// activation rows and of their scales that is three per wave.  The activation part of the stage is the same.
constexpr int ST_PRE_W_BYTES = 2 * W_BLOCK_BYTES;  // 18432
static_assert(ST_PRE_W_BYTES == ST_OFF_A, "both layouts put the activation behind 18 KB of weights and scales");
constexpr int ST_PRE_NPIECES = 3;

// a wave's fragments of one stage: for each of its two 64-chunks (2 kh, 2 kh + 1) 32 packed elements
// of a weight row and of an activation row (the lane's half of the chunk) and the two block scales of each
struct StageFrags {
  uint4 w[2], x[2];
  uint32_t ws[2], xs[2];
  float wfac[2];
};

// acc[c] += W . Xhat^T over the wave's two chunks of a stage (decode in registers)
__device__ __forceinline__ void stream_multiply(const StageFrags &cur, f32x16 (&acc)[2]) {
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const f16x2 wsc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(cur.ws[c], cur.wfac[c], false);
    const f16x2 xsc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(cur.xs[c], 1.0f, false);
    acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode_dword<false>(cur.w[c].x, wsc), decode_dword<false>(cur.x[c].x, xsc), acc[c], 0, 0, 0);
    acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode_dword<false>(cur.w[c].y, wsc), decode_dword<false>(cur.x[c].y, xsc), acc[c], 0, 0, 0);
    acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode_dword<true>(cur.w[c].z, wsc), decode_dword<true>(cur.x[c].z, xsc), acc[c], 0, 0, 0);
    acc[c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode_dword<true>(cur.w[c].w, wsc), decode_dword<true>(cur.x[c].w, xsc), acc[c], 0, 0, 0);
  }
}

// End of the LDS-ring kernels, after the last LDS-DMA has landed and every wave has passed a barrier:
// the two chunk sums of a wave, then the NK k parts of each of the NWN row groups (through `xch_base`,
// always in this order), then either the fp32 partial sums of this K range or the finished outputs
// (times gsA * gsB, plus bias).
template <int D_DT, int BIAS_DT, int NK = 2, int NWN = 4>
__device__ __forceinline__ void stream_finish(f32x16 (&acc)[2], const SkinnyArgs &a, char *xch_base, float gs_a, int wn, int kh,
                                              int lane, int64_t n0) {
  const int half = lane >> 5, r32 = lane & 31;
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[0][e] += acc[1][e];
  // the NK k parts of a row group meet in the waves of part 0, added in the order of the parts
  if (kh != 0) {
    float4 *xch = reinterpret_cast<float4 *>(xch_base) + (((kh - 1) * NWN + wn) * 64 + lane) * 4;
#pragma unroll
    for (int g = 0; g < 4; ++g) xch[g] = make_float4(acc[0][4 * g], acc[0][4 * g + 1], acc[0][4 * g + 2], acc[0][4 * g + 3]);
  }
  __syncthreads();
  if (kh != 0) return;
#pragma unroll
  for (int k = 1; k < NK; ++k) {
    const float4 *xch = reinterpret_cast<const float4 *>(xch_base) + (((k - 1) * NWN + wn) * 64 + lane) * 4;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const float4 o = xch[g];
      acc[0][4 * g] += o.x; acc[0][4 * g + 1] += o.y; acc[0][4 * g + 2] += o.z; acc[0][4 * g + 3] += o.w;
    }
  }

  // acc: lane <-> m = r32, element e <-> n = (e >> 2) * 8 + half * 4 + (e & 3): four consecutive n per group
  const int m = r32;
  if (m >= (int)a.M) return;
  const int64_t nw = n0 + wn * 32;
  if (a.split_k > 1) {
    float *pp = a.partial + ((int64_t)blockIdx.y * a.M + m) * a.N;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int64_t n = nw + g * 8 + half * 4;
      if (n + 3 < a.N && (a.N & 3) == 0) {
        *reinterpret_cast<float4 *>(pp + n) = make_float4(acc[0][4 * g], acc[0][4 * g + 1], acc[0][4 * g + 2], acc[0][4 * g + 3]);
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (n + q < a.N) pp[n + q] = acc[0][4 * g + q];
      }
    }
    return;
  }
  using DE = Elem<D_DT>;
  typename DE::T *Dp = static_cast<typename DE::T *>(a.D);
  const float scale = gs_a * (*a.B_gs);
  // a lane's four consecutive outputs of a group leave as one 8- or 16-byte store where the rows allow it
  const bool vec_ok = (a.N & 3) == 0 && ((uintptr_t)a.D & 15) == 0;
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int64_t n = nw + g * 8 + half * 4;
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = acc[0][4 * g + q] * scale;
      if constexpr (BIAS_DT != BIAS_NONE) v[q] += n + q < a.N ? Elem<BIAS_DT>::load(a.bias, n + q) : 0.0f;
    }
    typename DE::T *dst = Dp + (int64_t)m * a.N + n;
    if (vec_ok && n + 3 < a.N) {
      if constexpr (sizeof(typename DE::T) == 2)
        *reinterpret_cast<uint2 *>(dst) = make_uint2(DE::cvt2(v[0], v[1]), DE::cvt2(v[2], v[3]));
      else
        *reinterpret_cast<float4 *>(dst) = make_float4(v[0], v[1], v[2], v[3]);
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (n + q < a.N) dst[q] = DE::cvt(v[q]);
    }
  }
}

template <int D_DT, int BIAS_DT, bool PRE, int MR, bool TAIL>
__global__ __launch_bounds__(ST_THREADS, 1) void linear_nvfp4_stream_kernel(SkinnyArgs a) {
  static_assert(MR == 32 || MR == 16, "activation rows per stage");
  constexpr int NPIECES = PRE ? ST_PRE_NPIECES : ST_NPIECES;
  constexpr int OFF_A = ST_OFF_A, OFF_SFA = st_off_sfa(MR);
  constexpr int ST_PS = st_stages(MR), ST_STAGE_BYTES = st_stage_bytes(MR);
  extern __shared__ __attribute__((aligned(16))) char stlds[];
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, r32 = lane & 31;
  const int swave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = swave & 3, kh = swave >> 2;
  const int64_t n0 = (int64_t)blockIdx.x * ST_BN;
  const int nst_all = (int)ceil_div(a.K, ST_BK);
  const int s0 = (int)((int64_t)nst_all * blockIdx.y / a.split_k);
  const int nst = (int)((int64_t)nst_all * (blockIdx.y + 1) / a.split_k) - s0;  // >= 1: split_k <= stages
  const StageWalk<TAIL> walk{s0, (int)(a.K >> 6)};
  const int64_t kb = a.K >> 1;
  // Workgroup b walks its stages starting at stage b % nst and wraps around.  In step, every workgroup
  // would ask for the same 128-byte column of its rows at the same time; with a row pitch that is a
  // power of two (K = 8192: 4096 bytes) all those addresses fall on the same few memory channels.
  const int rot = (int)(blockIdx.x % (unsigned)nst);
  auto stage_of = [&](int step) {
    const int p = step + rot;
    return p >= nst ? p - nst : p;
  };

  // LDS holds row-major 128-byte rows (lane l of a transfer lands at 16 l: eight rows per transfer);
  // the eight 16-byte pieces of row r sit at positions piece ^ (r & 7), which spreads a fragment read
  // (one piece of each of 32 rows) over all LDS banks.  Unswizzled those reads fall on a quarter of the
  // banks and, issued by eight waves every stage, held the transfers back (40 us against 31 us on
  // N = 28672, K = 8192).
  // --- this wave's transfers of a stage: lane offsets (loop invariant), LDS destinations, sources
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)stlds;
  // weights (and, from an image, their scales)
  uint32_t offW[3];
  const uint8_t *srcW;
  int64_t strideW;
  uint32_t ldsW;
  if constexpr (PRE) {
    // transfers 2 swave, 2 swave + 1 of the stage's 18 contiguous kilobytes; waves 0 and 1 also 16, 17
    offW[0] = (uint32_t)(swave * 2048 + lane * 16);
    offW[1] = offW[0] + 1024;
    offW[2] = (uint32_t)((16 + swave) * 1024 + lane * 16);
    strideW = walk.step(W_BLOCK_BYTES / 2);  // (K % 128 == 0: a stage starts at a whole block)
    srcW = uniform_ptr(a.B + (int64_t)blockIdx.x * (a.K / W_BLOCK_K) * W_BLOCK_BYTES + walk.start(strideW));
    ldsW = (uint32_t)__builtin_amdgcn_readfirstlane(swave * 2048);
  } else {
    // weight rows swave * 16 + {0..7}, {8..15}, 128 B each
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int loc = swave * 16 + q * 8 + (lane >> 3);
      int64_t row = n0 + loc;
      row = row < a.N ? row : a.N - 1;  // rows past N read the last row; their outputs are never stored
      offW[q] = (uint32_t)((row - n0) * kb + ((lane & 7) ^ (loc & 7)) * 16);
    }
    offW[2] = 0;
    strideW = walk.step(ST_ROW / 4);
    srcW = uniform_ptr(a.B + n0 * kb + walk.start(strideW));
    ldsW = (uint32_t)__builtin_amdgcn_readfirstlane(ST_OFF_B + swave * 2048);
  }
  // weight scales from the scale tensor: chunk swave / 2, rows (swave % 2) * 64 + lane of the tile
  uint32_t offS = 0, ldsS = 0;
  int64_t strideS = 0;
  const uint8_t *srcS = nullptr;
  if constexpr (!PRE) {
    int64_t srow = n0 + (swave & 1) * 64 + lane;
    srow = srow < a.Np ? srow : a.Np - 1;
    offS = (uint32_t)(srow * 4);
    strideS = walk.step(a.Np * 4);  // chunk planes
    srcS = uniform_ptr(reinterpret_cast<const uint8_t *>(a.B_sf) + (int64_t)(swave >> 1) * a.Np * 4 + walk.start(strideS));
    ldsS = (uint32_t)__builtin_amdgcn_readfirstlane(ST_OFF_SFB + (swave >> 1) * (ST_BN * 4) + (swave & 1) * 256);
  }
  // activation: MR / 8 waves take the packed rows w * 8 + {0..7}; the scale dwords are one transfer for
  // MR = 16 (lane = chunk x row) and two for MR = 32 (chunks 2 p + {0, 1}, p = 0, 1).  From an image waves
  // 0 and 1 have their third weight transfer first.  The waves left over repeat a scale transfer: every wave
  // issues the same count.
  constexpr int A_FIRST = PRE ? 2 : 0;  // first wave of those that move the rows
  constexpr int A_WAVES = MR / 8;
  const bool moves_rows = swave >= A_FIRST && swave < A_FIRST + A_WAVES;
  uint32_t off4 = 0, lds4 = 0;
  const uint8_t *src4 = nullptr;
  int64_t stride4 = 0;
  if (moves_rows) {
    const int loc = (swave - A_FIRST) * 8 + (lane >> 3);
    const int64_t row = loc < a.M ? loc : a.M - 1;  // rows past M read row M - 1; their outputs are never stored
    off4 = (uint32_t)(row * kb + ((lane & 7) ^ (loc & 7)) * 16);
    stride4 = walk.step(ST_ROW / 4);
    src4 = uniform_ptr(a.Aq + walk.start(stride4));
    lds4 = (uint32_t)__builtin_amdgcn_readfirstlane(OFF_A + (swave - A_FIRST) * 1024);
  } else if (!PRE || swave >= 2) {
    stride4 = walk.step(a.Mp * 4);
    src4 = uniform_ptr(a.A_sf + walk.start(stride4));
    if constexpr (MR == 32) {
      const int pair = swave & 1;  // chunks 2 pair, 2 pair + 1
      const int64_t row = r32 < a.Mp ? r32 : a.Mp - 1;
      off4 = (uint32_t)(((2 * pair + half) * a.Mp + row) * 4);
      lds4 = (uint32_t)__builtin_amdgcn_readfirstlane(OFF_SFA + pair * 256);
    } else {
      off4 = (uint32_t)(((lane >> 4) * a.Mp + (lane & 15)) * 4);  // Mp >= 16
      lds4 = (uint32_t)__builtin_amdgcn_readfirstlane(OFF_SFA);
    }
  }
  auto issue_stage = [&](int slot, int step) {  // step: position in this workgroup's order of stages
    const int st = stage_of(step);
    const uint32_t base = lds_base + slot * ST_STAGE_BYTES;
    const uint8_t *pw = srcW + walk.offset(st, strideW);
    dma16(pw, offW[0], base, ldsW);
    dma16(pw, offW[1], base, ldsW + 1024);
    if constexpr (PRE) {
      if (swave < 2)
        dma16(pw, offW[2], base, (uint32_t)__builtin_amdgcn_readfirstlane((16 + swave) * 1024));
      else if (moves_rows)
        dma16(src4 + walk.offset(st, stride4), off4, base, lds4);
      else
        dma4(src4 + walk.offset(st, stride4), off4, base, lds4);
    } else {
      dma4(srcS + walk.offset(st, strideS), offS, base, ldsS);
      if (moves_rows)
        dma16(src4 + walk.offset(st, stride4), off4, base, lds4);
      else
        dma4(src4 + walk.offset(st, stride4), off4, base, lds4);
    }
  };

  const int wrow_l = wn * 32 + r32;
  const int xrow = r32 & (MR - 1);  // lanes of rows past MR read a staged row; their outputs are never stored
  int wf_off[2], xf_off[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int piece = kh * 4 + c * 2 + half;
    if constexpr (PRE)  // block kh of the stage; 64-byte rows, piece p of a chunk pair at p ^ ((r >> 1) & 3)
      wf_off[c] = kh * W_BLOCK_BYTES + wrow_l * 64 + (((c * 2 + half) ^ ((wrow_l >> 1) & 3)) * 16);
    else
      wf_off[c] = ST_OFF_B + wrow_l * ST_ROW + ((piece ^ (wrow_l & 7)) * 16);
    xf_off[c] = OFF_A + xrow * ST_ROW + ((piece ^ (xrow & 7)) * 16);
  }
  // scale planes of the wave's two chunks: `ws_pitch` bytes apart
  constexpr int ws_pitch = PRE ? W_BLOCK_ROWS * 4 : ST_BN * 4;
  const int ws_off = (PRE ? kh * W_BLOCK_BYTES + W_BLOCK_DATA : ST_OFF_SFB + (kh * 2) * (ST_BN * 4)) + wrow_l * 4 + half * 2;
  const int xs_off = OFF_SFA + (kh * 2) * (MR * 4) + xrow * 4 + half * 2;
  auto load_frags = [&](int slot, int step) {
    const char *st = stlds + slot * ST_STAGE_BYTES;
    StageFrags f;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      f.w[c] = *reinterpret_cast<const uint4 *>(st + wf_off[c]);
      f.x[c] = *reinterpret_cast<const uint4 *>(st + xf_off[c]);
      f.ws[c] = *reinterpret_cast<const uint16_t *>(st + ws_off + c * ws_pitch);
      f.xs[c] = *reinterpret_cast<const uint16_t *>(st + xs_off + c * (MR * 4));
      f.wfac[c] = walk.weight_factor(stage_of(step), 2 * kh + c);
    }
    return f;
  };

  f32x16 acc[2];  // one per chunk of the pair: two independent accumulation chains
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[c][e] = 0.0f;

  // prologue: stages 0 .. PS-2 in flight (past the range: the last stage again, into slots nobody
  // reads), stages 0 and 1 landed, fragments of stage 0 in registers
  const int last = nst - 1;
#pragma unroll
  for (int d = 0; d < ST_PS - 1; ++d) issue_stage(d, d < last ? d : last);
  wait_vmcnt<(ST_PS - 3) * NPIECES>();
  __syncthreads();
  StageFrags cur = load_frags(0, 0);

  int slot_next = 1, slot_dma = ST_PS - 1;
  for (int s = 0; s < nst; ++s) {
    // fragments of the next stage (it landed before the previous barrier) travel from LDS while this
    // stage is decoded and multiplied (past the range: a stage nobody uses)
    const StageFrags nxt = load_frags(slot_next, s + 1 < nst ? s + 1 : s);
    stream_multiply(cur, acc);
    // refill the slot of the stage before this one (everybody read it before the previous barrier)
    const int sd = s + ST_PS - 1;
    issue_stage(slot_dma, sd < last ? sd : last);
    wait_vmcnt<(ST_PS - 3) * NPIECES>();  // own transfers of stage s + 2 have landed
    __syncthreads();
    cur = nxt;
    slot_next = slot_next + 1 == ST_PS ? 0 : slot_next + 1;
    slot_dma = slot_dma + 1 == ST_PS ? 0 : slot_dma + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS-DMA may land after this point: the ring is reused
  __syncthreads();
  stream_finish<D_DT, BIAS_DT>(acc, a, stlds, *a.A_gs, wn, kh, lane, n0);
}

// ===========================================================================
// The LDS-ring kernel with 64 weight rows per workgroup, for weights with so few rows that 128-row
// tiles leave CUs idle or force a K split with partial sums and a second launch (N = 14336: 112
// tiles of 128 rows, 224 of 64).  Same ring, swizzle, stage order and arithmetic; wave (wn, kq) =
// (wave % 2, wave / 2) takes weight rows 32 wn .. 32 wn + 31 and chunk kq of every stage, and the four
// k parts of a row group meet through LDS at the end.  A stage is 13.5 KB (64 weight rows, 32
// activation rows, their scales), ten of them make the ring; three transfers per wave per stage.
// Plain layout only.
// ===========================================================================
constexpr int S6_BN = 64;
constexpr int S6_PS = 10;
constexpr int S6_NPIECES = 3;
constexpr int S6_OFF_B = 0;
constexpr int S6_OFF_A = S6_OFF_B + S6_BN * ST_ROW;      // 32 packed activation rows
constexpr int S6_OFF_SFB = S6_OFF_A + 32 * ST_ROW;       // weight scale dwords [chunk][64 rows]
constexpr int S6_OFF_SFA = S6_OFF_SFB + 4 * S6_BN * 4;   // activation scale dwords [chunk][32 rows]
constexpr int S6_STAGE_BYTES = S6_OFF_SFA + 4 * 32 * 4;  // 13824
constexpr int S6_LDS_BYTES = S6_PS * S6_STAGE_BYTES;
static_assert(S6_LDS_BYTES <= 160 * 1024, "the ring must fit in the CU's LDS");
static_assert((S6_PS - 3) * S6_NPIECES <= 63, "the wait counts must fit the 6-bit counter");
static_assert(S6_LDS_BYTES >= 3 * 2 * 64 * 16 * 4, "the ring doubles as the exchange buffer of the four k parts");

template <int D_DT, int BIAS_DT, bool TAIL>
__global__ __launch_bounds__(ST_THREADS, 1) void linear_nvfp4_stream64_kernel(SkinnyArgs a) {
  extern __shared__ __attribute__((aligned(16))) char stlds[];
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5, r32 = lane & 31;
  const int swave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = swave & 1, kq = swave >> 1;
  const int64_t n0 = (int64_t)blockIdx.x * S6_BN;
  const int nst_all = (int)ceil_div(a.K, ST_BK);
  const int s0 = (int)((int64_t)nst_all * blockIdx.y / a.split_k);
  const int nst = (int)((int64_t)nst_all * (blockIdx.y + 1) / a.split_k) - s0;  // >= 1: split_k <= stages
  const StageWalk<TAIL> walk{s0, (int)(a.K >> 6)};
  const int64_t kb = a.K >> 1;
  const int rot = (int)(blockIdx.x % (unsigned)nst);  // stages are walked from stage b % nst on (see linear_nvfp4_stream_kernel)
  auto stage_of = [&](int step) {
    const int p = step + rot;
    return p >= nst ? p - nst : p;
  };
  const uint32_t lds_base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char *)stlds;
  // (1) weight rows swave * 8 + {0..7}, 128 B each, piece p of row r at position p ^ (r & 7)
  uint32_t offW;
  {
    const int loc = swave * 8 + (lane >> 3);
    int64_t row = n0 + loc;
    row = row < a.N ? row : a.N - 1;  // rows past N read the last row; their outputs are never stored
    offW = (uint32_t)((row - n0) * kb + ((lane & 7) ^ (loc & 7)) * 16);
  }
  const uint8_t *srcW = uniform_ptr(a.B + n0 * kb + walk.start(walk.step(ST_ROW / 4)));
  const uint32_t ldsW = (uint32_t)__builtin_amdgcn_readfirstlane(S6_OFF_B + swave * 1024);
  // (2) waves 0..3: weight scale dwords of chunk swave, rows n0 + lane; waves 4..7: packed activation
  //     rows (swave - 4) * 8 + {0..7}
  uint32_t off2, lds2;
  const uint8_t *src2;
  int64_t stride2;
  if (swave < 4) {
    int64_t srow = n0 + lane;
    srow = srow < a.Np ? srow : a.Np - 1;
    off2 = (uint32_t)(srow * 4);
    stride2 = walk.step(a.Np * 4);  // chunk planes
    src2 = uniform_ptr(reinterpret_cast<const uint8_t *>(a.B_sf) + (int64_t)swave * a.Np * 4 + walk.start(stride2));
    lds2 = (uint32_t)__builtin_amdgcn_readfirstlane(S6_OFF_SFB + swave * (S6_BN * 4));
  } else {
    const int loc = (swave - 4) * 8 + (lane >> 3);
    const int64_t row = loc < a.M ? loc : a.M - 1;  // rows past M read row M - 1; their outputs are never stored
    off2 = (uint32_t)(row * kb + ((lane & 7) ^ (loc & 7)) * 16);
    stride2 = walk.step(ST_ROW / 4);
    src2 = uniform_ptr(a.Aq + walk.start(stride2));
    lds2 = (uint32_t)__builtin_amdgcn_readfirstlane(S6_OFF_A + (swave - 4) * 1024);
  }
  // (3) activation scales of chunks 2 p + {0, 1}, p = swave % 2 (waves 2..7 repeat the transfers of waves
  //     0 and 1: every wave issues the same count)
  const int pair = swave & 1;
  const int64_t arow = r32 < a.Mp ? r32 : a.Mp - 1;
  const uint32_t off3 = (uint32_t)(((2 * pair + half) * a.Mp + arow) * 4);
  const int64_t stride3 = walk.step(a.Mp * 4);
  const uint8_t *src3 = uniform_ptr(a.A_sf + walk.start(stride3));
  const uint32_t lds3 = (uint32_t)__builtin_amdgcn_readfirstlane(S6_OFF_SFA + pair * 256);
  auto issue_stage = [&](int slot, int step) {  // step: position in this workgroup's order of stages
    const int st = stage_of(step);
    const uint32_t base = lds_base + slot * S6_STAGE_BYTES;
    dma16(srcW + walk.offset(st, walk.step(ST_ROW / 4)), offW, base, ldsW);
    if (swave < 4)
      dma4(src2 + walk.offset(st, stride2), off2, base, lds2);
    else
      dma16(src2 + walk.offset(st, stride2), off2, base, lds2);
    dma4(src3 + walk.offset(st, stride3), off3, base, lds3);
  };

  // this wave's fragments of a stage: chunk kq, 32 packed elements of a weight row and of an activation
  // row (the lane's half of the chunk) and the two block scales of each
  struct Frags {
    uint4 w, x;
    uint32_t ws, xs;
    float wfac;
  };
  const int wrow_l = wn * 32 + r32;
  const int piece = kq * 2 + half;
  const int wf_off = S6_OFF_B + wrow_l * ST_ROW + ((piece ^ (wrow_l & 7)) * 16);
  const int xf_off = S6_OFF_A + r32 * ST_ROW + ((piece ^ (r32 & 7)) * 16);
  const int ws_off = S6_OFF_SFB + kq * (S6_BN * 4) + wrow_l * 4 + half * 2;
  const int xs_off = S6_OFF_SFA + kq * (32 * 4) + r32 * 4 + half * 2;
  auto load_frags = [&](int slot, int step) {
    const char *st = stlds + slot * S6_STAGE_BYTES;
    Frags f;
    f.wfac = walk.weight_factor(stage_of(step), kq);
    f.w = *reinterpret_cast<const uint4 *>(st + wf_off);
    f.x = *reinterpret_cast<const uint4 *>(st + xf_off);
    f.ws = *reinterpret_cast<const uint16_t *>(st + ws_off);
    f.xs = *reinterpret_cast<const uint16_t *>(st + xs_off);
    return f;
  };

  f32x16 acc[2];  // two independent accumulation chains: the first and the second half of the chunk
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[c][e] = 0.0f;

  const int last = nst - 1;
#pragma unroll
  for (int d = 0; d < S6_PS - 1; ++d) issue_stage(d, d < last ? d : last);
  wait_vmcnt<(S6_PS - 3) * S6_NPIECES>();
  __syncthreads();
  Frags cur = load_frags(0, 0);

  int slot_next = 1, slot_dma = S6_PS - 1;
  for (int s = 0; s < nst; ++s) {
    const Frags nxt = load_frags(slot_next, s + 1 < nst ? s + 1 : s);  // it landed before the previous barrier
    const f16x2 wsc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(cur.ws, cur.wfac, false);
    const f16x2 xsc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(cur.xs, 1.0f, false);
    acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode_dword<false>(cur.w.x, wsc), decode_dword<false>(cur.x.x, xsc), acc[0], 0, 0, 0);
    acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode_dword<false>(cur.w.y, wsc), decode_dword<false>(cur.x.y, xsc), acc[0], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode_dword<true>(cur.w.z, wsc), decode_dword<true>(cur.x.z, xsc), acc[1], 0, 0, 0);
    acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(decode_dword<true>(cur.w.w, wsc), decode_dword<true>(cur.x.w, xsc), acc[1], 0, 0, 0);
    const int sd = s + S6_PS - 1;
    issue_stage(slot_dma, sd < last ? sd : last);
    wait_vmcnt<(S6_PS - 3) * S6_NPIECES>();  // own transfers of stage s + 2 have landed
    __syncthreads();
    cur = nxt;
    slot_next = slot_next + 1 == S6_PS ? 0 : slot_next + 1;
    slot_dma = slot_dma + 1 == S6_PS ? 0 : slot_dma + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no LDS-DMA may land after this point: the ring is reused
  __syncthreads();
  stream_finish<D_DT, BIAS_DT, 4, 2>(acc, a, stlds, *a.A_gs, wn, kq, lane, n0);
}

// ===========================================================================
// Decode-sized linear (1 <= M <= 32, K % 64 == 0, K >= 256) with 16 weight rows per workgroup and all of K in it: weights with too
// few rows for the LDS-ring kernels, which split their K over workgroups and add the parts in a second launch.
//
// Eight waves take the 128-k steps of a row in turn.  Nothing is shared between them, so nothing goes through LDS: lane (row r,
// quarter g) loads the 16 bytes [32 g, 32 g + 32) of the step of its weight row - four lanes a 64-byte run - with the two block
// scales, and the same of activation row r, three steps ahead, and has with each dword the operand of one v_mfma_f32_16x16x32_f16 (the
// order of k is free as long as both sides share it).  The eight sums meet through LDS in the order of the waves.
// A step's second half that K does not have is read from its first one, with weight scales so small that they round to zero.
// Bound by the latency of what is in flight: at 16 x 4096 x 14336, one workgroup a CU, 36.1 MiB are read for 31.6 of operands, at 3.6 TB/s,
// and the counters show a SIMD's vector port busy for 40 % of the time and its matrix core for 8 %.  The activation, read and decoded again by
// every workgroup, as many bytes as its weights (M <= 16; twice as many above), adds a tenth from M = 1 to 16.
// 16 x 4096 x 14336, weights from HBM, 17.8 -> 11.4 us (64 rows, K split in four, and the second launch before), M = 1 15.8 -> 10.4; 16 x 4096 x 4096 10.2 -> 5.1; 1 x 20000 x 2880 23.4 -> 11.2; 32 x 1024 x 1024
// 7.6 -> 3.2.  Three steps ahead and two workgroups on a CU: two more cost 0.7 us at 16 x 4096 x 14336 in registers, sixteen waves 2.5 us at
// 1 x 14336 x 4096, four waves 3 us at 16 x 4096 x 14336; loads past the caches lose where the activation is read again.
// On a weight image a wave's step is one kilobyte of a block and its scales lie behind it: 16 x 4096 x 14336 10.1 us (plain 11.2), 16 x 14336 x 4096
// 10.9 (12.5), 8 x 20480 x 8192 23.4 (26.8); the ring kernel, which took all of M <= 32 there, 18.1, 16.1 and 38.7.
// ===========================================================================
constexpr int R16_DEPTH = 3;

// MT: tiles of 16 activation rows.  TAIL: K is no multiple of 128.  PRE: B is a weight image, whose blocks hold a step of 128 rows each.
template <int D_DT, int BIAS_DT, int MT, bool TAIL, bool PRE>
__global__ __launch_bounds__(64 * R16_WAVES, 2) void linear_nvfp4_rows16_kernel(SkinnyArgs a) {
  static_assert(!(PRE && TAIL), "an image has whole steps");
  __shared__ float4 part[R16_WAVES][MT][64];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 15, g = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * R16_ROWS, kb = a.K >> 1;
  const int nst = (int)ceil_div(a.K, R16_STEP);
  const int cnt = (nst - wave + R16_WAVES - 1) / R16_WAVES;  // steps of this wave; none where K is short
  const int wr = n0 + r < a.N ? r : (int)(a.N - 1 - n0);  // rows past N read the last row; their outputs are never stored
  const uint8_t *const w_src = uniform_ptr(PRE ? a.B + n0 / W_BLOCK_ROWS * nst * W_BLOCK_BYTES : a.B + n0 * kb);
  const uint8_t *const ws_src = uniform_ptr(PRE ? nullptr : reinterpret_cast<const uint8_t *>(a.B_sf) + n0 * 4);
  const int in_block = (int)(n0 % W_BLOCK_ROWS) + r;  // PRE: rows past N exist (zeros)
  const uint32_t w_row = PRE ? in_block * (W_BLOCK_K / 2) + ((g ^ ((in_block >> 1) & 3)) * 16) : (uint32_t)(wr * kb);
  const uint32_t ws_row = PRE ? W_BLOCK_DATA + (g >> 1) * (W_BLOCK_ROWS * 4) + in_block * 4 + (g & 1) * 2 : (uint32_t)(wr * 4);
  uint32_t x_row[MT], xs_row[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = i * 16 + r < a.M ? i * 16 + r : (int)a.M - 1;  // rows past M likewise
    x_row[i] = (uint32_t)(m * kb), xs_row[i] = (uint32_t)(m * 4);
  }
  struct Step {
    uint4 w, x[MT];
    uint32_t ws, xs[MT];
  };
  auto load = [&](Step &st, int t) {
    const int s = wave + t * R16_WAVES;
    const uint32_t gg = TAIL && s == nst - 1 ? g & 1 : g;
    const int64_t at = (int64_t)s * (R16_STEP / 2);
    if constexpr (PRE) {
      st.w = *reinterpret_cast<const uint4 *>(w_src + (int64_t)s * W_BLOCK_BYTES + w_row);
      st.ws = *reinterpret_cast<const uint16_t *>(w_src + (int64_t)s * W_BLOCK_BYTES + ws_row);
    } else {
      st.w = *reinterpret_cast<const uint4 *>(w_src + at + (w_row + gg * 16));
      st.ws = *reinterpret_cast<const uint16_t *>(ws_src + (int64_t)(2 * s) * a.Np * 4 + ((gg >> 1) * (uint32_t)a.Np * 4 + ws_row + (gg & 1) * 2));
    }
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      st.x[i] = *reinterpret_cast<const uint4 *>(a.Aq + at + (x_row[i] + gg * 16));
      st.xs[i] = *reinterpret_cast<const uint16_t *>(a.A_sf + (int64_t)(2 * s) * a.Mp * 4 + ((gg >> 1) * (uint32_t)a.Mp * 4 + xs_row[i] + (gg & 1) * 2));
    }
  };
  f32x4 acc[MT][2];  // two independent accumulation chains
#pragma unroll
  for (int i = 0; i < MT; ++i) acc[i][0] = acc[i][1] = (f32x4)(0.0f);
  auto multiply = [&](const Step &st, int t) {
    const float fac = TAIL && wave + t * R16_WAVES == nst - 1 && g >= 2 ? 0x1p-60f : 1.0f;
    const f16x2 wsc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(st.ws, fac, false);
    const f16x8 w0 = decode_dword<false>(st.w.x, wsc), w1 = decode_dword<false>(st.w.y, wsc);
    const f16x8 w2 = decode_dword<true>(st.w.z, wsc), w3 = decode_dword<true>(st.w.w, wsc);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const f16x2 xsc = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(st.xs[i], 1.0f, false);
      acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w0, decode_dword<false>(st.x[i].x, xsc), acc[i][0], 0, 0, 0);
      acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w1, decode_dword<false>(st.x[i].y, xsc), acc[i][1], 0, 0, 0);
      acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w2, decode_dword<true>(st.x[i].z, xsc), acc[i][0], 0, 0, 0);
      acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(w3, decode_dword<true>(st.x[i].w, xsc), acc[i][1], 0, 0, 0);
    }
  };
  Step ring[R16_DEPTH];
#pragma unroll
  for (int d = 0; d < R16_DEPTH; ++d)
    if (d < cnt) load(ring[d], d);
  int t = 0;
  for (; t + R16_DEPTH < cnt; t += R16_DEPTH) {
#pragma unroll
    for (int d = 0; d < R16_DEPTH; ++d) {
      multiply(ring[d], t + d);
      if (t + d + R16_DEPTH < cnt) load(ring[d], t + d + R16_DEPTH);
    }
  }
#pragma unroll
  for (int d = 0; d < R16_DEPTH; ++d)
    if (t + d < cnt) multiply(ring[d], t + d);

  rows16_finish<D_DT, BIAS_DT, MT>(acc, part, a.D, a.bias, (*a.A_gs) * (*a.B_gs), a.M, a.N, n0);
}

// CUs that the decode plans count on; a process without a GPU may ask for scratch sizes, too
static int64_t decode_cu_count() {
  const int n = device_cu_count();
  return n > 0 ? n : 256;
}

// Plan of a decode-sized linear: which kernel, its K split and the fp32 scratch it needs.
enum { DECODE_REGISTERS = 1, DECODE_LDS_RING = 2, DECODE_LDS_RING64 = 3, DECODE_ROWS16 = 4, DECODE_ROWS16_LDS = 5 };
struct SkinnyPlan {
  int kind;                // DECODE_REGISTERS: linear_nvfp4_skinny_kernel; DECODE_LDS_RING: linear_nvfp4_stream_kernel;
                           // DECODE_LDS_RING64: linear_nvfp4_stream64_kernel
  int ks_len;              // register kernel: k per workgroup (256, 512 or 1024)
  int split_k;             // K ranges; > 1 needs `partial_bytes` of fp32 scratch
  int64_t partial_bytes, groups;
  int lds_bytes;
  // linear_nvfp4_rows16_kernel runs instead, and needs no scratch.  The rest of the plan is what the entry points go on asking of
  // their callers for these shapes.
  bool rows16;
  bool fused;  // and so it does, with the quantizer in it, in a fused call
  bool lds_x;  // and the kernel of the fused call runs a linear alone, too
};
static std::atomic<int> g_forced_decode_kernel{0};  // ac4k_set_linear_tuning: 0 = by shape

// Register kernel: K slices of up to 1024, halved until about 768 workgroups are in flight.
static void plan_registers(int64_t M, int64_t N, int64_t K, SkinnyPlan &p) {
  int ks = 1024;
  const int f = g_forced_skinny_ks.load(std::memory_order_relaxed);
  if (f == 256 || f == 512 || f == 1024) ks = f;
  while (ks > SK_STEP && K % ks != 0) ks >>= 1;
  p.kind = DECODE_REGISTERS;
  p.groups = ceil_div(N, SK_ROWS);
  // short problems: use smaller slices to get enough workgroups in flight
  while (ks > SK_STEP && p.groups * (K / ks) < 768) ks >>= 1;
  p.ks_len = ks;
  p.split_k = (int)(K / ks);
  p.partial_bytes = p.split_k > 1 ? (int64_t)p.split_k * M * N * 4 : 0;
  p.lds_bytes = (int)M * ((M > 16 && ks == 1024 ? 512 : ks) * 2 + 16);
}

// LDS-ring kernel: one K range per 128-row tile when the tiles alone fill the GPU; otherwise the
// smallest number of ranges that gives about 200 workgroups, each range at least two stages long.
static void plan_lds_ring(int64_t M, int64_t N, int64_t K, SkinnyPlan &p, int rows = ST_BN) {
  p.kind = rows == ST_BN ? DECODE_LDS_RING : DECODE_LDS_RING64;
  p.groups = ceil_div(N, rows);
  const int64_t stages = ceil_div(K, ST_BK);
  int64_t splits = 1;
  if (const int f = g_forced_skinny_ks.load(std::memory_order_relaxed)) {  // forced length of a K range
    splits = K / f;
  } else if (p.groups < 192) {
    splits = ceil_div(200, p.groups);
    if (splits > stages / 2) splits = stages / 2;
    if (splits > 32) splits = 32;
  }
  if (splits < 1) splits = 1;
  if (splits > stages) splits = stages;
  p.ks_len = 0;
  p.split_k = (int)splits;
  p.partial_bytes = splits > 1 ? splits * M * N * 4 : 0;
  p.lds_bytes = rows == ST_BN ? st_lds_bytes(M <= 16 ? 16 : 32) : S6_LDS_BYTES;
}

// Shapes of the decode-sized kernels (K % 64 == 0, the register kernel K % 256 == 0) and the choice between them.  The
// register kernel has all its loads in flight at once and four workgroups per CU, which wins while M
// is small and the problem needs a K split anyway (few row tiles, long K); it pays for partial sums
// and a second launch, and its registers run out as M grows.  The LDS-ring kernels take nearly the
// same time for every M <= 32 and need no second launch when their row tiles alone fill the GPU:
// 128-row tiles when there are 192 of them, 64-row tiles for narrower weights.
// Measured on one box, linear alone, weights from HBM, register / ring 128 / ring 64 in us:
//   N = 28672, K = 8192 (224 / 448 tiles):  M = 1 31.0 / 32.4 / 41.3, M = 8 35.1 / 33.6 / 41.6, M = 16 40.4 / 35.5 / 42.7, M = 32 45.5 / 37.3 / 44.3
//   N = 14336, K = 4096 (112 / 224 tiles):  M = 1 14.0 / 15.5 / 13.8, M = 8 14.5 / 15.8 / 14.2, M = 16 17.6 / 16.4 / 13.9, M = 32 22.1 / 17.2 / 14.9
//   N = 4096, K = 14336 (32 / 64 tiles):    M = 1 15.1 / 16.8 / 16.2, M = 8 16.3 / 17.3 / 16.3, M = 16 18.7 / 17.5 / 16.9, M = 32 22.9 / 17.8 / 17.1
// Hence: with 192 tiles of 128 rows and more, 128-row tiles from M = 8 on; otherwise 64-row tiles when
// there are 192 of those, or from M = 8 on; the register kernel in the remaining cases.  A K that is no multiple of
// 256 takes the ring kernels for every M.
//
// 16-row workgroups take what they are faster at by these estimates (us, weights from HBM, fitted to 27 shapes of N = 128 to 57344,
// K = 512 to 16384 and M = 1 to 32; `million`: of weights).  They grow with M, which the ring kernels hardly notice, and a wave
// has its steps of K one after the other; the ring kernels run in whole rounds of workgroups and, like the register kernel, pay for
// a K split.  Both sides as measured (other kernel / 16 rows): M = 16, 4096 x 14336 17.8 / 11.4, 8192 x 8192 18.7 / 13.2, 10240 x 10240
// 33.5 / 23.5, 14336 x 4096 14.2 / 12.5, 28672 x 8192 33.5 / 41.0, 16384 x 16384 42.7 / 47.0; M = 32, 4096 x 14336 18.2 / 16.6, 14336 x 4096
// 14.5 / 17.7, 128 x 8192 7.8 / 9.8, 1000 x 1024 7.6 / 3.3; M = 1, 20480 x 8192 41.5 / 23.2, 28672 x 8192 29.2 / 30.0, 300 x 14336 7.8 / 8.8.
//
// The register kernel has two costs because it is planned in two ranges: below 12288 rows, K in short slices, and from 24576 rows (192
// groups of 128) on.
// `start`: what a fused call saves by quantizing the activation in these workgroups.
static bool rows16_faster(int64_t M, int64_t N, int64_t K, const SkinnyPlan &p, double start) {
  const double million = 1e-6 * (double)N * (double)K, steps = (double)ceil_div(ceil_div(K, R16_STEP), R16_WAVES);
  const double stream = M <= 16 ? 0.114 + 0.0031 * (double)M : 0.150 + 0.0023 * (double)M, chain = M <= 16 ? 0.45 + 0.007 * (double)M : 0.87;
  const double rows16 = 2.5 - start + fmax(stream * million, chain * steps);
  if (p.kind == DECODE_REGISTERS)
    return rows16 < (N >= 24576 ? 7.5 + (0.0925 + 0.0018 * (double)M) * million : 5.3 + 0.15 * million);
  if (p.split_k > 1) return rows16 < 7.6 + 0.16 * million;
  const double rounds = (double)ceil_div(p.groups, decode_cu_count());
  return rows16 < rounds * (5.0 + (p.kind == DECODE_LDS_RING ? 0.88 : 0.54) * (double)ceil_div(K, ST_BK));
}

static bool forced_decode_kernel() {
  return g_forced_decode_kernel.load(std::memory_order_relaxed) != 0 || g_forced_skinny_ks.load(std::memory_order_relaxed) != 0;
}

// Shapes whose fused call runs one launch: the activation fits into the registers and the LDS of a workgroup, and 16-row workgroups are
// faster than the other kernels with the quantizer's launch in front of these.  Every workgroup quantizes all of it, which costs the
// more beside its 16 weight rows the more rows the activation has; in a grid of two rounds and less that is hidden (us in a graph,
// two launches / one: 8 x 28672 x 2048 15.6 / 17.7, 16 x 28672 x 1024 11.5 / 14.6; 4 x 28672 x 4096 22.2 / 21.5, 8 x 6144 x 2048 8.0 / 7.3,
// 32 x 8192 x 512 6.7 / 6.1).
//
// A fused call is quantize and linear bit for bit, so a linear of these shapes sums like it.  Where linear_nvfp4_rows16_kernel is not the
// fastest for it - M = 1 or 2 on few rows of long K and on N >= 24576, K >= 8192 - the kernel of the fused call takes the quantized
// activation (`lds_x`), decodes it once a workgroup and has more weights in flight.  Linear alone, weights from HBM, one call after the other,
// register kernel / linear_nvfp4_rows16_kernel / this: 1 x 28672 x 8192 29.5 / 30.2 / 27.9 us, 2 x 28672 x 8192 30.5 / 30.8 / 28.9, 1 x 28672 x 10240
// 37.3 / 38.1 / 34.1, 1 x 24576 x 12288 37.6 / 37.9 / 33.9, 1 x 256 x 8192 6.6 / 5.8 / 5.5, 1 x 512 x 12288 7.5 / 7.6 / 6.7, 1 x 1536 x 16384 10.9 /
// 10.6 / 9.1; where linear_nvfp4_rows16_kernel is faster than the others, M above 4 or shorter K, the two are mostly alike (1 x 14336 x 4096
// 10.3 / 10.6, 16 x 4096 x 1024 3.9 / 4.0, 1 x 4096 x 14336 10.3 / 10.0).
static bool fused_rows16(int64_t M, int64_t N, int64_t K, const SkinnyPlan &p) {
  return M * K <= FUSED_ELEMS && K % SK_STEP == 0 && (M <= 4 || ceil_div(N, R16_ROWS) <= 2 * decode_cu_count()) && rows16_faster(M, N, K, p, 2.5);
}

static bool skinny_plan(int64_t M, int64_t N, int64_t K, SkinnyPlan &p) {
  if (M < 1 || M > 32 || K < SK_STEP || K % 64 != 0 || N < 1) return false;
  const bool ring_ok = (K >> 1) * ST_BN < (1ll << 31) && N < (1ll << 27);  // 32-bit lane offsets
  const bool whole = K % SK_STEP == 0;
  if (!whole && !ring_ok) return false;
  int kind = g_forced_decode_kernel.load(std::memory_order_relaxed);
  if (kind == 0 || (kind == DECODE_REGISTERS && !whole)) {
    if (!whole)
      kind = ceil_div(N, ST_BN) >= 192 ? DECODE_LDS_RING : DECODE_LDS_RING64;
    else if (ceil_div(N, ST_BN) >= 192)
      kind = M >= 8 ? DECODE_LDS_RING : DECODE_REGISTERS;
    else
      kind = (M >= 8 || ceil_div(N, S6_BN) >= 192) ? DECODE_LDS_RING64 : DECODE_REGISTERS;
  }
  if (kind == DECODE_LDS_RING64 && ring_ok)
    plan_lds_ring(M, N, K, p, S6_BN);
  else if (kind == DECODE_LDS_RING && ring_ok)
    plan_lds_ring(M, N, K, p);
  else
    plan_registers(M, N, K, p);
  // (ring_ok: 32-bit lane offsets, as in the ring kernels)
  const bool rows16_ok = !forced_decode_kernel() && ring_ok && rows16_grid_ok(N);
  p.fused = rows16_ok && fused_rows16(M, N, K, p);
  p.rows16 = rows16_ok && rows16_faster(M, N, K, p, 0.0);
  p.lds_x = p.fused && !p.rows16 && M <= 16;
  p.rows16 |= p.fused;
  return true;
}

template <int D_DT, int BIAS_DT, int MAX_IT>
static int launch_skinny_it(const SkinnyArgs &a, const SkinnyPlan &p, hipStream_t st) {
  auto *kern = linear_nvfp4_skinny_kernel<D_DT, BIAS_DT, MAX_IT>;
  static std::atomic<uint32_t> lds_ok{0};
  if (int rc = allow_dynamic_lds(kern, lds_ok, 32 * (1024 * 2 + 16))) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)p.split_k, (unsigned)p.groups), dim3(256), p.lds_bytes, st, a);
  return 0;
}

template <int D_DT, int BIAS_DT, bool PRE, int MR>
static int launch_ring(const SkinnyArgs &a, const SkinnyPlan &p, hipStream_t st) {
  const bool tail = a.K % ST_BK != 0;
  auto *kern = tail ? linear_nvfp4_stream_kernel<D_DT, BIAS_DT, PRE, MR, true> : linear_nvfp4_stream_kernel<D_DT, BIAS_DT, PRE, MR, false>;
  static std::atomic<uint32_t> lds_ok[2];
  if (int rc = allow_dynamic_lds(kern, lds_ok[tail], st_lds_bytes(MR))) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)p.groups, (unsigned)p.split_k), dim3(ST_THREADS), st_lds_bytes(MR), st, a);
  return 0;
}

template <int D_DT, int BIAS_DT>
static int launch_skinny(const SkinnyArgs &a, const SkinnyPlan &p, hipStream_t st) {
  if (p.lds_x)
    return launch_fused_rows16({a.D, nullptr, const_cast<uint8_t *>(a.Aq), const_cast<uint8_t *>(a.A_sf), const_cast<float *>(a.A_gs), a.B, a.B_sf, a.B_gs,
                                a.bias, a.M, a.N, a.K, a.Mp, a.Np}, D_DT, BIAS_DT, st);
  if (p.rows16) {
    const bool tail = a.K % R16_STEP != 0;
    auto *kern = a.M <= 16 ? tail ? linear_nvfp4_rows16_kernel<D_DT, BIAS_DT, 1, true, false> : linear_nvfp4_rows16_kernel<D_DT, BIAS_DT, 1, false, false>
                           : tail ? linear_nvfp4_rows16_kernel<D_DT, BIAS_DT, 2, true, false> : linear_nvfp4_rows16_kernel<D_DT, BIAS_DT, 2, false, false>;
    if (a.prepacked) kern = a.M <= 16 ? linear_nvfp4_rows16_kernel<D_DT, BIAS_DT, 1, false, true> : linear_nvfp4_rows16_kernel<D_DT, BIAS_DT, 2, false, true>;
    hipLaunchKernelGGL(kern, dim3((unsigned)ceil_div(a.N, R16_ROWS)), dim3(64 * R16_WAVES), 0, st, a);
    return 0;
  }
  if (p.kind == DECODE_LDS_RING) {
    int rc;
    if (a.M <= 16)
      rc = a.prepacked ? launch_ring<D_DT, BIAS_DT, true, 16>(a, p, st) : launch_ring<D_DT, BIAS_DT, false, 16>(a, p, st);
    else
      rc = a.prepacked ? launch_ring<D_DT, BIAS_DT, true, 32>(a, p, st) : launch_ring<D_DT, BIAS_DT, false, 32>(a, p, st);
    if (rc) return rc;
  } else if (p.kind == DECODE_LDS_RING64) {
    const bool tail = a.K % ST_BK != 0;
    auto *kern = tail ? linear_nvfp4_stream64_kernel<D_DT, BIAS_DT, true> : linear_nvfp4_stream64_kernel<D_DT, BIAS_DT, false>;
    static std::atomic<uint32_t> lds_ok[2];
    if (int rc = allow_dynamic_lds(kern, lds_ok[tail], S6_LDS_BYTES)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)p.groups, (unsigned)p.split_k), dim3(ST_THREADS), S6_LDS_BYTES, st, a);
  } else {
    int rc;
    if (a.M <= 8) rc = launch_skinny_it<D_DT, BIAS_DT, 1>(a, p, st);
    else if (a.M <= 16) rc = launch_skinny_it<D_DT, BIAS_DT, 2>(a, p, st);
    else rc = launch_skinny_it<D_DT, BIAS_DT, 4>(a, p, st);
    if (rc) return rc;
  }
  if (p.split_k > 1) launch_reduce<D_DT, BIAS_DT>(a, st);
  return 0;
}

template <int D_DT>
static int dispatch_skinny_bias(const SkinnyArgs &a, const SkinnyPlan &p, int bias_dtype, hipStream_t st) {
  if (!a.bias) return launch_skinny<D_DT, BIAS_NONE>(a, p, st);
  switch (bias_dtype) {
    case AC4K_DTYPE_BF16: return launch_skinny<D_DT, AC4K_DTYPE_BF16>(a, p, st);
    case AC4K_DTYPE_FP16: return launch_skinny<D_DT, AC4K_DTYPE_FP16>(a, p, st);
    case AC4K_DTYPE_FP32: return launch_skinny<D_DT, AC4K_DTYPE_FP32>(a, p, st);
  }
  return set_error("bias must be bfloat16, half or float (dtype tag %d)", bias_dtype);
}

static int dispatch_skinny(const SkinnyArgs &a, const SkinnyPlan &p, int d_dtype, int bias_dtype, hipStream_t st) {
  switch (d_dtype) {
    case AC4K_DTYPE_BF16: return dispatch_skinny_bias<AC4K_DTYPE_BF16>(a, p, bias_dtype, st);
    case AC4K_DTYPE_FP16: return dispatch_skinny_bias<AC4K_DTYPE_FP16>(a, p, bias_dtype, st);
    case AC4K_DTYPE_FP32: return dispatch_skinny_bias<AC4K_DTYPE_FP32>(a, p, bias_dtype, st);
  }
  return set_error("d must be bfloat16, half or float (dtype tag %d)", d_dtype);
}

// shapes the packed-LDS kernel takes: whole 64-chunks, 16-byte aligned rows, 32-bit lane offsets
// (256 operand rows in the loop, 4 output rows of up to 4-byte elements in the epilogue)
static bool packed_kernel_ok(const LinearArgs &a) {
  return a.K % 64 == 0 && a.K >= P_BK && (((uintptr_t)a.A | (uintptr_t)a.B) & 15) == 0 && (a.K >> 1) * 256 < (1ll << 31) &&
         a.N < (1ll << 27);
}

// Decode-sized shapes through the entry point that has no scratch: the plan of the workspace entry point
// when it needs none (one K range), otherwise the LDS-ring kernel with one K range per tile - fewer
// workgroups than the split plan, still the weights streamed once instead of the 128x128 tile kernel.
static bool noscratch_skinny_plan(const LinearArgs &a, SkinnyPlan &p) {
  if (!skinny_plan(a.M, a.N, a.K, p) || (((uintptr_t)a.A | (uintptr_t)a.B) & 15) != 0) return false;
  if (p.rows16 || p.partial_bytes == 0) return true;
  if (!((a.K >> 1) * ST_BN < (1ll << 31) && a.N < (1ll << 27))) return false;  // the ring kernels' 32-bit lane offsets
  p.kind = ceil_div(a.N, ST_BN) >= 192 ? DECODE_LDS_RING : DECODE_LDS_RING64;
  p.groups = ceil_div(a.N, p.kind == DECODE_LDS_RING ? ST_BN : S6_BN);
  p.ks_len = 0;
  p.split_k = 1;
  p.partial_bytes = 0;
  p.lds_bytes = p.kind == DECODE_LDS_RING ? st_lds_bytes(a.M <= 16 ? 16 : 32) : S6_LDS_BYTES;
  return true;
}

// Decode-sized M goes to the weight-streaming kernels, 32 < M <= 128 to the K-split-waves kernel, larger
// M to the packed-operand tile kernel, each whenever its layout conditions hold; the 128x128 kernel,
// which has no condition beyond K % 16 == 0, takes everything else.
template <int D_DT, int BIAS_DT>
static int launch_linear(const LinearArgs &a, hipStream_t st) {
  SkinnyPlan sp;
  if (noscratch_skinny_plan(a, sp)) {
    const SkinnyArgs sa{a.D, a.A, reinterpret_cast<const uint8_t *>(a.A_sf), a.Mp, a.B, a.B_sf, a.A_gs, a.B_gs, a.bias, nullptr,
                        a.M, a.N, a.K, a.Np, sp.ks_len, sp.split_k};
    return launch_skinny<D_DT, BIAS_DT>(sa, sp, st);
  }
  if (ksplit_shape(a.M, a.N, a.K) && ksplit_aligned(a))  // all of M in one tile, one K range (no scratch here)
    return launch_ksplit<D_DT, BIAS_DT>(a, ksplit_plan(a.M, a.N, a.K, false), SplitK{nullptr, 1}, st);
  if (a.M > 32 && a.N >= 128 && packed_kernel_ok(a)) return launch_tile256p<D_DT, BIAS_DT>(a, st);
  const int64_t ntiles = ceil_div(a.M, T_BM) * ceil_div(a.N, T_BN);
  hipLaunchKernelGGL((linear_nvfp4_tile128_kernel<D_DT, BIAS_DT>), dim3((unsigned)ntiles), dim3(256), 0, st, a);
  return 0;
}

template <int D_DT>
static int dispatch_bias(const LinearArgs &a, int bias_dtype, hipStream_t st) {
  if (!a.bias) return launch_linear<D_DT, BIAS_NONE>(a, st);
  switch (bias_dtype) {
    case AC4K_DTYPE_BF16: return launch_linear<D_DT, AC4K_DTYPE_BF16>(a, st);
    case AC4K_DTYPE_FP16: return launch_linear<D_DT, AC4K_DTYPE_FP16>(a, st);
    case AC4K_DTYPE_FP32: return launch_linear<D_DT, AC4K_DTYPE_FP32>(a, st);
  }
  return set_error("bias must be bfloat16, half or float (dtype tag %d)", bias_dtype);
}

}  // namespace ac4k

using namespace ac4k;

extern "C" __attribute__((visibility("default"))) int ac4k_linear_nvfp4(void *D, int d_dtype, const void *A, const void *A_sf, const float *A_gs,
                                 const void *B, const void *B_sf, const float *B_gs, const void *bias,
                                 int bias_dtype, int64_t M, int64_t N, int64_t K, ac4k_stream_t stream) {
  AC4K_REQUIRE(D && A && A_sf && A_gs && B && B_sf && B_gs, "null pointer argument");
  AC4K_REQUIRE(M >= 1 && N >= 1 && K >= 1, "M, N, K must be positive (M=%lld N=%lld K=%lld)", (long long)M,
               (long long)N, (long long)K);
  AC4K_REQUIRE(K % 16 == 0, "A size(1)*2 must be multiple of 16 but see %lld", (long long)K);
  AC4K_REQUIRE(((uintptr_t)A & 7) == 0 && ((uintptr_t)B & 7) == 0 && ((uintptr_t)A_sf & 3) == 0 &&
                   ((uintptr_t)B_sf & 3) == 0,
               "A/B must be 8-byte aligned and the scale tensors 4-byte aligned");
  AC4K_REQUIRE(ceil_div(M, T_BM) * ceil_div(N, T_BN) < (1ll << 31), "problem too large");
  LinearArgs a{D,
               static_cast<const uint8_t *>(A),
               static_cast<const uint8_t *>(B),
               static_cast<const uint32_t *>(A_sf),
               static_cast<const uint32_t *>(B_sf),
               A_gs,
               B_gs,
               bias,
               M,
               N,
               K,
               align_up(M, 16),
               align_up(N, 16)};
  hipStream_t st = (hipStream_t)stream;
  int rc;
  switch (d_dtype) {
    case AC4K_DTYPE_BF16: rc = dispatch_bias<AC4K_DTYPE_BF16>(a, bias_dtype, st); break;
    case AC4K_DTYPE_FP16: rc = dispatch_bias<AC4K_DTYPE_FP16>(a, bias_dtype, st); break;
    case AC4K_DTYPE_FP32: rc = dispatch_bias<AC4K_DTYPE_FP32>(a, bias_dtype, st); break;
    default: return set_error("d must be bfloat16, half or float (dtype tag %d)", d_dtype);
  }
  if (rc) return rc;
  return check_launch("ac4k_linear_nvfp4");
}

namespace ac4k {

// Split-K for problems with too few output tiles to fill the GPU (32 < M, few tiles, long K): the
// K-split-waves kernel (M <= 128) or the packed-LDS tile kernel runs `splits` K ranges per tile into
// fp32 partial buffers in the workspace and skinny_reduce_kernel adds them.
struct MidPlan {
  bool has_ksplit;   // the shape suits the K-split-waves kernel (taken when the pointers are aligned for it)
  KsplitPlan kp;
  TilePlan tp;       // the plan of the tile kernel where the shape does not
  int64_t bytes;     // scratch that the entry points ask for
};
// shapes the workspace entry point takes with 32 < M
static bool mid_plan(int64_t M, int64_t N, int64_t K, MidPlan &p) {
  if (M <= 32 || N < 128 || K % 64 != 0 || K < P_BK || (K >> 1) * 256 >= (1ll << 31) || N >= (1ll << 27)) return false;
  p.has_ksplit = ksplit_shape(M, N, K);
  if (p.has_ksplit) {
    p.kp = ksplit_plan(M, N, K, true);
    p.bytes = p.kp.partial_bytes;
    return true;
  }
  p.bytes = tile_scratch_bytes(M, N, K);
  if (p.bytes > 0) p.tp = tile_plan(M, N, K, p.bytes);
  return p.bytes > 0;
}

// `partial_bytes` of scratch at `partial` (possibly none): the K-split-waves kernel when the shape and the
// pointers suit it, else the tile kernel, split along K when the scratch holds its partial sums
template <int D_DT, int BIAS_DT>
static int launch_mid(const LinearArgs &a, const MidPlan &p, float *partial, int64_t partial_bytes, hipStream_t st) {
  int splits;
  if (p.has_ksplit && ksplit_aligned(a)) {
    splits = p.kp.splits;
    if (int rc = launch_ksplit<D_DT, BIAS_DT>(a, p.kp, SplitK{splits > 1 ? partial : nullptr, splits}, st)) return rc;
  } else {
    TilePlan tp = p.has_ksplit ? tile_plan(a.M, a.N, a.K, tile_scratch_bytes(a.M, a.N, a.K)) : p.tp;
    if (tp.partial_bytes > partial_bytes) tp = tile_plan(a.M, a.N, a.K, 0);
    splits = tp.splits;
    if (int rc = launch_tile_plan<D_DT, BIAS_DT>(a, tp, SplitK{splits > 1 ? partial : nullptr, splits}, st)) return rc;
  }
  if (splits > 1) {
    SkinnyArgs r{a.D, nullptr, nullptr, 0, nullptr, nullptr, a.A_gs, a.B_gs, a.bias, partial, a.M, a.N, a.K, a.Np, 0, splits};
    launch_reduce<D_DT, BIAS_DT>(r, st);
  }
  return 0;
}

template <int D_DT>
static int dispatch_mid_bias(const LinearArgs &a, const MidPlan &p, float *partial, int64_t partial_bytes, int bias_dtype,
                             hipStream_t st) {
  if (!a.bias) return launch_mid<D_DT, BIAS_NONE>(a, p, partial, partial_bytes, st);
  switch (bias_dtype) {
    case AC4K_DTYPE_BF16: return launch_mid<D_DT, AC4K_DTYPE_BF16>(a, p, partial, partial_bytes, st);
    case AC4K_DTYPE_FP16: return launch_mid<D_DT, AC4K_DTYPE_FP16>(a, p, partial, partial_bytes, st);
    case AC4K_DTYPE_FP32: return launch_mid<D_DT, AC4K_DTYPE_FP32>(a, p, partial, partial_bytes, st);
  }
  return set_error("bias must be bfloat16, half or float (dtype tag %d)", bias_dtype);
}

static int dispatch_mid(const LinearArgs &a, const MidPlan &p, float *partial, int64_t partial_bytes, int d_dtype,
                        int bias_dtype, hipStream_t st) {
  switch (d_dtype) {
    case AC4K_DTYPE_BF16: return dispatch_mid_bias<AC4K_DTYPE_BF16>(a, p, partial, partial_bytes, bias_dtype, st);
    case AC4K_DTYPE_FP16: return dispatch_mid_bias<AC4K_DTYPE_FP16>(a, p, partial, partial_bytes, bias_dtype, st);
    case AC4K_DTYPE_FP32: return dispatch_mid_bias<AC4K_DTYPE_FP32>(a, p, partial, partial_bytes, bias_dtype, st);
  }
  return set_error("d must be bfloat16, half or float (dtype tag %d)", d_dtype);
}

// one K range of the tile kernel with a given plan (the entry point of the weight image)
template <int D_DT>
static int dispatch_prepacked_bias(const LinearArgs &a, const TilePlan &p, int bias_dtype, hipStream_t st) {
  const SplitK one{nullptr, 1};
  if (!a.bias) return launch_tile_plan<D_DT, BIAS_NONE>(a, p, one, st);
  switch (bias_dtype) {
    case AC4K_DTYPE_BF16: return launch_tile_plan<D_DT, AC4K_DTYPE_BF16>(a, p, one, st);
    case AC4K_DTYPE_FP16: return launch_tile_plan<D_DT, AC4K_DTYPE_FP16>(a, p, one, st);
    case AC4K_DTYPE_FP32: return launch_tile_plan<D_DT, AC4K_DTYPE_FP32>(a, p, one, st);
  }
  return set_error("bias must be bfloat16, half or float (dtype tag %d)", bias_dtype);
}

// shared tail of the two decode-sized entry points: packed activation in, partial sums in the workspace
static int run_skinny(void *D, int d_dtype, const void *Aq, const void *A_sf, const float *A_gs, const void *B,
                      const void *B_sf, const float *B_gs, const void *bias, int bias_dtype, int64_t M, int64_t N,
                      int64_t K, const SkinnyPlan &p, void *workspace, hipStream_t st) {
  SkinnyArgs a{D,
               static_cast<const uint8_t *>(Aq),
               static_cast<const uint8_t *>(A_sf),
               align_up(M, 16),
               static_cast<const uint8_t *>(B),
               static_cast<const uint32_t *>(B_sf),
               A_gs,
               B_gs,
               bias,
               static_cast<float *>(workspace),
               M,
               N,
               K,
               align_up(N, 16),
               p.ks_len,
               p.split_k};
  return dispatch_skinny(a, p, d_dtype, bias_dtype, st);
}

static int check_skinny(const SkinnyPlan &p, bool ok, const void *B, void *workspace, int64_t workspace_bytes) {
  AC4K_REQUIRE(ok, "no workspace-assisted path for this shape: decode-sized shapes need 1 <= M <= 32 and K a multiple of 256");
  AC4K_REQUIRE(((uintptr_t)B & 15) == 0, "weights must be 16-byte aligned");
  if (p.partial_bytes > 0) {  // one K range per tile needs no scratch
    AC4K_REQUIRE(workspace && ((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
    AC4K_REQUIRE(workspace_bytes >= p.partial_bytes, "workspace too small: %lld bytes needed", (long long)p.partial_bytes);
  }
  return 0;
}

}  // namespace ac4k

extern "C" __attribute__((visibility("default"))) int64_t ac4k_linear_nvfp4_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  SkinnyPlan p;
  if (skinny_plan(M, N, K, p)) return p.partial_bytes;
  MidPlan mp;
  if (mid_plan(M, N, K, mp)) return mp.bytes;
  return 0;
}

extern "C" __attribute__((visibility("default"))) int64_t ac4k_linear_nvfp4_scratch_bytes(int64_t M, int64_t N, int64_t K) {
  SkinnyPlan p;
  if (skinny_plan(M, N, K, p)) return p.rows16 ? 0 : p.partial_bytes;
  MidPlan mp;
  if (mid_plan(M, N, K, mp)) return mp.has_ksplit || mp.tp.splits > 1 ? mp.bytes : 0;
  return 0;
}

namespace ac4k {

// K that the `skinny` entry points take: whole stages of the kernels they began with
static bool skinny_entry_k(int64_t M, int64_t K) { return K % (M > 32 ? P_BK : SK_STEP) == 0; }

}  // namespace ac4k

extern "C" __attribute__((visibility("default"))) int ac4k_debug_linear_decode_kernel(int64_t M, int64_t N, int64_t K, int *fused_launches) {
  SkinnyPlan p;
  const bool ok = skinny_plan(M, N, K, p);
  if (fused_launches) *fused_launches = !ok || !skinny_entry_k(M, K) ? 0 : p.fused ? 1 : p.rows16 || p.split_k == 1 ? 2 : 3;
  return !ok ? 0 : p.lds_x ? DECODE_ROWS16_LDS : p.rows16 ? DECODE_ROWS16 : p.kind;
}

extern "C" __attribute__((visibility("default"))) int64_t ac4k_linear_nvfp4_skinny_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  return skinny_entry_k(M, K) ? ac4k_linear_nvfp4_workspace_bytes(M, N, K) : 0;
}

namespace ac4k {

// body of the two workspace-assisted entry points (caller's workspace / the library's static array)
static int linear_skinny_impl(void *D, int d_dtype, const void *A, const void *A_sf, const float *A_gs, const void *B,
                              const void *B_sf, const float *B_gs, const void *bias, int bias_dtype, int64_t M,
                              int64_t N, int64_t K, void *workspace, int64_t workspace_bytes, hipStream_t st,
                              const char *what) {
  AC4K_REQUIRE(D && A && A_sf && A_gs && B && B_sf && B_gs, "null pointer argument");
  AC4K_REQUIRE(M >= 1 && N >= 1 && K >= 1, "M, N, K must be positive (M=%lld N=%lld K=%lld)", (long long)M,
               (long long)N, (long long)K);
  MidPlan mp;
  if (M > 32 && skinny_entry_k(M, K) && mid_plan(M, N, K, mp)) {  // few tiles, long K: split-K
    AC4K_REQUIRE((((uintptr_t)A | (uintptr_t)B) & 15) == 0 && (((uintptr_t)A_sf | (uintptr_t)B_sf) & 3) == 0,
                 "A and B must be 16-byte aligned and the scale tensors 4-byte aligned");
    if (mp.bytes > 0) {  // one K range per tile needs no scratch
      AC4K_REQUIRE(workspace && ((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
      AC4K_REQUIRE(workspace_bytes >= mp.bytes, "workspace too small: %lld bytes needed", (long long)mp.bytes);
    }
    LinearArgs la{D, static_cast<const uint8_t *>(A), static_cast<const uint8_t *>(B),
                  static_cast<const uint32_t *>(A_sf), static_cast<const uint32_t *>(B_sf), A_gs, B_gs, bias,
                  M, N, K, align_up(M, 16), align_up(N, 16)};
    if (int rc = dispatch_mid(la, mp, static_cast<float *>(workspace), workspace ? workspace_bytes : 0, d_dtype, bias_dtype, st))
      return rc;
    return check_launch(what);
  }
  SkinnyPlan p;
  const bool ok = skinny_entry_k(M, K) && skinny_plan(M, N, K, p);
  if (int rc = check_skinny(p, ok, B, workspace, workspace_bytes)) return rc;
  AC4K_REQUIRE(((uintptr_t)A & 15) == 0, "A must be 16-byte aligned");
  if (int rc = run_skinny(D, d_dtype, A, A_sf, A_gs, B, B_sf, B_gs, bias, bias_dtype, M, N, K, p, workspace, st))
    return rc;
  return check_launch(what);
}

// ---------------------------------------------------------------------------
// Scratch of the entry point that allocates nothing: one array per GPU, held until the process ends.
// In host code the array's name is only a handle: its device address comes from hipGetSymbolAddress,
// once per device with that device current, and that pointer is what the kernels are given.
// ---------------------------------------------------------------------------
constexpr int64_t STATIC_SCRATCH_BYTES = AC4K_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];

static int static_scratch(void **ptr_out) {
  constexpr int MAX_DEV = 64;
  static void *ptrs[MAX_DEV] = {};
  static std::mutex mu;
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return set_error("hipGetDevice: %s", hipGetErrorString(e));
  AC4K_REQUIRE(dev >= 0 && dev < MAX_DEV, "device index %d out of range", dev);
  std::lock_guard<std::mutex> lock(mu);
  if (!ptrs[dev]) {
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p) return set_error("hipGetSymbolAddress(scratch): %s", hipGetErrorString(e));
    ptrs[dev] = p;
  }
  *ptr_out = ptrs[dev];
  return 0;
}

}  // namespace ac4k

extern "C" __attribute__((visibility("default"))) int ac4k_linear_nvfp4_skinny(void *D, int d_dtype, const void *A, const void *A_sf, const float *A_gs,
                                        const void *B, const void *B_sf, const float *B_gs, const void *bias,
                                        int bias_dtype, int64_t M, int64_t N, int64_t K, void *workspace,
                                        int64_t workspace_bytes, ac4k_stream_t stream) {
  return linear_skinny_impl(D, d_dtype, A, A_sf, A_gs, B, B_sf, B_gs, bias, bias_dtype, M, N, K, workspace,
                            workspace_bytes, (hipStream_t)stream, "ac4k_linear_nvfp4_skinny");
}

extern "C" __attribute__((visibility("default"))) int ac4k_linear_nvfp4_workspace(void *D, int d_dtype, const void *A, const void *A_sf, const float *A_gs,
                                        const void *B, const void *B_sf, const float *B_gs, const void *bias,
                                        int bias_dtype, int64_t M, int64_t N, int64_t K, void *workspace,
                                        int64_t workspace_bytes, ac4k_stream_t stream) {
  // what the kernels that split K do not take runs without scratch, for every K alike: shapes that need none, operands that
  // are not aligned for them, and everything that ac4k_linear_nvfp4 refuses with its own message
  SkinnyPlan p;
  MidPlan mp;
  const bool aligned = D && A && A_sf && A_gs && B && B_sf && B_gs && (((uintptr_t)A | (uintptr_t)B) & 15) == 0 &&
                       (((uintptr_t)A_sf | (uintptr_t)B_sf) & 3) == 0;
  const bool skinny = aligned && skinny_plan(M, N, K, p);
  const bool mid = aligned && !skinny && mid_plan(M, N, K, mp);
  const int64_t need = skinny ? p.partial_bytes : mid ? mp.bytes : 0;
  if (need == 0) return ac4k_linear_nvfp4(D, d_dtype, A, A_sf, A_gs, B, B_sf, B_gs, bias, bias_dtype, M, N, K, stream);
  AC4K_REQUIRE(workspace && ((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
  AC4K_REQUIRE(workspace_bytes >= need, "workspace too small: %lld bytes needed", (long long)need);
  int rc;
  if (skinny) {
    rc = run_skinny(D, d_dtype, A, A_sf, A_gs, B, B_sf, B_gs, bias, bias_dtype, M, N, K, p, workspace, (hipStream_t)stream);
  } else {
    LinearArgs la{D, static_cast<const uint8_t *>(A), static_cast<const uint8_t *>(B),
                  static_cast<const uint32_t *>(A_sf), static_cast<const uint32_t *>(B_sf), A_gs, B_gs, bias,
                  M, N, K, align_up(M, 16), align_up(N, 16)};
    rc = dispatch_mid(la, mp, static_cast<float *>(workspace), workspace_bytes, d_dtype, bias_dtype, (hipStream_t)stream);
  }
  if (rc) return rc;
  return check_launch("ac4k_linear_nvfp4_workspace");
}

extern "C" __attribute__((visibility("default"))) int ac4k_linear_nvfp4_skinny_static(void *D, int d_dtype, const void *A, const void *A_sf,
                                               const float *A_gs, const void *B, const void *B_sf,
                                               const float *B_gs, const void *bias, int bias_dtype, int64_t M,
                                               int64_t N, int64_t K, ac4k_stream_t stream) {
  AC4K_REQUIRE(M >= 1 && N >= 1 && K >= 1, "M, N, K must be positive (M=%lld N=%lld K=%lld)", (long long)M,
               (long long)N, (long long)K);
  const int64_t need = ac4k_linear_nvfp4_skinny_workspace_bytes(M, N, K);
  AC4K_REQUIRE(need <= STATIC_SCRATCH_BYTES,
               "shape needs %lld bytes of scratch, the static scratch holds %lld: use ac4k_linear_nvfp4_skinny with a "
               "workspace of the caller",
               (long long)need, (long long)STATIC_SCRATCH_BYTES);
  void *ws = nullptr;
  if (int rc = static_scratch(&ws)) return rc;
  // the partial sums are written before they are read: nothing in the array has to start at zero
  return linear_skinny_impl(D, d_dtype, A, A_sf, A_gs, B, B_sf, B_gs, bias, bias_dtype, M, N, K, ws,
                            STATIC_SCRATCH_BYTES, (hipStream_t)stream, "ac4k_linear_nvfp4_skinny_static");
}

namespace ac4k {

// One workgroup writes one block of the weight image: 128 rows x 64 packed bytes (rows past N zero),
// piece p of row r at position p ^ ((r >> 1) & 3), then the scale dwords [2 chunks][128 rows].
__global__ __launch_bounds__(256) void prepack_weight_kernel(uint8_t *image, const uint8_t *B, const uint32_t *B_sf,
                                                             int64_t N, int64_t K, int64_t Np) {
  const int64_t kt = blockIdx.x, band = blockIdx.y;
  uint8_t *blk = image + (band * gridDim.x + kt) * W_BLOCK_BYTES;
  const int t = threadIdx.x;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = (t + i * 256) >> 2, pc = t & 3;
    const int64_t row = band * W_BLOCK_ROWS + r;
    uint4 v = make_uint4(0, 0, 0, 0);
    if (row < N) v = *reinterpret_cast<const uint4 *>(B + row * (K >> 1) + kt * (W_BLOCK_K / 2) + pc * 16);
    *reinterpret_cast<uint4 *>(blk + r * (W_BLOCK_K / 2) + ((pc ^ ((r >> 1) & 3)) * 16)) = v;
  }
  const int c = t >> 7, r = t & 127;
  const int64_t row = band * W_BLOCK_ROWS + r;
  reinterpret_cast<uint32_t *>(blk + W_BLOCK_DATA)[c * W_BLOCK_ROWS + r] = row < N ? B_sf[(kt * 2 + c) * Np + row] : 0u;
}

static int64_t weight_image_bytes(int64_t N, int64_t K) {
  if (N < 1 || K < W_BLOCK_K || K % W_BLOCK_K != 0) return 0;
  return ceil_div(N, W_BLOCK_ROWS) * (K / W_BLOCK_K) * W_BLOCK_BYTES;
}

// How a linear on a weight image runs: the LDS-ring kernel or 16-row workgroups for decode-sized M (K >= 256), the K-split-waves
// kernel for 32 < M <= 128, the tile kernel otherwise, split along K when the workspace entry point of the plain
// layout would split too.
struct PrepackedPlan {
  bool ring, mid;
  SkinnyPlan sp;
  KsplitPlan kp;
  TilePlan tp;
  int64_t partial_bytes;
};
// 16-row workgroups on an image, where a step of a wave's rows is one run of a kilobyte, against its ring kernel, by these estimates (us,
// weights from HBM, fitted to 160 shapes of N = 256 to 28672, K = 256 to 16384 and M = 1 to 32).  Ring / 16 rows as measured:
// M = 1, 4096 x 4096 10.5 / 4.3, 28672 x 8192 32.3 / 28.1; M = 8, 28672 x 8192 32.5 / 31.2; M = 16, 4096 x 14336 18.1 / 10.1, 14336 x 4096 16.1 / 10.9,
// 28672 x 8192 33.0 / 35.0, 27264 x 256 5.3 / 4.7; M = 20, 12288 x 12288 39.5 / 30.6, 27264 x 256 5.4 / 6.9, 28672 x 4096 21.0 / 24.1; M = 32,
// 4096 x 14336 17.8 / 14.8, 2688 x 14208 14.8 / 11.8, 14336 x 14336 33.5 / 47.6, 256 x 14336 10.4 / 12.4.
// Two tiles of activation rows (M > 16): two workgroups on a CU have their steps nearly one after the other (24 x 4096 x 8192 8.8 us, 4112 rows 13.3), and
// the estimates have to differ by more than they err: of 423 shapes of M = 17 to 32 383 take 16 rows, four of these 3 to
// 5 % slower than the ring (394 and 13 by 2 to 18 % without the two: 31 x 320 x 14080 10.7 / 12.7, 29 x 22656 x 512 6.7 / 7.7).
static bool rows16_faster_image(int64_t M, int64_t N, int64_t K, const SkinnyPlan &p) {
  const double m = (double)M, cus = (double)decode_cu_count(), million = 1e-6 * (double)N * (double)K;
  const double steps = (double)ceil_div(ceil_div(K, R16_STEP), R16_WAVES), wgs = (double)ceil_div(N, R16_ROWS) / (2.0 * cus);
  const double last = wgs > 1.0 && wgs < 2.0 ? sqrt(2.0 / wgs) : 1.0;  // a second round that is not full
  const double rows16 = M <= 16 ? fmax(0.35 * wgs + (0.10 + 0.0022 * m) * million, (0.37 + 0.003 * m) * steps)
                                : fmax(last * (wgs + (0.126 + 0.0016 * m) * million), (wgs > 0.5 ? 1.8 : 1.0) * (0.5 + 0.006 * m) * steps);
  const double rounds = ceil((double)(p.groups * p.split_k) / cus), stages = (double)ceil_div(ceil_div(K, ST_BK), p.split_k);
  const double ring = 4.2 + 0.03 * m + 0.8 * stages + 0.3 * fmin(stages, 8.0);
  return (M <= 16 ? 1.0 : 1.1) * (2.5 + rows16) < rounds * ring + (p.split_k > 1 ? 4.0 : 0.0);
}

static bool prepacked_plan(int64_t M, int64_t N, int64_t K, PrepackedPlan &p) {
  const int64_t bytes = weight_image_bytes(N, K);
  if (M < 1 || bytes == 0 || bytes >= (1ll << 32) || (K >> 1) * 256 >= (1ll << 31) || N >= (1ll << 27)) return false;
  p.ring = M <= 32 && K >= ST_BK;
  p.mid = !p.ring && ksplit_shape(M, N, K);
  if (p.ring) {
    plan_lds_ring(M, N, K, p.sp);
    p.sp.rows16 = !forced_decode_kernel() && rows16_faster_image(M, N, K, p.sp);
    p.sp.fused = p.sp.lds_x = false;
    p.partial_bytes = p.sp.rows16 ? 0 : p.sp.partial_bytes;
  } else if (p.mid) {
    p.kp = ksplit_plan(M, N, K, true);
    p.partial_bytes = p.kp.partial_bytes;
  } else {
    p.partial_bytes = tile_scratch_bytes(M, N, K);
    p.tp = tile_plan(M, N, K, p.partial_bytes);
  }
  return true;
}

}  // namespace ac4k

extern "C" __attribute__((visibility("default"))) int64_t ac4k_prepack_weight_nvfp4_bytes(int64_t N, int64_t K) {
  const int64_t bytes = weight_image_bytes(N, K);
  return bytes < (1ll << 32) ? bytes : 0;
}

extern "C" __attribute__((visibility("default"))) int ac4k_prepack_weight_nvfp4(void *image, const void *B, const void *B_sf, int64_t N, int64_t K,
                                                                                ac4k_stream_t stream) {
  AC4K_REQUIRE(image && B && B_sf, "null pointer argument");
  const int64_t bytes = ac4k_prepack_weight_nvfp4_bytes(N, K);
  AC4K_REQUIRE(bytes > 0, "no weight image for N = %lld, K = %lld: K must be a multiple of 128 and the image smaller than 4 GiB",
               (long long)N, (long long)K);
  AC4K_REQUIRE((((uintptr_t)image | (uintptr_t)B) & 15) == 0 && ((uintptr_t)B_sf & 3) == 0,
               "image and B must be 16-byte aligned, B_sf 4-byte aligned");
  hipLaunchKernelGGL(prepack_weight_kernel, dim3((unsigned)(K / W_BLOCK_K), (unsigned)ceil_div(N, W_BLOCK_ROWS)), dim3(256), 0,
                     (hipStream_t)stream, static_cast<uint8_t *>(image), static_cast<const uint8_t *>(B),
                     static_cast<const uint32_t *>(B_sf), N, K, align_up(N, 16));
  return check_launch("ac4k_prepack_weight_nvfp4");
}

extern "C" __attribute__((visibility("default"))) int64_t ac4k_linear_nvfp4_prepacked_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  PrepackedPlan p;
  return prepacked_plan(M, N, K, p) ? p.partial_bytes : 0;
}

extern "C" __attribute__((visibility("default"))) int ac4k_debug_linear_prepacked_decode_kernel(int64_t M, int64_t N, int64_t K) {
  PrepackedPlan p;
  if (!prepacked_plan(M, N, K, p) || !p.ring) return 0;
  return p.sp.rows16 ? DECODE_ROWS16 : DECODE_LDS_RING;
}

extern "C" __attribute__((visibility("default"))) int ac4k_linear_nvfp4_prepacked(void *D, int d_dtype, const void *A, const void *A_sf, const float *A_gs,
                                                                                  const void *W_image, const float *B_gs, const void *bias,
                                                                                  int bias_dtype, int64_t M, int64_t N, int64_t K, void *workspace,
                                                                                  int64_t workspace_bytes, ac4k_stream_t stream) {
  AC4K_REQUIRE(D && A && A_sf && A_gs && W_image && B_gs, "null pointer argument");
  AC4K_REQUIRE(M >= 1 && N >= 1, "M and N must be positive (M = %lld, N = %lld)", (long long)M, (long long)N);
  PrepackedPlan p;
  AC4K_REQUIRE(prepacked_plan(M, N, K, p), "no weight image for N = %lld, K = %lld (ac4k_prepack_weight_nvfp4_bytes returns 0)",
               (long long)N, (long long)K);
  AC4K_REQUIRE((((uintptr_t)A | (uintptr_t)W_image) & 15) == 0 && ((uintptr_t)A_sf & 3) == 0,
               "A and the weight image must be 16-byte aligned, A_sf 4-byte aligned");
  AC4K_REQUIRE(ceil_div(M, 128) * ceil_div(N, 64) < (1ll << 31), "problem too large");
  if (p.partial_bytes > 0) {
    AC4K_REQUIRE(workspace && ((uintptr_t)workspace & 255) == 0, "workspace must be 256-byte aligned");
    AC4K_REQUIRE(workspace_bytes >= p.partial_bytes, "workspace too small: %lld bytes needed", (long long)p.partial_bytes);
  }
  hipStream_t st = (hipStream_t)stream;
  if (p.ring) {
    SkinnyArgs a{D, static_cast<const uint8_t *>(A), static_cast<const uint8_t *>(A_sf), align_up(M, 16),
                 static_cast<const uint8_t *>(W_image), nullptr, A_gs, B_gs, bias, static_cast<float *>(workspace),
                 M, N, K, align_up(N, 16), 0, p.sp.split_k, 1};
    if (int rc = dispatch_skinny(a, p.sp, d_dtype, bias_dtype, st)) return rc;
    return check_launch("ac4k_linear_nvfp4_prepacked");
  }
  LinearArgs la{D, static_cast<const uint8_t *>(A), static_cast<const uint8_t *>(W_image),
                static_cast<const uint32_t *>(A_sf), nullptr, A_gs, B_gs, bias,
                M, N, K, align_up(M, 16), align_up(N, 16), 1};
  int rc;
  if (p.mid || p.tp.splits > 1) {
    rc = dispatch_mid(la, MidPlan{p.mid, p.mid ? p.kp : KsplitPlan{0, 0, 1, 0}, p.tp, p.partial_bytes},
                      static_cast<float *>(workspace), workspace_bytes, d_dtype, bias_dtype, st);
  } else {
    switch (d_dtype) {
      case AC4K_DTYPE_BF16: rc = dispatch_prepacked_bias<AC4K_DTYPE_BF16>(la, p.tp, bias_dtype, st); break;
      case AC4K_DTYPE_FP16: rc = dispatch_prepacked_bias<AC4K_DTYPE_FP16>(la, p.tp, bias_dtype, st); break;
      case AC4K_DTYPE_FP32: rc = dispatch_prepacked_bias<AC4K_DTYPE_FP32>(la, p.tp, bias_dtype, st); break;
      default: return set_error("d must be bfloat16, half or float (dtype tag %d)", d_dtype);
    }
  }
  if (rc) return rc;
  return check_launch("ac4k_linear_nvfp4_prepacked");
}

namespace ac4k {

static bool overlap(const void *a, int64_t a_bytes, const void *b, int64_t b_bytes) {
  return (uintptr_t)a < (uintptr_t)b + (uintptr_t)b_bytes && (uintptr_t)b < (uintptr_t)a + (uintptr_t)a_bytes;
}

}  // namespace ac4k

extern "C" __attribute__((visibility("default"))) int ac4k_linear_nvfp4_fused_bf16(void *D, int d_dtype, const void *X, void *X_q, void *X_sf,
                                            float *X_gs, const void *B, const void *B_sf, const float *B_gs,
                                            const void *bias, int bias_dtype, int64_t M, int64_t N, int64_t K,
                                            void *workspace, int64_t workspace_bytes, ac4k_stream_t stream) {
  AC4K_REQUIRE(D && X && X_q && X_sf && X_gs && B && B_sf && B_gs, "null pointer argument");
  AC4K_REQUIRE(M >= 1 && M <= 32, "the fused skinny linear takes 1 <= M <= 32 (got %lld)", (long long)M);
  AC4K_REQUIRE(N >= 1 && K >= 1, "N and K must be positive (N=%lld K=%lld)", (long long)N, (long long)K);
  SkinnyPlan p;
  const bool ok = skinny_entry_k(M, K) && skinny_plan(M, N, K, p);
  if (int rc = check_skinny(p, ok, B, workspace, workspace_bytes)) return rc;
  hipStream_t st = (hipStream_t)stream;
  AC4K_REQUIRE(((uintptr_t)X & 15) == 0, "activation must be 16-byte aligned");
  // (one launch reads X to its end while it stores: outputs over X, as in a linear in place, need the order of two)
  if (p.fused && (((uintptr_t)X_q | (uintptr_t)B) & 15) == 0 && (((uintptr_t)X_sf | (uintptr_t)B_sf) & 3) == 0 &&
      !overlap(X, M * K * 2, D, M * N * (d_dtype == AC4K_DTYPE_FP32 ? 4 : 2)) && !overlap(X, M * K * 2, X_q, M * K / 2) &&
      !overlap(X, M * K * 2, X_sf, K / 64 * align_up(M, 16) * 4) && !overlap(X, M * K * 2, X_gs, 4)) {
    const FusedArgs a{D, static_cast<const uint16_t *>(X), static_cast<uint8_t *>(X_q), static_cast<uint8_t *>(X_sf), X_gs,
                      static_cast<const uint8_t *>(B), static_cast<const uint32_t *>(B_sf), B_gs, bias, M, N, K, align_up(M, 16), align_up(N, 16)};
    if (int rc = launch_fused_rows16(a, d_dtype, bias_dtype, st)) return rc;
    return check_launch("ac4k_linear_nvfp4_fused_bf16");
  }
  if (int rc = ac4k_quantize_nvfp4_bf16(X_q, X_sf, X_gs, X, 1, 1, M, K, 0, 0, K, 1, 0, 2688.0f, stream)) return rc;
  if (int rc = run_skinny(D, d_dtype, X_q, X_sf, X_gs, B, B_sf, B_gs, bias, bias_dtype, M, N, K, p, workspace,
                          st))
    return rc;
  return check_launch("ac4k_linear_nvfp4_fused_bf16");
}

extern "C" __attribute__((visibility("default"))) int ac4k_set_linear_tuning(int mi, int nj, int splits, int skinny_ks,
                                                                          int decode_kernel) {
  // every argument is checked before any is stored: a rejected call changes nothing
  AC4K_REQUIRE(decode_kernel >= 0 && decode_kernel <= 3,
               "decode_kernel must be 0 (by shape), 1 (register kernel), 2 (LDS-ring kernel) or 3 (LDS-ring kernel with "
               "64-row tiles) (got %d)", decode_kernel);
  const bool no_plan = mi == 0 && nj == 0 && splits == 0;
  AC4K_REQUIRE(no_plan || (mi >= 2 && mi <= 4 && (nj == 1 || nj == 2 || nj == 4) && !(mi != 2 && nj == 1) && splits >= 1 &&
                           splits <= 0xffff),
               "tile plan must be mi in {2,3,4}, nj in {1,2,4} (1 with mi = 2), 1 <= splits (got %d,%d,%d)", mi, nj, splits);
  AC4K_REQUIRE(skinny_ks >= 0 && skinny_ks % 256 == 0, "skinny_ks must be 0 (automatic) or a multiple of 256 (got %d)",
               skinny_ks);
  ac4k::g_forced_decode_kernel.store(decode_kernel);
  ac4k::g_forced_tile_plan.store(no_plan ? 0u : (uint32_t)mi | ((uint32_t)nj << 8) | ((uint32_t)splits << 16));
  ac4k::g_forced_skinny_ks.store(skinny_ks);
  return 0;
}

#ifdef AC4K_LINEAR_TIMELINE
// Timeline build only: copies the per-workgroup stamps of the last tile / K-split-waves launch to host
// memory ([8192][6]: 100 MHz ticks at kernel entry, loop entry, loop exit, kernel exit; shader cycles in
// the loop; XCC and hardware id for the tile kernel).  Synchronises the device.
extern "C" __attribute__((visibility("default"))) int ac4k_debug_linear_timeline(uint64_t *host_out) {
  hipError_t e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpyFromSymbol(host_out, HIP_SYMBOL(ac4k::g_linear_timeline), sizeof(uint64_t) * 8192 * 6);
  return e == hipSuccess ? 0 : ac4k::set_error("ac4k_debug_linear_timeline: %s", hipGetErrorString(e));
}
#endif
