// NVFP4 attention forward for gfx950, head dims up to 128:  O = softmax(Q K^T * sm_scale) V on NVFP4 operands.
//
// Math contract of the reference kernel (lib/cuda/sm120/mha_nvfp4.cu:336-905, host checks :911-1077,
// interface include/ac4k_kernel/ops.h:12-16):
//   S = (Qhat . Khat^T) * (q_gs * k_gs * sm_scale), accumulated in fp32                          :586-598
//   online softmax over kv tiles of 128; kv positions past Nkv inside the last tile have S = 0,
//   enter the row maximum and P, and are taken out of the row sum again                          :600-700
//   P is quantized to NVFP4 on the fly with the global scale 1/2688; its 16-blocks are the kv
//   positions {8g + 4h + j} (g, j = 0..3) of a 32-group, h = 0, 1 - the sets that the swizzle of
//   quantize(v, 3, N_dim, swizzle=True) makes contiguous in V                                    :248-319
//   O = (sum over tiles of Phat . Vhat^T, rescaled) * ((1/l) * (1/2688) * v_gs) -> bf16          :705-830
// A workgroup (eight waves) owns 256, 128 or 64 query rows.  Per kv tile of 128 the packed K rows and the packed V rows (V
// is stored [d][kv]) are fetched once per workgroup, decoded once to exact fp16 and written to LDS, from where all waves
// read their MFMA operands.  Two LDS buffers alternate, one barrier per tile.  Decoded rows are 256 bytes at a pitch of
// 272, so that the 16-byte fragment reads of 16 lanes fall on 64 different banks.
//
// The MFMAs are issued so that a lane owns ONE query row: S^T = Khat . Qhat^T and O^T = Vhat . Phat^T
// (v_mfma_f32_32x32x16_f16, exact fp16 decode as in the linear).  Lane (r, h) of a wave then holds, per
// 32-row kv fragment, the 16 values S[r][8g + 4h + j]: exactly one P block, so its maximum, scale and
// nibbles are formed inside the lane, and the row maximum and row sum need one exchange between the two
// halves of the wave.  The k slots of the second product are paired through the stored (swizzled) order
// of V: slot s of step t holds kv position 8 (2t + (s>>1 & 1)) + 4h + 2 (s>>2) + (s & 1).
#include "attention_quantize.h"

#include <atomic>
#include <type_traits>

namespace ac4k {

struct MhaArgs {
  uint16_t *O;
  int64_t o_b, o_h, o_n, o_d;  // element strides of O [B, H, Nq, 128]
  const uint8_t *q, *k, *v, *q_sf, *k_sf, *v_sf;
  const float *q_gs, *k_gs, *v_gs;
  uint32_t H, head0;                  // heads; first head of the launch, of those of all batches
  int64_t Nq, Nkv, Nqp, Nkvp, Nkv64;  // padded: rows of the Q / K scale planes (16), stored kv length of V (64)
  int chunks, Dv, Dvp;                   // 64-chunks of a Q / K row (1 or 2), rows of V, rows of a V scale plane (16)
  float sm_scale;
  int o_vec;  // O rows are contiguous along d, 16-byte aligned, Dv % 8 == 0: rows leave as 16-byte pieces
};

constexpr float MHA_LOG2E = 1.4426950408889634f;
constexpr float MHA_P_ALPHA = 2688.0f;  // 1 / (global scale of P)

// Work of a launch: blocks of 256 query rows of all heads, one after the other.  The first `full` blocks are a workgroup
// each; what is behind them is cut into workgroups of 256 / tail rows.
struct MhaWork {
  uint32_t full, blocks, cut;  // full: a multiple of the number of XCDs; blocks and cut workgroups per head
};
struct MhaTile {
  int64_t block, head, b;  // block: in units of the rows of this workgroup
};
// Workgroups are dealt to the eight XCDs in turn: a run of consecutive blocks of one head is given to one XCD, whose L2 then
// fetches the K and V of that head once for all of them, instead of all eight XCDs fetching those of every head
// (4096 x 40 x 128 int8 x fp8: 262 -> 260 us, 4096 x 8: 59.3 -> 58.3).
__device__ __forceinline__ MhaTile mha_tile(const MhaWork &w, uint32_t H, uint32_t head0, uint32_t tail, uint32_t per_head) {
  const uint32_t first = blockIdx.x < w.full ? 0 : w.full, L = blockIdx.x - first;
  const uint32_t T = blockIdx.x < w.full ? w.full : gridDim.x - w.full;
  const uint32_t xcd = L & 7, q = T >> 3, rem = T & 7;
  const uint32_t id = (xcd < rem ? xcd * (q + 1) : rem * (q + 1) + (xcd - rem) * q) + (L >> 3) + first * tail;
  const uint32_t local = id / per_head, bh = local + head0;
  return MhaTile{id - local * per_head, bh % H, bh / H};
}

// Plan of a launch.  A workgroup that splits its tiles over 2 or 4 waves needs `tile_us` per kv tile and `fixed_us` for
// everything else.  Either whole rounds of unsplit workgroups and behind them the rest, cut so that the last round ends
// soonest; or all of it cut alike, which leaves out the rows that the last block of a head does not have (windows of 49
// tokens: 64 rows a workgroup instead of 256).
struct MhaCost {
  float fixed_us[3], tile_us[3];  // split 1, 2, 4
};
struct MhaPlan {
  MhaWork work;
  unsigned grid;
  int tail;  // 1, 2, 4
  float us;
};
static int64_t mha_cus() { return device_cu_count() >= 8 ? device_cu_count() / 8 * 8 : 256; }
static MhaPlan mha_plan(const MhaCost &c, int64_t heads, int64_t Nq, int64_t ntiles) {
  const int64_t cus = mha_cus();
  const int64_t blocks = ceil_div(Nq, 256), T = heads * blocks, full = T / cus * cus, left = T - full;
  auto rounds_us = [&](int64_t wgs, int i) { return (float)ceil_div(wgs, cus) * (c.fixed_us[i] + (float)ntiles * c.tile_us[i]); };
  MhaPlan p{{0, (uint32_t)blocks, 0}, 0, 1, 0.0f};
  auto offer = [&](float us, int64_t first, int64_t wgs, int64_t cut, int i) {
    if ((p.grid && us >= p.us) || first + wgs >= (1ll << 23)) return;  // (2^23 workgroups of 512 threads: more than a launch carries)
    p.us = us, p.tail = 1 << i, p.grid = (unsigned)(first + wgs);
    p.work.full = (uint32_t)first, p.work.cut = (uint32_t)cut;
  };
  for (int i = 0; i < (left ? 3 : 1) && full; ++i) offer(rounds_us(full, 0) + rounds_us(left << i, i), full, left << i, blocks << i, i);
  for (int i = 0; i < 3; ++i) {  // (beside whole rounds only where it gains more than the costs are good for)
    const int64_t cut = ceil_div(Nq << i, 256);
    offer(rounds_us(heads * cut, i) * (full ? 1.05f : 1.0f), 0, heads * cut, cut, i);
  }
  return p;
}
// Workgroups of four waves, 128 rows or 128 / split, all alike: a CU holds two of them, and one that has it to itself is faster.
struct Mha4Cost {
  MhaCost alone, shared;
};
static MhaPlan mha4_plan(const Mha4Cost &c, int64_t heads, int64_t Nq, int64_t ntiles) {
  const int64_t cus = mha_cus();
  MhaPlan p{{0, 0, 0}, 0, 1, 0.0f};
  for (int i = 0; i < 3; ++i) {
    const int64_t cut = ceil_div(Nq << i, 128), wgs = heads * cut, rounds = ceil_div(wgs, 2 * cus);
    const MhaCost &m = wgs <= cus ? c.alone : c.shared;
    const float us = (float)rounds * (m.fixed_us[i] + (float)ntiles * m.tile_us[i]);
    if ((p.grid && us >= p.us) || wgs >= (1ll << 24)) continue;  // (2^24 workgroups of 256 threads: more than a launch carries)
    p = MhaPlan{{0, 0, (uint32_t)cut}, (unsigned)wgs, 1 << i, us};
  }
  return p;
}

// eight nibbles times the block scale -> eight fp16 (exact)
__device__ __forceinline__ f16x8 mha_decode8(uint32_t w, f16x2 sc) {
  const f16x2 d0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 0) * sc;
  const f16x2 d1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 1) * sc;
  const f16x2 d2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 2) * sc;
  const f16x2 d3 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp4(w, 1.0f, 3) * sc;
  return (f16x8){d0.x, d0.y, d1.x, d1.y, d2.x, d2.y, d3.x, d3.y};
}

// A row-major packed row of Q: the lane's 32 elements [32 h, 32 h + 32) of 64-chunk c, and the two block
// scales that go with them, decoded into the four 16-k operands of that chunk.
__device__ __forceinline__ void mha_load_row_chunk(const uint8_t *row, const uint8_t *sf_chunk_row, int c, int h,
                                                   f16x8 (&out)[4]) {
  const uint4 w = *reinterpret_cast<const uint4 *>(row + c * 32 + h * 16);
  const uint32_t sc = *reinterpret_cast<const uint16_t *>(sf_chunk_row + 2 * h);
  const f16x2 s2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(sc, 1.0f, false);
  const f16x2 lo = {s2.x, s2.x}, hi = {s2.y, s2.y};
  out[0] = mha_decode8(w.x, lo);
  out[1] = mha_decode8(w.y, lo);
  out[2] = mha_decode8(w.z, hi);
  out[3] = mha_decode8(w.w, hi);
}

// dword i (0..7) of two 16-byte pieces; i is a constant after unrolling
__device__ __forceinline__ uint32_t mha_dword(const uint4 &a, const uint4 &b, int i) {
  switch (i) {
    case 0: return a.x;
    case 1: return a.y;
    case 2: return a.z;
    case 3: return a.w;
    case 4: return b.x;
    case 5: return b.y;
    case 6: return b.z;
    default: return b.w;
  }
}

// both halves of the wave (lanes 0-31 and 32-63) receive op(x of the lower half, x of the upper half)
// (v_permlane32_swap of x with itself: {lower, lower} and {upper, upper})
__device__ __forceinline__ float mha_halves_max(float x) {
  const u32x2 s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __builtin_fmaxf(__uint_as_float(s.x), __uint_as_float(s.y));
}
__device__ __forceinline__ int mha_halves_imax(int x) {
  const u32x2 s = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
  return (int)s.x > (int)s.y ? (int)s.x : (int)s.y;
}
__device__ __forceinline__ int mha_halves_imin(int x) {
  const u32x2 s = __builtin_amdgcn_permlane32_swap((uint32_t)x, (uint32_t)x, false, false);
  return (int)s.x < (int)s.y ? (int)s.x : (int)s.y;
}
__device__ __forceinline__ float mha_halves_sum(float x) {
  const u32x2 s = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(s.x) + __uint_as_float(s.y);
}

// Output of one wave: NFD fragments of O^T, head dims from d0 on, in the MFMA accumulator layout (lane (r, h) owns query
// row r of the wave: OT[fd][e] is head dim d0 + 32 fd + 8 (e >> 2) + 4 h + (e & 3)), already scaled, as bf16 bits in
// ob[fd][e].  Vector path (rows of O contiguous along d, 16-byte aligned, Dv % 8 == 0): the wave's 32 x (32 NFD) tile goes
// through LDS (32 * mha_out_pitch(NFD) bytes at `stage`, the wave's own) and leaves as 16-byte pieces of adjacent lanes,
// whole rows of the tile; otherwise element by element.
constexpr int mha_out_pitch(int nfd) { return nfd * 64 + 8; }  // bytes per row of the staged tile (8: bank spread)
constexpr int MHA_OUT_LDS = 32 * mha_out_pitch(4);
template <int NFD>
__device__ __forceinline__ void mha_store_rows(uint16_t *o_base, int64_t o_n, int64_t o_d, int o_vec, int64_t row0,
                                               int64_t Nq, int Dv, int d0, int lane, uint8_t *stage,
                                               const uint16_t (&ob)[NFD][16]) {
  constexpr int PITCH = mha_out_pitch(NFD), LPR = NFD * 4;  // lanes per row of the staged tile
  const int r = lane & 31, h = lane >> 5;
  if (o_vec) {
#pragma unroll
    for (int fd = 0; fd < NFD; ++fd)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4)
        *reinterpret_cast<uint2 *>(stage + r * PITCH + (fd * 32 + q4 * 8 + h * 4) * 2) =
            make_uint2(ob[fd][4 * q4] | ((uint32_t)ob[fd][4 * q4 + 1] << 16), ob[fd][4 * q4 + 2] | ((uint32_t)ob[fd][4 * q4 + 3] << 16));
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int p = 0; p < 2 * NFD; ++p) {
      const int row = p * (64 / LPR) + lane / LPR, d = (lane % LPR) * 8;
      const uint4 w = *reinterpret_cast<const uint4 *>(stage + row * PITCH + d * 2);
      if (row0 + row < Nq && d0 + d < Dv) *reinterpret_cast<uint4 *>(o_base + (row0 + row) * o_n + d0 + d) = w;
    }
  } else if (row0 + r < Nq) {
    uint16_t *orow = o_base + (row0 + r) * o_n;
#pragma unroll
    for (int fd = 0; fd < NFD; ++fd)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int d = d0 + fd * 32 + (e >> 2) * 8 + h * 4 + (e & 3);
        if (d < Dv) orow[d * o_d] = ob[fd][e];
      }
  }
}

// The parts of O and of the row sum of the SPLIT waves of a group meet: every wave leaves its part in LDS and adds up, in
// order, those of its 128 / SPLIT head dims (OT[0 ..] afterwards).  o_lds: 8 * 16 KB, l_lds: 1 KB.
template <int SPLIT>
__device__ __forceinline__ void mha_meet(f32x16 (&OT)[4], float &l_run, float *o_lds, float *l_lds, int group, int part, int lane) {
  constexpr int NFD = 4 / SPLIT;
  o_lds += lane;  // [wave][64 values][lane]
  l_lds += group * (SPLIT * 32) + (lane & 31);
#pragma unroll
  for (int fd = 0; fd < 4; ++fd)
#pragma unroll
    for (int e = 0; e < 16; ++e) o_lds[(group * SPLIT + part) * 4096 + (fd * 16 + e) * 64] = OT[fd][e];
  l_lds[part * 32] = l_run;
  __syncthreads();
  l_run = 0.0f;
#pragma unroll
  for (int q = 0; q < SPLIT; ++q) {
#pragma unroll
    for (int fd = 0; fd < NFD; ++fd)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float o = o_lds[(group * SPLIT + q) * 4096 + ((part * NFD + fd) * 16 + e) * 64];
        OT[fd][e] = q == 0 ? o : OT[fd][e] + o;
      }
    l_run += l_lds[q * 32];
  }
  __syncthreads();  // what follows lies over the parts
}

constexpr int MHA_PITCH = 272;                   // bytes per decoded row in LDS: 128 fp16 + 16 (bank spread)
constexpr int MHA_TILE_LDS = 128 * MHA_PITCH;    // one decoded operand tile: K 128 kv rows, V 128 d rows
constexpr int MHA_STAT_LDS = 4 * MHA_TILE_LDS;   // K tiles j & 1, V tiles j & 1; behind them the row maxima and sums of split tiles
constexpr int MHA_LUT_LDS = MHA_STAT_LDS + 2 * 256 * 4;  // exact reciprocals of the e4m3 values, as in the quantizer
constexpr int MHA_LDS = MHA_LUT_LDS + 128 * 4;
static_assert(8 * 16384 <= MHA_STAT_LDS && 8 * MHA_OUT_LDS <= MHA_STAT_LDS, "the parts of O and the staged output fit below the maxima");

// Eight waves, two per SIMD; a wave owns 32 query rows and 1 / SPLIT of the kv positions of every tile (see the INT8 x FP8
// kernel below, which has the same structure).  A tile step runs, in the order written out,
//   O += Vhat . Phat of tile i - 1  |  maxima, exp2, NVFP4 of tile i  |  S of tile i + 1
// and decodes K of tile i + 2 and V of tile i, which were fetched a step earlier, into LDS.
// Priorities fall as a wave gets on with P, as in the INT8 x FP8 kernel, so that the two waves of a SIMD stay side by side: whole calls on
// 16384 x 40 x 128 5468 -> 5337 us, 4096 x 40 418 -> 410, 2048 x 4 on 4096 keys 72 -> 69.
// (The multiplier of a P block inside the exponent instead of 16 multiplications gains another 3 %, but moves values across
// rounding boundaries of P.)
// Bound by vector-instruction issue - 551 instructions per tile and wave beside 64 MFMAs; at 8192 x 40 x 128 the counters show the
// vector port busy for 73 % of a SIMD's time and the matrix core for 49 % - and by power: the clock is 1.9 GHz there.  Kernel alone, same box, before (128 or 256 rows, no pipeline, no split) and now: 16384 x 40 x 128 6042 -> 5410 us
// (1016 TFLOP/s; 1085 on a cooler box), 4096 x 40 422 -> 370, 8192 x 4 194 -> 165, 3000 x 24 214 -> 162, 512 x 2 on 8192
// keys 191 -> 107, 75600 x 1 5250 -> 3676.
// TILES: 1 and 2 for calls of so many kv tiles, 0 for any number.  The step in front of the first tile and the one behind the
// last are then not there - multiplying by zeros and fetching a tile again - which made the pipeline slower than one tile after
// the other at those lengths.  Kernels of their own: written out for every length, or behind a branch in this one, they cost
// the loop registers (2 %, and spills).  Kernel alone, us, before the pipeline / with its loop / now: 8192 heads of 49 x 49, D = 32,
// 240 / 209 / 168 (workgroups of 64 rows); 1024 heads of 256 x 256, D = 64, 55.5 / 58.5 / 49.5; 40 heads of 16384 x 200 148 / 152 / 130.
template <int SPLIT, int TILES>
__device__ __forceinline__ void mha_nvfp4_block(const MhaArgs &a, const MhaTile &wg) {
  constexpr int NF = 4 / SPLIT;  // 32-row fragments of a tile per wave
  constexpr int ROWS = 256 / SPLIT;
  constexpr int RING = 4;        // MFMA operands in flight from LDS
  extern __shared__ __attribute__((aligned(16))) uint8_t mha_lds[];
  if (wg.block * ROWS >= a.Nq) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, h = lane >> 5;
  const int group = wave / SPLIT, part = wave % SPLIT;
  // staging role: row srow of the tile, 64-chunk sc, half sh of the chunk (K: elements 32 sh.. of the chunk, V: 32-group
  // 2 sc + sh)
  const int srow = threadIdx.x >> 2, sc = (threadIdx.x >> 1) & 1, sh = threadIdx.x & 1;
  const int64_t bh = wg.b * a.H + wg.head;
  const int64_t m = wg.block * ROWS + group * 32 + r;  // this lane's query row
  const int64_t mq = m < a.Nq ? m : a.Nq - 1;          // rows past Nq read the last row; never stored
  const int ntiles = (int)((a.Nkv + 127) / 128);
  const int k_last = (int)(a.Nkv - 1 - (int64_t)(ntiles - 1) * 128);             // last kv row of the last tile
  const int v_chunks_last = (int)(a.Nkv64 / 64 - (int64_t)(ntiles - 1) * 2);     // 64-chunks of V in the last tile: 1 or 2

  // What does not exist is read from a place that does and decoded with a scale of zero: kv rows past Nkv, the second
  // chunk of head dims up to 64, columns of V past its stored length.  Rows of V past Dv are never stored.
  const int64_t qk_row = a.chunks * 32;  // packed bytes of a Q / K row
  const int ksc_mask = sc < a.chunks ? 0xffff : 0, kchunk = sc < a.chunks ? sc : 0;
  const uint8_t *k_src = a.k + bh * a.Nkv * qk_row + kchunk * 32 + sh * 16;
  const uint8_t *ksf_src = a.k_sf + (bh * a.chunks + kchunk) * a.Nkvp * 4 + sh * 2;
  const int vrow = srow < a.Dv ? srow : a.Dv - 1;
  const uint8_t *v_src = a.v + (bh * a.Dv + vrow) * (a.Nkv64 / 2) + sh * 16;
  const uint8_t *vsf_src = a.v_sf + (bh * (a.Nkv64 / 64) * a.Dvp + vrow) * 4 + sh * 2;
  uint4 fk, fv;         // fetched, packed
  uint32_t fksc, fvsc;  // and the two scale bytes that go with them
  auto fetch_k = [&](int tile) {
    const bool last = tile >= ntiles - 1;
    if (last) tile = ntiles - 1;
    const int row = !last || srow < k_last ? srow : k_last;
    const int64_t n = (int64_t)tile * 128 + row;
    fk = *reinterpret_cast<const uint4 *>(k_src + n * qk_row);
    fksc = *reinterpret_cast<const uint16_t *>(ksf_src + n * 4);
    fksc &= last && srow > k_last ? 0 : ksc_mask;
  };
  auto fetch_v = [&](int tile) {
    const bool last = tile >= ntiles - 1;
    if (last) tile = ntiles - 1;
    const bool there = !last || sc < v_chunks_last;
    const int64_t chunk = (int64_t)tile * 2 + (there ? sc : 0);
    fv = *reinterpret_cast<const uint4 *>(v_src + chunk * 32);
    fvsc = *reinterpret_cast<const uint16_t *>(vsf_src + chunk * a.Dvp * 4);
    fvsc &= there ? 0xffff : 0;
  };
  // Decode, piece by piece (0..3 of K, 4..7 of V), into the tile buffers `buf`.  V: the thread's 32-group holds 16 stored
  // bytes; operand piece (t, hh) takes the t-th 16-bit halves of its dwords 2 hh and 2 hh + 1, and the scale of stored
  // block hh.
  uint8_t *const kd = mha_lds + srow * MHA_PITCH + sc * 128 + sh * 64, *const vd = kd + 2 * MHA_TILE_LDS;
  auto stage_piece = [&](int buf, int piece) {
    const f16x2 s2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(piece < 4 ? fksc : fvsc, 1.0f, false);
    const f16x2 b0 = {s2.x, s2.x}, b1 = {s2.y, s2.y};
    const int j = piece & 3;
    if (piece < 4) {
      const uint32_t w = j == 0 ? fk.x : j == 1 ? fk.y : j == 2 ? fk.z : fk.w;
      *reinterpret_cast<f16x8 *>(kd + buf * MHA_TILE_LDS + j * 16) = mha_decode8(w, j < 2 ? b0 : b1);
    } else {
      const uint32_t w = j == 0 ? (fv.x & 0xffffu) | (fv.y << 16) : j == 1 ? (fv.z & 0xffffu) | (fv.w << 16)
                       : j == 2 ? (fv.x >> 16) | (fv.y & 0xffff0000u) : (fv.z >> 16) | (fv.w & 0xffff0000u);
      *reinterpret_cast<f16x8 *>(vd + buf * MHA_TILE_LDS + j * 16) = mha_decode8(w, j & 1 ? b1 : b0);
    }
  };

  float *const lut = reinterpret_cast<float *>(mha_lds + MHA_LUT_LDS);
  if (threadIdx.x < 128) lut[threadIdx.x] = g_rcp_e4m3.v[threadIdx.x];
  if constexpr (TILES != 1) {
    fetch_k(1);  // (both in flight together: the registers of V are free)
    fv = fk, fvsc = fksc;
  }
  fetch_k(0);
  if constexpr (TILES == 1) fetch_v(0);
  // Qhat of the lane's row: 8 operands of 16 k (chunk c, sub-step s), kept for the whole kernel
  f16x8 QF[2][4];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
#pragma unroll
    for (int s = 0; s < 4; ++s) QF[c][s] = (f16x8)((_Float16)0);
    if (c < a.chunks)
      mha_load_row_chunk(a.q + (bh * a.Nq + mq) * qk_row, a.q_sf + ((bh * a.chunks + c) * a.Nqp + mq) * 4, c, h, QF[c]);
  }
  // exp2 argument = S * cs - (row maximum of S) * cs with cs = q_gs * k_gs * sm_scale * log2(e); a negative cs is
  // moved into Q so that the row maximum can be taken over the raw dot products
  float cs = (*a.q_gs) * (*a.k_gs) * a.sm_scale * MHA_LOG2E;
  if (cs < 0.0f) {
    cs = -cs;
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int s = 0; s < 4; ++s) QF[c][s] = -QF[c][s];
  }
#pragma unroll
  for (int p = 0; p < 4; ++p) stage_piece(0, p);
  if constexpr (TILES != 1) {
    fk = fv, fksc = fvsc;
    fetch_v(0);
  }
  float ml_run = -__builtin_inff(), l_run = 0.0f;  // running row maximum (in log2 units) and row sum
  float alpha = 1.0f;                              // factor of O and l that the last tile's maximum asks for
  f32x16 OT[4];  // O^T: d = 32 fd + 8 (e >> 2) + 4 h + (e & 3), for the lane's query row
#pragma unroll
  for (int fd = 0; fd < 4; ++fd) OT[fd] = (f32x16)(0.0f);
  uint32_t PW[2 * NF];  // P of a tile: eight nibbles per (fragment, step of 16 kv positions)
  uint32_t pcode[NF];   // and its block scales
  if constexpr (TILES == 0) {
#pragma unroll
    for (int f = 0; f < NF; ++f) PW[2 * f] = PW[2 * f + 1] = pcode[f] = 0;
    // V of the tile in front of the first one: zeros, and so is its P
#pragma unroll
    for (int j = 0; j < 4; ++j) *reinterpret_cast<uint4 *>(vd + MHA_TILE_LDS + j * 16) = make_uint4(0, 0, 0, 0);
  }
  if constexpr (TILES != 1) {
#pragma unroll
    for (int p = 0; p < 4; ++p) stage_piece(1, p);
  }
  if constexpr (TILES == 0) fetch_k(2);
  __syncthreads();

  f32x16 ST[NF];  // S^T of the tile at hand
  float bmax[NF];
  auto rescale = [&]() {
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {  // else no row of this wave raised its maximum
#pragma unroll
      for (int fd = 0; fd < 4; ++fd)
#pragma unroll
        for (int e = 0; e < 16; ++e) OT[fd][e] *= alpha;
    }
  };
  // operands: K for step t = 8 (fragment) + (16 columns), V for step u = 8 (fragment) + 4 (16 kv positions) + (32 rows of d)
  const uint8_t *const k_lane = mha_lds + (part * NF * 32 + r) * MHA_PITCH + h * 64;
  const uint8_t *const v_lane = mha_lds + 2 * MHA_TILE_LDS + r * MHA_PITCH + h * 16 + part * NF * 64;
  auto k_operand = [&](int buf, int t) {
    return *reinterpret_cast<const f16x8 *>(k_lane + buf * MHA_TILE_LDS + (t >> 3) * 32 * MHA_PITCH + ((t >> 2) & 1) * 128 + (t & 3) * 16);
  };
  auto v_operand = [&](int buf, int u) {
    return *reinterpret_cast<const f16x8 *>(v_lane + buf * MHA_TILE_LDS + (u & 3) * 32 * MHA_PITCH + (u >> 3) * 64 + ((u >> 2) & 1) * 32);
  };
  auto p_operand = [&](int g) {  // g = 2 (fragment) + (16 kv positions)
    const f16x2 s2 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(pcode[g >> 1], 1.0f, false);
    return mha_decode8(PW[g], (f16x2){s2.x, s2.x});
  };
  // row maxima of a tile's parts, two tiles in turn: [tile & 1][group][part][row]
  float *mx_lds = reinterpret_cast<float *>(mha_lds + MHA_STAT_LDS) + group * (SPLIT * 32) + r;
  // maxima of the raw values per fragment = per P block: exp2 and the scaling are monotonic, so the largest p of a block
  // is the p of its largest raw value, bit for bit
  auto part_maximum = [&](int parity) {
    float mx = -__builtin_inff();
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      bmax[f] = ST[f][0];
#pragma unroll
      for (int e = 1; e < 16; ++e) bmax[f] = __builtin_fmaxf(bmax[f], ST[f][e]);
      mx = __builtin_fmaxf(mx, bmax[f]);
    }
    mx_lds[parity * 256 + part * 32] = mha_halves_max(mx);  // (both halves of the wave write the same value)
  };
#pragma unroll
  for (int t = 0; t < 8 * NF; ++t)
    ST[t >> 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k_operand(0, t), QF[(t >> 2) & 1][t & 3], (t & 7) == 0 ? (f32x16)(0.0f) : ST[t >> 3], 0, 0, 0);
  if constexpr (SPLIT > 1) part_maximum(0);
  __syncthreads();

  auto tile_step = [&](auto first_tag, auto last_tag, int i) {
    constexpr bool FIRST = decltype(first_tag)::value, LAST = decltype(last_tag)::value;  // no tile in front of / behind this one
    const int buf = i & 1;
    f16x8 VF[RING], PF;
    __builtin_amdgcn_s_setprio(3);
    if constexpr (!FIRST) {
#pragma unroll
      for (int u = 0; u < RING; ++u) VF[u] = v_operand(buf ^ 1, u);
      rescale();
      PF = p_operand(0);
    }
    // ---- all but the last fragment of O of the tile before; under it the decoding of what was fetched and (SPLIT 1) the
    // maxima of this tile
    constexpr int PVA = 8 * (NF - 1), PIECE0 = TILES != 0 ? 4 : 0;
    if constexpr (NF == 1) {
#pragma unroll
      for (int p = PIECE0; p < 8; ++p) stage_piece(buf, p);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < PVA; ++u) {
      if constexpr (!FIRST) {
        OT[u & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(VF[u % RING], PF, OT[u & 3], 0, 0, 0);
        VF[u % RING] = v_operand(buf ^ 1, u + RING);
        if ((u & 3) == 3) PF = p_operand((u >> 2) + 1);
      }
      if (SPLIT == 1 && u < 16) {
        float &b = bmax[(u >> 2) % NF];
#pragma unroll
        for (int e = 4 * (u & 3); e < 4 * (u & 3) + 4; ++e) b = e == 0 ? ST[(u >> 2) % NF][0] : __builtin_fmaxf(b, ST[(u >> 2) % NF][e]);
        asm volatile("" : "+v"(b));
      }
      if (NF == 4 && (u % 3) == 2 && u / 3 >= PIECE0) stage_piece(buf, u / 3);
      if (NF == 2 && u >= PIECE0) stage_piece(buf, u);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (TILES == 0) fetch_k(i + 3);
    if constexpr (!LAST) fetch_v(i + 1);
    float mx;
    if constexpr (SPLIT == 1) {
      mx = mha_halves_max(__builtin_fmaxf(__builtin_fmaxf(bmax[0], bmax[1 % NF]), __builtin_fmaxf(bmax[2 % NF], bmax[3 % NF])));
    } else {
      mx = mx_lds[buf * 256];
#pragma unroll
      for (int q = 1; q < SPLIT; ++q) mx = __builtin_fmaxf(mx, mx_lds[buf * 256 + q * 32]);
    }
    const float ml = __builtin_fmaxf(ml_run, mx * cs);
    alpha = __builtin_amdgcn_exp2f(ml_run - ml);
    ml_run = ml;
    // block scales: e4m3(2688 * (largest p / 6)), saturated at 448, and the multiplier 2688 / scale, 0 for code 0.  ml is
    // rounded and the argument below is not, so with maxima of 2^20 and more it exceeds zero by up to half an ulp of ml and
    // the product reaches the 464 that the conversion turns into NaN.  A largest p held at 1 gives the code of 448, which is
    // where the product saturates (the compiler makes it the output modifier of the exp2).
    float o[NF];
    uint32_t code[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
      const float bm = __builtin_amdgcn_fmed3f(__builtin_amdgcn_exp2f(__builtin_fmaf(bmax[f], cs, -ml)), 0.0f, 1.0f);
      code[f] = (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(MHA_P_ALPHA * (bm * 0.16666666666666666f), 0.0f, 0, false) & 0x7f;
      o[f] = MHA_P_ALPHA * lut[code[f]];
    }
    // ---- P of this tile; under it the last fragment of O of the tile before and S of the next one
    float lsum = 0.0f;
    f16x8 KF[RING];
    uint32_t w;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int st = 0; st < 8 * NF + 8; ++st) {
      if (st == 2 * NF) __builtin_amdgcn_s_setprio(2);
      if (st == 5 * NF) __builtin_amdgcn_s_setprio(1);
      if (st == 8 * NF) __builtin_amdgcn_s_setprio(0);
      if (st < 8) {
        const int u = PVA + st;
        if constexpr (!FIRST) {
          OT[u & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(VF[u % RING], PF, OT[u & 3], 0, 0, 0);
          if (st + RING < 8) VF[u % RING] = v_operand(buf ^ 1, u + RING);
          if (st == 3) PF = p_operand(2 * NF - 1);
        }
        if (!LAST && st + RING >= 8) KF[st % RING] = k_operand(buf ^ 1, st + RING - 8);
      } else if constexpr (!LAST) {
        const int t = st - 8;
        ST[t >> 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(KF[t % RING], QF[(t >> 2) & 1][t & 3], (t & 7) == 0 ? (f32x16)(0.0f) : ST[t >> 3], 0, 0, 0);
        if (t + RING < 8 * NF) KF[t % RING] = k_operand(buf ^ 1, t + RING);
      }
      if (st < 8 * NF) {
        // two values of fragment f, in the order in which the stored nibbles of V come (see the header)
        const int f = st >> 3, t = (st >> 2) & 1, j = st & 3, e = 8 * t + (j == 0 ? 0 : j == 1 ? 4 : j == 2 ? 2 : 6);
        const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(ST[f][e], cs, -ml));
        const float p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(ST[f][e + 1], cs, -ml));
        lsum += p0;
        lsum += p1;
        if (j == 0) {
          asm volatile("" : "=v"(w));  // (any value: all four bytes are written)
          w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, p0 * o[f], p1 * o[f], 1.0f, 0);
        } else if (j == 1) w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, p0 * o[f], p1 * o[f], 1.0f, 1);
        else if (j == 2) w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, p0 * o[f], p1 * o[f], 1.0f, 2);
        else w = __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(w, p0 * o[f], p1 * o[f], 1.0f, 3);
        asm volatile("" : "+v"(w), "+v"(lsum));
        if (j == 3) PW[2 * f + t] = w;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) pcode[f] = code[f];
    l_run = __builtin_fmaf(l_run, alpha, mha_halves_sum(lsum));
    if constexpr (SPLIT > 1 && !LAST) part_maximum(buf ^ 1);
    __syncthreads();
  };
  if constexpr (TILES == 0) {
    for (int i = 0; i < ntiles; ++i) tile_step(std::false_type{}, std::false_type{}, i);
  } else if constexpr (TILES == 1) {
    tile_step(std::true_type{}, std::true_type{}, 0);
  } else {
    tile_step(std::true_type{}, std::false_type{}, 0);
    tile_step(std::false_type{}, std::true_type{}, 1);
  }
  rescale();
#pragma unroll
  for (int u = 0; u < 8 * NF; ++u)
    OT[u & 3] = __builtin_amdgcn_mfma_f32_32x32x16_f16(v_operand((ntiles - 1) & 1, u), p_operand(u >> 2), OT[u & 3], 0, 0, 0);
  __syncthreads();  // what follows lies over the tile buffers

  // The parts of O meet: every wave leaves its part in LDS and adds up, in order, those of 128 / SPLIT head dims.
  constexpr int NFD = 4 / SPLIT;
  const int d0 = part * NFD * 32;
  if constexpr (SPLIT > 1)
    mha_meet<SPLIT>(OT, l_run, reinterpret_cast<float *>(mha_lds), reinterpret_cast<float *>(mha_lds + MHA_STAT_LDS), group, part, lane);

  // the zero-filled kv positions of the last tile each added exp(0 - m) to the row sum
  if (a.Nkv % 128 != 0) l_run -= (float)(128 - a.Nkv % 128) / __builtin_amdgcn_exp2f(ml_run);
  // ---- O = O * ((1/l) * (1/2688) * v_gs) -> bf16
  const float scale = (1.0f / l_run) * (1.0f / MHA_P_ALPHA) * (*a.v_gs);
  uint16_t ob[NFD][16];
#pragma unroll
  for (int fd = 0; fd < NFD; ++fd)
#pragma unroll
    for (int e = 0; e < 16; ++e) ob[fd][e] = __builtin_bit_cast(uint16_t, (__bf16)(OT[fd][e] * scale));
  mha_store_rows<NFD>(a.O + wg.b * a.o_b + wg.head * a.o_h, a.o_n, a.o_d, a.o_vec, wg.block * ROWS + group * 32, a.Nq, a.Dv, d0,
                      lane, mha_lds + wave * MHA_OUT_LDS, ob);
}

// (two bodies in one kernel, so that the workgroups of the last round start as the ones in front of them end)
template <int TAIL, int TILES>
__global__ __launch_bounds__(512, 1) void mha_nvfp4_fwd_kernel(MhaArgs a, MhaWork w) {
  if (TAIL == 1 || blockIdx.x < w.full) mha_nvfp4_block<1, TILES>(a, mha_tile(w, a.H, a.head0, 1, w.blocks));
  else mha_nvfp4_block<TAIL, TILES>(a, mha_tile(w, a.H, a.head0, TAIL, w.cut));
}

// ---------------------------------------------------------------------------------------------------------------
// INT8 (QK) x FP8 (PV) attention forward, head dims up to 128 (lib/cuda/sm120/mha_int8_x_fp8.cu:346-975; host :979-1137;
// interface include/ac4k_kernel/ops.h:18-21):
//   S = Q . K^T in int32 (exact); s = float(S) * ((sm_scale * log2e) * q_sf[row / q_block] * k_sf[tile])   :476,657-677
//   kv positions past Nkv are -inf                                                                    :679-700
//   m = max(rowmax(s) - 7.5, m_old); p = exp2(s - m); l = l * exp2(m_old - m) + sum(p)                 :702-776
//   P -> e4m3 per element (cvt.rn.satfinite, no scales); O = O * exp2(m_old - m) + Phat . Vhat^T        :323-345,828-880
//   O * ((1 / l) * v_sf[d]) -> bf16                                                                   :886-905
// The product Phat . Vhat^T is accumulated in fp32 here (the reference's MMA accumulates each tile in fp16).
// Like in the NVFP4 kernel above a lane owns one query row (S^T = K . Q^T with v_mfma_i32_32x32x32_i8,
// O^T = Vhat . Phat^T with v_mfma_scale_f32_32x32x64_f8f6f4 on e4m3 operands, scales 2^0), but nothing has to be decoded: the int8 rows of K and the
// e4m3 rows of V go from global memory into LDS as they are, and from there into the MFMAs.  V is stored with the
// 16-group swizzle of quantize(v, 3, N_dim, swizzle=True, precision="fp8e4m3"): stored byte 8 h + 4 (j >> 1) + 2 q
// + (j & 1) of a 16-group holds kv position 8 q + 4 h + j, so the eight positions that lane half h owns in a
// 16-group are the contiguous stored bytes [8 h, 8 h + 8): four such pieces are the lane's share of one MFMA operand.

struct Mha8Args {
  uint16_t *O;
  int64_t o_b, o_h, o_n, o_d;  // element strides of O [B, H, Nq, 128]
  const int8_t *q, *k;
  const uint8_t *v;
  const float *q_sf, *k_sf, *v_sf;
  uint32_t H, head0;                 // heads; first head of the launch, of those of all batches
  int64_t Nq, Nkv, Nkv16, nqb, nkb;  // stored kv length of V (16), scales per head of Q and K
  int Dp, Dv, Dvp;                      // bytes of a Q / K row (head dim padded to 16), rows of V, scales of V per head (16)
  int q_block;
  float sm_scale;
  int o_vec;
};

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

// LDS: K tiles j & 1 of 128 rows of 128 bytes, the 16-byte piece p of row n at p ^ ((n >> 1) & 7) (bank spread); behind them V
// tiles j & 1 of 128 d rows at a pitch of 144 bytes
constexpr int MHA8_K_LDS = 128 * 128;
constexpr int MHA8_PITCH = 144;
constexpr int MHA8_V_LDS = 128 * MHA8_PITCH;
// split tiles: row maxima and sums behind the tile buffers and behind the parts of O of all waves
constexpr int mha8_stat_lds(int waves, int split) {
  return split == 1 || waves * 16384 < 2 * MHA8_K_LDS + 2 * MHA8_V_LDS ? 2 * MHA8_K_LDS + 2 * MHA8_V_LDS : waves * 16384;
}
constexpr int mha8_lds_bytes(int waves, int split) { return mha8_stat_lds(waves, split) + (split == 1 ? 0 : 2 * 512 * 4); }
static_assert(8 * MHA_OUT_LDS <= mha8_lds_bytes(8, 1) && 2 * mha8_lds_bytes(4, 4) <= 160 * 1024);
constexpr float MHA8_EXP_OFFSET = 7.5f;
// start of S: the bits of 1 / (2 pi), the inline constant whose mantissa (2292099 of 2^23) leaves room for every S on both sides;
// 1 / the unit of its last place
constexpr int MHA8_S_BIAS = 0x3e22f983;
constexpr float MHA8_S_UNIT = 67108864.0f;  // 2^26
static_assert((MHA8_S_BIAS & 0x7fffff) > 128 * 128 * 128 && (MHA8_S_BIAS & 0x7fffff) + 128 * 128 * 128 < 0x800000);

// Two waves per SIMD; a wave owns 32 query rows and 1 / SPLIT of the kv positions of every tile: SPLIT waves
// share a group of query rows, 32 * WAVES / SPLIT rows per workgroup.  What a shared group needs per tile is the row maximum
// over the whole tile, which goes through LDS with the barrier that ends the tile; the partial sums of O and of the row
// meet at the end.  The maxima, and with them every rounding of P, are those of the unsplit tile; the sums of O and of the row
// are added in another order, so equal rows of two launches, or of the cut and the uncut part of one, may differ by an fp32
// rounding (outputs 2e-5 apart, relative).
//
// A tile step is a software pipeline over three tiles, written out in the order in which it issues (the compiler's
// scheduler keeps an MFMA and the vector instructions that could run under it apart):
//   O += Vhat . Phat of tile i - 1  |  exp2, e4m3 of tile i  |  S of tile i + 1, into the registers that the scores of
//   tile i leave one 32-row fragment after the other; under its last fragment the maxima of the others
// K arrives by LDS-DMA two tiles ahead, V through registers one tile ahead.
// Bound by the issue of vector instructions (about 350 per tile and wave beside 24 MFMAs; two waves share a SIMD and take 8.3 cycles for
// an exp2, 9.6 for a pair of e4m3, 4.3 for a maximum or an integer conversion, 2.4 to 2.9 for an addition or fma, which they issue
// together; at 8192 x 40 x 128 the vector port is busy for 86 % of a SIMD's time, the matrix core for 41 %) and, where the whole GPU is
// busy for long, by power (2.0 GHz there).
// Of the two waves of a SIMD the older one is served first: it ran a whole step alone, at the rate of one wave, and then waited at
// the barrier for half of the next.  A wave therefore lowers its priority as it gets on with a step, which keeps the two side by side:
// 16384 x 40 x 128 5270 -> 4955 cycles per tile of both (priorities that alternate step by step 5160 to 5220).
// The whole call on 16384 x 40 x 128 3474 -> 3301 us with all of it (moving the maxima and the conversion alone 3446), 4096 x 40 284 -> 277,
// 3000 x 2 x 24 x 64 194 -> 188.  The conversion and the maxima cost less than they save in the clock: power takes back about a third.
// TILES as above, with eight waves, where they gained the same: 8192 heads of 49 x 49, D = 32, 209 / 179 / 144 us; 1024 heads of 256 x 256,
// D = 64, 42 / 44 / 41.5; 40 heads of 16384 x 200 133 / 122 / 114.
// WAVES: eight, or four and two workgroups on a CU, which wait for their barriers and their ends one under the other's work, but
// fetch every tile of K and V twice per CU.  Whole rounds of many tiles go to eight (kernel alone, us, eight / four: 40 heads of 4096 x
// 4096 224 / 250, 24 of 4096 x 8192 260 / 277); short loops and grids that leave CUs idle, which finer cuts fill, to four (2 heads of 4096 x 8192 70 / 63,
// 3 of 2111 x 7000 61 / 56, 24 of 2637 x 2637 75 / 65; whole calls on 40 heads of 16384 x 77 134 -> 120).
template <int WAVES, int SPLIT, int TILES>
__device__ __forceinline__ void mha_int8_x_fp8_block(const Mha8Args &a, const MhaTile &wg) {
  constexpr int NF = 4 / SPLIT;             // 32-row fragments of a tile per wave
  constexpr int NPV = SPLIT == 1 ? 2 : 1;   // P.V operands of 64 kv positions per wave (SPLIT 4: half of one, zeros behind)
  constexpr int ROWS = WAVES * 32 / SPLIT;
  constexpr int KT = 16 / WAVES, VT = WAVES / 2, VP = 8 / VT;  // transfers of K per wave; threads on a row of V, their 16-groups
  extern __shared__ __attribute__((aligned(16))) uint8_t mha_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r = lane & 31, h = lane >> 5;
  const int group = wave / SPLIT, part = wave % SPLIT;
  const int srow = threadIdx.x / VT, sv = threadIdx.x % VT;  // staging role for V: row of the tile, part of it
  if (wg.block * ROWS >= a.Nq) return;
  const int64_t bh = wg.b * a.H + wg.head;
  const int64_t m = wg.block * ROWS + group * 32 + r;  // this lane's query row
  const int64_t mq = m < a.Nq ? m : a.Nq - 1;          // rows past Nq read the last row; never stored
  const int ntiles = (int)a.nkb;
  // last kv row and last 16-group of V that exist in the last tile
  const int k_last = (int)(a.Nkv - 1 - (int64_t)(ntiles - 1) * 128), v_last = (int)(a.Nkv16 - 16 - (int64_t)(ntiles - 1) * 128);

  // What does not exist is read from a place that does, with no test in the loop: rows of K past Nkv repeat the last row
  // (no other maximum, and P is set to zero), columns of K past the head dim (those of Q are zero), columns of V past its
  // stored length (P is zero there) and rows of V past Dv (never stored).
  const int8_t *k_head = a.k + bh * a.Nkv * a.Dp;
  // K goes from global memory straight into LDS: transfer t of 16 lands in the eight rows from 8 t on, lane l in position
  // l % 8 of row l / 8, so it fetches the 16-byte piece that belongs there
  const int kpiece = (lane & 7) ^ (lane >> 4);  // even t; ^ 4 for odd t
  const uint32_t kcol[2] = {(uint32_t)(kpiece * 16 < a.Dp ? kpiece * 16 : 0), (uint32_t)((kpiece ^ 4) * 16 < a.Dp ? (kpiece ^ 4) * 16 : 0)};
  const uint32_t krow = (uint32_t)((wave * 8 * KT + (lane >> 3)) * a.Dp);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)mha_lds;
  auto fetch_k = [&](int tile, int buf) {
    if (tile >= ntiles) tile = ntiles - 1;
    const int8_t *src = k_head + (int64_t)tile * 128 * a.Dp;
    const uint32_t last_off = (uint32_t)((tile < ntiles - 1 ? 127 : k_last) * a.Dp);
#pragma unroll
    for (int j = 0; j < KT; ++j) {
      const uint32_t off = krow + (uint32_t)(j * 8 * a.Dp);
      dma16(src, (off < last_off ? off : last_off) + kcol[j & 1], lds0 + buf * MHA8_K_LDS, (uint32_t)((wave * KT + j) * 1024));
    }
  };
  struct Piece {
    uint4 g[VP];
  };
  const uint8_t *v_row = a.v + (bh * a.Dv + (srow < a.Dv ? srow : a.Dv - 1)) * a.Nkv16;
  auto fetch_v = [&](int tile, Piece &v) {  // tiles in turn
    const int last = tile < ntiles - 1 ? 112 : v_last;
#pragma unroll
    for (int j = 0; j < VP; ++j) {
      const int c = (sv * VP + j) * 16;
      v.g[j] = *reinterpret_cast<const uint4 *>(v_row + (c < last ? c : last));
    }
    v_row += 128;
  };
  // V: the thread's 16-groups regrouped in pairs so that the 8-byte pieces of lane half hh of both are one 16-byte run at
  // 32 (pair) + 16 hh
  auto stage_v = [&](int buf, const Piece &v) {
    uint8_t *vd = mha_lds + 2 * MHA8_K_LDS + buf * MHA8_V_LDS + srow * MHA8_PITCH + sv * VP * 16;
#pragma unroll
    for (int j = 0; j < VP; j += 2) {
      *reinterpret_cast<uint4 *>(vd + j * 16) = make_uint4(v.g[j].x, v.g[j].y, v.g[j + 1].x, v.g[j + 1].y);
      *reinterpret_cast<uint4 *>(vd + j * 16 + 16) = make_uint4(v.g[j].z, v.g[j].w, v.g[j + 1].z, v.g[j + 1].w);
    }
  };

  Piece vp;
  fetch_k(0, 0);
  if constexpr (TILES == 1) fetch_v(0, vp);
  else fetch_k(1, 1);
  // Q of the lane's row: the 16 bytes [32 s + 16 h, +16) of k-step s, kept for the whole kernel
  i32x4 QF[4];
#pragma unroll
  for (int s4 = 0; s4 < 4; ++s4) {
    QF[s4] = (i32x4)(0);
    if (s4 * 32 + h * 16 < a.Dp) QF[s4] = *reinterpret_cast<const i32x4 *>(a.q + (bh * a.Nq + mq) * a.Dp + s4 * 32 + h * 16);
  }
  const float qs = (a.sm_scale * MHA_LOG2E) * a.q_sf[bh * a.nqb + mq / a.q_block];
  const float *ksf_src = a.k_sf + bh * a.nkb;
  // A negative product of scales turns the order of the scores of a tile around, and one near the end of the range (2^100) does not take
  // the unit of S.  The quantizers write none; operands that hold one anywhere take a loop of their own.
  bool negative = !(qs >= 0.0f);
  for (int t = lane; t < ntiles; t += 64) negative |= !(ksf_src[t] >= 0.0f && qs * ksf_src[t] < 0x1p100f);
  negative = __builtin_amdgcn_ballot_w64(negative) != 0;
  float ksf_next = ksf_src[0];

  float m_run = -__builtin_inff(), l_run = 0.0f;  // running maximum (held 7.5 below the row maximum) and row sum
  float alpha = 1.0f;                             // factor of O and l that the last tile's maximum asks for
  f32x16 OT[4];  // O^T: d = 32 fd + 8 (e >> 2) + 4 h + (e & 3), for the lane's query row
#pragma unroll
  for (int fd = 0; fd < 4; ++fd) OT[fd] = (f32x16)(0.0f);
  i32x8 P[NPV];  // P of a tile as e4m3, MFMA operands of 64 kv positions (SPLIT 4: 32, and zeros)
#pragma unroll
  for (int j = 0; j < NPV; ++j) P[j] = (i32x8)(0);
  if constexpr (TILES == 0) {  // V of the tile in front of the first one: zeros, and so is its P
    Piece z;
#pragma unroll
    for (int j = 0; j < VP; ++j) z.g[j] = make_uint4(0, 0, 0, 0);
    stage_v(1, z);
  }
  wait_vmcnt<0>();
  __syncthreads();

  i32x16 SI[NF];  // S^T of the tile at hand
  auto rescale = [&]() {
    if (__builtin_amdgcn_ballot_w64(alpha != 1.0f)) {  // else no row of this wave raised its maximum
#pragma unroll
      for (int fd = 0; fd < 4; ++fd)
#pragma unroll
        for (int e = 0; e < 16; ++e) OT[fd][e] *= alpha;
    }
  };
  // O^T += Vhat . Phat^T: one MFMA (k = 64: v_mfma_scale_f32_32x32x64_f8f6f4 with unit scales; lane half h supplies 32
  // of the 64 k slots) per 64 kv positions and 32 rows of d; step st = 4 (64 kv positions) + (32 rows of d)
  const uint8_t *v_lane = mha_lds + 2 * MHA8_K_LDS + r * MHA8_PITCH + h * 16 + part * NF * 32;
  auto v_operand = [&](int buf, int st) {
    const uint8_t *p = v_lane + buf * MHA8_V_LDS + (st & 3) * 32 * MHA8_PITCH + (st >> 2) * 64;
    const uint4 va = *reinterpret_cast<const uint4 *>(p);
    const uint4 vc = SPLIT == 4 ? make_uint4(0, 0, 0, 0) : *reinterpret_cast<const uint4 *>(p + 32);
    return (i32x8){(int)va.x, (int)va.y, (int)va.z, (int)va.w, (int)vc.x, (int)vc.y, (int)vc.z, (int)vc.w};
  };
  auto pv_mfma = [](i32x8 v, i32x8 p, f32x16 o) {
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(v, p, o, 0, 0, 0, 0x7f7f7f7f, 0, 0x7f7f7f7f);
  };
  // K for step t = 4 (fragment of 32 kv positions) + (32 columns) of S^T = K . Q^T
  const int kswz = (part * NF * 32 + r) * 128 + ((h ^ ((r >> 1) & 7)) << 4);
  auto k_rows = [&](int buf, const uint8_t *(&kb)[4]) {
#pragma unroll
    for (int s4 = 0; s4 < 4; ++s4) kb[s4] = mha_lds + buf * MHA8_K_LDS + (kswz ^ (s4 * 32));
  };
  auto k_operand = [](const uint8_t *const (&kb)[4], int t) {
    return *reinterpret_cast<const i32x4 *>(kb[t & 3] + (t >> 2) * 4096);
  };
  // A score as a float.  Scales of one sign and of ordinary size: S starts at the bits of a float, MHA8_S_BIAS, so that its bits, read as a
  // float, are that number + S units of its last place (no sum leaves the binade).  Taking the number off again is exact, as is the unit, a
  // power of two, in the scale: the scores are those of a conversion, bit for bit, by an addition that two waves of a SIMD issue
  // together (2.4 cycles a wave) where the conversion of an integer takes 4.3.
  auto score = [&](auto negative_tag, int s) {
    return decltype(negative_tag)::value ? (float)s : __int_as_float(s) - __int_as_float(MHA8_S_BIAS);
  };
  // extrema over the scores of fragments
  int hi, lo;
  auto extremum = [&](auto negative_tag, int f) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      hi = SI[f][e] > hi ? SI[f][e] : hi;
      if (decltype(negative_tag)::value) lo = SI[f][e] < lo ? SI[f][e] : lo;
    }
    asm volatile("" : "+v"(hi));
  };
  // maxima (minima) of a tile's parts, two tiles in turn: [tile & 1][max, min][group][part][row]
  int *mx_lds = reinterpret_cast<int *>(mha_lds + mha8_stat_lds(WAVES, SPLIT)) + group * (SPLIT * 32) + r;
  auto part_extremum = [&](auto negative_tag, int parity) {  // (the last fragment's; the others are in hi and lo)
    constexpr bool NEG = decltype(negative_tag)::value;
    if (NF == 1) hi = lo = SI[0][0];
    extremum(negative_tag, NF - 1);
    mx_lds[parity * 512 + part * 32] = mha_halves_imax(hi);  // (both halves of the wave write the same value)
    if (NEG) mx_lds[parity * 512 + 256 + part * 32] = mha_halves_imin(lo);
  };
  // (in registers of its own: folded into the first MFMA of one fragment, but copied from scalars for four of them in a loop)
  i32x16 start = (i32x16)(MHA8_S_BIAS);
  auto first_scores = [&](auto negative_tag) {
    if (!decltype(negative_tag)::value) asm volatile("" : "+v"(start));
    constexpr bool NEG = decltype(negative_tag)::value;
    const uint8_t *kb[4];
    k_rows(0, kb);
#pragma unroll
    for (int t = 0; t < 4 * NF; ++t)
      SI[t >> 2] = __builtin_amdgcn_mfma_i32_32x32x32_i8(k_operand(kb, t), QF[t & 3], (t & 3) == 0 ? (i32x16)(NEG ? 0 : MHA8_S_BIAS) : SI[t >> 2], 0, 0, 0);
    hi = lo = SI[0][0];
#pragma unroll
    for (int f = 0; f < NF - 1; ++f) extremum(negative_tag, f);
    if constexpr (SPLIT > 1) part_extremum(negative_tag, 0);
    __syncthreads();
  };

  // One kv tile i.  TAIL: the last, partial one, where P of the positions past Nkv is zero.
  auto tile_step = [&](auto negative_tag, auto tail_tag, auto first_tag, auto last_tag, int i) {
    constexpr bool FIRST = decltype(first_tag)::value, LAST = decltype(last_tag)::value;  // no tile in front of / behind this one
    constexpr bool NEG = decltype(negative_tag)::value, TAIL = decltype(tail_tag)::value;
    constexpr int PV0 = SPLIT == 1 ? 1 : 0;  // steps of O in front of P
    const int buf = i & 1;
    __builtin_amdgcn_s_setprio(3);
    float qk = qs * ksf_next;
    // (here, not behind the loads below: the compiler does not count the transfers of K, and its wait for a load in front of
    // them would be a wait for them too)
    asm volatile("" : "+v"(qk));
    if constexpr (!LAST) ksf_next = ksf_src[i + 1 < ntiles ? i + 1 : i];
    asm volatile("" ::: "memory");
    i32x8 VF[2];
    if constexpr (!FIRST) {
      VF[0] = v_operand(buf ^ 1, 0);
      VF[1] = v_operand(buf ^ 1, 1);
    }
    if constexpr (TILES == 0) fetch_k(i + 2, buf);
    if constexpr (TILES != 1) fetch_v(i, vp);
    if constexpr (!FIRST) rescale();
    __builtin_amdgcn_sched_barrier(0);
    // ---- maxima.  The maximum of s = float(S) * qk is taken over the integers S (the conversion keeps their order):
    // qk >= 0 keeps it too, qk < 0 reverses it.  SPLIT 1: those of the last fragment; the step before took the others.
    if constexpr (SPLIT == 1) {
      if constexpr (FIRST || NF == 1) hi = lo = SI[0][0];
      if constexpr (!FIRST) OT[0] = pv_mfma(VF[0], P[0], OT[0]), VF[0] = v_operand(buf ^ 1, 2);
#pragma unroll
      for (int f = FIRST ? 0 : NF - 1; f < NF; ++f) extremum(negative_tag, f);
      hi = mha_halves_imax(hi);
      if (NEG) lo = mha_halves_imin(lo);
    } else {
      hi = mx_lds[buf * 512];
      if (NEG) lo = mx_lds[buf * 512 + 256];
#pragma unroll
      for (int q = 1; q < SPLIT; ++q) {
        const int up = mx_lds[buf * 512 + q * 32];
        hi = up > hi ? up : hi;
        if (NEG) {
          const int down = mx_lds[buf * 512 + 256 + q * 32];
          lo = down < lo ? down : lo;
        }
      }
    }
    const float qk1 = NEG ? qk : qk * MHA8_S_UNIT;
    const float smax = score(negative_tag, NEG && qk < 0.0f ? lo : hi) * qk1;
    const float m_new = __builtin_fmaxf(smax - MHA8_EXP_OFFSET, m_run);
    alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    // ---- P of this tile, under it (the rest of) O of the tile before and S of the next one
    const int left = k_last + 1 - part * NF * 32 - h * 4;  // TAIL: kv positions that exist, from the lane's first one on
    const uint8_t *kb[4];
    k_rows(buf ^ 1, kb);
    float lsum = 0.0f;
    int w0, w1;
    i32x8 PN[NPV];  // P of this tile (SPLIT 1 and 2 write all of it)
#pragma unroll
    for (int j = 0; j < NPV; ++j) PN[j] = P[j];
    i32x4 KF[2];
#pragma unroll
    for (int st = 0; st < 4 * NF + 4; ++st) {  // step st: P of the st-th group of four scores; a part of O; a part of S, st - 4
      if (st == NF) __builtin_amdgcn_s_setprio(2);
      if (st == NF * 9 / 4) __builtin_amdgcn_s_setprio(1);
      if (st == NF * 7 / 2) __builtin_amdgcn_s_setprio(0);
      if constexpr (!FIRST) {
        const int u = st + PV0;
        if (u < 4 * NPV) {
          OT[u & 3] = pv_mfma(VF[u & 1], P[u >> 2], OT[u & 3]);
          if (u + 2 < 4 * NPV) VF[u & 1] = v_operand(buf ^ 1, u + 2);
        }
      }
      if constexpr (!LAST) {
        if (st == 2 || st == 3) KF[st & 1] = k_operand(kb, st - 2);
        if (st >= 4) {
          const int t = st - 4, f = t >> 2, s4 = t & 3;
          SI[f] = __builtin_amdgcn_mfma_i32_32x32x32_i8(KF[t & 1], QF[s4], s4 == 0 ? (NEG ? (i32x16)(0) : start) : SI[f], 0, 0, 0);
          if (t + 2 < 4 * NF) KF[t & 1] = k_operand(kb, t + 2);
        }
      }
      if (st < 4 * NF) {
        const int f = st >> 2, q = st & 3;
        float p[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          p[e] = __builtin_amdgcn_exp2f(__builtin_fmaf(score(negative_tag, SI[f][4 * q + e]), qk1, -m_new));  // p <= 2^7.5
          if (TAIL && f * 32 + q * 8 + e >= left) p[e] = 0.0f;
          lsum += p[e];
        }
        // the lane's two 16-group halves of the fragment, in the stored order of V: e = {0, 1, 4, 5, 2, 3, 6, 7}
        if (q & 1) {
          w0 = __builtin_amdgcn_cvt_pk_fp8_f32(p[0], p[1], w0, true);
          w1 = __builtin_amdgcn_cvt_pk_fp8_f32(p[2], p[3], w1, true);
        } else {
          asm volatile("" : "=v"(w0), "=v"(w1));  // (any value: both halves are written)
          w0 = __builtin_amdgcn_cvt_pk_fp8_f32(p[0], p[1], w0, false);
          w1 = __builtin_amdgcn_cvt_pk_fp8_f32(p[2], p[3], w1, false);
        }
        asm volatile("" : "+v"(lsum), "+v"(w0), "+v"(w1));
        if (q & 1) {
          PN[f >> 1][4 * (f & 1) + 2 * (q >> 1)] = w0;
          PN[f >> 1][4 * (f & 1) + 2 * (q >> 1) + 1] = w1;
        }
      } else if constexpr (!LAST) {  // under S of the last fragment, the extrema of the others
        const int f = st - 4 * NF;
        if (f == 0) hi = lo = SI[0][0];
        if (f < NF - 1) extremum(negative_tag, f);
        if (f == 3) stage_v(buf, vp);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LAST) stage_v(buf, vp);
#pragma unroll
    for (int j = 0; j < NPV; ++j) P[j] = PN[j];
    l_run = __builtin_fmaf(l_run, alpha, mha_halves_sum(lsum));
    if constexpr (SPLIT > 1 && !LAST) part_extremum(negative_tag, buf ^ 1);
    wait_vmcnt<0>();  // the transfers of K
    __syncthreads();
  };
  using No = std::false_type;
  using Yes = std::true_type;
  auto all_tiles = [&](auto negative_tag) {
    first_scores(negative_tag);
    int i = 0;
    for (; i < (int)(a.Nkv / 128); ++i) tile_step(negative_tag, No{}, No{}, No{}, i);
    if (i < ntiles) tile_step(negative_tag, Yes{}, No{}, No{}, i);
  };
  // (the probability keeps the registers of the loop that runs)
  if constexpr (TILES == 1) {  // (a code for both signs and both ends)
    first_scores(Yes{});
    tile_step(Yes{}, Yes{}, Yes{}, Yes{}, 0);
  } else if constexpr (TILES == 2) {
    first_scores(Yes{});
    tile_step(Yes{}, No{}, Yes{}, No{}, 0);
    tile_step(Yes{}, Yes{}, No{}, Yes{}, 1);
  } else if (__builtin_expect_with_probability(negative, 0, 0.99999)) {
    all_tiles(Yes{});
  } else {
    all_tiles(No{});
  }
  rescale();
#pragma unroll
  for (int st = 0; st < 4 * NPV; ++st) OT[st & 3] = pv_mfma(v_operand((ntiles - 1) & 1, st), P[st >> 2], OT[st & 3]);
  __syncthreads();  // what follows lies over the tile buffers

  // The parts of O meet: every wave leaves its part in LDS and adds up, in order, those of 128 / SPLIT head dims.
  constexpr int NFD = 4 / SPLIT;
  const int d0 = part * NFD * 32;
  if constexpr (SPLIT > 1)
    mha_meet<SPLIT>(OT, l_run, reinterpret_cast<float *>(mha_lds), reinterpret_cast<float *>(mha_lds + mha8_stat_lds(WAVES, SPLIT)), group, part, lane);

  // ---- O = O * ((1 / l) * v_sf[d]) -> bf16
  const float rl = 1.0f / l_run;
  const float *vsf = a.v_sf + bh * a.Dvp;
  uint16_t ob[NFD][16];
#pragma unroll
  for (int fd = 0; fd < NFD; ++fd)
#pragma unroll
    for (int q4 = 0; q4 < 4; ++q4) {
      const int d = d0 + fd * 32 + q4 * 8 + h * 4;  // four consecutive head dims; the scale row is padded to 16
      const float4 sv = d < a.Dvp ? *reinterpret_cast<const float4 *>(vsf + d) : make_float4(0.f, 0.f, 0.f, 0.f);
      const float sc[4] = {rl * sv.x, rl * sv.y, rl * sv.z, rl * sv.w};
#pragma unroll
      for (int e = 0; e < 4; ++e) ob[fd][4 * q4 + e] = __builtin_bit_cast(uint16_t, (__bf16)(OT[fd][4 * q4 + e] * sc[e]));
    }
  mha_store_rows<NFD>(a.O + wg.b * a.o_b + wg.head * a.o_h, a.o_n, a.o_d, a.o_vec, wg.block * ROWS + group * 32, a.Nq, a.Dv, d0,
                      lane, mha_lds + wave * MHA_OUT_LDS, ob);
}

// (two bodies in one kernel, so that the workgroups of the last round start as the ones in front of them end)
template <int TAIL>
__global__ __launch_bounds__(512, 1) void mha_int8_x_fp8_fwd_kernel(Mha8Args a, MhaWork w) {
  if (TAIL == 1 || blockIdx.x < w.full) mha_int8_x_fp8_block<8, 1, 0>(a, mha_tile(w, a.H, a.head0, 1, w.blocks));
  else mha_int8_x_fp8_block<8, TAIL, 0>(a, mha_tile(w, a.H, a.head0, TAIL, w.cut));
}
template <int SPLIT, int TILES>
__global__ __launch_bounds__(256, 2) void mha_int8_x_fp8_fwd4_kernel(Mha8Args a, MhaWork w) {
  mha_int8_x_fp8_block<4, SPLIT, TILES>(a, mha_tile(w, a.H, a.head0, SPLIT, w.cut));
}

// Per-token-block int8 quantizer in front of it (python/ac4k_kernel/ops/attention.py:18-99, a Triton kernel in the
// reference): one scale = max|x| / 127 per block of `block` tokens of a head (all D columns), y = int8(trunc(x /
// scale)), 0 where the scale is 0; y is [B, H, N, Dp] with pad columns 0, the scales [B, H, ceil(N / block)].
__global__ __launch_bounds__(256) void quantize_int8_token_block_kernel(int8_t *__restrict__ y, float *__restrict__ scale,
                                                                        const uint16_t *__restrict__ x, int64_t s_b,
                                                                        int64_t s_h, int64_t s_n, int64_t H, int64_t N,
                                                                        int D, int Dp, int block, int vec) {
  __shared__ uint32_t wmax[4];
  const int64_t nb = gridDim.x, blk = blockIdx.x, head = blockIdx.y, b = blockIdx.z;
  const int64_t n0 = blk * block;
  const int rows = (int)((N - n0) < block ? (N - n0) : block);
  const uint16_t *src = x + b * s_b + head * s_h + n0 * s_n;
  int8_t *dst = y + ((b * H + head) * N + n0) * Dp;
  uint32_t mx = 0;
  // rows of whole 16-byte vectors (D % 8 == 0, aligned), at most eight vectors per thread: the block is read once,
  // into registers
  const int vpr = D / 8, nvec = rows * vpr;
  if (vec && nvec <= 8 * 256) {
    uint4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = threadIdx.x + j * 256;
      v[j] = make_uint4(0, 0, 0, 0);
      if (i < nvec) v[j] = ld_stream_u4(src + (int64_t)(i / vpr) * s_n + (i % vpr) * 8);
      mx = umax32(mx, absmax_bf16x8(v[j]));
    }
    mx = group_umax<64>(mx);
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
    __syncthreads();
    mx = umax32(umax32(wmax[0], wmax[1]), umax32(wmax[2], wmax[3]));
    const Int8BlockScale sc(mx);
    if (threadIdx.x == 0) scale[(b * H + head) * nb + blk] = sc.scale;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int i = threadIdx.x + j * 256;
      if (i < nvec) *reinterpret_cast<uint2 *>(dst + (int64_t)(i / vpr) * Dp + (i % vpr) * 8) = sc.quantize8(v[j]);
    }
    if (Dp != D) {  // D % 16 == 8: eight pad columns per row
      for (int rr = threadIdx.x; rr < rows; rr += 256) *reinterpret_cast<uint2 *>(dst + (int64_t)rr * Dp + D) = make_uint2(0, 0);
    }
    return;
  }
  for (int i = threadIdx.x; i < rows * D; i += 256) mx = umax32(mx, src[(int64_t)(i / D) * s_n + i % D] & 0x7fffu);
  mx = group_umax<64>(mx);
  if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = mx;
  __syncthreads();
  mx = umax32(umax32(wmax[0], wmax[1]), umax32(wmax[2], wmax[3]));
  const float sc = bf16_bits_to_f32(mx) / 127.0f;
  if (threadIdx.x == 0) scale[(b * H + head) * nb + blk] = sc;
  for (int i = threadIdx.x; i < rows * Dp; i += 256) {
    const int rr = i / Dp, c = i % Dp;
    float q = 0.0f;
    if (c < D && sc != 0.0f) q = bf16_bits_to_f32(src[(int64_t)rr * s_n + c]) / sc;
    dst[i] = (int8_t)(int)q;  // toward zero; |q| <= 127 up to rounding
  }
}

// one kernel per number of tiles (any, 1, 2) and cut (1, 2, 4)
static void (*const mha_nvfp4_kernels[3][3])(MhaArgs, MhaWork) = {
    {mha_nvfp4_fwd_kernel<1, 0>, mha_nvfp4_fwd_kernel<2, 0>, mha_nvfp4_fwd_kernel<4, 0>},
    {mha_nvfp4_fwd_kernel<1, 1>, mha_nvfp4_fwd_kernel<2, 1>, mha_nvfp4_fwd_kernel<4, 1>},
    {mha_nvfp4_fwd_kernel<1, 2>, mha_nvfp4_fwd_kernel<2, 2>, mha_nvfp4_fwd_kernel<4, 2>}};
// (row 0: eight waves.  One and two tiles always run four: kernel alone, us, eight / four: 8192 heads of 49 x 49, D = 32, 143 / 75; of
// 64 x 64 151 / 81, of 128 x 128 211 / 124, D = 64; 1024 of 256 x 256, D = 64, 40.5 / 36.9; 40 of 4096 x 77 27.4 / 22.8, of 16384 x 200
// 114 / 98; 300 of 200 x 200, D = 64, 16.7 / 16.6)
static void (*const mha_int8_x_fp8_kernels[4][3])(Mha8Args, MhaWork) = {
    {mha_int8_x_fp8_fwd_kernel<1>, mha_int8_x_fp8_fwd_kernel<2>, mha_int8_x_fp8_fwd_kernel<4>},
    {mha_int8_x_fp8_fwd4_kernel<1, 1>, mha_int8_x_fp8_fwd4_kernel<2, 1>, mha_int8_x_fp8_fwd4_kernel<4, 1>},
    {mha_int8_x_fp8_fwd4_kernel<1, 2>, mha_int8_x_fp8_fwd4_kernel<2, 2>, mha_int8_x_fp8_fwd4_kernel<4, 2>},
    {mha_int8_x_fp8_fwd4_kernel<1, 0>, mha_int8_x_fp8_fwd4_kernel<2, 0>, mha_int8_x_fp8_fwd4_kernel<4, 0>}};

// A launch carries fewer than 2^32 threads along a grid dim: from 2^31 on the heads go out in several launches, each planned
// by itself.
constexpr int64_t MHA_MAX_BLOCKS = 1 << 22;
static int64_t mha_heads_per_launch(int64_t Nq) {
  const int64_t blocks = ceil_div(Nq, 256);
  return blocks < MHA_MAX_BLOCKS ? MHA_MAX_BLOCKS / blocks : 1;
}

template <typename Args>
static int mha_launch(const Args &a, const MhaPlan &p, void (*kern)(Args, MhaWork), std::atomic<uint32_t> &lds_done, int lds, int threads,
                      hipStream_t st) {
  // more than 64 KB of dynamic LDS has to be allowed once per device and kernel
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = 0;
  const uint32_t bit = 1u << (dev & 31);
  if (!(lds_done.load(std::memory_order_relaxed) & bit)) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (e != hipSuccess) return set_error("hipFuncSetAttribute(LDS=%d): %s", lds, hipGetErrorString(e));
    lds_done.fetch_or(bit, std::memory_order_relaxed);
  }
  hipLaunchKernelGGL(kern, dim3(p.grid), dim3(threads), lds, st, a, p.work);
  return 0;
}

}  // namespace ac4k

using namespace ac4k;

extern "C" __attribute__((visibility("default"))) int ac4k_mha_nvfp4_fwd(
    void *O, int64_t o_b_stride, int64_t o_h_stride, int64_t o_n_stride, int64_t o_d_stride, const void *q, const void *q_sf,
    const float *q_gs, const void *k, const void *k_sf, const float *k_gs, const void *v, const void *v_sf, const float *v_gs,
    int64_t B, int64_t H, int64_t Nq, int64_t Nkv, int64_t Dqk, int64_t Dv, float sm_scale, ac4k_stream_t stream) {
  AC4K_REQUIRE(O && q && q_sf && q_gs && k && k_sf && k_gs && v && v_sf && v_gs, "null pointer argument");
  AC4K_REQUIRE(B >= 1 && H >= 1 && Nq >= 1 && Nkv >= 1, "B, H, Nq, Nkv must be positive (B=%lld H=%lld Nq=%lld Nkv=%lld)",
               (long long)B, (long long)H, (long long)Nq, (long long)Nkv);
  AC4K_REQUIRE(Dqk % 16 == 0, "Dqk must be multiple of 16");
  AC4K_REQUIRE(Dqk <= 128 && Dv <= 128, "Dqk and Dv must not exceed 128");
  AC4K_REQUIRE(Dqk % 64 == 0 && Dqk >= 64 && Dv >= 1,
               "Dqk must be 64 or 128 (packed rows of whole 64-chunks, as the quantizer writes them) and Dv positive (Dqk=%lld Dv=%lld)",
               (long long)Dqk, (long long)Dv);
  AC4K_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 15) == 0 && (((uintptr_t)q_sf | (uintptr_t)k_sf | (uintptr_t)v_sf) & 3) == 0,
               "q, k, v must be 16-byte aligned and the scale tensors 4-byte aligned");
  AC4K_REQUIRE(H <= 65535 && B <= 65535 && ceil_div(Nq, 128) < (1ll << 31), "problem too large");
  AC4K_REQUIRE(o_b_stride >= 0 && o_h_stride >= 0 && o_n_stride >= 1 && o_d_stride >= 1, "strides of O must be positive");
  MhaArgs a{static_cast<uint16_t *>(O), o_b_stride, o_h_stride, o_n_stride, o_d_stride,
            static_cast<const uint8_t *>(q), static_cast<const uint8_t *>(k), static_cast<const uint8_t *>(v),
            static_cast<const uint8_t *>(q_sf), static_cast<const uint8_t *>(k_sf), static_cast<const uint8_t *>(v_sf),
            q_gs, k_gs, v_gs, (uint32_t)H, 0, Nq, Nkv, align_up(Nq, 16), align_up(Nkv, 16), align_up(Nkv, 64), (int)(Dqk / 64), (int)Dv,
            (int)align_up(Dv, 16), sm_scale,
            (o_d_stride == 1 && Dv % 8 == 0 && ((uintptr_t)O & 15) == 0 && o_b_stride % 8 == 0 && o_h_stride % 8 == 0 && o_n_stride % 8 == 0) ? 1 : 0};
  // measured: 512 x 2 x 128 to 8192 x 4 x 128 and 16384 x 40 on 4096 to 16384 keys
  static constexpr MhaCost cost{{5.0f, 6.0f, 5.5f}, {3.9f, 2.35f, 1.6f}};
  static std::atomic<uint32_t> lds_done[3][3];
  const int64_t ntiles = ceil_div(Nkv, 128), heads = B * H, most = mha_heads_per_launch(Nq);
  for (int64_t head0 = 0; head0 < heads; head0 += most) {
    const MhaPlan p = mha_plan(cost, heads - head0 < most ? heads - head0 : most, Nq, ntiles);
    const int tiles = ntiles <= 2 ? (int)ntiles : 0;
    a.head0 = (uint32_t)head0;
    if (int rc = mha_launch(a, p, mha_nvfp4_kernels[tiles][p.tail >> 1], lds_done[tiles][p.tail >> 1], MHA_LDS, 512, (hipStream_t)stream)) return rc;
  }
  return check_launch("ac4k_mha_nvfp4_fwd");
}

// Replaces ac4k::mha_int8_x_fp8_fwd (lib/cuda/sm120/mha_int8_x_fp8.cu:979-1137).
extern "C" __attribute__((visibility("default"))) int ac4k_mha_int8_x_fp8_fwd(
    void *O, int64_t o_b_stride, int64_t o_h_stride, int64_t o_n_stride, int64_t o_d_stride, const void *q,
    const float *q_sf, int q_quantize_block_size, const void *k, const float *k_sf, int k_quantize_block_size, const void *v,
    const float *v_sf, int64_t B, int64_t H, int64_t Nq, int64_t Nkv, int64_t Dqk, int64_t Dv, float sm_scale,
    ac4k_stream_t stream) {
  AC4K_REQUIRE(O && q && q_sf && k && k_sf && v && v_sf, "null pointer argument");
  AC4K_REQUIRE(B >= 1 && H >= 1 && Nq >= 1 && Nkv >= 1, "B, H, Nq, Nkv must be positive (B=%lld H=%lld Nq=%lld Nkv=%lld)",
               (long long)B, (long long)H, (long long)Nq, (long long)Nkv);
  AC4K_REQUIRE(Dqk % 16 == 0, "Dqk must be multiple of 16");
  AC4K_REQUIRE(Dqk <= 128 && Dv <= 128, "Dqk and Dv must not exceed 128");
  AC4K_REQUIRE(q_quantize_block_size == 32 || q_quantize_block_size == 64, "q_quantize_block_size must be 32 or 64 (got %d)",
               q_quantize_block_size);
  AC4K_REQUIRE(k_quantize_block_size == 128, "k_quantize_block_size must be 128 (got %d)", k_quantize_block_size);
  AC4K_REQUIRE(Dqk >= 16 && Dv >= 1, "Dqk and Dv must be positive");
  AC4K_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)v_sf) & 15) == 0,
               "q, k, v and v_sf must be 16-byte aligned");
  AC4K_REQUIRE(H <= 65535 && B <= 65535 && ceil_div(Nq, 128) < (1ll << 31), "problem too large");
  AC4K_REQUIRE(o_b_stride >= 0 && o_h_stride >= 0 && o_n_stride >= 1 && o_d_stride >= 1, "strides of O must be positive");
  Mha8Args a{static_cast<uint16_t *>(O), o_b_stride, o_h_stride, o_n_stride, o_d_stride,
             static_cast<const int8_t *>(q), static_cast<const int8_t *>(k), static_cast<const uint8_t *>(v),
             q_sf, k_sf, v_sf, (uint32_t)H, 0, Nq, Nkv, align_up(Nkv, 16), ceil_div(Nq, q_quantize_block_size), ceil_div(Nkv, 128),
             (int)Dqk, (int)Dv, (int)align_up(Dv, 16), q_quantize_block_size, sm_scale,
             (o_d_stride == 1 && Dv % 8 == 0 && ((uintptr_t)O & 15) == 0 && o_b_stride % 8 == 0 && o_h_stride % 8 == 0 && o_n_stride % 8 == 0) ? 1 : 0};
  // measured: 4096 rows of 1 to 40 heads on 1024 and 8192 keys, D = 128, every split of both kernels
  static constexpr MhaCost cost{{6.7f, 5.0f, 4.1f}, {2.36f, 1.43f, 1.06f}};
  static constexpr Mha4Cost cost4{{{2.9f, 2.7f, 2.1f}, {1.50f, 1.10f, 0.905f}}, {{6.7f, 4.7f, 4.3f}, {2.50f, 1.55f, 1.21f}}};
  static std::atomic<uint32_t> lds_done[4][3];
  const int64_t ntiles = ceil_div(Nkv, 128), heads = B * H, most = mha_heads_per_launch(Nq);
  for (int64_t head0 = 0; head0 < heads; head0 += most) {
    const int64_t n = heads - head0 < most ? heads - head0 : most;
    MhaPlan p = mha4_plan(cost4, n, Nq, ntiles);
    int kind = ntiles <= 2 ? (int)ntiles : 3;
    if (ntiles > 2) {
      const MhaPlan p8 = mha_plan(cost, n, Nq, ntiles);
      if (p8.us <= p.us) p = p8, kind = 0;
    }
    a.head0 = (uint32_t)head0;
    const int waves = kind == 0 ? 8 : 4;
    if (int rc = mha_launch(a, p, mha_int8_x_fp8_kernels[kind][p.tail >> 1], lds_done[kind][p.tail >> 1],
                            mha8_lds_bytes(waves, p.tail), waves * 64, (hipStream_t)stream)) return rc;
  }
  return check_launch("ac4k_mha_int8_x_fp8_fwd");
}

// Replaces _int8_quantize / _triton_block_token_quantize (python/ac4k_kernel/ops/attention.py:18-99): x bf16 with element
// strides (s_b, s_h, s_n, 1) over [B, H, N, D] -> y int8 [B, H, N, align_up(D, 16)], scale fp32 [B, H, ceil(N / block)].
extern "C" __attribute__((visibility("default"))) int ac4k_quantize_int8_token_block_bf16(
    void *y, float *scale, const void *x, int64_t B, int64_t H, int64_t N, int64_t D, int64_t s_b, int64_t s_h, int64_t s_n,
    int block, ac4k_stream_t stream) {
  AC4K_REQUIRE(y && scale && x, "null pointer argument");
  AC4K_REQUIRE(B >= 1 && H >= 1 && N >= 1 && D >= 1, "B, H, N, D must be positive");
  AC4K_REQUIRE(block >= 16 && (block & (block - 1)) == 0, "the block size must be a power of two, at least 16 (got %d)", block);
  AC4K_REQUIRE(D <= 1024 && block <= 1024, "D and the block size must not exceed 1024");
  AC4K_REQUIRE(H <= 65535 && B <= 65535 && ceil_div(N, (int64_t)block) < (1ll << 31), "problem too large");
  hipLaunchKernelGGL(quantize_int8_token_block_kernel, dim3((unsigned)ceil_div(N, (int64_t)block), (unsigned)H, (unsigned)B),
                     dim3(256), 0, (hipStream_t)stream, static_cast<int8_t *>(y), scale, static_cast<const uint16_t *>(x), s_b,
                     s_h, s_n, H, N, (int)D, (int)align_up(D, 16), block,
                     (D % 8 == 0 && ((uintptr_t)x & 15) == 0 && s_b % 8 == 0 && s_h % 8 == 0 && s_n % 8 == 0) ? 1 : 0);
  return check_launch("ac4k_quantize_int8_token_block_bf16");
}

// Whole attention calls on bf16 operands: the quantizers of attention_quantize.hip, then the forward on their outputs.
// q_tile: query rows that a workgroup of the quantizers takes, beside 128 keys and 256 positions of V; 2^24 workgroups of
// 256 threads would be 2^32 threads, more than a launch carries
static int attention_check_sizes(int64_t B, int64_t H, int64_t Nq, int64_t Nkv, int64_t Dqk, int64_t Dv, int q_tile) {
  AC4K_REQUIRE(B >= 1 && H >= 1 && Nq >= 1 && Nkv >= 1, "B, H, Nq, Nkv must be positive (B=%lld H=%lld Nq=%lld Nkv=%lld)",
               (long long)B, (long long)H, (long long)Nq, (long long)Nkv);
  AC4K_REQUIRE(Dqk >= 8 && Dqk <= 128 && Dv >= 8 && Dv <= 128, "Dqk and Dv must be 8 to 128");
  AC4K_REQUIRE(H <= 65535 && B <= 65535 && Nq < (1ll << 30) && Nkv < (1ll << 30) &&
               B * H * (ceil_div(Nq, (int64_t)q_tile) + ceil_div(Nkv, 128) + ceil_div(Nkv, 256)) < (1ll << 24), "problem too large");
  return 0;
}
template <typename Args>
static int attention_operands(Args &a, const void *q, int64_t q_b, int64_t q_h, int64_t q_n, const void *k, int64_t k_b, int64_t k_h,
                              int64_t k_n, const void *v, int64_t v_b, int64_t v_h, int64_t v_n, const void *workspace) {
  AC4K_REQUIRE(q && k && v && workspace, "null pointer argument");
  AC4K_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v) & 1) == 0 && ((uintptr_t)workspace & 15) == 0,
               "q, k, v must be 2-byte aligned and the workspace 16-byte aligned");
  AC4K_REQUIRE(q_b >= 0 && q_h >= 0 && q_n >= 0 && k_b >= 0 && k_h >= 0 && k_n >= 0 && v_b >= 0 && v_h >= 0 && v_n >= 0,
               "strides of q, k and v must not be negative");
  a.q = {static_cast<const uint16_t *>(q), q_b, q_h, q_n};
  a.k = {static_cast<const uint16_t *>(k), k_b, k_h, k_n};
  a.v = {static_cast<const uint16_t *>(v), v_b, v_h, v_n};
  return 0;
}

// Replaces _int8_x_fp8_attention (python/ac4k_kernel/ops/attention.py:137-190): the quantizers of attention_quantize.hip,
// then ac4k_mha_int8_x_fp8_fwd on their outputs.
static int attention_int8_args(AttnQuantArgs &a, int64_t B, int64_t H, int64_t Nq, int64_t Nkv, int64_t Dqk, int64_t Dv) {
  if (int rc = attention_check_sizes(B, H, Nq, Nkv, Dqk, Dv, AQ_Q_BLOCK)) return rc;
  a = AttnQuantArgs{};
  a.B = (int)B, a.H = (int)H, a.Nq = (int)Nq, a.Nkv = (int)Nkv, a.D = (int)Dqk, a.Dv = (int)Dv;
  return 0;
}

extern "C" __attribute__((visibility("default"))) int64_t ac4k_attention_int8_x_fp8_workspace_bytes(
    int64_t B, int64_t H, int64_t Nq, int64_t Nkv, int64_t Dqk, int64_t Dv) {
  AttnQuantArgs a;
  if (attention_int8_args(a, B, H, Nq, Nkv, Dqk, Dv)) return -1;
  return attn_quant_layout(a, nullptr);
}

// checks and plan of the quantizers; rc != 0: the call is refused
static int attention_int8_plan(AttnQuantArgs &a, const void *q, int64_t q_b, int64_t q_h, int64_t q_n, const void *k, int64_t k_b, int64_t k_h,
                               int64_t k_n, const void *v, int64_t v_b, int64_t v_h, int64_t v_n, int64_t B, int64_t H, int64_t Nq, int64_t Nkv,
                               int64_t Dqk, int64_t Dv, float v_scale_max, void *workspace, int64_t workspace_bytes) {
  if (int rc = attention_int8_args(a, B, H, Nq, Nkv, Dqk, Dv)) return rc;
  if (int rc = attention_operands(a, q, q_b, q_h, q_n, k, k_b, k_h, k_n, v, v_b, v_h, v_n, workspace)) return rc;
  AC4K_REQUIRE(v_scale_max > 0.0f, "v_scale_max must be positive");
  const int64_t need = attn_quant_layout(a, workspace);
  AC4K_REQUIRE(workspace_bytes >= need, "workspace too small: %lld bytes, %lld needed", (long long)workspace_bytes, (long long)need);
  a.v_smax = v_scale_max;
  attn_quant_plan(a);
  return 0;
}

extern "C" __attribute__((visibility("default"))) int64_t ac4k_debug_attention_quantize_int8_x_fp8(
    const void *q, int64_t q_b_stride, int64_t q_h_stride, int64_t q_n_stride, const void *k, int64_t k_b_stride, int64_t k_h_stride,
    int64_t k_n_stride, const void *v, int64_t v_b_stride, int64_t v_h_stride, int64_t v_n_stride, int64_t B, int64_t H, int64_t Nq,
    int64_t Nkv, int64_t Dqk, int64_t Dv, float v_scale_max, void *workspace, int64_t workspace_bytes, int two_launches, int *launches,
    ac4k_stream_t stream) {
  AttnQuantArgs a;
  if (attention_int8_plan(a, q, q_b_stride, q_h_stride, q_n_stride, k, k_b_stride, k_h_stride, k_n_stride, v, v_b_stride, v_h_stride,
                          v_n_stride, B, H, Nq, Nkv, Dqk, Dv, v_scale_max, workspace, workspace_bytes)) return -1;
  if (two_launches) a.classes = 0;
  launch_attn_quant(a, (hipStream_t)stream);
  if (launches) *launches = a.classes > 0 ? 1 : 2;
  return check_launch("ac4k_debug_attention_quantize_int8_x_fp8") ? -1 : (char *)a.ksum - (char *)workspace;
}

extern "C" __attribute__((visibility("default"))) int ac4k_attention_int8_x_fp8_bf16(
    void *O, int64_t o_b_stride, int64_t o_h_stride, int64_t o_n_stride, int64_t o_d_stride, const void *q, int64_t q_b_stride,
    int64_t q_h_stride, int64_t q_n_stride, const void *k, int64_t k_b_stride, int64_t k_h_stride, int64_t k_n_stride,
    const void *v, int64_t v_b_stride, int64_t v_h_stride, int64_t v_n_stride, int64_t B, int64_t H, int64_t Nq, int64_t Nkv,
    int64_t Dqk, int64_t Dv, float v_scale_max, float sm_scale, void *workspace, int64_t workspace_bytes, ac4k_stream_t stream) {
  AC4K_REQUIRE(O, "null pointer argument");
  AttnQuantArgs a;
  if (int rc = attention_int8_plan(a, q, q_b_stride, q_h_stride, q_n_stride, k, k_b_stride, k_h_stride, k_n_stride, v, v_b_stride,
                                   v_h_stride, v_n_stride, B, H, Nq, Nkv, Dqk, Dv, v_scale_max, workspace, workspace_bytes)) return rc;
  launch_attn_quant(a, (hipStream_t)stream);
  if (int rc = check_launch("ac4k_attention_int8_x_fp8_bf16")) return rc;
  return ac4k_mha_int8_x_fp8_fwd(O, o_b_stride, o_h_stride, o_n_stride, o_d_stride, a.q8, a.q_sf, AQ_Q_BLOCK, a.k8, a.k_sf, AQ_K_BLOCK,
                                 a.v8, a.v_sf, B, H, Nq, Nkv, a.Dp, Dv, sm_scale, stream);
}

// Replaces _nvfp4_attention (python/ac4k_kernel/ops/attention.py:100-133).
static int attention_nvfp4_args(AttnNvfp4Args &a, int64_t B, int64_t H, int64_t Nq, int64_t Nkv, int64_t Dqk, int64_t Dv) {
  if (int rc = attention_check_sizes(B, H, Nq, Nkv, Dqk, Dv, 128)) return rc;
  a = AttnNvfp4Args{};
  a.B = (int)B, a.H = (int)H, a.Nq = (int)Nq, a.Nkv = (int)Nkv, a.D = (int)Dqk, a.Dv = (int)Dv;
  return 0;
}

extern "C" __attribute__((visibility("default"))) int64_t ac4k_attention_nvfp4_workspace_bytes(int64_t B, int64_t H, int64_t Nq,
                                                                                               int64_t Nkv, int64_t Dqk, int64_t Dv) {
  AttnNvfp4Args a;
  if (attention_nvfp4_args(a, B, H, Nq, Nkv, Dqk, Dv)) return -1;
  return attn_nvfp4_layout(a, nullptr);
}

extern "C" __attribute__((visibility("default"))) int ac4k_attention_nvfp4_bf16(
    void *O, int64_t o_b_stride, int64_t o_h_stride, int64_t o_n_stride, int64_t o_d_stride, const void *q, int64_t q_b_stride,
    int64_t q_h_stride, int64_t q_n_stride, const void *k, int64_t k_b_stride, int64_t k_h_stride, int64_t k_n_stride,
    const void *v, int64_t v_b_stride, int64_t v_h_stride, int64_t v_n_stride, int64_t B, int64_t H, int64_t Nq, int64_t Nkv,
    int64_t Dqk, int64_t Dv, float max_scale, float sm_scale, void *workspace, int64_t workspace_bytes, ac4k_stream_t stream) {
  AC4K_REQUIRE(O, "null pointer argument");
  AttnNvfp4Args a;
  if (int rc = attention_nvfp4_args(a, B, H, Nq, Nkv, Dqk, Dv)) return rc;
  if (int rc = attention_operands(a, q, q_b_stride, q_h_stride, q_n_stride, k, k_b_stride, k_h_stride, k_n_stride, v, v_b_stride,
                                  v_h_stride, v_n_stride, workspace)) return rc;
  // the maxima are taken over the whole tensors: [B,N,H,D] or [B,H,N,D] without gaps (dims of one element carry any stride)
  auto dense = [&](const AttnOperand &t, int64_t N, int64_t D) {
    const bool bnhd = (t.s_h == D || H == 1) && (t.s_n == H * D || N == 1), bhnd = (t.s_n == D || N == 1) && (t.s_h == N * D || H == 1);
    return (bnhd || bhnd) && (t.s_b == H * N * D || B == 1);
  };
  AC4K_REQUIRE(dense(a.q, Nq, Dqk) && dense(a.k, Nkv, Dqk) && dense(a.v, Nkv, Dv), "q, k and v must be dense");
  a.max_scale = max_scale;
  const int64_t need = attn_nvfp4_layout(a, workspace);
  AC4K_REQUIRE(workspace_bytes >= need, "workspace too small: %lld bytes, %lld needed", (long long)workspace_bytes, (long long)need);
  launch_attn_nvfp4(a, (hipStream_t)stream);
  if (int rc = check_launch("ac4k_attention_nvfp4_bf16")) return rc;
  return ac4k_mha_nvfp4_fwd(O, o_b_stride, o_h_stride, o_n_stride, o_d_stride, a.q4, a.q_sf, a.gs, a.k4, a.k_sf, a.gs + 1, a.v4, a.v_sf,
                            a.gs + 2, B, H, Nq, Nkv, a.Dp, Dv, sm_scale, stream);
}
