// Pieces shared by the Q4_K matrix-core kernels (the prefill GEMM and the routed-expert kernels):
// direct HBM -> LDS loads, the power-of-two row scale of the fp16 activation copies, the
// in-register super-block decode (src/core/numerics/quant.cpp:58-70,656-675) and the tile loop.
#pragma once

#include <type_traits>

#include "qmm_device.hpp"

namespace qmm {
namespace {

// Largest |v| over a 256-thread workgroup (every thread returns it).
__device__ __forceinline__ float block_amax(float v, float* red) {
  v = wave_max(v);
  if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const float r = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  __syncthreads();
  return r;
}

// Power-of-two scale that brings a row with largest magnitude `amax` to [1024, 2048): the
// fp16 copy then neither overflows nor loses small values to subnormals, and the scaling itself
// is exact.  Zero rows (and non-finite ones) get scale 1.
__device__ __forceinline__ float row_scale_for(float amax) {
  const uint32_t e = (bit_cast<uint32_t>(amax) >> 23) & 0xFFu;
  if (e == 0u || e == 0xFFu) return 1.0f;
  const int se = static_cast<int>(e) - 10;
  return bit_cast<float>(static_cast<uint32_t>(se < 1 ? 1 : se) << 23);
}

__device__ __forceinline__ half8_t to_f16_group(const float4& lo, const float4& hi, float inv) {
  // the order 0,2,1,3,4,6,5,7 inside each group of 8 (what the in-register weight decode yields)
  half8_t v;
  v[0] = static_cast<_Float16>(lo.x * inv), v[1] = static_cast<_Float16>(lo.z * inv);
  v[2] = static_cast<_Float16>(lo.y * inv), v[3] = static_cast<_Float16>(lo.w * inv);
  v[4] = static_cast<_Float16>(hi.x * inv), v[5] = static_cast<_Float16>(hi.z * inv);
  v[6] = static_cast<_Float16>(hi.y * inv), v[7] = static_cast<_Float16>(hi.w * inv);
  return v;
}

// body(integral_constant<int, 0>) ... body(integral_constant<int, N - 1>), in order.
template <int N, int I = 0, typename F>
__device__ __forceinline__ void unrolled(F&& body) {
  if constexpr (I < N) {
    body(std::integral_constant<int, I>{});
    unrolled<N, I + 1>(body);
  }
}

// Two packed fp16 weights RN16(fma(q, dsc, ndmm)) from the nibbles (low: HI = 0, high: HI = 1) of
// bytes 0 and 2 of `x`.  A nibble masked in place inside a 16-bit half is the fp16 subnormal
// q * 2^-24 (16 q * 2^-24 for a high nibble), which the mixed-precision multiply-add reads as it
// is: `dsc24` is d*sc * 2^24 (d*sc * 2^20 for high nibbles), so the fp32 result is exactly
// DequantizeQ4K's and one instruction per weight forms it and rounds it to fp16.
template <int HI>
__device__ __forceinline__ half2_t decode_pair(uint32_t x, float dsc24, float ndmm) {
  const half2_t q = bit_cast<half2_t>(x & (HI ? 0x00F000F0u : 0x000F000Fu));
  return half2_t{static_cast<_Float16>(fmaf(static_cast<float>(q[0]), dsc24, ndmm)),
                 static_cast<_Float16>(fmaf(static_cast<float>(q[1]), dsc24, ndmm))};
}

// The 6-bit scales and mins of a super-block, one byte each (src/core/numerics/quant.cpp:58-70):
// sc[0], mn[0] hold sub-blocks 0..3, sc[1], mn[1] sub-blocks 4..7.
struct ScaleBytes {
  uint32_t sc[2], mn[2];
};
__device__ __forceinline__ ScaleBytes unpack_scales(uint32_t s0, uint32_t s1, uint32_t s2) {
  ScaleBytes r;
  r.sc[0] = s0 & 0x3F3F3F3Fu;
  r.mn[0] = s1 & 0x3F3F3F3Fu;
  r.sc[1] = (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
  r.mn[1] = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
  return r;
}

// (d * sc * 2^24, -(dmin * mn)) of sub-block SB in fp32, both exact (11-bit header times 6-bit
// integer; the 2^24 undoes the subnormal reading of the nibbles in decode_pair).  Odd sub-blocks
// live in the high nibbles, which read as 16 q: their factor is 2^20.
struct ScaleMin {
  float dsc, ndmm;
};
template <int SB>
__device__ __forceinline__ ScaleMin scale_min_f32(const ScaleBytes& sbytes, float d, float ndmin) {
  const float sc = static_cast<float>((sbytes.sc[SB >> 2] >> (8 * (SB & 3))) & 0xFFu);
  const float mn = static_cast<float>((sbytes.mn[SB >> 2] >> (8 * (SB & 3))) & 0xFFu);
  return ScaleMin{d * sc * ((SB & 1) ? 0x1p20f : 0x1p24f), ndmin * mn};
}

// Header of the super-block at `raw` (a lane's weight row inside a raw LDS stage): d, -dmin and
// the unpacked 6-bit scales and mins.
struct BlockHead {
  float d, ndmin;
  ScaleBytes sbytes;
};
__device__ __forceinline__ BlockHead block_head(const uint4& head) {
  return BlockHead{half_bits_to_float(head.x & 0xFFFFu), -half_bits_to_float(head.x >> 16),
                   unpack_scales(head.y, head.z, head.w)};
}
__device__ __forceinline__ BlockHead load_block_head(const uint8_t* raw) {
  return block_head(*reinterpret_cast<const uint4*>(raw));
}

// Sub-block SB lives in the low (even SB) or high nibbles of bytes (SB/2)*32 + [0,32) of the quants
// (src/core/numerics/quant.cpp:656-675): the sixteen bytes of K half `kg`, which serve SB and SB ^ 1.
template <int SB>
__device__ __forceinline__ void load_nibbles(const uint8_t* raw, uint32_t kg, uint32_t (&qw)[4]) {
  const uint4 q = *reinterpret_cast<const uint4*>(raw + 16 + (SB >> 1) * 32 + kg * 16u);
  qw[0] = q.x, qw[1] = q.y, qw[2] = q.z, qw[3] = q.w;
}

// The B operand of matrix step `tt` of a sub-block (32 weights of one row) for a lane of K half `kg`: the weights
// 16kg + 8tt + [0,8) in the order 0,2,1,3,4,6,5,7 (any assignment of the sub-block's K positions to matrix steps and lane
// halves will do as long as the activation fragments follow it; this one lets a lane take its sixteen bytes with ONE
// 16-byte LDS read, which sixteen lanes 144 bytes apart make without a bank conflict, where two 8-byte reads a lane put
// lanes l and l + 16 on the same banks).  HI: its nibbles are the high ones.
template <int HI>
__device__ __forceinline__ half8_t decode_eight(uint32_t x, uint32_t y, const ScaleMin& sm) {
  const half2_t p0 = decode_pair<HI>(x, sm.dsc, sm.ndmm), p1 = decode_pair<HI>(x >> 8, sm.dsc, sm.ndmm);
  const half2_t p2 = decode_pair<HI>(y, sm.dsc, sm.ndmm), p3 = decode_pair<HI>(y >> 8, sm.dsc, sm.ndmm);
  return half8_t{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}
template <int HI>
__device__ __forceinline__ half8_t decode_step(const uint32_t (&qw)[4], int tt, const ScaleMin& sm) {
  return decode_eight<HI>(qw[2 * tt], qw[2 * tt + 1], sm);
}

// Both steps of sub-block SB; an odd one decodes the bytes its even predecessor loaded, so `qw` (the words) and `qs8` (the
// same shifted down one byte, for bytes 1 and 3) are carried from that call.
template <int SB>
__device__ __forceinline__ void decode_subblock(const uint8_t* raw, uint32_t kg, const BlockHead& h, uint32_t (&qw)[4],
                                                uint32_t (&qs8)[4], half8_t (&b)[2]) {
  constexpr int kHi = SB & 1;
  const ScaleMin sm = scale_min_f32<SB>(h.sbytes, h.d, h.ndmin);
  if (kHi == 0) {
    load_nibbles<SB>(raw, kg, qw);
#pragma unroll
    for (int x = 0; x < 4; ++x) qs8[x] = qw[x] >> 8;
  }
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const half2_t p0 = decode_pair<kHi>(qw[2 * tt], sm.dsc, sm.ndmm), p1 = decode_pair<kHi>(qs8[2 * tt], sm.dsc, sm.ndmm);
    const half2_t p2 = decode_pair<kHi>(qw[2 * tt + 1], sm.dsc, sm.ndmm), p3 = decode_pair<kHi>(qs8[2 * tt + 1], sm.dsc, sm.ndmm);
    b[tt] = half8_t{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
  }
}

// Wavefronts of a BM x BN tile whose wavefronts each own WM rows x WN columns.
template <int BM, int BN, int WM, int WN>
constexpr int tile_waves() { return (BM / WM) * (BN / WN); }

// A wavefront's sums: WM / 32 by WN / 32 matrix tiles.
template <int WM, int WN>
using TileSums = float16_t[WM / 32][WN / 32];

// The sums of one BM x BN tile of C at (m0, n0) over `blocks` super-blocks of K from the matrix's block `blk0` on.  A
// wavefront owns WM rows x WN columns of it.  Every MFMA takes its activation fragment from LDS (1 KB a
// wavefront, against 128 bytes a clock for the whole CU, which four SIMDs running 32-clock MFMAs
// would need in full); with WN = 64 a fragment read feeds two MFMAs.  The price is that the
// BM / WM wavefronts that share a column range each decode its weights.
//
// PAIR: the tile's columns are BN / 2 of either matrix, gate weights `w` and up weights `w_up`, and a wavefront's two column
// tiles the same columns of both, so that silu(A Wg^T) * (A Wu^T) is formed in its registers: no product goes to memory, and
// the activations are read once.
//
// No direct load is in flight when it returns; LDS may be used again after a barrier.
template <int BM, int BN, int WM, int WN, bool PAIR = false, int KSETS = 1>
__device__ __forceinline__ void q4k_tile_sums(TileSums<WM / KSETS, WN>& out, const _Float16* __restrict__ a16, const uint8_t* __restrict__ w,
                                              uint32_t m, uint32_t n, uint32_t k, uint32_t m0, uint32_t n0, uint32_t blk0,
                                              uint32_t blocks, const uint8_t* __restrict__ w_up = nullptr) {
  constexpr int kWaves = tile_waves<BM, BN, WM, WN>() * KSETS;
  constexpr int kWavesN = BN / WN;
  constexpr int kTI = WM / 32, kTJ = WN / 32;      // MFMA tiles per wavefront: rows x columns
  constexpr int kABlk = BM / 16 / kWaves;          // 1 KB activation blocks a wavefront loads per step
  constexpr int kWL = (BN * 9 + 64 * kWaves - 1) / (64 * kWaves);  // 1 KB weight blocks per super-block
  constexpr uint32_t kAStage = BM * 64, kWStage = kWL * kWaves * 1024;
  constexpr uint32_t kJRows = PAIR ? BN / 2 : 32;  // weight rows from a wavefront's column tile to its next
  static_assert(!PAIR || (kTJ == 2 && BN * 9 % 128 == 0), "a load block lies in one matrix");
  static_assert(KSETS == 1 || (KSETS == 2 && WM == BM && kTI % 2 == 0 && !PAIR), "two sets share a tile of one row of wavefronts");
  static_assert(KSETS == 1 || (kTJ == 2 && (kWavesN & (kWavesN - 1)) == 0), "two sets: one decode in each half of a slice, partners a bit apart");
  static_assert(BM % WM == 0 && BN % WN == 0 && WM % 32 == 0 && WN % 32 == 0 && BM % (16 * kWaves) == 0, "tile shape");
  __shared__ __attribute__((aligned(16))) uint8_t lds[4 * kAStage + 2 * kWStage];

  const uint32_t t = threadIdx.x, lane = t & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t wave_m = KSETS == 2 ? 0u : wave / kWavesN, wave_n = wave % kWavesN, set = wave / kWavesN;
  const uint32_t l32 = lane & 31u, kg = lane >> 5;
  const uint32_t row_blocks = k / 256;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) uint8_t*)lds));
  const uint8_t* a_tile = reinterpret_cast<const uint8_t*>(a16) + static_cast<size_t>(m0) * k * 2 + blk0 * 512u;
  const uint8_t* w_tile = w + (static_cast<size_t>(n0) * row_blocks + blk0) * 144;
  const uint8_t* up_tile = PAIR ? w_up + (static_cast<size_t>(n0) * row_blocks + blk0) * 144 : nullptr;

  // Direct loads.  Activation block L of a step (1 KB, rows 16L..16L+15, four 16-byte chunks
  // a row): lane p fetches row 16L + p/4, chunk (p%4) ^ ((row>>2)&3).  Weight chunk q of a
  // super-block column (q = 9*row + part, 144 bytes a row): the tile's blocks are copied as
  // they lie, 64 chunks a load; chunks past the tile repeat its last chunk into spare LDS.
  // Rows past the matrix edge are clamped to the last row (never stored).
  uint32_t a_src[kABlk], w_src[kWL];
#pragma unroll
  for (int i = 0; i < kABlk; ++i) {
    const uint32_t row = 16u * (wave * kABlk + i) + lane / 4u;
    const uint32_t chunk = (lane % 4u) ^ ((row >> 2) & 3u);
    a_src[i] = (m0 + row < m ? row : m - 1u - m0) * (k * 2u) + chunk * 16u;
  }
#pragma unroll
  for (int i = 0; i < kWL; ++i) {
    uint32_t q = (wave * kWL + i) * 64u + lane;
    q = q < BN * 9u ? q : BN * 9u - 1u;
    const uint32_t row = PAIR ? q / 9u % (BN / 2) : q / 9u, part = q % 9u;
    w_src[i] = (n0 + row < n ? row : n - 1u - n0) * (row_blocks * 144u) + part * 16u;
  }
  auto issue_a = [&](uint32_t stage, uint32_t slice) {      // slice = 32 K values = 64 bytes a row
    const uint8_t* g = a_tile + slice * 64u;
#pragma unroll
    for (int i = 0; i < kABlk; ++i) direct_load16(g, a_src[i], lds_base + stage * kAStage + (wave * kABlk + i) * 1024u);
  };
  auto issue_w = [&](uint32_t stage, uint32_t block) {
#pragma unroll
    for (int i = 0; i < kWL; ++i) {
      const uint8_t* g = (PAIR && (wave * kWL + i) * 128u >= BN * 9u ? up_tile : w_tile) + block * 144u;
      direct_load16(g, w_src[i], lds_base + 4 * kAStage + stage * kWStage + (wave * kWL + i) * 1024u);
    }
  };

  float16_t held[KSETS == 2 ? kTI : 1][KSETS == 2 ? kTJ : 1];
  auto& acc = [&]() -> auto& {
    if constexpr (KSETS == 2) return held;
    else return out;
  }();
#pragma unroll
  for (int i = 0; i < kTI; ++i)
#pragma unroll
    for (int j = 0; j < kTJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  // This lane's first weight row inside a raw stage (column tile j is 32 rows further), and its
  // activation fragment offsets: MFMA step t of a slice takes chunk 2kg + t of the row
  // (k = 16kg + 8t + [0,8), the positions decode_step gives the step).
  const uint32_t w_row = (wave_n * (PAIR ? 32u : WN) + l32) * 144u;
  uint32_t a_fr[2];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) a_fr[tt] = (wave_m * WM + l32) * 64u + (((kg * 2u + tt) ^ ((l32 >> 2) & 3u)) * 16u);

  const uint32_t slices = blocks * 8u;

  // AHEAD: one half of a slice's matrix instructions (one step of the slice) go with the making of the next half's operands:
  // activation fragments read from LDS, weights decoded.  A wavefront issues in order, so what lies between two matrix
  // instructions runs under the first of them.  2048 rows of 2 x 17408 x 5120 with silu 775 -> 765 us, the matrix cores
  // being held down by power.  Otherwise a slice's operands are made in the slice: where a half has few matrix instructions to
  // put the making between and a CU holds several workgroups, they hide what waits, the start and the end are shorter, and
  // the compiler keeps most of the decode's multiply-adds in fp32 and converts two numbers at once, which takes less of the
  // vector unit than multiply-adds that round to fp16.  Ahead it took longer by: 17 rows of 17408 x 1536 3 %, 100 rows of 17408 x
  // 1280 7, gate and up of 128 rows of 8192 x 4096 4 (53.6 / 51.5 us), 256 rows with two of 16 experts of 2048 x 4096 7 (171 / 160);
  // but 33 to 64 rows, one wavefront of two matrix tiles, 2 % less.
  constexpr bool AHEAD = KSETS == 2 || kTI * kTJ >= 8 || (kWaves == 1 && kTI == 2);
  half8_t a0[kTI], a1[kTI], b0[kTJ], b1[kTJ];
  BlockHead head[kTJ];
  ScaleMin sm[kTJ];
  uint32_t qw[kTJ][4];
  auto read_a = [&](uint32_t slice, int tt, half8_t (&f)[kTI]) {
    const uint8_t* a_stage = lds + (slice & 3u) * kAStage + a_fr[tt];
#pragma unroll
    for (int i = 0; i < kTI; ++i) f[i] = *reinterpret_cast<const half8_t*>(a_stage + i * 32 * 64);
  };
  auto multiply = [&](const half8_t (&af)[kTI], const half8_t (&bf)[kTJ]) {
#pragma unroll
    for (int i = 0; i < kTI; ++i)
#pragma unroll
      for (int j = 0; j < kTJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], bf[j], acc[i][j], 0, 0, 0);
  };
  auto interleave = [&](auto reads_c) {
    constexpr int kReads = decltype(reads_c)::value, kMfmas = kTI * kTJ, kValu = (kTJ * 20 + kMfmas - 1) / kMfmas;
    unrolled<kMfmas>([&](auto at) {
      constexpr int q = decltype(at)::value, reads = (q + 1) * kReads / kMfmas - q * kReads / kMfmas;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                           // a matrix instruction,
      if constexpr (reads > 0) __builtin_amdgcn_sched_group_barrier(0x100, reads, 0);   // its share of the LDS reads
      __builtin_amdgcn_sched_group_barrier(0x002, kValu, 0);                       // and of the decode
    });
  };

  auto interleave_half = [&](auto reads_c) {
    constexpr int kReads = decltype(reads_c)::value, kMfmas = kTI * kTJ / 2;
    unrolled<kMfmas>([&](auto at) {
      constexpr int q = decltype(at)::value, reads = (q + 1) * kReads / kMfmas - q * kReads / kMfmas;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if constexpr (reads > 0) __builtin_amdgcn_sched_group_barrier(0x100, reads, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
    });
  };

  if constexpr (!AHEAD) {
    // Prologue: first super-block and three activation slices in flight, then the first of each is waited for.
    issue_w(0, 0);
    issue_a(0, 0);
    issue_a(1, 1);
    issue_a(2, 2);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kABlk) : "memory");
    for (uint32_t blk = 0; blk < blocks; ++blk) {
      const uint8_t* raw = lds + 4 * kAStage + (blk & 1u) * kWStage + w_row;
      const bool more = blk + 1 < blocks;        // uniform
      BlockHead head[kTJ];
      uint32_t qw[kTJ][4], qs8[kTJ][4];
#pragma unroll
      for (int j = 0; j < kTJ; ++j) head[j] = load_block_head(raw + j * kJRows * 144);
      unrolled<8>([&](auto step) {
        constexpr int sb = decltype(step)::value;
        const uint32_t slice = blk * 8u + sb;
        if (sb == 0 && more) issue_w((blk + 1u) & 1u, blk + 1u);
        issue_a((slice + 3u) & 3u, slice + 3u < slices ? slice + 3u : slices - 1u);
        half8_t b[kTJ][2];
#pragma unroll
        for (int j = 0; j < kTJ; ++j) decode_subblock<sb>(raw + j * kJRows * 144, kg, head[j], qw[j], qs8[j], b[j]);
        const uint8_t* a_stage = lds + (slice & 3u) * kAStage;
#pragma unroll
        for (int tt = 0; tt < 2; ++tt) {
#pragma unroll
          for (int i = 0; i < kTI; ++i) {
            const half8_t af = *reinterpret_cast<const half8_t*>(a_stage + a_fr[tt] + i * 32 * 64);
#pragma unroll
            for (int j = 0; j < kTJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af, b[j][tt], acc[i][j], 0, 0, 0);
          }
        }
        // Publish slice + 1: every direct load older than the two youngest activation slices (and, in the two steps after a
        // weight refill was issued, older than that refill) has landed; this wavefront's LDS reads of the stage about to be
        // refilled are done.
        if (sb <= 1 && more) {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kABlk + kWL) : "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kABlk) : "memory");
        }
      });
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no direct load may outlive the workgroup
    return;
  }

  // Prologue: two super-blocks and four activation slices in flight, then the first of each is waited for.
  issue_w(0, 0);
  issue_a(0, 0);
  if (blocks > 1) issue_w(1, 1);
  issue_a(1, 1);
  issue_a(2, 2);
  issue_a(3, 3);
  if (blocks > 1) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * kABlk + kWL) : "memory");
  else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * kABlk) : "memory");
  if constexpr (KSETS == 2) {
    // Two sets of wavefronts share the tile: set t takes step t of every slice, so that a wavefront owns all of the tile's
    // rows (a weight is decoded once, where two wavefronts one above the other would each decode it) without owning half
    // as many columns.  The decode is what bounds the tile: a multiply-add that rounds to fp16 takes the vector unit 9.6
    // clocks (48 of them between eight matrix instructions 485 clocks; fp32 ones 305), and with a wavefront a SIMD every
    // instruction takes an issue slot of four.  A slice of a 128 x 128 tile alone on its CU: wavefronts of 64 x 64 362 ns,
    // two sets 329, with their LDS reads and decode between the matrix instructions 265.
    uint32_t a_step = set == 0u ? a_fr[0] : a_fr[1];
    auto read_step = [&](uint32_t slice, half8_t (&f)[kTI]) {
      const uint8_t* a_stage = lds + (slice & 3u) * kAStage + a_step;
#pragma unroll
      for (int i = 0; i < kTI; ++i) f[i] = *reinterpret_cast<const half8_t*>(a_stage + i * 32 * 64);
    };
    uint32_t qs[kTJ][2], qn[kTJ][2];
    uint4 hn[kTJ];
    auto load_step = [&](auto sb, const uint8_t* raw) {       // this set's eight of the sixteen bytes of sub-blocks sb, sb + 1
#pragma unroll
      for (int j = 0; j < kTJ; ++j) {
        const uint2 q = *reinterpret_cast<const uint2*>(raw + j * kJRows * 144 + 16 + (decltype(sb)::value >> 1) * 32 + kg * 16u + set * 8u);
        qn[j][0] = q.x, qn[j][1] = q.y;
      }
    };
    {
      const uint8_t* raw = lds + 4 * kAStage + w_row;
      read_step(0, a0);
      load_step(std::integral_constant<int, 0>{}, raw);
#pragma unroll
      for (int j = 0; j < kTJ; ++j) {
        qs[j][0] = qn[j][0], qs[j][1] = qn[j][1];
        head[j] = load_block_head(raw + j * kJRows * 144);
        b0[j] = decode_eight<0>(qs[j][0], qs[j][1], scale_min_f32<0>(head[j].sbytes, head[j].d, head[j].ndmin));
      }
    }
    for (uint32_t blk = 0; blk < blocks; ++blk) {
      unrolled<8>([&](auto step) {
        constexpr int sb = decltype(step)::value, next = (sb + 1) & 7;
        const uint32_t slice = blk * 8u + sb;
        half8_t (&ac)[kTI] = (sb & 1) ? a1 : a0;
        half8_t (&an)[kTI] = (sb & 1) ? a0 : a1;
        half8_t (&bc)[kTJ] = (sb & 1) ? b1 : b0;
        half8_t (&bn)[kTJ] = (sb & 1) ? b0 : b1;
        auto decode_next = [&](int j) {
          if constexpr (sb == 7) head[j] = block_head(hn[j]);
          if constexpr (sb & 1) qs[j][0] = qn[j][0], qs[j][1] = qn[j][1];
          bn[j] = decode_eight<next & 1>(qs[j][0], qs[j][1], scale_min_f32<next>(head[j].sbytes, head[j].d, head[j].ndmin));
        };
        // Publish slice + 1, as below; every wavefront has read its fragments of `slice`, whose stage takes slice + 4.
        if ((sb == 7 && blk + 2 < blocks) || (sb == 0 && blk > 0 && blk + 1 < blocks)) {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kABlk + kWL) : "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kABlk) : "memory");
        }
        // Half of the matrix instructions over the LDS reads (fragments of the next slice, weights of the next two) and half
        // of the decode; the direct loads; the rest.
        const uint8_t* raw = lds + 4 * kAStage + ((blk + (sb == 6 ? 1u : 0u)) & 1u) * kWStage + w_row;
        read_step(slice + 1u, an);
        if constexpr (sb % 2 == 0) load_step(std::integral_constant<int, (sb + 2) & 7>{}, raw);
        if constexpr (sb == 6) {
#pragma unroll
          for (int j = 0; j < kTJ; ++j) hn[j] = *reinterpret_cast<const uint4*>(raw + j * kJRows * 144);
        }
        decode_next(0);
        auto multiply_rows = [&](int i0) {
#pragma unroll
          for (int i = i0; i < i0 + kTI / 2; ++i)
#pragma unroll
            for (int j = 0; j < kTJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ac[i], bc[j], acc[i][j], 0, 0, 0);
        };
        multiply_rows(0);
        interleave_half(std::integral_constant<int, kTI + (sb == 6 ? 2 * kTJ : sb % 2 == 0 ? kTJ : 0)>{});
        __builtin_amdgcn_sched_barrier(0);
        if (sb == 6 && blk + 2 < blocks) issue_w(blk & 1u, blk + 2u);
        issue_a(slice & 3u, slice + 4u < slices ? slice + 4u : slices - 1u);
        decode_next(1);
        multiply_rows(kTI / 2);
        interleave_half(std::integral_constant<int, 0>{});
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    // Each set keeps half of the rows and hands the other half to the other set.
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    constexpr int kKeep = kTI / 2;
    static_assert(kWaves * kKeep * kTJ * 4096 <= sizeof(lds), "the halves fit LDS");
    float4_t* mine = reinterpret_cast<float4_t*>(lds) + wave * (kKeep * kTJ * 256u) + lane;
    const float4_t* theirs = reinterpret_cast<const float4_t*>(lds) + (wave ^ kWavesN) * (kKeep * kTJ * 256u) + lane;
#pragma unroll
    for (int i = 0; i < kKeep; ++i)
#pragma unroll
      for (int j = 0; j < kTJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float4_t v;
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = set == 0u ? held[i + kKeep][j][4 * q + e] : held[i][j][4 * q + e];
          mine[((i * kTJ + j) * 4 + q) * 64] = v;
        }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kKeep; ++i)
#pragma unroll
      for (int j = 0; j < kTJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float4_t v = theirs[((i * kTJ + j) * 4 + q) * 64];
#pragma unroll
          for (int e = 0; e < 4; ++e) out[i][j][4 * q + e] = (set == 0u ? held[i][j][4 * q + e] : held[i + kKeep][j][4 * q + e]) + v[e];
        }
    return;
  } else {
  {
    const uint8_t* raw = lds + 4 * kAStage + w_row;
    read_a(0, 0, a0);
#pragma unroll
    for (int j = 0; j < kTJ; ++j) {
      head[j] = load_block_head(raw + j * kJRows * 144);
      load_nibbles<0>(raw + j * kJRows * 144, kg, qw[j]);
      sm[j] = scale_min_f32<0>(head[j].sbytes, head[j].d, head[j].ndmin);
      b0[j] = decode_step<0>(qw[j], 0, sm[j]);
    }
  }

  for (uint32_t blk = 0; blk < blocks; ++blk) {
    unrolled<8>([&](auto step) {
      constexpr int sb = decltype(step)::value, next = (sb + 1) & 7;
      const uint32_t slice = blk * 8u + sb;
      // First half: step 0; made meanwhile: step 1, and the bytes that the next slice's weights come from.
      const uint8_t* raw = lds + 4 * kAStage + ((blk + (sb == 7 ? 1u : 0u)) & 1u) * kWStage + w_row;
      uint32_t qn[kTJ][4];
      uint4 hn[kTJ];
      read_a(slice, 1, a1);
#pragma unroll
      for (int j = 0; j < kTJ; ++j) {
        if constexpr (sb == 7) hn[j] = *reinterpret_cast<const uint4*>(raw + j * kJRows * 144);
        if constexpr (sb & 1) load_nibbles<next>(raw + j * kJRows * 144, kg, qn[j]);
        b1[j] = decode_step<sb & 1>(qw[j], 1, sm[j]);
      }
      multiply(a0, b0);
      interleave(std::integral_constant<int, kTI + (sb == 7 ? 2 * kTJ : sb & 1 ? kTJ : 0)>{});
      __builtin_amdgcn_sched_barrier(0);

      // Publish slice + 1: every direct load older than the two youngest activation slices (and, in the two steps after a
      // weight refill was issued, older than that refill) has landed; every wavefront has read all of `slice`, whose stage
      // takes slice + 4, and after step 6 of a super-block all of its weights, whose stage takes the one after the next.
      if ((sb == 7 && blk + 2 < blocks) || (sb == 0 && blk > 0 && blk + 1 < blocks)) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kABlk + kWL) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kABlk) : "memory");
      }
      if (sb == 6 && blk + 2 < blocks) issue_w(blk & 1u, blk + 2u);
      issue_a(slice & 3u, slice + 4u < slices ? slice + 4u : slices - 1u);

      // Second half: step 1; made meanwhile: step 0 of the next slice (after the last one: of a stage that nobody needs).
      read_a(slice + 1u, 0, a0);
#pragma unroll
      for (int j = 0; j < kTJ; ++j) {
        if constexpr (sb == 7) head[j] = block_head(hn[j]);
        if constexpr (sb & 1) {
#pragma unroll
          for (int x = 0; x < 4; ++x) qw[j][x] = qn[j][x];
        }
        sm[j] = scale_min_f32<next>(head[j].sbytes, head[j].d, head[j].ndmin);
        b0[j] = decode_step<next & 1>(qw[j], 0, sm[j]);
      }
      multiply(a1, b1);
      interleave(std::integral_constant<int, kTI>{});
      __builtin_amdgcn_sched_barrier(0);
    });
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no direct load may outlive the workgroup
  }
}

// Stores a tile's sums times their rows' scales; rows from m and columns from n_end on are not stored.  A lane holds column
// l32 and rows (e/4)*8 + kg*4 + e%4 of each 32 x 32 tile; the four row scales of each e/4 group are one 16-byte load (the
// scale array is padded, so rows past m read something harmless).
template <int BM, int BN, int WM, int WN, bool PAIR = false>
__device__ __forceinline__ void q4k_tile_store(const TileSums<WM, WN>& acc, const float* __restrict__ a_scale, float* __restrict__ c,
                                               uint32_t m, uint32_t n, uint32_t m0, uint32_t n0, uint32_t n_end) {
  constexpr int kWavesN = BN / WN, kTI = WM / 32, kTJ = WN / 32;
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t wave_m = wave / kWavesN, wave_n = wave % kWavesN, l32 = lane & 31u, kg = lane >> 5;
#pragma unroll
  for (int i = 0; i < kTI; ++i) {
    const uint32_t row0 = m0 + wave_m * WM + i * 32u + kg * 4u;
    float4 sc[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) sc[q] = *reinterpret_cast<const float4*>(a_scale + row0 + q * 8u);
    if constexpr (PAIR) {
      const uint32_t col = n0 + wave_n * 32u + l32;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t row = row0 + (e >> 2) * 8u + (e & 3u);
        const float4 s4 = sc[e >> 2];
        const float rs = (e & 3) == 0 ? s4.x : (e & 3) == 1 ? s4.y : (e & 3) == 2 ? s4.z : s4.w;
        const float gate = acc[i][0][e] * rs, up = acc[i][1][e] * rs;
        if (row < m && col < n_end) c[static_cast<size_t>(row) * n + col] = (gate / (1.0f + expf(-gate))) * up;
      }
      continue;
    }
#pragma unroll
    for (int j = 0; j < kTJ; ++j) {
      const uint32_t col = n0 + wave_n * WN + j * 32u + l32;
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t row = row0 + (e >> 2) * 8u + (e & 3u);
        const float4 s4 = sc[e >> 2];
        const float rs = (e & 3) == 0 ? s4.x : (e & 3) == 1 ? s4.y : (e & 3) == 2 ? s4.z : s4.w;
        if (row < m && col < n_end) c[static_cast<size_t>(row) * n + col] = acc[i][j][e] * rs;
      }
    }
  }
}

// One tile, all of K.
template <int BM, int BN, int WM, int WN, bool PAIR = false>
__device__ __forceinline__ void q4k_gemm_tile(const _Float16* __restrict__ a16, const float* __restrict__ a_scale,
                                              const uint8_t* __restrict__ w, float* __restrict__ c, uint32_t m, uint32_t n,
                                              uint32_t k, uint32_t m0, uint32_t n0, uint32_t n_end,
                                              const uint8_t* __restrict__ w_up = nullptr) {
  TileSums<WM, WN> acc;
  q4k_tile_sums<BM, BN, WM, WN, PAIR>(acc, a16, w, m, n, k, m0, n0, 0u, k / 256u, w_up);
  q4k_tile_store<BM, BN, WM, WN, PAIR>(acc, a_scale, c, m, n, m0, n0, n_end);
}

}  // namespace
}  // namespace qmm
