// "gemm_fp8" from 17 rows up on the matrix cores: C (m x n fp32) = A (m x k fp32) . W^T diag(s), W = n rows of
// k E4M3 bytes with one fp32 scale a row (include/tessera/backend.hpp:191-194,504-512; reference kernel
// src/backends/rocm/rocm_kernels_basic.cpp:1039-1064, one thread an output).
//
// Precision.  The contract is fp32 activations and exact weights.  Every E4M3 code is an fp16 number, so the
// weights are converted in registers without loss; a row of A becomes two fp16 terms under a power of two that
// brings its largest magnitude to [2^14, 2^15): hi = RN16(x / s), lo = RN16(2^11 (x / s - hi)), x / s = hi + 2^-11 lo.
// That misses an element by at most 2^-23 of itself down to 2^-28 of the row's largest, and by 2^-50 of the
// largest below.  Products of an 11-bit and a 4-bit significand are exact; v_mfma_f32_32x32x16_f16 adds them up,
// and its additions are what costs precision: one chain of both terms over 5120 weights was measured at 6.2e-7 of
// the float64 result in the 2-norm, against 1.2e-7 for the multiply-add kernel's short chains.  So an output has
// four sums: the second term's products, worth 2^-11 each, in one of their own, the first term's for 128 weights
// at a time, those of 1024, and the total.  Measured 0.91e-7 (k = 1024) to 1.22e-7 (k = 17408), the multiply-add
// kernel 0.94e-7 and 1.48e-7; with eight columns of the activations 1000 times the others 1.11e-7 and 1.35e-7
// against 0.92e-7 and 1.44e-7 (64 weights at a time: 1.06e-7, but 58.4 us instead of 56.2 at 300 x 6144 x 5120).
// (The scaled 8-bit instruction would take the codes as they are but aligns an instruction's products to the
// largest before it adds them: 1.5e-5.)
//
// Three launches: rows to terms, the product, and the sum of the K parts where K is split.  A workgroup of four
// wavefronts owns BM x 128 of C and walks its part of K 64 at a time: both terms (BM x 128 bytes each, whole
// cache lines: with 32 at a time the L1 fetched every line two to four times and the product was 1.4 times as
// long) and the codes (128 x 64 bytes) travel HBM -> LDS by direct loads into a ring of stages; a wavefront
// converts the codes of its columns once per stage and uses them against both terms of all its rows.  Whatever
// part of the chip one round of tiles leaves idle is filled by splitting K (fp8_plan); the partial sums are added
// in part order by a last launch: no atomics, the same bits every time.  What bounds it: at 300 x 6144 x 5120 the
// matrix cores are busy 41 % of the product's cycles, vector instructions issue in 27 %, and a wavefront, alone on its SIMD,
// waits in 25 % (direct loads, barrier) and for issue in 29 %; neither a deeper ring (five stages) nor a tile that reads
// less LDS changes it.  A short stack of rows is bound by the weight stream.  Half a step's operands are read and
// converted between the matrix instructions of the half before: 57.2 -> 54.0 us with the rows' conversion.
// 300 x 6144 x 5120: 1108 -> 56 us against 75 four-row passes of the multiply-add kernel; 17 rows 68 -> 16 us.

#include <type_traits>

#include "q4k_tile.hpp"
#include "qmm_kernels.hpp"

namespace qmm {
namespace {

// One workgroup per row: fp32 -> the two terms and the row's power of two.  The maximum is taken over the
// finite elements, so that an infinity or a NaN stays itself in the first term (with a zero second one) and the
// row's other elements do not overflow.  NV > 0: the row is held in registers (k <= 1024 NV); 0: read twice.
template <int NV>
__global__ __launch_bounds__(256) void rows_to_f16_terms_kernel(const float* __restrict__ src, _Float16* __restrict__ dst,
                                                                float* __restrict__ scale, uint32_t cols, size_t plane) {
  typedef _Float16 half4_t __attribute__((ext_vector_type(4)));
  __shared__ float red[4];
  const float4* in = reinterpret_cast<const float4*>(src + static_cast<size_t>(blockIdx.x) * cols);
  const uint32_t groups = cols / 4u;
  float amax = 0.0f;
  float4 held[NV > 0 ? NV : 1];
  auto scan = [&](const float4& v) {
    const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t mag = bit_cast<uint32_t>(e[i]) & 0x7FFFFFFFu;
      amax = mag < 0x7F800000u ? fmaxf(amax, bit_cast<float>(mag)) : amax;
    }
  };
  if constexpr (NV > 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const uint32_t g = threadIdx.x + j * 256u;
      held[j] = g < groups ? in[g] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) scan(held[j]);
  } else {
    for (uint32_t g = threadIdx.x; g < groups; g += 256u) scan(in[g]);
  }
  amax = block_amax(amax, red);
  // exponent of the scale: amax / s in [2^14, 2^15); both s and 1 / s normal
  const int e = static_cast<int>(bit_cast<uint32_t>(amax) >> 23);
  const int se = amax == 0.0f ? 127 : (e - 14 < 1 ? 1 : e - 14);
  const float s = bit_cast<float>(static_cast<uint32_t>(se) << 23);
  const float inv = bit_cast<float>(static_cast<uint32_t>(254 - se) << 23);
  _Float16* out = dst + static_cast<size_t>(blockIdx.x) * cols;
  auto emit = [&](const float4& v, uint32_t g) {
    const float x[4] = {v.x * inv, v.y * inv, v.z * inv, v.w * inv};
    half4_t hi, lo;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      hi[i] = static_cast<_Float16>(x[i]);
      const float rest = (x[i] - static_cast<float>(hi[i])) * 0x1p11f;
      lo[i] = static_cast<_Float16>(fabsf(x[i]) < 65504.0f ? rest : 0.0f);   // (NaN compares false)
    }
    *reinterpret_cast<half4_t*>(out + g * 4u) = hi;
    *reinterpret_cast<half4_t*>(out + plane + g * 4u) = lo;
  };
  if constexpr (NV > 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const uint32_t g = threadIdx.x + j * 256u;
      if (g < groups) emit(held[j], g);
    }
  } else {
    for (uint32_t g = threadIdx.x; g < groups; g += 256u) emit(in[g], g);
  }
  if (threadIdx.x == 0) scale[blockIdx.x] = s;
}

constexpr uint32_t kBN = 128;
constexpr uint32_t kStepK = 64, kRunSteps = 2, kAccSteps = 16;

// BM x 128 of C, or of one K part's partial sums (`part` set: [parts][m][n], unscaled).  A wavefront owns
// WM rows x WN columns; STAGES = depth of the ring.
template <int BM, int WM, int WN, int STAGES>
__global__ __launch_bounds__(256, 2) void fp8_gemm_kernel(const _Float16* __restrict__ a16, size_t plane,
                                                          const float* __restrict__ a_scale, const uint8_t* __restrict__ w,
                                                          const float* __restrict__ w_scale, float* __restrict__ c,
                                                          float* __restrict__ part, uint32_t m, uint32_t n, uint32_t k,
                                                          uint32_t steps_per_part) {
  constexpr int kWavesN = kBN / WN, kTI = WM / 32, kTJ = WN / 32;
  static_assert((BM / WM) * kWavesN == 4, "four wavefronts");
  constexpr int kABlk = 2 * BM / 8 / 4, kWBlk = kBN / 16 / 4;   // 1 KB blocks a wavefront brings per stage: both terms, codes
  constexpr int kDma = kABlk + kWBlk;
  constexpr uint32_t kTermStage = BM * 128, kWBase = 2 * kTermStage, kStage = kWBase + kBN * 64;
  __shared__ __attribute__((aligned(16))) uint8_t lds[STAGES * kStage];

  // Workgroups go round the eight XCDs; neighbours in (row tile, column tile, K part) order share weights, so
  // each XCD takes one contiguous run of that order.
  const uint32_t tiles_m = (m + BM - 1) / BM, tiles_n = (n + kBN - 1) / kBN;
  const uint32_t xcd = blockIdx.x % 8u, per = gridDim.x / 8u, extra = gridDim.x % 8u;
  const uint32_t idx = xcd * per + (xcd < extra ? xcd : extra) + blockIdx.x / 8u;
  const uint32_t m0 = (idx % tiles_m) * BM, n0 = (idx / tiles_m % tiles_n) * kBN, z = idx / (tiles_m * tiles_n);
  const uint32_t steps = k / kStepK, s0 = z * steps_per_part;
  const uint32_t count = steps - s0 < steps_per_part ? steps - s0 : steps_per_part;

  const uint32_t t = threadIdx.x, lane = t & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t wave_m = wave / kWavesN, wave_n = wave % kWavesN;
  const uint32_t l32 = lane & 31u, kg = lane >> 5;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) uint8_t*)lds));
  const uint8_t* a_tile = reinterpret_cast<const uint8_t*>(a16 + static_cast<size_t>(m0) * k + s0 * kStepK);
  const uint8_t* w_tile = w + static_cast<size_t>(n0) * k + s0 * kStepK;

  // Term block L of a stage (rows 8L.. of one term, eight 16-byte chunks a row): lane p fetches row 8L + p/8,
  // chunk (p%8) ^ ((row>>1)&7).  Code block L (rows 16L.., four chunks a row): row 16L + p/4, chunk (p%4) ^
  // ((row>>2)&3).  Rows past the matrix edge repeat the last one (never stored).
  uint32_t a_src[kABlk], w_src[kWBlk];
#pragma unroll
  for (int i = 0; i < kABlk; ++i) {
    const uint32_t row = 8u * ((wave * kABlk + i) % (BM / 8)) + lane / 8u;
    a_src[i] = (m0 + row < m ? row : m - 1u - m0) * (k * 2u) + (((lane % 8u) ^ ((row >> 1) & 7u)) * 16u);
  }
#pragma unroll
  for (int i = 0; i < kWBlk; ++i) {
    const uint32_t row = 16u * (wave * kWBlk + i) + lane / 4u;
    w_src[i] = (n0 + row < n ? row : n - 1u - n0) * k + (((lane % 4u) ^ ((row >> 2) & 3u)) * 16u);
  }
  auto issue = [&](uint32_t stage, uint32_t step_any) {
    const uint32_t step = __builtin_amdgcn_readfirstlane(step_any);
#pragma unroll
    for (int i = 0; i < kABlk; ++i) {
      const uint32_t blk = wave * kABlk + i;
      const uint8_t* term = blk >= BM / 8 ? a_tile + plane * 2u : a_tile;
      direct_load16(term + step * (kStepK * 2u), a_src[i], lds_base + stage * kStage + blk * 1024u);
    }
#pragma unroll
    for (int i = 0; i < kWBlk; ++i)
      direct_load16(w_tile + step * kStepK, w_src[i], lds_base + stage * kStage + kWBase + (wave * kWBlk + i) * 1024u);
  };

  // Four sums an output: `run` takes the first term's products of kRunSteps steps and is then added to `acc`, which
  // takes kAccSteps steps and is added to `total`; `low` takes the second term's, worth 2^-11 each, from end to end.
  float16_t total[kTI][kTJ], acc[kTI][kTJ], run[kTI][kTJ], low[kTI][kTJ];
#pragma unroll
  for (int i = 0; i < kTI; ++i)
#pragma unroll
    for (int j = 0; j < kTJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) total[i][j][e] = acc[i][j][e] = run[i][j][e] = low[i][j][e] = 0.0f;
  // A lane of K half kg supplies k = 16 (2 h + kg) + 8 tt + [0, 8) to matrix step 2 h + tt: half tt of chunk
  // 2 h + kg of the codes, chunk 2 (2 h + kg) + tt of a term's row.
  uint32_t a_fr[4], w_fr[2];
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q)
    a_fr[q] = (wave_m * WM + l32) * 128u + (((2u * (2u * (q >> 1) + kg) + (q & 1u)) ^ ((l32 >> 1) & 7u)) * 16u);
#pragma unroll
  for (uint32_t h = 0; h < 2; ++h) w_fr[h] = kWBase + (wave_n * WN + l32) * 64u + (((2u * h + kg) ^ ((l32 >> 2) & 3u)) * 16u);

  // The operands of half a step.
  struct Frag {
    half8_t b[kTJ][2], hi[kTI][2], lo[kTI][2];
  };
  uint4 codes[kTJ];
  auto read = [&](const uint8_t* stage, int h, Frag& f) {
#pragma unroll
    for (int j = 0; j < kTJ; ++j) codes[j] = *reinterpret_cast<const uint4*>(stage + w_fr[h] + j * 32 * 64);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int i = 0; i < kTI; ++i) {
        const uint8_t* at = stage + a_fr[2 * h + tt] + i * 32 * 128;
        f.hi[i][tt] = *reinterpret_cast<const half8_t*>(at);
        f.lo[i][tt] = *reinterpret_cast<const half8_t*>(at + kTermStage);
      }
  };
  auto convert = [&](int tt, Frag& f) {
#pragma unroll
    for (int j = 0; j < kTJ; ++j) {
      const uint32_t words[2] = {tt == 0 ? codes[j].x : codes[j].z, tt == 0 ? codes[j].y : codes[j].w};
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const half2_t p0 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(words[i], 1.0f, false);
        const half2_t p1 = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(words[i], 1.0f, true);
        f.b[j][tt][4 * i] = p0[0], f.b[j][tt][4 * i + 1] = p0[1], f.b[j][tt][4 * i + 2] = p1[0], f.b[j][tt][4 * i + 3] = p1[1];
      }
      asm volatile("" : "+v"(f.b[j][tt]));      // here, not where it is used
    }
  };
  // Half a step: the matrix instructions of `f`, and the operands `g` of the next half made meanwhile.  With a wavefront a
  // SIMD nothing hides what waits, so the order is fixed: reads, half of the matrix instructions, and the conversions
  // between the others; no two in a row into the same sums.  With `first` the second term's instructions go first, and
  // under them the run that has ended is added.
  auto half_step = [&](const Frag& f, const uint8_t* stage, int h, Frag& g, auto first) {
    constexpr bool FIRST = decltype(first)::value;
    read(stage, h, g);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int tt = FIRST ? q & 1 : q >> 1;
      const bool second_term = FIRST ? q < 2 : (q & 1) == 0;
      if (q >= 2) {
        convert(q - 2, g);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < kTI; ++i)
#pragma unroll
        for (int j = 0; j < kTJ; ++j) {
          if (second_term) low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.lo[i][tt], f.b[j][tt], low[i][j], 0, 0, 0);
          else run[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.hi[i][tt], f.b[j][tt], run[i][j], 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
          if (FIRST && q < 2) {
            constexpr int kEach = 8;      // of the 16 sums of each matrix tile, twice as many instructions as tiles
#pragma unroll
            for (int e = 0; e < kEach; ++e) {
              const int at = q * kEach + e;
              acc[i][j][at] += run[i][j][at], run[i][j][at] = 0.0f;
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
    }
  };

#pragma unroll
  for (int i = 0; i < STAGES; ++i) issue(i, static_cast<uint32_t>(i) < count ? i : count - 1u);
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 1) * kDma) : "memory");
  uint32_t rd = 0, step = 0;
  Frag f0, f1;
  read(lds, 0, f0);
  convert(0, f0);
  convert(1, f0);
  // Between a step's halves every wavefront has read all of its stage, which is asked for again, and the next stage has
  // landed.  (After the last step: operands of a stage that nobody needs.)
  auto one_step = [&](auto first) {
    half_step(f0, lds + rd * kStage, 1, f1, first);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 2) * kDma) : "memory");
    issue(rd, step + STAGES < count ? step + STAGES : count - 1u);
    rd = rd + 1u == STAGES ? 0u : rd + 1u;
    half_step(f1, lds + rd * kStage, 0, f0, std::false_type{});
    return ++step == count;
  };
  auto add_acc = [&]() {
#pragma unroll
    for (int i = 0; i < kTI; ++i)
#pragma unroll
      for (int j = 0; j < kTJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) total[i][j][e] += acc[i][j][e], acc[i][j][e] = 0.0f;
  };
  static_assert(kRunSteps == 2, "the loop's steps");
  for (;;) {
    const bool last = one_step(std::true_type{});
    if (step % kAccSteps == 1u && step != 1u) add_acc();
    if (last || one_step(std::false_type{})) break;
  }
  if (count % kRunSteps == 0u) {      // the last run, as the step after it would have
#pragma unroll
    for (int i = 0; i < kTI; ++i)
#pragma unroll
      for (int j = 0; j < kTJ; ++j)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] += run[i][j][e], run[i][j][e] = 0.0f;
    if (count % kAccSteps == 0u) add_acc();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no direct load may outlive the workgroup

  // lane: column l32, rows (e/4)*8 + kg*4 + e%4 of each 32 x 32 tile
  float* out = part != nullptr ? part + static_cast<size_t>(z) * m * n : c;
#pragma unroll
  for (int j = 0; j < kTJ; ++j) {
    const uint32_t col = n0 + wave_n * WN + j * 32u + l32;
    const float ws = part != nullptr ? 1.0f : w_scale[col < n ? col : n - 1u];
#pragma unroll
    for (int i = 0; i < kTI; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t row = m0 + wave_m * WM + i * 32u + (e >> 2) * 8u + kg * 4u + (e & 3u);
        if (row >= m || col >= n) continue;
        const float sum = total[i][j][e] + (acc[i][j][e] + fmaf(low[i][j][e], 0x1p-11f, run[i][j][e]));
        out[static_cast<size_t>(row) * n + col] = part != nullptr ? sum : sum * a_scale[row] * ws;
      }
  }
}

// The K parts' sums in part order, under the row's power of two and the weight row's scale.  VEC outputs a thread.
template <int VEC>
__global__ __launch_bounds__(256) void fp8_reduce_kernel(const float* __restrict__ part, const float* __restrict__ a_scale,
                                                         const float* __restrict__ w_scale, float* __restrict__ c, uint32_t n,
                                                         uint32_t parts, size_t region) {
  const uint32_t row = blockIdx.y, col = (blockIdx.x * 256u + threadIdx.x) * VEC;
  if (col >= n) return;
  const float* src = part + static_cast<size_t>(row) * n + col;
  float* dst = c + static_cast<size_t>(row) * n + col;
  const float rs = a_scale[row];
  if constexpr (VEC == 4) {
    float4 sum = *reinterpret_cast<const float4*>(src);
    for (uint32_t z = 1; z < parts; ++z) {
      const float4 v = *reinterpret_cast<const float4*>(src + z * region);
      sum.x += v.x, sum.y += v.y, sum.z += v.z, sum.w += v.w;
    }
    *reinterpret_cast<float4*>(dst) = make_float4(sum.x * rs * w_scale[col], sum.y * rs * w_scale[col + 1],
                                                  sum.z * rs * w_scale[col + 2], sum.w * rs * w_scale[col + 3]);
  } else {
    float sum = src[0];
    for (uint32_t z = 1; z < parts; ++z) sum += src[z * region];
    dst[0] = sum * rs * w_scale[col];
  }
}

struct Fp8Plan {
  uint32_t bm, parts, steps_per_part;
};

// Row tile and K parts with the smallest estimate of the launch: the workgroups of the fullest CU one after
// another (two on a CU take as long as one after the other), then the launch that adds the parts and the traffic of their
// sums.  A 64-wide step of 32 rows counts as 0.36 us, of 64 rows 0.58, as measured with 1 to 4 a CU when a step's operands were made
// in the step; as they are made now a step takes 0.33 and 0.51, two on a CU 0.97 of 64 rows, the same in proportion.
// 17 x 6144 x 5120: one part 33, five 16 us; 300 x 512 x 5120: 54 and, with eight, 21 us.  A part keeps at least
// four steps, and the parts' sums fit `room` bytes.  (Tiles of 128 rows were no faster up to 1024 rows and leave no
// registers for the sums.)
Fp8Plan fp8_plan(uint32_t m, uint32_t n, uint32_t k, size_t room, float* estimate) {
  const uint32_t cus = static_cast<uint32_t>(num_cus()), steps = k / kStepK, tiles_n = (n + kBN - 1u) / kBN;
  Fp8Plan best{64u, 1u, steps};
  float best_us = 1e30f;
  for (uint32_t bm = 32; bm <= 64; bm *= 2) {
    const uint64_t tiles = static_cast<uint64_t>((m + bm - 1u) / bm) * tiles_n;
    const float step_us = bm == 32u ? 0.36f : 0.58f;
    for (uint32_t parts = 1; parts == 1u || (parts <= 16u && steps / parts >= 4u); ++parts) {
      const uint32_t spp = (steps + parts - 1u) / parts, real = (steps + spp - 1u) / spp;
      if (real > 1u && static_cast<size_t>(real) * m * n * 4 > room) break;
      const uint64_t rounds = (tiles * real + cus - 1u) / cus;
      float us = static_cast<float>(rounds) * static_cast<float>(spp) * step_us;
      if (real > 1u) us += 3.5f + static_cast<float>(real) * static_cast<float>(m) * static_cast<float>(n) * 1.6e-6f;
      if (us < best_us) best_us = us, best = Fp8Plan{bm, real, spp};
    }
  }
  *estimate = best_us;
  return best;
}

size_t terms_bytes(uint64_t m, uint64_t k) {
  return static_cast<size_t>(m) * k * 4 + ((static_cast<size_t>(m) * 4 + 255) & ~size_t{255});
}

// Rows of one go: all where their terms fit the scratch, else the multiple of 64 (fewer where not even 64 fit)
// with the smallest sum of estimates.  The limit of 128 MB costs nothing up to 8192 rows; with 32 MB 300 x 5120 x
// 17408, whose terms take 21 MB, has no room for the sums of K parts (162 us, without a limit 137), with 64 MB 512
// rows have room for some of them only (220, without 201).
uint32_t fp8_rows(uint32_t m, uint32_t n, uint32_t k, size_t limit) {
  if (terms_bytes(m, k) <= limit) return m;
  uint32_t most = static_cast<uint32_t>((limit - 256) / (static_cast<size_t>(k) * 4 + 4));
  if (most < 64u) return most;
  most = most / 64u * 64u;
  uint32_t best = most;
  float best_us = 1e30f;
  for (uint32_t rows = most; rows >= 64u && rows * 2u >= most; rows -= 64u) {
    float each = 0.0f, last = 0.0f;
    fp8_plan(rows, n, k, limit - terms_bytes(rows, k), &each);
    const uint32_t left = m % rows;
    if (left != 0u) fp8_plan(left, n, k, limit - terms_bytes(left, k), &last);
    const float us = static_cast<float>(m / rows) * each + last;
    if (us < best_us) best_us = us, best = rows;
  }
  return best;
}

// One go of m rows (their terms fit the scratch): the terms, the product, the parts' sums.
hipError_t launch_rows(const float* a, const uint8_t* w, const float* w_scale, float* c, void* scratch, size_t limit, uint32_t m,
                       uint32_t n, uint32_t k, hipStream_t stream) {
  float us;
  const Fp8Plan pl = fp8_plan(m, n, k, limit - terms_bytes(m, k), &us);
  _Float16* a16 = static_cast<_Float16*>(scratch);
  const size_t plane = static_cast<size_t>(m) * k;
  float* a_scale = reinterpret_cast<float*>(a16 + 2 * plane);
  float* part = pl.parts > 1 ? reinterpret_cast<float*>(static_cast<uint8_t*>(scratch) + terms_bytes(m, k)) : nullptr;
  if (k <= 2048u) hipLaunchKernelGGL(rows_to_f16_terms_kernel<2>, dim3(m), dim3(256), 0, stream, a, a16, a_scale, k, plane);
  else if (k <= 8192u) hipLaunchKernelGGL(rows_to_f16_terms_kernel<8>, dim3(m), dim3(256), 0, stream, a, a16, a_scale, k, plane);
  else hipLaunchKernelGGL(rows_to_f16_terms_kernel<0>, dim3(m), dim3(256), 0, stream, a, a16, a_scale, k, plane);
  const uint32_t grid = ((m + pl.bm - 1u) / pl.bm) * ((n + kBN - 1u) / kBN) * pl.parts;
  if (pl.bm == 32u) {
    hipLaunchKernelGGL((fp8_gemm_kernel<32, 32, 32, 4>), dim3(grid), dim3(256), 0, stream, a16, plane, a_scale, w, w_scale, c, part,
                       m, n, k, pl.steps_per_part);
  } else {
    hipLaunchKernelGGL((fp8_gemm_kernel<64, 32, 64, 3>), dim3(grid), dim3(256), 0, stream, a16, plane, a_scale, w, w_scale, c, part,
                       m, n, k, pl.steps_per_part);
  }
  if (part != nullptr) {
    const size_t region = static_cast<size_t>(m) * n;
    if (n % 4u == 0u && reinterpret_cast<uintptr_t>(c) % 16u == 0u) {
      hipLaunchKernelGGL(fp8_reduce_kernel<4>, dim3((n + 1023u) / 1024u, m), dim3(256), 0, stream, part, a_scale, w_scale, c, n,
                         pl.parts, region);
    } else {
      hipLaunchKernelGGL(fp8_reduce_kernel<1>, dim3((n + 255u) / 256u, m), dim3(256), 0, stream, part, a_scale, w_scale, c, n,
                         pl.parts, region);
    }
  }
  return hipGetLastError();
}

}  // namespace

bool gemm_fp8_f16_supported(uint64_t m, uint64_t n, uint64_t k) {
  return m >= 17 && k % 64 == 0 && k <= (1u << 20) && n <= (1u << 30) && m <= 65535u && m * n < (1ull << 40);
}

size_t gemm_fp8_f16_scratch_bytes(uint64_t m, uint64_t n, uint64_t k, size_t limit) {
  const uint32_t rows = fp8_rows(static_cast<uint32_t>(m), static_cast<uint32_t>(n), static_cast<uint32_t>(k), limit);
  size_t most = 0;
  for (const uint32_t part : {rows, static_cast<uint32_t>(m % rows)}) {
    if (part == 0u) continue;
    float us;
    const Fp8Plan pl = fp8_plan(part, static_cast<uint32_t>(n), static_cast<uint32_t>(k), limit - terms_bytes(part, k), &us);
    const size_t bytes = terms_bytes(part, k) + (pl.parts > 1 ? static_cast<size_t>(pl.parts) * part * n * 4 : 0);
    most = bytes > most ? bytes : most;
  }
  return most;
}

hipError_t launch_fp8_f16_gemm(const float* a, const uint8_t* w, const float* w_scale, float* c, void* scratch, size_t limit,
                               uint32_t m, uint32_t n, uint32_t k, hipStream_t stream) {
  const uint32_t rows = fp8_rows(m, n, k, limit);
  for (uint32_t r = 0; r < m; r += rows) {
    const hipError_t e = launch_rows(a + static_cast<size_t>(r) * k, w, w_scale, c + static_cast<size_t>(r) * n, scratch, limit,
                                     m - r < rows ? m - r : rows, n, k, stream);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace qmm
