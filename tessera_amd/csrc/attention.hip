// Softmax attention over a key/value cache: the "attention" ids, their flash-decoding forms and the
// merge of those.  Contracts: include/tessera/backend.hpp:162-179,284-333,429-475,679-705; CPU
// statements src/core/numerics/attention.cpp.
//
// Precision.  Scores and sums are fp32 in every variant.  Where the contraction runs on the fp16
// matrix instruction, the fp32 side (queries, then weights times the values' scales) enters as two fp16
// terms of a value x that a power of two brings below 2^15: hi = RN16(x), lo = RN16(2^11 (x - hi)), whose
// sums meet as hi + 2^-11 lo.  That misses x by at most 2^-23 of itself while |x| >= 2^-14 and by 2^-36
// below.  A query element is brought under its head's largest and keeps that precision down to 2^-28 of it; a
// weight, under the largest of the row so far, down to 2^-18 of it, and what is smaller is off by 2^-40 of it.
// The cache's side enters exactly: an fp16 number, or the integer or E4M3 code, whose scale multiplies
// the fp32 score (keys) or the fp32 weight (values).

#include <type_traits>

#include "qmm_device.hpp"
#include "qmm_kernels.hpp"
#include "launch_rules.hpp"

namespace qmm {
namespace {

// How keys and values are stored.  The quantized kinds hold codes and one fp32 scale per key row (all
// kv heads of a position), and an element is code * scale as in AttentionQ8Ref / AttentionQ4Ref /
// AttentionFp8Ref (src/core/numerics/attention.cpp:45-121).
enum class KvKind { F32, F16, Q8, Q4, Fp8 };
constexpr int kv_bits(KvKind k) { return k == KvKind::F32 ? 32 : k == KvKind::F16 ? 16 : k == KvKind::Q4 ? 4 : 8; }
constexpr bool kv_quantized(KvKind k) { return k == KvKind::Q8 || k == KvKind::Q4 || k == KvKind::Fp8; }

// SPLIT (the flash-decoding ids, src/backends/rocm/rocm_kernels_basic.cpp:275-440): the part s of
// (row, head) is chunk s of ceil(span / split) keys of the row's key range; it leaves the unnormalized
// sum, the chunk's largest score and its sum of weights in pacc / pmax / psum at index
// (row * heads + head) * split + s (an empty chunk: 0, -1e30, 0); attention_combine_kernel merges them.
struct SplitOut {
  float *pacc, *pmax, *psum;
  uint64_t split;   // 0: no parts, `out` receives the rows
};

struct AttentionArgs {
  const float* q;
  const void *k, *v;
  const float *k_scale, *v_scale;
  float* out;
  SplitOut part;
  uint64_t rows, n, q_base, row_base, window;
  uint32_t heads, kv_heads, head_dim, causal;
};

// Keys [start, last] that query row i sees.
__device__ __forceinline__ void key_range(const AttentionArgs& a, uint64_t i, uint64_t& start, uint64_t& last) {
  const uint64_t pos = a.q_base + i;
  last = a.causal != 0 ? (pos >= a.n ? a.n - 1 : pos) : a.n - 1;
  start = 0;
  if (a.causal != 0) {
    start = (a.window != 0 && pos + 1 > a.window) ? pos + 1 - a.window : 0;
    if (start > last) start = last;
  }
}
// Chunk s of that range; false: the chunk is empty.
__device__ __forceinline__ bool key_chunk(const AttentionArgs& a, uint64_t s, uint64_t& start, uint64_t& last) {
  const uint64_t chunk = (last + 1 - start + a.part.split - 1) / a.part.split;
  start += s * chunk;
  if (start > last) return false;
  last = start + chunk - 1 < last ? start + chunk - 1 : last;
  return true;
}

// ---- few query rows: one workgroup per (row, kv head, chunk) -------------------------------------
//
// Bound by reading the cache.  A kv head's keys and values are read once for all the query heads that
// share it (up to eight a workgroup; sixteen over an fp32 cache), each wavefront taking every NW-th tile
// of 32 keys on its own, with no barrier and no LDS before the final merge of the wavefronts:
//   S^T = K Q^T on v_mfma_f32_16x16x32_f16, keys as matrix rows, columns 2h and 2h + 1 the hi and lo
//   term of head h, so a lane ends up with scores of 4 + 4 keys of its column and its neighbour's
//   column is the other term.  O^T = V^T P^T takes those lanes' weights as they stand (slots 8g..8g+3
//   of lane group g are keys 4g.. of the tile's first half, the next four of its second half), and a
//   lane reads whole runs of eight keys' values, of which a byte permute per register pair makes the
//   key-major operand: no transposition through LDS.
// The loads of a tile's keys are under way during the previous tile's softmax and values, its values'
// during the scores.  Over an fp32 cache the same shape runs on v_mfma_f32_16x16x4_f32, tiles of 16 keys.
// One row against 9301 int8 keys of 4 heads of 256 in 64 parts: 16 us (one element a load: 86 us).
template <int BYTES>
__device__ __forceinline__ void load_run(const uint8_t* p, uint32_t (&r)[(BYTES + 3) / 4]) {
  if constexpr (BYTES == 1) {
    r[0] = *p;
  } else if constexpr (BYTES == 2) {
    r[0] = *reinterpret_cast<const uint16_t*>(p);
  } else if constexpr (BYTES == 4) {
    r[0] = *reinterpret_cast<const uint32_t*>(p);
  } else if constexpr (BYTES == 8) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    r[0] = v.x, r[1] = v.y;
  } else {
#pragma unroll
    for (int i = 0; i < BYTES / 16; ++i) {
      const uint4 v = load_u4(p + 16 * i);
      r[4 * i] = v.x, r[4 * i + 1] = v.y, r[4 * i + 2] = v.z, r[4 * i + 3] = v.w;
    }
  }
}

__device__ __forceinline__ half2_t as_half2(uint32_t v) { return bit_cast<half2_t>(v); }
__device__ __forceinline__ uint32_t as_bits(half2_t v) { return bit_cast<uint32_t>(v); }
// Two bytes 128 + code in the low bytes of halves -> the codes as fp16 (1024 + u is the half 0x6400 | u).
__device__ __forceinline__ uint32_t halves_from_biased_bytes(uint32_t v) {
  return as_bits(as_half2(v | 0x64006400u) - half2_t{static_cast<_Float16>(1152.0f), static_cast<_Float16>(1152.0f)});
}
// Two nibbles in the low bits of halves (two's complement) -> the codes as fp16.
__device__ __forceinline__ uint32_t halves_from_nibbles(uint32_t v) {
  return as_bits(as_half2((v & 0x000F000Fu) ^ 0x64086408u) - half2_t{static_cast<_Float16>(1032.0f), static_cast<_Float16>(1032.0f)});
}
__device__ __forceinline__ uint32_t perm(uint32_t hi, uint32_t lo, uint32_t sel) { return __builtin_amdgcn_perm(hi, lo, sel); }

// Eight elements of one key (`w`: their run) as a matrix operand, in the order kq_dim.
template <KvKind KV>
__device__ __forceinline__ half8_t key_operand(const uint32_t* w) {
  uint4 r;
  if constexpr (KV == KvKind::F16) {
    r = uint4{w[0], w[1], w[2], w[3]};
  } else if constexpr (KV == KvKind::Q8) {
    const uint32_t a = w[0] ^ 0x80808080u, b = w[1] ^ 0x80808080u;
    r = uint4{halves_from_biased_bytes(perm(0, a, 0x0C010C00)), halves_from_biased_bytes(perm(0, a, 0x0C030C02)),
              halves_from_biased_bytes(perm(0, b, 0x0C010C00)), halves_from_biased_bytes(perm(0, b, 0x0C030C02))};
  } else if constexpr (KV == KvKind::Q4) {
    const uint32_t a = perm(0, w[0], 0x0C010C00), b = perm(0, w[0], 0x0C030C02);
    r = uint4{halves_from_nibbles(a), halves_from_nibbles(a >> 4), halves_from_nibbles(b), halves_from_nibbles(b >> 4)};
  } else {
    r = uint4{as_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[0], 1.0f, false)), as_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[0], 1.0f, true)),
              as_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[1], 1.0f, false)), as_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w[1], 1.0f, true))};
  }
  return bit_cast<half8_t>(r);
}
// The element of a run of eight that sits in slot e of key_operand: 4-bit codes come low nibbles of two
// bytes first.
template <KvKind KV>
__device__ constexpr int kq_dim(int e) {
  if (KV != KvKind::Q4) return e;
  const int order[8] = {0, 2, 1, 3, 4, 6, 5, 7};
  return order[e];
}

// Element j of the runs of two keys as a pair of fp16 numbers (the first key in the low half).
template <KvKind KV>
__device__ __forceinline__ uint32_t value_pair(const uint32_t* k0, const uint32_t* k1, int j) {
  if constexpr (KV == KvKind::F16) {
    return perm(k1[j / 2], k0[j / 2], (j & 1) ? 0x07060302u : 0x05040100u);
  } else if constexpr (KV == KvKind::Q8) {
    const uint32_t b = static_cast<uint32_t>(j & 3);
    return halves_from_biased_bytes(perm(k1[j / 4], k0[j / 4], 0x0C000C00u | ((4u + b) << 16) | b) ^ 0x00800080u);
  } else if constexpr (KV == KvKind::Q4) {
    const uint32_t b = static_cast<uint32_t>(j & 7) / 2u;
    const uint32_t t = perm(k1[j / 8], k0[j / 8], 0x0C000C00u | ((4u + b) << 16) | b);
    return halves_from_nibbles((j & 1) ? t >> 4 : t);
  } else {
    const uint32_t b = static_cast<uint32_t>(j & 3);
    return as_bits(__builtin_amdgcn_cvt_scalef32_pk_f16_fp8(perm(k1[j / 4], k0[j / 4], 0x0C0C0000u | ((4u + b) << 8) | b), 1.0f, false));
  }
}

// Maximum / sum over the four groups of sixteen lanes; every lane returns it.
__device__ __forceinline__ float groups_max(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(bit_cast<uint32_t>(v), bit_cast<uint32_t>(v), false, false);
  v = fmaxf(bit_cast<float>(a[0]), bit_cast<float>(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(bit_cast<uint32_t>(v), bit_cast<uint32_t>(v), false, false);
  return fmaxf(bit_cast<float>(b[0]), bit_cast<float>(b[1]));
}
__device__ __forceinline__ float groups_sum(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(bit_cast<uint32_t>(v), bit_cast<uint32_t>(v), false, false);
  v = bit_cast<float>(a[0]) + bit_cast<float>(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(bit_cast<uint32_t>(v), bit_cast<uint32_t>(v), false, false);
  return bit_cast<float>(b[0]) + bit_cast<float>(b[1]);
}
// The value of the neighbouring lane (lane ^ 1).
__device__ __forceinline__ float other_term(float v) {
  return bit_cast<float>(__builtin_amdgcn_update_dpp(0, bit_cast<int>(v), 0xB1, 0xF, 0xF, false));
}
// 2^(target - exponent of v) for v > 0, within what fp32 can hold.
__device__ __forceinline__ float power_of_two_to(float v, int target) {
  const int e = static_cast<int>(bit_cast<uint32_t>(v) >> 23 & 255u);
  const int s = 254 + target - e;
  return bit_cast<float>(static_cast<uint32_t>(s > 254 ? 254 : s < 1 ? 1 : s) << 23);
}

constexpr float kLog2E = 1.44269504088896340736f, kLn2 = 0.69314718055994530942f;

// What weights are taken relative to: the largest score, or 0 where every score so far is -inf (the weights
// are then 0, not exp(-inf + inf)).
__device__ __forceinline__ float reference_score(float largest) { return largest == -INFINITY ? 0.0f : largest; }
// A second term's sum where the cache's side may hold infinities: infinity times the (possibly zero or
// negative) second term says nothing that the first term's sum does not.
__device__ __forceinline__ float finite_or_zero(float v) { return __builtin_isfinite(v) ? v : 0.0f; }

// Query heads a workgroup takes at once, and what its wavefronts hand to the merge.
template <KvKind KV>
constexpr int rows_heads() { return KV == KvKind::F32 ? 16 : 8; }
template <KvKind KV, int DP, int NW>
struct RowsShared {
  float m[NW][rows_heads<KV>()], l[NW][rows_heads<KV>()], scale[rows_heads<KV>()];
  alignas(16) float o[NW][rows_heads<KV>()][16][DP / 16 + 4];
};

// A part without keys, of heads head0 .. head0 + here - 1 of a row.
template <int THREADS>
__device__ __forceinline__ void empty_part(const AttentionArgs& a, uint64_t row, uint32_t head0, uint32_t here, uint64_t s_part) {
  const uint32_t t = threadIdx.x, D = a.head_dim;
  const uint64_t split = a.part.split;
  for (uint32_t i = t; i < here * D; i += THREADS) a.part.pacc[((row * a.heads + head0 + i / D) * split + s_part) * D + i % D] = 0.0f;
  if (t < here) {
    const uint64_t at = (row * a.heads + head0 + t) * split + s_part;
    a.part.pmax[at] = -1e30f, a.part.psum[at] = 0.0f;
  }
}

// Heads head0 .. head0 + here - 1 (at most rows_heads, all of key head kv) of query row `row` over keys start .. last:
// part s_part of the row, or all of it.  KEYS: keys a tile, 16 where the registers of 32 are not to be had.
template <KvKind KV, int DP, int NW, int KEYS = KV == KvKind::F32 ? 16 : 32>
__device__ __forceinline__ void attend_row(const AttentionArgs& a, uint64_t row, uint32_t kv, uint32_t head0, uint32_t here,
                                           uint64_t start, uint64_t last, uint64_t s_part, RowsShared<KV, DP, NW>& merge) {
  constexpr bool F32 = KV == KvKind::F32, QUANT = kv_quantized(KV);
  constexpr int BITS = kv_bits(KV);
  constexpr int CE = F32 ? 4 : 128 / BITS < DP / 4 ? 128 / BITS : DP / 4;   // elements of a key a lane loads at once
  constexpr int RUNS = DP / (4 * CE);                              // such loads a key row
  constexpr int STEPS = F32 ? DP / 4 : DP / 32;                    // matrix instructions over head_dim
  constexpr int CHAINS = F32 ? STEPS / 4 : STEPS / 2 < 1 ? 1 : STEPS / 2;   // sums of a score
  constexpr int VE = DP / 16;                                      // elements of a value row a lane holds
  constexpr int KW = CE * BITS / 32, VW = (VE * BITS + 31) / 32;   // dwords of those
  constexpr int HALVES = KEYS / 16;

  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6, r = lane & 15u, g = lane >> 4;
  const uint64_t split = a.part.split == 0 ? 1 : a.part.split;
  const uint32_t D = a.head_dim;

  const uint64_t stride = static_cast<uint64_t>(a.kv_heads) * D * BITS / 8;
  const uint8_t* kb = static_cast<const uint8_t*>(a.k) + static_cast<uint64_t>(kv) * D * BITS / 8;
  const uint8_t* vb = static_cast<const uint8_t*>(a.v) + static_cast<uint64_t>(kv) * D * BITS / 8;
  uint32_t kr[HALVES][RUNS][KW], vr[4 * HALVES][VW];
  float ksv[4 * HALVES], vsv[4 * HALVES];
  // Rows past the range's end are read as its last row: finite numbers that get the weight 0.
  auto key_at = [&](uint64_t j) { return j < last ? j : last; };
  auto load_keys = [&](uint64_t j0) {
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      const uint8_t* p = kb + key_at(j0 + 16 * h + r) * stride;
#pragma unroll
      for (int i = 0; i < RUNS; ++i) {
        const uint32_t d = (i * 4 + g) * CE;
        if (d < D) {
          load_run<CE * BITS / 8>(p + d * BITS / 8, kr[h][i]);
        } else {
#pragma unroll
          for (int w = 0; w < KW; ++w) kr[h][i][w] = 0u;
        }
      }
    }
    if constexpr (QUANT) {
#pragma unroll
      for (int e = 0; e < 4 * HALVES; ++e) ksv[e] = a.k_scale[key_at(j0 + 16 * (e / 4) + 4 * g + e % 4)];
    }
  };
  auto load_values = [&](uint64_t j0) {
#pragma unroll
    for (int e = 0; e < 4 * HALVES; ++e) {
      const uint64_t key = key_at(j0 + 16 * (e / 4) + 4 * g + e % 4);
      if (r * VE < D) {
        load_run<VE * BITS / 8>(vb + key * stride + r * VE * BITS / 8, vr[e]);
      } else {
#pragma unroll
        for (int w = 0; w < VW; ++w) vr[e][w] = 0u;
      }
      if constexpr (QUANT) vsv[e] = a.v_scale[key];
    }
  };
  const uint64_t first = start + wave * KEYS;
  if (first <= last) {
    load_keys(first);
    load_values(first);
  }

  // The query operand: column r is head r (fp32) or the term r % 2 of head r / 2.
  const uint32_t column_head = F32 ? r : r / 2u;
  const bool second = !F32 && (r & 1u) != 0u;                      // this lane's column is a second term
  const float term_down = second ? 0x1p-11f : 1.0f;
  // Of the two terms of x and of y this lane's: hi, or 2^11 (x - hi).  (x and y are kept apart from their conversions, which
  // make two numbers at once: a multiply-add that rounds to fp16 takes the vector unit twice a conversion's time.  Not where
  // the registers are just enough, KEYS = 16.)
  auto terms_of = [&](float x, float y) {
    constexpr bool APART = F32 || KEYS == 32;
    if constexpr (APART) asm("" : "+v"(x), "+v"(y));
    const half2_t hi = {static_cast<_Float16>(x), static_cast<_Float16>(y)};
    if constexpr (!APART) {
      return half2_t{second ? static_cast<_Float16>((x - static_cast<float>(hi[0])) * 0x1p11f) : hi[0],
                     second ? static_cast<_Float16>((y - static_cast<float>(hi[1])) * 0x1p11f) : hi[1]};
    }
    float low_x = (x - static_cast<float>(hi[0])) * 0x1p11f, low_y = (y - static_cast<float>(hi[1])) * 0x1p11f;
    asm("" : "+v"(low_x), "+v"(low_y));
    const half2_t lo = {static_cast<_Float16>(low_x), static_cast<_Float16>(low_y)};
    return bit_cast<half2_t>(second ? bit_cast<uint32_t>(lo) : bit_cast<uint32_t>(hi));
  };
  const float* qp = a.q + ((a.row_base + row) * a.heads + head0 + (column_head < here ? column_head : here - 1u)) * D;
  float qf[F32 ? STEPS : 1];
  half8_t qh[F32 ? 1 : STEPS];
  // A column's scores are kept as the matrix instructions leave them, s; score_scale s is in units of log2.  Only
  // differences from the largest are brought to those units, so that rounding goes with their size.
  float score_scale = kLog2E / sqrtf(static_cast<float>(D));
  if constexpr (F32) {
#pragma unroll
    for (int i = 0; i < RUNS; ++i) {
      const uint32_t d = (i * 4 + g) * CE;
      const float4 x = d < D ? *reinterpret_cast<const float4*>(qp + d) : float4{0.0f, 0.0f, 0.0f, 0.0f};
      qf[4 * i] = x.x, qf[4 * i + 1] = x.y, qf[4 * i + 2] = x.z, qf[4 * i + 3] = x.w;
    }
  } else {
    float raw[STEPS][8], most = 0.0f;
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const uint32_t d = ((i * 8 / CE) * 4 + g) * CE + i * 8 % CE;
      const float4 x = d < D ? *reinterpret_cast<const float4*>(qp + d) : float4{0.0f, 0.0f, 0.0f, 0.0f};
      const float4 y = d < D ? *reinterpret_cast<const float4*>(qp + d + 4) : float4{0.0f, 0.0f, 0.0f, 0.0f};
      raw[i][0] = x.x, raw[i][1] = x.y, raw[i][2] = x.z, raw[i][3] = x.w;
      raw[i][4] = y.x, raw[i][5] = y.y, raw[i][6] = y.z, raw[i][7] = y.w;
#pragma unroll
      for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(raw[i][e]));
    }
    most = groups_max(most);
    const float up = most == 0.0f ? 1.0f : power_of_two_to(most, 14);
    score_scale /= up;
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const half2_t pair = terms_of(raw[i][kq_dim<KV>(e)] * up, raw[i][kq_dim<KV>(e + 1)] * up);
        qh[i][e] = pair[0], qh[i][e + 1] = pair[1];
      }
    }
  }

  float4_t o[VE];
#pragma unroll
  for (int j = 0; j < VE; ++j) o[j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float run_max = -INFINITY, run_sum = 0.0f;
  float lane_most = 0.0f, value_up = F32 ? 1.0f : QUANT ? power_of_two_to(0.0f, 14) : 0x1p14f;
  for (uint64_t j0 = first; j0 <= last; j0 += NW * KEYS) {
    const bool more = j0 + NW * KEYS <= last;
    float s[4 * HALVES];
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      // One matrix instruction after another on one sum rounds at every step: CHAINS sums, added pairwise.
      float4_t sums[CHAINS];
#pragma unroll
      for (int c = 0; c < CHAINS; ++c) sums[c] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < STEPS; ++i) {
        float4_t& acc = sums[i * CHAINS / STEPS];
        if constexpr (F32) {
          acc = __builtin_amdgcn_mfma_f32_16x16x4f32(bit_cast<float>(kr[h][i / 4][i % 4]), qf[i], acc, 0, 0, 0);
        } else {
          acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(key_operand<KV>(&kr[h][i * 8 / CE][i * 8 % CE * BITS / 32]), qh[i], acc, 0, 0, 0);
        }
      }
#pragma unroll
      for (int c = CHAINS / 2; c > 0; c /= 2) {
#pragma unroll
        for (int i = 0; i < c; ++i) sums[i] += sums[i + c];
      }
      const float4_t acc = sums[0];
#pragma unroll
      for (int e = 0; e < 4; ++e) s[4 * h + e] = acc[e] * term_down;
    }
    float own[4 * HALVES], all = 0.0f;
#pragma unroll
    for (int e = 0; e < 4 * HALVES; ++e) {
      own[e] = s[e];
      if constexpr (!F32) s[e] += other_term(s[e]);
      if constexpr (QUANT) s[e] *= ksv[e];
      all += s[e];
    }
    if constexpr (QUANT) {
      // A key with an infinite scale is NaN where its code is 0; its score is formed from the codes' sum, which is not.
      float scale_most = ksv[0];
#pragma unroll
      for (int e = 1; e < 4 * HALVES; ++e) scale_most = fmaxf(scale_most, ksv[e]);
      if (__any(scale_most == INFINITY)) {
#pragma unroll
        for (int e = 0; e < 4 * HALVES; ++e) s[e] = ksv[e] == INFINITY ? NAN : s[e];
      }
    }
    if (more) load_keys(j0 + NW * KEYS);
    if constexpr (KV == KvKind::F16) {
      if (__any(!(fabsf(all) < INFINITY))) {       // infinities among the keys
#pragma unroll
        for (int e = 0; e < 4 * HALVES; ++e) {
          const float x = second ? finite_or_zero(own[e]) : own[e];
          s[e] = x + other_term(x);
        }
      }
    }
    const bool past = j0 + KEYS - 1 > last;        // the range ends inside this tile
    if (past) {
#pragma unroll
      for (int e = 0; e < 4 * HALVES; ++e) {
        const bool none = j0 + 16 * (e / 4) + 4 * g + e % 4 > last;
        s[e] = none ? -INFINITY : s[e];
        if constexpr (QUANT) vsv[e] = none ? 0.0f : vsv[e];
      }
    }

    float most = s[0];
#pragma unroll
    for (int e = 1; e < 4 * HALVES; ++e) most = fmaxf(most, s[e]);
    const float m_new = fmaxf(run_max, groups_max(most));
    const float m_ref = reference_score(m_new);
    float corr = __builtin_amdgcn_exp2f((run_max - m_ref) * score_scale);   // 0 on the first tile (run_max = -inf)
    run_max = m_new;
    float sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 4 * HALVES; ++e) {
      s[e] = __builtin_amdgcn_exp2f((s[e] - m_ref) * score_scale);
      sum += s[e];
    }
    run_sum = fmaf(corr, run_sum, sum);
    if constexpr (QUANT) {
      // The values' scales enter the weights.  The power of two keeps the largest contribution so far between
      // 2^4 and 2^15.  It is looked at when a new largest score has made the old contributions smaller, and when a
      // scale of this tile would leave the range under the largest weight, 1 (known before the weights are).
      float scale_most = fabsf(vsv[0]);
#pragma unroll
      for (int e = 1; e < 4 * HALVES; ++e) scale_most = fmaxf(scale_most, fabsf(vsv[e]));
      lane_most *= corr;
#pragma unroll
      for (int e = 0; e < 4 * HALVES; ++e) {
        s[e] *= vsv[e];
        lane_most = fmaxf(lane_most, fabsf(s[e]));
      }
      if (__any(corr != 1.0f || !(scale_most * value_up < 0x1p15f))) {
        const float largest = groups_max(lane_most), scaled = largest * value_up;
        if (largest > 0.0f && !(scaled >= 0x1p4f && scaled < 0x1p15f)) {
          const float up = power_of_two_to(largest, 12);
          corr *= up / value_up;
          value_up = up;
        }
      }
#pragma unroll
      for (int e = 0; e < 4 * HALVES; ++e) s[e] *= value_up;
    } else if constexpr (!F32) {
#pragma unroll
      for (int e = 0; e < 4 * HALVES; ++e) s[e] *= value_up;
    }
    if (__any(corr != 1.0f)) {
#pragma unroll
      for (int j = 0; j < VE; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e) o[j][e] *= corr;
      }
    }
    if constexpr (!QUANT) {
      // Rows past the range's end stand for no key: infinite elements of the one read in their place would
      // not vanish under the weight 0.
      if (past) {
#pragma unroll
        for (int e = 0; e < 4 * HALVES; ++e) {
          const bool none = j0 + 16 * (e / 4) + 4 * g + e % 4 > last;
#pragma unroll
          for (int w = 0; w < VW; ++w) vr[e][w] = none ? 0u : vr[e][w];
        }
      }
    }
    if constexpr (F32) {
#pragma unroll
      for (int j = 0; j < VE; ++j) {
        float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};   // the tile's own sum, for the reason of CHAINS
#pragma unroll
        for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(bit_cast<float>(vr[e][j]), s[e], acc, 0, 0, 0);
        o[j] += acc;
      }
    } else {
      half8_t p;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        const half2_t pair = e < 4 * HALVES ? terms_of(s[e % (4 * HALVES)], s[(e + 1) % (4 * HALVES)]) : half2_t{};
        p[e] = pair[0], p[e + 1] = pair[1];
      }
#pragma unroll
      for (int j = 0; j < VE; ++j) {
        uint4 w = {value_pair<KV>(vr[0], vr[1], j), value_pair<KV>(vr[2], vr[3], j), 0u, 0u};
        if constexpr (HALVES == 2) w.z = value_pair<KV>(vr[4], vr[5], j), w.w = value_pair<KV>(vr[6], vr[7], j);
        o[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bit_cast<half8_t>(w), p, o[j], 0, 0, 0);
      }
    }
    if (more) load_values(j0 + NW * KEYS);
  }

  // Merge of the wavefronts: everyone's sum under the largest score of all, added in wavefront order.
  run_sum = groups_sum(run_sum);
  const bool writer = !second;
  if (g == 0u && writer) merge.m[wave][column_head] = run_max, merge.l[wave][column_head] = run_sum;
  if (t < 16u && writer) merge.scale[column_head] = score_scale;
  __syncthreads();
  float top = merge.m[0][column_head];
#pragma unroll
  for (int w = 1; w < NW; ++w) top = fmaxf(top, merge.m[w][column_head]);
  const float f = __builtin_amdgcn_exp2f((run_max - reference_score(top)) * score_scale) / value_up;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int j = 0; j < VE; j += 4) {
      float4 x;
      float* xs = &x.x;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float own = o[j + c][e];
        if constexpr (!F32) own = second ? finite_or_zero(own) : own;
        own *= term_down;
        xs[c] = (F32 ? own : own + other_term(own)) * f;
      }
      if (writer) *reinterpret_cast<float4*>(&merge.o[wave][column_head][4 * g + e][j]) = x;
    }
  }
  __syncthreads();
  for (uint32_t i = t; i < here * D; i += NW * 64u) {
    const uint32_t h = i / D, d = i % D;
    float m = merge.m[0][h];
#pragma unroll
    for (int w = 1; w < NW; ++w) m = fmaxf(m, merge.m[w][h]);
    float sum = 0.0f, acc = 0.0f;
    const float m_ref = reference_score(m), scale = merge.scale[h];
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      sum = fmaf(__builtin_amdgcn_exp2f((merge.m[w][h] - m_ref) * scale), merge.l[w][h], sum);
      acc += merge.o[w][h][d / VE][d % VE];
    }
    if (a.part.split != 0) {
      const uint64_t at = (row * a.heads + head0 + h) * split + s_part;
      // The part's largest score in natural units is rounded; the sums move by what that took from it.
      const float natural = scale * kLn2, largest = m * natural;
      const float moved = m == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(fmaf(m, natural, -largest) * kLog2E);
      a.part.pacc[at * D + d] = acc * moved;
      if (d == 0) a.part.pmax[at] = largest, a.part.psum[at] = sum * moved;
    } else {
      a.out[((a.row_base + row) * a.heads + head0 + h) * D + d] = acc / sum;
    }
  }
}

template <KvKind KV, int DP, int NW>
__global__ __launch_bounds__(NW * 64, 1) void attention_rows_kernel(AttentionArgs a) {
  constexpr uint32_t kHeads = rows_heads<KV>();
  __shared__ RowsShared<KV, DP, NW> merge;
  const uint32_t group = a.heads / a.kv_heads, blocks = (group + kHeads - 1) / kHeads;
  const uint64_t split = a.part.split == 0 ? 1 : a.part.split;
  const uint64_t rest = blockIdx.x / split, row_kv = rest / blocks;
  const uint32_t first = static_cast<uint32_t>(rest % blocks) * kHeads, kv = static_cast<uint32_t>(row_kv % a.kv_heads);
  const uint32_t head0 = kv * group + first, here = group - first < kHeads ? group - first : kHeads;
  const uint64_t row = row_kv / a.kv_heads, s_part = blockIdx.x % split;
  uint64_t start, last;
  key_range(a, row, start, last);
  if (a.part.split != 0 && !key_chunk(a, s_part, start, last)) {   // workgroup-uniform
    empty_part<NW * 64>(a, row, head0, here, s_part);
    return;
  }
  attend_row<KV, DP, NW>(a, row, kv, head0, here, start, last, s_part, merge);
}

// ---- many query rows: a workgroup shares its keys among 64 (row, head) pairs ---------------------
//
// The pairs of a key head, `group` to a row, are the columns of the contractions.  A workgroup owns 64 of them
// and walks the keys that any of them sees, 64 at a time: they are made fp16 (exactly: an fp16 number or a code)
// once, on their way into LDS, keys row by row and values transposed, and every column's two terms meet the same
// operand read.  Eight wavefronts, two a SIMD: four groups of 16 columns times two halves of a tile's keys, each
// wavefront with its own running maximum and sums, merged at the end, and its queries' terms in registers.
//   S^T = K Q^T and O^T = V^T P^T on v_mfma_f32_16x16x32_f16, a lane's weights taken as they stand, as in
//   attend_row, but with a column a pair and both of its terms in one lane.  Row r of block j of O^T stands for
//   element VE r + j, so that a lane ends up with runs of a row of the result.
// A tile's contribution, the second terms' sum brought down by 2^-11 and the first terms' added to it, is summed by
// itself and added to the running sum, so that rounding there goes with a few terms and not with the number of keys.
// 512 rows of 24 heads of 256 on 2512 fp16 keys of 4: 121 us among other calls (432 with a workgroup a row and key head,
// which read each key for six columns), back to back 107 (417), int8 keys 121 (439).  Vector instructions issue in 56 % of
// the cycles, the matrix cores are busy in 34 %, LDS in 30 %; a wavefront waits in 37 % of its own, at the tile's barrier
// and for operands.  STAGGERED: the values' operands are read two groups ahead, the second terms' matrix instructions go one, and
// the running sums are scaled by the multiply-add that adds to them: 512 rows on 2512 keys back to back, 24 heads of 256 106.9 ->
// 103.4 us, int8 119.9 -> 116.0, 24 of 128 int8 77.3 -> 74.0.  fp16 keys of heads of 128 (65 to 128) keep a group after the other:
// 24 heads 60.7 us, staggered 63.6.
// Infinities and NaN are not kept apart here.  Whatever meets one ends with a sum that is not finite, or sets
// `special`; the workgroup's columns are then done again with attend_row.
template <int DP>
struct TileShared {
  static constexpr uint32_t kKeyBytes = 64 * DP * 2, kStage = 2 * kKeyBytes;
  alignas(16) uint8_t stage[2][kStage];        // 64 keys, then two times 32 keys' values transposed
  float scales[2][2][64];                      // keys', values'
  float most[64], sum[64], up[64];             // the second halves'
  uint32_t special;
};

template <KvKind KV, int DP>
__global__ __launch_bounds__(512, 2) void attention_tile_kernel(AttentionArgs a) {
  constexpr bool QUANT = kv_quantized(KV);
  constexpr int BITS = kv_bits(KV);
  constexpr int STEPS = DP / 32, CHAINS = STEPS / 2;               // matrix instructions of a score, its sums (as in attend_row)
  constexpr int VE = DP / 16, RE = DP / 32;                        // elements of a row of the result, of a value run
  constexpr int GROUP = DP == 256 ? 2 : 4;                                         // operands read at once
  constexpr int CHUNKS = DP / 8;                                   // runs of eight elements of a key
  constexpr int KLOADS = 64 * CHUNKS / 512;
  constexpr int KW = 8 * BITS / 32, VW = (RE * BITS + 31) / 32;
  using Shared = TileShared<DP>;
  union Lds {
    Shared tile;
    RowsShared<KV, DP, 8> rows;
    __device__ Lds() {}
  };
  __shared__ Lds lds;
  Shared& sh = lds.tile;

  const uint32_t t = threadIdx.x, lane = t & 63u, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t r = lane & 15u, g = lane >> 4, col_group = wave & 3u, half = wave >> 2;
  const uint32_t D = a.head_dim, group = a.heads / a.kv_heads;
  const uint32_t split = a.part.split == 0 ? 1u : static_cast<uint32_t>(a.part.split), units = gridDim.x / a.kv_heads;
  const uint32_t kv = blockIdx.x % a.kv_heads, unit = units - 1u - blockIdx.x / a.kv_heads, s_part = unit % split;
  const uint32_t columns = static_cast<uint32_t>(a.rows * group);  // fewer than 2^29, as a grid has fewer than 2^32 threads
  const uint32_t c0 = unit / split * 64u;                          // the longest first
  const uint32_t c_end = c0 + 64u < columns ? c0 + 64u : columns;
  // A value the compiler takes for a new one: at head size 256, where the registers are just enough, what is needed
  // only now and then or after the walk over the keys is formed from the thread's number again, not held.
  auto again = [](uint32_t v) {
    if constexpr (DP == 256) asm volatile("" : "+v"(v));
    return v;
  };
  // This lane's column of the workgroup's, past the last one the last.
  struct Column {
    uint64_t row;
    uint32_t head;
  };
  auto column = [&]() {
    const uint32_t at = c0 + col_group * 16u + (again(t) & 15u), col = at < c_end ? at : c_end - 1u;
    return Column{col / group, kv * group + col % group};
  };
  const Column mine = column();
  uint64_t first_key, last_key;
  key_range(a, mine.row, first_key, last_key);
  const uint32_t start = static_cast<uint32_t>(first_key), last = static_cast<uint32_t>(last_key);
  key_range(a, c0 / group, first_key, last_key);
  uint32_t wg_start = static_cast<uint32_t>(first_key);
  const uint32_t first_row_last = static_cast<uint32_t>(last_key);
  key_range(a, (c_end - 1) / group, first_key, last_key);
  uint32_t wg_last = static_cast<uint32_t>(last_key);
  const uint32_t last_row_start = static_cast<uint32_t>(first_key);
  // Calls f(row, first head, heads) for the workgroup's columns, rows_heads of a row at most at a time.
  auto for_rows = [&](auto f) {
    for (uint32_t c = c0; c < c_end;) {
      const uint32_t h = c % group;
      uint32_t here = group - h < rows_heads<KV>() ? group - h : rows_heads<KV>();
      if (here > c_end - c) here = c_end - c;
      f(c / group, kv * group + h, here);
      c += here;
    }
  };
  if (split > 1u) {                                                // whole tiles of the workgroup's keys a part
    const uint32_t chunk = ((wg_last - wg_start + split) / split + 63u) / 64u * 64u;
    if (s_part * chunk > wg_last - wg_start) {
      for_rows([&](uint64_t i, uint32_t head0, uint32_t here) { empty_part<512>(a, i, head0, here, s_part); });
      return;
    }
    wg_start += s_part * chunk;
    if (wg_last - wg_start >= chunk) wg_last = wg_start + chunk - 1u;
  }

  const uint64_t stride = static_cast<uint64_t>(a.kv_heads) * D * BITS / 8;
  const uint8_t* kb = static_cast<const uint8_t*>(a.k) + static_cast<uint64_t>(kv) * D * BITS / 8;
  const uint8_t* vb = static_cast<const uint8_t*>(a.v) + static_cast<uint64_t>(kv) * D * BITS / 8;
  uint32_t kr[KLOADS][KW], vr[4][VW];
  float sr = 0.0f;
  // This thread's share of a tile's loads: chunk k_chunk of keys k_key + (512 / CHUNKS) i, elements RE v_run.. of keys
  // 4 v_four.. (lanes l and l + 16 write the halves of a chunk).  Elements past head_dim are read as the row's first: the
  // queries are 0 there, of the result they are not stored.
  struct Share {
    uint32_t k_key, k_chunk, v_run, v_four, k_elem, v_elem;
  };
  auto share_of = [&](uint32_t thread) {
    Share s;
    s.k_key = thread / CHUNKS, s.k_chunk = thread % CHUNKS;
    s.v_run = (thread & 15u) * 2u + (thread >> 5 & 1u), s.v_four = half * 8u + (thread >> 4 & 1u) * 4u + col_group;
    s.k_elem = s.k_chunk * 8u < D ? s.k_chunk * BITS : 0u, s.v_elem = s.v_run * RE < D ? s.v_run * RE * BITS / 8 : 0u;
    return s;
  };
  const Share own_share = share_of(t);
  const uint32_t stride32 = static_cast<uint32_t>(stride);
  const uint32_t k_off = own_share.k_key * stride32 + own_share.k_elem, v_off = own_share.v_four * 4u * stride32 + own_share.v_elem;
  auto fetch = [&](uint32_t j0) {
    const uint32_t left = wg_last - j0;
    const uint8_t *k_tile = kb + j0 * stride, *v_tile = vb + j0 * stride;
    if (left >= 63u) {
#pragma unroll
      for (int i = 0; i < KLOADS; ++i) load_run<BITS>(k_tile + i * (512 / CHUNKS) * stride + k_off, kr[i]);
#pragma unroll
      for (int e = 0; e < 4; ++e) load_run<RE * BITS / 8>(v_tile + e * stride + v_off, vr[e]);
    } else {
      // The last tile: keys past the range's end are read as its last one; no column sees them.
      const Share late = share_of(again(t));
#pragma unroll
      for (int i = 0; i < KLOADS; ++i) {
        const uint32_t key = late.k_key + i * (512u / CHUNKS);
        load_run<BITS>(k_tile + (key < left ? key : left) * stride32 + late.k_elem, kr[i]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t key = late.v_four * 4u + e;
        load_run<RE * BITS / 8>(v_tile + (key < left ? key : left) * stride32 + late.v_elem, vr[e]);
      }
    }
    if constexpr (QUANT) {
      const uint32_t key = t & 63u;
      if (t < 128u) sr = (t < 64u ? a.k_scale : a.v_scale)[j0 + (key < left ? key : left)];
    }
  };
  // A key's row in LDS: its chunks of sixteen bytes at c ^ swizzle, so that neighbouring keys' chunks fall on
  // different banks; 256 bytes hold 16 chunks.
  auto key_swizzle = [](uint32_t key) { return CHUNKS >= 16 ? key & 15u : (key >> 1) & 7u; };
  auto value_place = [](uint32_t row, uint32_t chunk) { return (row & 3u) * 256u + (row >> 2) * 64u + ((chunk ^ (row & 3u)) * 16u); };
  auto stash = [&](uint32_t b) {
    uint8_t* keys = sh.stage[b];
#pragma unroll
    for (int i = 0; i < KLOADS; ++i) {
      const uint32_t key = own_share.k_key + i * (512u / CHUNKS);
      *reinterpret_cast<half8_t*>(keys + key * (DP * 2u) + ((own_share.k_chunk ^ key_swizzle(key)) * 16u)) = key_operand<KV>(kr[i]);
    }
    // Row r of block j of a half's values: four chunks of sixteen bytes, chunk c of keys 4c.. and 16 + 4c.. at
    // c ^ r % 4; the rows in the order 0, 4, 8, 12, 1, .., which with that puts sixteen lanes on sixteen bank groups.
    const uint32_t vrow = own_share.v_run >> 1, four = own_share.v_four & 7u;
    uint8_t* values = keys + Shared::kKeyBytes + half * (DP * 64u) + (own_share.v_run & 1u) * (RE * 1024u) + value_place(vrow, four & 3u) + (four >> 2) * 8u;
#pragma unroll
    for (int j = 0; j < RE; ++j) {
      *reinterpret_cast<uint2*>(values + j * 1024u) = uint2{value_pair<KV>(vr[0], vr[1], j), value_pair<KV>(vr[2], vr[3], j)};
    }
    if constexpr (QUANT) {
      if (t < 128u) {
        sh.scales[b][t >> 6][t & 63u] = sr;
        if (t < 64u && !(fabsf(sr) < INFINITY)) sh.special = 1u;   // such a key's score says nothing of its weight here
      }
    }
  };

  if (t == 0) sh.special = 0u;
  fetch(wg_start);

  // The queries' terms.
  half8_t q_hi[STEPS], q_lo[STEPS];
  float score_scale = kLog2E / sqrtf(static_cast<float>(D));
  {
    const float* qp = a.q + ((a.row_base + mine.row) * a.heads + mine.head) * D;
    float raw[STEPS][8], most = 0.0f;
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const uint32_t d = i * 32u + g * 8u;
      const float4 x = d < D ? *reinterpret_cast<const float4*>(qp + d) : float4{0.0f, 0.0f, 0.0f, 0.0f};
      const float4 y = d < D ? *reinterpret_cast<const float4*>(qp + d + 4) : float4{0.0f, 0.0f, 0.0f, 0.0f};
      raw[i][0] = x.x, raw[i][1] = x.y, raw[i][2] = x.z, raw[i][3] = x.w;
      raw[i][4] = y.x, raw[i][5] = y.y, raw[i][6] = y.z, raw[i][7] = y.w;
#pragma unroll
      for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(raw[i][e]));
    }
    most = groups_max(most);
    const float up = most == 0.0f ? 1.0f : power_of_two_to(most, 14);
    score_scale /= up;
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = raw[i][kq_dim<KV>(e)] * up;
        const _Float16 hi = static_cast<_Float16>(v);
        q_hi[i][e] = hi;
        q_lo[i][e] = static_cast<_Float16>((v - static_cast<float>(hi)) * 0x1p11f);
      }
    }
  }
  __syncthreads();                                                 // `special` is set up
  stash(0);
  if (wg_last - wg_start >= 64u) fetch(wg_start + 64u);
  __syncthreads();

  float4_t o[VE];
#pragma unroll
  for (int j = 0; j < VE; ++j) o[j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  float run_max = -INFINITY, run_sum = 0.0f;
  float lane_most = 0.0f, value_up = QUANT ? power_of_two_to(0.0f, 14) : 0x1p14f;
  const uint32_t key_row = (half * 32u + r) * (DP * 2u), key_swz = key_swizzle(r);
  const uint32_t value_row = Shared::kKeyBytes + half * (DP * 64u) + value_place(r, g);
  // A tile's loads are under way for the whole of the tile before it, and it goes to LDS after that one's scores.
  for (uint32_t j0 = wg_start, b = 0; j0 <= wg_last; j0 += 64u, b ^= 1u) {
    const uint8_t* stage = sh.stage[b];

    // Element 4 h + e of a lane: key 16 h + 4 g + e of the wavefront's 32.  Operands are read a group ahead of
    // their matrix instructions; the barriers keep the compiler from moving each read to its use.
    float s[8];
    float4_t hi[CHAINS], lo;
    half8_t kf[2][GROUP];
    auto read_keys = [&](int n, half8_t (&f)[GROUP]) {
#pragma unroll
      for (int i = 0; i < GROUP; ++i) {
        const uint32_t h = (n * GROUP + i) / STEPS, step = (n * GROUP + i) % STEPS;
        f[i] = *reinterpret_cast<const half8_t*>(stage + key_row + h * (16u * DP * 2u) + (((4u * step + g) ^ key_swz) * 16u));
      }
    };
    read_keys(0, kf[0]);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int n = 0; n < 2 * STEPS / GROUP; ++n) {
      if (n + 1 < 2 * STEPS / GROUP) read_keys(n + 1, kf[(n + 1) & 1]);
#pragma unroll
      for (int i = 0; i < GROUP; ++i) {
        const int h = (n * GROUP + i) / STEPS, step = (n * GROUP + i) % STEPS;
        if (step == 0) {
          lo = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int c = 0; c < CHAINS; ++c) hi[c] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        }
        hi[step % CHAINS] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[n & 1][i], q_hi[step], hi[step % CHAINS], 0, 0, 0);
        lo = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf[n & 1][i], q_lo[step], lo, 0, 0, 0);
        if (step == STEPS - 1) {
#pragma unroll
          for (int c = CHAINS / 2; c > 0; c /= 2) {
#pragma unroll
            for (int x = 0; x < c; ++x) hi[x] += hi[x + c];
          }
#pragma unroll
          for (int e = 0; e < 4; ++e) s[4 * h + e] = fmaf(lo[e], 0x1p-11f, hi[0][e]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (wg_last - j0 >= 64u) stash(b ^ 1u);
    if (wg_last - j0 >= 128u) fetch(j0 + 128u);
    // The values' operands: groups of BLOCKS blocks of O^T, read AHEAD groups before their matrix instructions.
    constexpr bool STAGGERED = QUANT || DP != 128;
    constexpr int BLOCKS = !STAGGERED ? GROUP : DP == 256 ? 1 : 2, GROUPS = VE / BLOCKS, AHEAD = STAGGERED ? 2 : 1;
    half8_t vf[AHEAD + 1][BLOCKS];
    auto read_values = [&](int n) {
#pragma unroll
      for (int i = 0; i < BLOCKS; ++i) vf[n % (AHEAD + 1)][i] = *reinterpret_cast<const half8_t*>(stage + value_row + (n * BLOCKS + i) * 1024u);
    };
    read_values(0);
    float vsv[8];
    if constexpr (QUANT) {
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const uint32_t at = half * 32u + h * 16u + g * 4u;
        const float4 ks = *reinterpret_cast<const float4*>(&sh.scales[b][0][at]), vs = *reinterpret_cast<const float4*>(&sh.scales[b][1][at]);
        s[4 * h] *= ks.x, s[4 * h + 1] *= ks.y, s[4 * h + 2] *= ks.z, s[4 * h + 3] *= ks.w;
        vsv[4 * h] = vs.x, vsv[4 * h + 1] = vs.y, vsv[4 * h + 2] = vs.z, vsv[4 * h + 3] = vs.w;
      }
    }
    if (j0 + 63 > first_row_last || j0 < last_row_start) {         // some column does not see some key of the tile
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t key = j0 + half * 32u + 16u * (e / 4) + 4u * g + e % 4;
        s[e] = key >= start && key <= last ? s[e] : -INFINITY;
      }
    }
    float most = s[0];
#pragma unroll
    for (int e = 1; e < 8; ++e) most = fmaxf(most, s[e]);
    const float m_new = fmaxf(run_max, groups_max(most));
    const float m_ref = reference_score(m_new);
    float corr = __builtin_amdgcn_exp2f((run_max - m_ref) * score_scale);   // 0 on the first tile (run_max = -inf)
    run_max = m_new;
    float sum = 0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      s[e] = __builtin_amdgcn_exp2f((s[e] - m_ref) * score_scale);
      sum += s[e];
    }
    run_sum = fmaf(corr, run_sum, sum);
    if constexpr (QUANT) {
      // As in attend_row: the power of two follows the largest contribution.
      float scale_most = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) scale_most = fmaxf(scale_most, fabsf(vsv[e]));
      lane_most *= corr;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        s[e] *= vsv[e];
        lane_most = fmaxf(lane_most, fabsf(s[e]));
      }
      if (__any(corr != 1.0f || !(scale_most * value_up < 0x1p15f))) {
        const float largest = groups_max(lane_most), scaled = largest * value_up;
        if (largest > 0.0f && !(scaled >= 0x1p9f && scaled < 0x1p15f)) {
          const float up = power_of_two_to(largest, 13);
          corr *= up / value_up;
          value_up = up;
        }
      }
    }
    // APART: x and the rests are kept apart from their conversions (a multiply that rounds to fp16 takes the vector unit twice a
    // conversion's time).  It leads for fp16 keys of heads of 64 and 256, elsewhere the compiler's own choice does (us, 512 rows on
    // 2512 keys, apart / not: fp16, 24 heads of 256 103.4 / 105.7, 16 of 64 30.9 / 31.3; int8, 32 of 64 56.3 / 54.7, 24 of 128 75.4 / 74.0).
    constexpr bool APART = !QUANT && STAGGERED;
    half8_t p_hi, p_lo;
    if constexpr (APART) {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float x = s[e] * value_up;
        asm("" : "+v"(x));
        s[e] = x;
        p_hi[e] = static_cast<_Float16>(x);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float x = (s[e] - static_cast<float>(p_hi[e])) * 0x1p11f;
        asm("" : "+v"(x));
        p_lo[e] = static_cast<_Float16>(x);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float x = s[e] * value_up;
        const _Float16 hi = static_cast<_Float16>(x);
        p_hi[e] = hi;
        p_lo[e] = static_cast<_Float16>((x - static_cast<float>(hi)) * 0x1p11f);
      }
    }
    if constexpr (STAGGERED) {
      // Group n of the operands: its second terms' sums with the first terms' of the group before and the running sums of
      // the one before that, so that no instruction waits for the matrix instruction that has just been issued.
      float4_t low[2][BLOCKS], own[2][BLOCKS];
#pragma unroll
      for (int n = 1; n < AHEAD && n < GROUPS; ++n) read_values(n);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < GROUPS + 2; ++n) {
        if (n < GROUPS) {
#pragma unroll
          for (int i = 0; i < BLOCKS; ++i) {
            low[n & 1][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[n % (AHEAD + 1)][i], p_lo, float4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
          }
        }
        if (n >= 1 && n - 1 < GROUPS) {
#pragma unroll
          for (int i = 0; i < BLOCKS; ++i) {
            float4_t x = low[(n - 1) & 1][i];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] *= 0x1p-11f;
            own[(n - 1) & 1][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[(n - 1) % (AHEAD + 1)][i], p_hi, x, 0, 0, 0);
          }
        }
        if (n >= 2) {
#pragma unroll
          for (int i = 0; i < BLOCKS; ++i) {
#pragma unroll
            for (int e = 0; e < 4; ++e) o[(n - 2) * BLOCKS + i][e] = fmaf(o[(n - 2) * BLOCKS + i][e], corr, own[n & 1][i][e]);
            asm volatile("" ::"v"(own[n & 1][i]));      // still held: the multiply-add writes o in place, not here
          }
        }
        if (n + AHEAD < GROUPS) read_values(n + AHEAD);      // where group n - 1 was
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      if (__any(corr != 1.0f)) {
#pragma unroll
        for (int j = 0; j < VE; ++j) {
#pragma unroll
          for (int e = 0; e < 4; ++e) o[j][e] *= corr;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = 0; n < GROUPS; ++n) {
        if (n + 1 < GROUPS) read_values(n + 1);
        float4_t acc[BLOCKS];
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[n & 1][i], p_lo, float4_t{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) {
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][e] *= 0x1p-11f;
          acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[n & 1][i], p_hi, acc[i], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < BLOCKS; ++i) o[n * BLOCKS + i] += acc[i];
      }
    }
    __syncthreads();
  }

  // Merge of the two halves' sums under the larger maximum; the lanes' shares of the sum of weights first.
  run_sum = groups_sum(run_sum);
  const uint32_t late = again(t), late_g = late >> 4 & 3u;
  float* other = reinterpret_cast<float*>(sh.stage[0]) + col_group * (VE * 256u) + (late & 63u);
  const uint32_t at = col_group * 16u + (late & 15u);
  if (half == 1u) {
    if (late_g == 0u) sh.most[at] = run_max, sh.sum[at] = run_sum, sh.up[at] = value_up;
#pragma unroll
    for (int j = 0; j < VE; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) other[(j * 4 + e) * 64] = o[j][e];
  }
  __syncthreads();
  if (half == 0u) {
    const float m1 = sh.most[at], most = fmaxf(run_max, m1), top = reference_score(most);
    const float w0 = __builtin_amdgcn_exp2f((run_max - top) * score_scale), w1 = __builtin_amdgcn_exp2f((m1 - top) * score_scale);
    const float total = fmaf(w1, sh.sum[at], w0 * run_sum);
    const float f0 = w0 / value_up, f1 = w1 / sh.up[at];
    bool finite = fabsf(total) < INFINITY && (split > 1u || total != 0.0f);
#pragma unroll
    for (int j = 0; j < VE; ++j) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float x = fmaf(other[(j * 4 + e) * 64], f1, o[j][e] * f0);
        finite = finite && fabsf(x) < INFINITY;
        other[(j * 4 + e) * 64] = x;
      }
    }
    if (!finite) sh.special = 1u;
    if (late_g == 0u) sh.most[at] = most, sh.sum[at] = total;
  }
  __syncthreads();
  // (the results only now: `out` may be q's memory, which attend_row reads)
  if (__builtin_amdgcn_readfirstlane(sh.special) != 0u) {          // workgroup-uniform
    for_rows([&](uint64_t i, uint32_t head0, uint32_t here) {
      uint64_t row_start, row_last;
      key_range(a, i, row_start, row_last);
      if (split > 1u) {
        row_start = row_start > wg_start ? row_start : wg_start, row_last = row_last < wg_last ? row_last : wg_last;
        if (row_start > row_last) {
          empty_part<512>(a, i, head0, here, s_part);
          return;
        }
      }
      __syncthreads();
      attend_row<KV, DP, 8, DP == 256 ? 16 : 32>(a, i, kv, head0, here, row_start, row_last, s_part, lds.rows);
    });
    return;
  }
  if (c0 + at >= c_end) return;
  const Column own = column();
  const float total = sh.sum[at];
  float* out = a.out + ((a.row_base + own.row) * a.heads + own.head) * D;
  float factor = 1.0f;
  if (split > 1u) {
    const uint64_t part = (own.row * a.heads + own.head) * split + s_part;
    out = a.part.pacc + part * D;
    // The part's largest score in natural units is rounded; the sums move by what that took from it.
    const float most = sh.most[at], natural = score_scale * kLn2, largest = most * natural;
    factor = most == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(fmaf(most, natural, -largest) * kLog2E);
    if (late_g == 0u && half == 0u) a.part.pmax[part] = fmaxf(largest, -1e30f), a.part.psum[part] = total * factor;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t e = half * 2u + i, d = (late_g * 4u + e) * VE;
#pragma unroll
    for (int j = 0; j < VE; j += 4) {
      float x[4];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float sum = other[((j + v) * 4 + e) * 64];
        x[v] = split > 1u ? sum * factor : sum / total;
      }
      if (d + j < D) *reinterpret_cast<float4*>(out + d + j) = float4{x[0], x[1], x[2], x[3]};
    }
  }
}

// ---- head sizes that the matrix kernels' 16-byte runs do not divide ------------------------------
//
// One workgroup of four wavefronts per (query row, head[, chunk]).  Keys are taken 64 at a time: a
// wavefront forms the score of a key with its lanes across head_dim (coalesced key reads, a sum over the
// wavefront), the first wavefront turns the 64 scores into weights against the running maximum, and
// thread e accumulates weight * v[key][e] (coalesced value reads).
template <KvKind KV>
__global__ __launch_bounds__(256) void attention_any_kernel(AttentionArgs a) {
  constexpr uint32_t kKeys = 64;
  __shared__ float sc[kKeys], wt[kKeys], bc[2];
  const uint32_t t = threadIdx.x, lane = t & 63u, wave = t >> 6;
  const uint64_t split = a.part.split == 0 ? 1 : a.part.split, at = blockIdx.x, rest = at / split;
  const uint64_t i = rest / a.heads, h = rest % a.heads, kv = h / (a.heads / a.kv_heads), D = a.head_dim;
  uint64_t start, last;
  key_range(a, i, start, last);
  if (a.part.split != 0 && !key_chunk(a, at % split, start, last)) {   // workgroup-uniform
    if (t < D) a.part.pacc[at * D + t] = 0.0f;
    if (t == 0) a.part.pmax[at] = -1e30f, a.part.psum[at] = 0.0f;
    return;
  }
  const float scale = 1.0f / sqrtf(static_cast<float>(D));
  const uint64_t qb = ((a.row_base + i) * a.heads + h) * D;
  auto kv_at = [&](const void* base, const float* row_scale, uint64_t key, uint64_t idx) {
    if constexpr (KV == KvKind::F16) {
      return half_bits_to_float(static_cast<const uint16_t*>(base)[idx]);
    } else if constexpr (KV == KvKind::F32) {
      return static_cast<const float*>(base)[idx];
    } else if constexpr (KV == KvKind::Q8) {
      return static_cast<float>(static_cast<const int8_t*>(base)[idx]) * row_scale[key];
    } else if constexpr (KV == KvKind::Q4) {
      const int nib = (static_cast<const uint8_t*>(base)[idx >> 1] >> ((idx & 1u) * 4u)) & 0xF;
      return static_cast<float>((nib & 8) ? nib - 16 : nib) * row_scale[key];
    } else {
      return e4m3_to_float(static_cast<const uint8_t*>(base)[idx]) * row_scale[key];
    }
  };
  float qr[4];                       // head_dim <= 256: up to four elements a lane
#pragma unroll
  for (int cc = 0; cc < 4; ++cc) qr[cc] = lane + 64u * cc < D ? a.q[qb + lane + 64u * cc] : 0.0f;

  float run_max = -INFINITY, run_sum = 0.0f, acc = 0.0f;
  for (uint64_t j0 = start; j0 <= last; j0 += kKeys) {
    const uint32_t count = last - j0 + 1 < kKeys ? static_cast<uint32_t>(last - j0 + 1) : kKeys;
    for (uint32_t kk = wave; kk < kKeys; kk += 4u) {
      float dot = 0.0f;
      if (kk < count) {
        const uint64_t kb = ((j0 + kk) * a.kv_heads + kv) * D;
#pragma unroll
        for (int cc = 0; cc < 4; ++cc) {
          if (lane + 64u * cc < D) dot = fmaf(qr[cc], kv_at(a.k, a.k_scale, j0 + kk, kb + lane + 64u * cc), dot);
        }
      }
      dot = wave_sum(dot);
      if (lane == 0) sc[kk] = kk < count ? dot * scale : -INFINITY;
    }
    __syncthreads();
    if (wave == 0) {
      const float s = sc[lane];
      const float m_new = fmaxf(run_max, wave_max(s));
      const float w = lane < count ? expf(s - reference_score(m_new)) : 0.0f;
      wt[lane] = w;
      const float l = wave_sum(w);
      if (lane == 0) {
        bc[0] = m_new;
        bc[1] = l;
      }
    }
    __syncthreads();
    const float m_new = bc[0];
    const float corr = expf(run_max - reference_score(m_new));      // 0 on the first tile (run_max = -inf)
    run_sum = fmaf(corr, run_sum, bc[1]);
    run_max = m_new;
    if (t < D) {
      float x = 0.0f;
      for (uint32_t kk = 0; kk < count; ++kk) {
        x = fmaf(wt[kk], kv_at(a.v, a.v_scale, j0 + kk, ((j0 + kk) * a.kv_heads + kv) * D + t), x);
      }
      acc = fmaf(corr, acc, x);
    }
    __syncthreads();
  }
  if (a.part.split != 0) {
    if (t < D) a.part.pacc[at * D + t] = acc;
    if (t == 0) a.part.pmax[at] = run_max, a.part.psum[at] = run_sum;
  } else {
    if (t < D) a.out[qb + t] = acc / run_sum;
  }
}

// out[row][head] = sum_s w_s pacc_s / sum_s w_s psum_s with w_s = exp(pmax_s - max_s pmax_s)
// (src/backends/rocm/rocm_kernels_basic.cpp:664-690).  One workgroup of WAVES wavefronts per (row, head), V
// consecutive elements a lane, the parts dealt to the wavefronts.  With few rows latency is all there is to it: a wavefront
// asks for four parts' sums before it knows their weights, which its lanes form for all of a round's parts at once.  24 rows
// of 256 over 64 parts: 5.9 us (four wavefronts, a weight formed by every lane for each part: 12.7).
template <int V, int WAVES>
__global__ __launch_bounds__(WAVES * 64) void attention_combine_kernel(const float* __restrict__ pacc, const float* __restrict__ pmax,
                                                                       const float* __restrict__ psum, float* __restrict__ out,
                                                                       uint32_t head_dim, uint32_t split) {
  constexpr uint32_t kRound = 4 * WAVES;                           // parts taken at once
  __shared__ float num[WAVES][64 * V + 1], den_s;
  const uint64_t at = blockIdx.x, base = at * split;
  const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), e0 = lane * V;
  float held[4][V];
  auto fetch = [&](uint32_t s0) {      // parts s0 + wave + WAVES i
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      const uint32_t s = s0 + wave + WAVES * i;
#pragma unroll
      for (int c = 0; c < V; ++c) held[i][c] = s < split && e0 + c < head_dim ? pacc[(base + s) * head_dim + e0 + c] : 0.0f;
    }
  };
  fetch(0);
  float first_max = lane < split ? pmax[base + lane] : -1e30f;
  float first_sum = lane < split ? psum[base + lane] : 0.0f;
  float top = fmaxf(first_max, -1e30f);
  for (uint32_t s = lane + 64u; s < split; s += 64u) top = fmaxf(top, pmax[base + s]);
  top = wave_max(top);
  float n[V] = {}, d = 0.0f;
  for (uint32_t s0 = 0; s0 < split; s0 += kRound) {
    if (s0 != 0u) {
      fetch(s0);
      first_max = s0 + lane < split ? pmax[base + s0 + lane] : -1e30f;
      first_sum = s0 + lane < split ? psum[base + s0 + lane] : 0.0f;
    }
    const bool here = lane < kRound && s0 + lane < split;
    const float w = here ? expf(first_max - top) : 0.0f;
    d = fmaf(w, here ? first_sum : 0.0f, d);
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      if (s0 + wave + WAVES * i >= split) break;                       // wave-uniform: nothing enters for a part that is not there
      const float part_w = bit_cast<float>(__builtin_amdgcn_readlane(bit_cast<int>(w), wave + WAVES * i));
#pragma unroll
      for (int c = 0; c < V; ++c) n[c] = fmaf(part_w, held[i][c], n[c]);
    }
  }
  d = wave_sum(d);
  if constexpr (WAVES == 1) {
#pragma unroll
    for (int c = 0; c < V; ++c) {
      if (e0 + c < head_dim) out[at * head_dim + e0 + c] = n[c] / d;
    }
    return;
  }
#pragma unroll
  for (int c = 0; c < V; ++c) num[wave][e0 + c] = n[c];
  if (threadIdx.x == 0) den_s = d;
  __syncthreads();
  if (threadIdx.x < head_dim) {
    float sum[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if constexpr (WAVES < 16) sum[q] = num[q % WAVES][threadIdx.x];
      else sum[q] = (num[4 * q][threadIdx.x] + num[4 * q + 1][threadIdx.x]) + (num[4 * q + 2][threadIdx.x] + num[4 * q + 3][threadIdx.x]);
    }
    out[at * head_dim + threadIdx.x] = ((sum[0] + sum[1]) + (sum[2] + sum[3])) / den_s;
  }
}

// ---- dispatch ------------------------------------------------------------------------------------

template <KvKind KV>
hipError_t launch_rows(const AttentionArgs& a, uint64_t m, hipStream_t stream) {
  constexpr uint32_t kHeads = KV == KvKind::F32 ? 16 : 8;
  const uint32_t group = a.heads / a.kv_heads, blocks = (group + kHeads - 1) / kHeads;
  const uint64_t split = a.part.split == 0 ? 1 : a.part.split;
  const uint64_t workgroups = m * a.kv_heads * blocks * split;
  const dim3 grid(static_cast<uint32_t>(workgroups));
  // Four wavefronts a workgroup take 128 keys at once; where a workgroup has more to do and the registers and the size of a
  // grid allow it, eight; with no more workgroups than CUs, five take the 129 to 160 keys that parts of 128 come to where they
  // do not divide the keys, and spare a time round (us, four / five: int8, 1200 keys in 9 parts, 4 key heads of 128 8.6 /
  // 7.9, 9301 in 64, 4 of 64 6.7 / 6.2; but two workgroups a CU, 9301 keys, 8 of 128 12.4 / 15.6).  Over an fp32 cache, whose wavefronts
  // take 16 keys at a time, up to 144: from there on all five go round twice (24 heads over 8 of 128, 140 keys 9.7 / 9.0, 160 9.7 /
  // 10.4; 9301 keys in 64 parts of 146, 8 heads over 1 of 128 11.0 / 11.5).
  const uint64_t each = (a.n + split - 1) / split;
  const bool wide = a.n / split > 160 && workgroups < kMaxGridThreads / 512u;
  const bool five = each > 128 && each <= (KV == KvKind::F32 ? 144 : 160) && workgroups <= static_cast<uint64_t>(num_cus());
  auto go = [&](auto kernel, uint32_t waves) { hipLaunchKernelGGL(kernel, grid, dim3(waves * 64u), 0, stream, a); };
  auto pick = [&](auto dim) {
    constexpr int DP = decltype(dim)::value;
    if (DP < 256 && five) go(attention_rows_kernel<KV, DP, DP < 256 ? 5 : 4>, 5);
    else if (DP < 256 && wide) go(attention_rows_kernel<KV, DP, DP < 256 ? 8 : 4>, 8);
    else go(attention_rows_kernel<KV, DP, 4>, 4);
  };
  if (a.head_dim <= 64) pick(std::integral_constant<int, 64>{});
  else if (a.head_dim <= 128) pick(std::integral_constant<int, 128>{});
  else pick(std::integral_constant<int, 256>{});
  return hipGetLastError();
}

// The runs that the lanes of the matrix kernels load divide a head's row: 16 bytes of a key (a quarter of the padded
// row where that is less), a sixteenth of the padded row of a value.
constexpr uint32_t padded_head(uint32_t head_dim) { return head_dim <= 64 ? 64 : head_dim <= 128 ? 128 : 256; }
template <KvKind KV>
bool runs_fit(uint32_t head_dim) {
  const uint32_t padded = padded_head(head_dim);
  const uint32_t run = KV == KvKind::F32 ? 4 : 128u / kv_bits(KV) < padded / 4 ? 128u / kv_bits(KV) : padded / 4;
  return head_dim % run == 0 && head_dim % (padded / 16) == 0;
}

// `a.part.split` parts of the keys (0: one, into `a.out`) for each 64 (row, head) pairs.
template <KvKind KV>
hipError_t launch_tiles(const AttentionArgs& a, hipStream_t stream) {
  const uint64_t split = a.part.split == 0 ? 1 : a.part.split;
  const AttentionCall call{a.rows, a.n, a.heads, a.kv_heads, a.head_dim, 0, false};
  const dim3 grid(static_cast<uint32_t>(attention_pairs64(call) * split));
  auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, dim3(512), 0, stream, a); };
  a.head_dim <= 64 ? go(attention_tile_kernel<KV, 64>) : a.head_dim <= 128 ? go(attention_tile_kernel<KV, 128>) : go(attention_tile_kernel<KV, 256>);
  return hipGetLastError();
}

// kind: 0 fp32, 1 fp16 keys and values; 2 int8, 3 4-bit, 4 E4M3 codes with one scale per key row.
template <class Go>
auto with_kind(uint32_t kind, Go&& go) {
  switch (kind) {
    case 0: return go(std::integral_constant<KvKind, KvKind::F32>{});
    case 1: return go(std::integral_constant<KvKind, KvKind::F16>{});
    case 2: return go(std::integral_constant<KvKind, KvKind::Q8>{});
    case 3: return go(std::integral_constant<KvKind, KvKind::Q4>{});
    default: return go(std::integral_constant<KvKind, KvKind::Fp8>{});
  }
}

hipError_t launch_attention_as(uint32_t kind, const AttentionArgs& a, uint64_t m, hipStream_t stream) {
  return with_kind(kind, [&](auto tag) {
    constexpr KvKind KV = decltype(tag)::value;
    if (runs_fit<KV>(a.head_dim)) return launch_rows<KV>(a, m, stream);
    const uint64_t parts = a.part.split == 0 ? 1 : a.part.split;
    hipLaunchKernelGGL(attention_any_kernel<KV>, dim3(static_cast<uint32_t>(m * a.heads * parts)), dim3(256), 0, stream, a);
    return hipGetLastError();
  });
}

AttentionArgs args_of(const float* q, const void* k, const void* v, const float* k_scale, const float* v_scale, float* out,
                      uint64_t n, uint64_t heads, uint64_t kv_heads, uint64_t head_dim, uint64_t q_base, uint64_t row_base,
                      uint64_t window, bool causal, uint64_t rows) {
  return AttentionArgs{q, k, v, k_scale, v_scale, out, SplitOut{}, rows, n, q_base, row_base, window, static_cast<uint32_t>(heads),
                       static_cast<uint32_t>(kv_heads), static_cast<uint32_t>(head_dim), causal ? 1u : 0u};
}

}  // namespace

uint64_t attention_parts(uint32_t kind, uint64_t m, uint64_t n, uint64_t heads, uint64_t kv_heads, uint64_t head_dim,
                         uint64_t q_base, uint64_t window, bool causal, const void* out, uint64_t most_parts) {
  if (kind == 0 || m < 17 || n >= (1u << 31) || reinterpret_cast<uintptr_t>(out) % 16 != 0) return 0;
  const uint32_t dim = static_cast<uint32_t>(head_dim);
  if (!with_kind(kind, [&](auto tag) { return runs_fit<decltype(tag)::value>(dim); })) return 0;
  if (kv_heads * head_dim * 2 >= (1u << 25)) return 0;             // a tile's rows lie within 2^31 bytes
  uint64_t keys = causal && q_base + m < n ? q_base + m : n;
  if (causal && window != 0 && window < keys) keys = window;
  const AttentionCall call{m, keys, heads, kv_heads, head_dim, padded_head(dim), kind != 1};
  if (attention_pairs64(call) >= kMaxGridThreads / 512u) return 0;
  return attention_rule(call, static_cast<uint64_t>(num_cus()), most_parts, kAttentionPartsMost);
}

size_t attention_parts_bytes(uint64_t m, uint64_t heads, uint64_t head_dim, uint64_t parts) {
  return attention_parts_size(m, heads, head_dim, parts);
}

// kind: 0 fp32, 1 fp16 keys and values; 2 int8, 3 4-bit, 4 E4M3 codes with one scale per key row (always causal).
hipError_t launch_attention(uint32_t kind, const float* q, const void* k, const void* v, const float* k_scale, const float* v_scale,
                            float* out, uint64_t m, uint64_t n, uint64_t heads, uint64_t kv_heads, uint64_t head_dim,
                            uint64_t q_base, uint64_t row_base, uint64_t window, bool causal, uint64_t parts, void* scratch,
                            hipStream_t stream) {
  AttentionArgs a = args_of(q, k, v, k_scale, v_scale, out, n, heads, kv_heads, head_dim, q_base, row_base, window, causal, m);
  if (parts == 0) return launch_attention_as(kind, a, m, stream);
  if (parts > 1) {
    float* acc = static_cast<float*>(scratch);
    float* most = acc + m * heads * parts * head_dim;
    a.part = SplitOut{acc, most, most + m * heads * parts, parts};
  }
  const hipError_t e = with_kind(kind, [&](auto tag) {
    if constexpr (decltype(tag)::value == KvKind::F32) return hipErrorInvalidValue;
    else return launch_tiles<decltype(tag)::value>(a, stream);
  });
  if (e != hipSuccess || parts == 1) return e;
  return launch_attention_combine(a.part.pacc, a.part.pmax, a.part.psum, out + row_base * heads * head_dim, m, heads, head_dim, parts, stream);
}

// The split-N form: kv_kind as launch_attention_as (0 fp32, 1 fp16, 2.. quantized with scales).
hipError_t launch_attention_split(const float* q, const void* k, const void* v, const float* k_scale, const float* v_scale,
                                  float* pacc, float* pmax, float* psum, uint64_t m, uint64_t n, uint64_t heads,
                                  uint64_t kv_heads, uint64_t head_dim, uint64_t q_base, uint64_t window, uint32_t kv_kind,
                                  bool causal, uint64_t split, hipStream_t stream) {
  AttentionArgs a = args_of(q, k, v, k_scale, v_scale, nullptr, n, heads, kv_heads, head_dim, q_base, 0, window, causal, m);
  a.part = SplitOut{pacc, pmax, psum, split};
  return launch_attention_as(kv_kind, a, m, stream);
}

hipError_t launch_attention_combine(const float* pacc, const float* pmax, const float* psum, float* out, uint64_t m,
                                    uint64_t heads, uint64_t head_dim, uint64_t split, hipStream_t stream) {
  auto go = [&](auto waves) {
    constexpr int W = decltype(waves)::value;
    auto with = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(m * heads)), dim3(W * 64), 0, stream, pacc, pmax, psum, out,
                         static_cast<uint32_t>(head_dim), static_cast<uint32_t>(split));
    };
    head_dim <= 64 ? with(attention_combine_kernel<1, W>) : head_dim <= 128 ? with(attention_combine_kernel<2, W>) : with(attention_combine_kernel<4, W>);
  };
  switch (combine_waves(m * heads, head_dim, split)) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    default: go(std::integral_constant<int, 16>{}); break;
  }
  return hipGetLastError();
}

}  // namespace qmm
