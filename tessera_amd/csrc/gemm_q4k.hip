// Q4_K prefill GEMM on MFMA: C (m x n fp32) = A (m x k) . deq(W)^T, W = n rows of k/256
// Q4_K super-blocks (src/core/numerics/quant.hpp:11-15; reference kernel
// src/backends/rocm/rocm_kernels_wmma.cpp:30-80,334-431, which stages A and the decoded
// weights in LDS as fp16 and accumulates in fp32).
//
// Two launches.  (1) The activations are converted once to fp16 in a workspace, each row divided
// by a power-of-two scale that the epilogue multiplies back, so the fp16 range is no limit (the
// reference converts them again in every workgroup; done once, the GEMM reads 2 bytes per
// activation instead of 4 and the conversion costs one pass over A).  (2) The GEMM proper:
// v_mfma_f32_32x32x16_f16, fp32 accumulate.
//
// Weights never exist dequantized in memory: the raw 144-byte super-blocks travel
// HBM -> LDS by direct loads, and each wavefront decodes the eight weights a lane owes the
// B operand of one MFMA straight from those bytes into registers.  The decode is the reference's:
// the fp32 value fma(q, d*sc, -(dmin*mn)) -- d*sc, dmin*mn and q*(d*sc) are exact in fp32, so this
// is DequantizeQ4K's value bit for bit -- rounded ONCE to fp16 (round to nearest even), which is
// what the reference's tensor-core tile stages (rocm_kernels_wmma.cpp:73-77).  A masked nibble
// pair masked in place is a pair of fp16 subnormals (q * 2^-24) that the mixed-precision
// multiply-add consumes directly, so two weights cost one mask and two multiply-adds that also
// round to fp16.  The nibble pairs come out of a dword in the order
// (k0,k2),(k1,k3); instead of un-shuffling them, the fp16 copy of A is written with the same
// order inside every group of 8, which a dot product cannot see.
//
// A wavefront owns WM rows x WN columns of the workgroup's tile.  Small tiles (a short stack of
// rows) use WN = 32 and all rows, so no two wavefronts decode the same weight; the 256 x 256
// prefill tile uses 128 x 64, where each activation fragment read from LDS feeds two MFMAs.
//
// K advances one 32-wide sub-block per step: activation slices (BM x 64 bytes) run through
// a four-stage XOR-swizzled LDS ring, raw weight super-blocks through a two-stage ring that
// is refilled once per eight steps; waits are counted by hand as in gemm_mxfp4.hip.

#include "q4k_tile.hpp"
#include "qmm_kernels.hpp"
#include "launch_rules.hpp"

namespace qmm {
namespace {

// One workgroup per destination row: fp32 row -> fp16 (round to nearest even) divided by the
// row's power-of-two scale, which goes to scale[row] and is multiplied back in the GEMM's
// epilogue.  With `pos` the rows are gathered: destination row pos[p] takes source row p / top_k.
// NV > 0: the row is held in registers between its maximum and its conversion (cols <= 2048 NV) and read once: 2048 rows
// of 17408 63 -> 46 us; 0: read twice.
template <int NV>
__device__ __forceinline__ void row_to_f16(const float* __restrict__ src, _Float16* __restrict__ dst, float* __restrict__ scale,
                                           uint32_t cols, uint32_t drow, uint32_t srow) {
  __shared__ float red[4];
  const uint32_t groups = cols / 8u;
  const float4* in = reinterpret_cast<const float4*>(src + static_cast<size_t>(srow) * cols);
  float amax = 0.0f;
  auto scan = [&](const float4& v) {
    amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fmaxf(fabsf(v.z), fabsf(v.w)), amax));
  };
  float4 held[NV > 0 ? 2 * NV : 1];
  if constexpr (NV > 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const uint32_t g = threadIdx.x + j * 256u;
      held[2 * j] = g < groups ? in[2 * g] : make_float4(0.f, 0.f, 0.f, 0.f);
      held[2 * j + 1] = g < groups ? in[2 * g + 1] : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int j = 0; j < 2 * NV; ++j) scan(held[j]);
  } else {
    for (uint32_t g = threadIdx.x; g < cols / 4u; g += 256u) scan(in[g]);
  }
  const float s = row_scale_for(block_amax(amax, red)), inv = 1.0f / s;
  half8_t* out = reinterpret_cast<half8_t*>(dst + static_cast<size_t>(drow) * cols);
  if constexpr (NV > 0) {
#pragma unroll
    for (int j = 0; j < NV; ++j) {
      const uint32_t g = threadIdx.x + j * 256u;
      if (g < groups) out[g] = to_f16_group(held[2 * j], held[2 * j + 1], inv);
    }
  } else {
    for (uint32_t g = threadIdx.x; g < groups; g += 256u) out[g] = to_f16_group(in[2 * g], in[2 * g + 1], inv);
  }
  if (threadIdx.x == 0) scale[drow] = s;
}
template <int NV>
__global__ __launch_bounds__(256) void rows_to_f16_kernel(const float* __restrict__ src, _Float16* __restrict__ dst,
                                                          float* __restrict__ scale, uint32_t cols,
                                                          const uint32_t* __restrict__ pos, uint32_t top_k) {
  const uint32_t p = blockIdx.x;
  row_to_f16<NV>(src, dst, scale, cols, pos != nullptr ? pos[p] : p, pos != nullptr ? p / top_k : p);
}
// How much of a row of `cols` a thread holds.
template <class F>
void with_row_registers(uint32_t cols, F&& f) {
  if (cols <= 2048u) f(std::integral_constant<int, 1>{});
  else if (cols <= 6144u) f(std::integral_constant<int, 3>{});
  else if (cols <= 18432u) f(std::integral_constant<int, 9>{});
  else f(std::integral_constant<int, 0>{});
}


template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void q4k_gemm_kernel(
    const _Float16* __restrict__ a16, const float* __restrict__ a_scale, const uint8_t* __restrict__ w,
    float* __restrict__ c, uint32_t m, uint32_t n, uint32_t k, uint32_t n_begin, uint32_t n_end) {
  const uint32_t tiles_n = (n_end - n_begin + BN - 1) / BN;
  const TileAt at = xcd_tile(blockIdx.x, (m + BM - 1) / BM, tiles_n);
  q4k_gemm_tile<BM, BN, WM, WN>(a16, a_scale, w, c, m, n, k, at.m * BM, n_begin + at.n * BN, n_end);
}

template <int BM, int BN, int WM = BM, int WN = 32>
void launch_range(const _Float16* a16, const float* a_scale, const uint8_t* w, float* c, uint32_t m, uint32_t n,
                  uint32_t k, uint32_t n_begin, uint32_t n_end, hipStream_t stream) {
  const uint32_t tiles = ((m + BM - 1) / BM) * ((n_end - n_begin + BN - 1) / BN);
  hipLaunchKernelGGL((q4k_gemm_kernel<BM, BN, WM, WN>), dim3(tiles), dim3(tile_waves<BM, BN, WM, WN>() * 64), 0, stream,
                     a16, a_scale, w, c, m, n, k, n_begin, n_end);
}

// silu(A Wg^T) * (A Wu^T) on columns n_begin .. n_end, BN / 2 of them a tile.
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void q4k_gate_up_kernel(
    const _Float16* __restrict__ a16, const float* __restrict__ a_scale, const uint8_t* __restrict__ gate, const uint8_t* __restrict__ up,
    float* __restrict__ c, uint32_t m, uint32_t n, uint32_t k, uint32_t n_begin, uint32_t n_end) {
  const uint32_t tiles_n = (n_end - n_begin + BN / 2 - 1) / (BN / 2);
  const TileAt at = xcd_tile(blockIdx.x, (m + BM - 1) / BM, tiles_n);
  q4k_gemm_tile<BM, BN, WM, WN, true>(a16, a_scale, gate, c, m, n, k, at.m * BM, n_begin + at.n * (BN / 2), n_end, up);
}

template <int BM, int BN, int WM, int WN>
void launch_pair_range(const _Float16* a16, const float* a_scale, const uint8_t* gate, const uint8_t* up, float* c, uint32_t m,
                       uint32_t n, uint32_t k, uint32_t n_begin, uint32_t n_end, hipStream_t stream) {
  const uint32_t tiles = ((m + BM - 1) / BM) * ((n_end - n_begin + BN / 2 - 1) / (BN / 2));
  hipLaunchKernelGGL((q4k_gate_up_kernel<BM, BN, WM, WN>), dim3(tiles), dim3(tile_waves<BM, BN, WM, WN>() * 64), 0, stream,
                     a16, a_scale, gate, up, c, m, n, k, n_begin, n_end);
}

}  // namespace

void launch_rows_to_f16(const float* src, _Float16* dst, float* scale, uint32_t rows, uint32_t cols, const uint32_t* pos,
                        uint32_t top_k, hipStream_t stream) {
  with_row_registers(cols, [&](auto nv) {
    hipLaunchKernelGGL(rows_to_f16_kernel<decltype(nv)::value>, dim3(rows), dim3(256), 0, stream, src, dst, scale, cols, pos, top_k);
  });
}

bool gemm_q4k_supported(uint64_t m, uint64_t k) { return k % 256 == 0 && k <= (1u << 20) && m * k < (1ull << 31); }

// fp16 copy of A, then one scale per row padded by a tile of rows (the epilogue reads scales in fours).
size_t gemm_q4k_workspace_bytes(uint64_t m, uint64_t k) { return static_cast<size_t>(m) * k * 2 + (static_cast<size_t>(m) + 256) * 4; }

// The feed forward's front half in one product: tiles of 128 columns of either matrix (gate_up_large_tiles).  2048 rows of
// 17408 x 5120: 858 us, as two products and silu_mul 940.
hipError_t launch_q4k_gate_up(const float* a, const uint8_t* gate, const uint8_t* up, float* c, void* workspace, uint32_t m,
                              uint32_t n, uint32_t k, hipStream_t stream) {
  _Float16* a16 = static_cast<_Float16*>(workspace);
  float* a_scale = reinterpret_cast<float*>(a16 + static_cast<size_t>(m) * k);
  launch_rows_to_f16(a, a16, a_scale, m, k, nullptr, 1u, stream);
  const uint32_t main_tn = gate_up_large_tiles(m, n, static_cast<uint32_t>(num_cus()));
  const uint32_t n_split = main_tn * 128u < n ? main_tn * 128u : n;
  if (n_split > 0) launch_pair_range<256, 256, 128, 64>(a16, a_scale, gate, up, c, m, n, k, 0u, n_split, stream);
  if (n_split < n) launch_pair_range<128, 128, 64, 64>(a16, a_scale, gate, up, c, m, n, k, n_split, n, stream);
  return hipGetLastError();
}

// ---- Q5_K / Q6_K prefill: weights decoded once to fp16, then a dense fp16 MFMA GEMM ----------
// Their blocks (176 and 210 bytes, the latter only 2-byte aligned) do not suit the in-register
// decode above, and they are the minority of a K-quant file's tensors, so the weights take a
// pre-pass: every value is formed exactly in fp32 as the reference decodes it and rounded once
// to fp16 (the same operand precision as the Q4_K path), in the 0,2,1,3,4,6,5,7 order that the
// activation copy uses.  The GEMM then streams both operands as 32-K slices through four-stage
// swizzled LDS rings.
namespace {

// Eight consecutive values of a group in the stored order 0,2,1,3,4,6,5,7.
__device__ __forceinline__ void store_perm8(_Float16* dst, const float (&v)[8]) {
  half8_t h;
  h[0] = static_cast<_Float16>(v[0]), h[1] = static_cast<_Float16>(v[2]);
  h[2] = static_cast<_Float16>(v[1]), h[3] = static_cast<_Float16>(v[3]);
  h[4] = static_cast<_Float16>(v[4]), h[5] = static_cast<_Float16>(v[6]);
  h[6] = static_cast<_Float16>(v[5]), h[7] = static_cast<_Float16>(v[7]);
  *reinterpret_cast<half8_t*>(dst) = h;
}

__device__ __forceinline__ uint64_t load8_a2(const uint8_t* p) {   // eight bytes from a 2-byte aligned address
  const uint16_t* q = reinterpret_cast<const uint16_t*>(p);
  return static_cast<uint64_t>(q[0]) | (static_cast<uint64_t>(q[1]) << 16) | (static_cast<uint64_t>(q[2]) << 32) |
         (static_cast<uint64_t>(q[3]) << 48);
}

// One thread per (block, half n, eight lanes l = 8o..8o+7): 32 values, four 16-byte stores
// (src/core/numerics/quant.cpp:421-450).
__device__ __forceinline__ void q6k_to_f16(const uint8_t* __restrict__ w, _Float16* __restrict__ out, uint64_t nitems, uint64_t t) {
  if (t >= nitems) return;
  const uint64_t blk = t >> 3;
  const uint32_t n = static_cast<uint32_t>(t >> 2) & 1u, o = static_cast<uint32_t>(t) & 3u, is = o >> 1;
  const uint8_t* base = w + blk * 210u;
  const uint64_t a = load8_a2(base + n * 64 + o * 8), b = load8_a2(base + n * 64 + 32 + o * 8);
  const uint64_t h = load8_a2(base + 128 + n * 32 + o * 8);
  const float d = half_bits_to_float(*reinterpret_cast<const uint16_t*>(base + 208));
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float ds = d * static_cast<float>(static_cast<int8_t>(base[192 + n * 8 + is + 2 * j]));
    const uint64_t lo = (j & 1) ? b : a;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t nib = static_cast<uint32_t>(lo >> (8 * i + 4 * (j >> 1))) & 15u;
      const uint32_t top = static_cast<uint32_t>(h >> (8 * i + 2 * j)) & 3u;
      v[i] = ds * static_cast<float>(static_cast<int>(nib | (top << 4)) - 32);
    }
    store_perm8(out + blk * 256 + n * 128 + 32 * j + o * 8, v);
  }
}

// One thread per (block, group g, eight lanes): 16 values, two 16-byte stores
// (src/core/numerics/quant.cpp:388-419).
__device__ __forceinline__ void q5k_to_f16(const uint8_t* __restrict__ w, _Float16* __restrict__ out, uint64_t nitems, uint64_t t) {
  if (t >= nitems) return;
  const uint64_t blk = t >> 4;
  const uint32_t g = static_cast<uint32_t>(t >> 2) & 3u, o = static_cast<uint32_t>(t) & 3u;
  const uint8_t* base = w + blk * 176u;
  const uint8_t* p = base + 4;
  auto scale_min = [&](uint32_t sb, uint32_t& sc, uint32_t& mn) {
    if (sb < 4) {
      sc = p[sb] & 63u;
      mn = p[sb + 4] & 63u;
    } else {
      sc = (p[sb + 4] & 15u) | ((p[sb - 4] >> 6) << 4);
      mn = (p[sb + 4] >> 4) | ((p[sb] >> 6) << 4);
    }
  };
  uint32_t sca, mna, scb, mnb;
  scale_min(2 * g, sca, mna);
  scale_min(2 * g + 1, scb, mnb);
  const uint32_t dd = *reinterpret_cast<const uint32_t*>(base);
  const float d = half_bits_to_float(dd & 0xFFFFu), dmin = half_bits_to_float(dd >> 16);
  const float d1 = d * static_cast<float>(sca), m1 = dmin * static_cast<float>(mna);
  const float d2 = d * static_cast<float>(scb), m2 = dmin * static_cast<float>(mnb);
  const uint64_t low = *reinterpret_cast<const uint64_t*>(base + 48 + g * 32 + o * 8);
  const uint64_t high = *reinterpret_cast<const uint64_t*>(base + 16 + o * 8);
  float v0[8], v1[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t lb = static_cast<uint32_t>(low >> (8 * i)) & 0xFFu, hb = static_cast<uint32_t>(high >> (8 * i)) & 0xFFu;
    v0[i] = d1 * static_cast<float>((lb & 15u) + (((hb >> (2 * g)) & 1u) << 4)) - m1;
    v1[i] = d2 * static_cast<float>((lb >> 4) + (((hb >> (2 * g + 1)) & 1u) << 4)) - m2;
  }
  store_perm8(out + blk * 256 + g * 64 + o * 8, v0);
  store_perm8(out + blk * 256 + g * 64 + 32 + o * 8, v1);
}

// Both operands in one launch: `rows` workgroups from `row0` on convert a row of A each, the others the weights.  Two launches one
// after the other cost a start and an end more: the product as a whole Q6_K 512 x 1024 x 5120 30.0 -> 27.8 us,
// 100 x 5120 x 5120 41.1 -> 38.4, 64 x 5120 x 17408 100 -> 93, Q5_K 200 x 2048 x 3072 31.9 -> 28.3.
template <int BITS, int NV>
__global__ __launch_bounds__(256) void operands_to_f16_kernel(const float* __restrict__ a, _Float16* __restrict__ a16,
                                                              float* __restrict__ a_scale, uint32_t rows, uint32_t row0, uint32_t cols,
                                                              const uint8_t* __restrict__ w, _Float16* __restrict__ w16, uint64_t nitems) {
  const uint32_t row = blockIdx.x - row0;
  if (row < rows) {        // workgroup-uniform
    row_to_f16<NV>(a, a16, a_scale, cols, row, row);
    return;
  }
  const uint64_t t = static_cast<uint64_t>(blockIdx.x < row0 ? blockIdx.x : blockIdx.x - rows) * 256u + threadIdx.x;
  if constexpr (BITS == 6) q6k_to_f16(w, w16, nitems, t);
  else q5k_to_f16(w, w16, nitems, t);
}

// How the two go (kquant_operands in launch_rules.hpp).
template <int BITS>
void launch_operands_to_f16(const float* a, _Float16* a16, float* a_scale, uint32_t m, uint32_t n, uint32_t k, const uint8_t* w,
                            _Float16* w16, hipStream_t stream) {
  const uint64_t items = static_cast<uint64_t>(n) * (k / 256u) * (BITS == 6 ? 8 : 16);
  const uint32_t groups = static_cast<uint32_t>((items + 255) / 256);     // below 2^20, as m is below 2^23 (gemm_kquant_f16_supported)
  auto go = [&](auto kernel, uint32_t rows, uint32_t row0) {
    hipLaunchKernelGGL(kernel, dim3(rows + groups), dim3(256), 0, stream, a, a16, a_scale, rows, row0, k, w, w16, items);
  };
  const KquantOperands how = kquant_operands(m, n, k, BITS);
  if (how == KquantOperands::Apart) {
    go(operands_to_f16_kernel<BITS, 0>, 0u, 0u);
    launch_rows_to_f16(a, a16, a_scale, m, k, nullptr, 1u, stream);
  } else if (how == KquantOperands::RowsTwice) {
    go(operands_to_f16_kernel<BITS, 0>, m, 0u);
  } else {
    with_row_registers(k, [&](auto nv) { go(operands_to_f16_kernel<BITS, decltype(nv)::value>, m, how == KquantOperands::RowsLast ? groups : 0u); });
  }
}

// C tile = A16 (rows scaled by a_scale) . W16^T, both operands fp16 row-major with row length k.
//
// A wavefront owns WM rows x WN columns.  An operand read from LDS is 1 KB a wavefront against 128 bytes a clock for the
// CU, and four SIMDs start a matrix instruction of 32 clocks each: 128 x 64 takes six reads to eight instructions, 64 x 96
// five to six (256 x 32, nine to eight, was bound by them: 160 tiles of 2048 rows x 5120 columns, K = 17408, 500 us).  The
// reads of a 16-wide K step go between the matrix instructions of the one before.
//
// The sums of one tile at (m0, n0) over `slices` 32-wide slices of K from slice0 on; no direct load is in flight when it
// returns.
template <int BM, int BN, int WM, int WN>
__device__ __forceinline__ void f16w_tile_sums(TileSums<WM, WN>& acc, const _Float16* __restrict__ a16, const _Float16* __restrict__ w16,
                                               uint32_t m, uint32_t n, uint32_t k, uint32_t m0, uint32_t n0, uint32_t slice0,
                                               uint32_t slices) {
  constexpr int kWavesN = BN / WN, kWaves = (BM / WM) * kWavesN, kTI = WM / 32, kTJ = WN / 32;
  constexpr int kABlk = BM / 16 / kWaves, kWBlk = (BN / 16 + kWaves - 1) / kWaves;   // 1 KB blocks per wavefront and slice
  constexpr int kDma = kABlk + kWBlk;
  constexpr uint32_t kAStage = BM * 64, kWStage = kWBlk * kWaves * 1024, kStage = kAStage + kWStage;
  static_assert(BM % (16 * kWaves) == 0 && BN % 16 == 0 && WM % 32 == 0 && WN % 32 == 0, "tile shape");
  __shared__ __attribute__((aligned(16))) uint8_t lds[4 * kStage];

  const uint32_t t = threadIdx.x, lane = t & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const uint32_t wave_m = wave / kWavesN, wave_n = wave % kWavesN;
  const uint32_t l32 = lane & 31u, kg = lane >> 5;
  const uint32_t lds_base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
      (__attribute__((address_space(3))) uint8_t*)lds));
  const uint8_t* a_tile = reinterpret_cast<const uint8_t*>(a16) + static_cast<size_t>(m0) * k * 2 + slice0 * 64u;
  const uint8_t* w_tile = reinterpret_cast<const uint8_t*>(w16) + static_cast<size_t>(n0) * k * 2 + slice0 * 64u;

  // Block L of a slice = rows 16L..16L+15, four 16-byte chunks a row: lane p fetches row
  // 16L + p/4, chunk (p%4) ^ ((row>>2)&3).  Rows past the matrix edge are clamped (never stored), and so are
  // those of blocks past the tile, which where BN / 16 does not divide go to spare LDS.
  uint32_t a_src[kABlk], w_src[kWBlk];
#pragma unroll
  for (int i = 0; i < kABlk; ++i) {
    const uint32_t row = 16u * (wave * kABlk + i) + lane / 4u;
    a_src[i] = (m0 + row < m ? row : m - 1u - m0) * (k * 2u) + (((lane % 4u) ^ ((row >> 2) & 3u)) * 16u);
  }
#pragma unroll
  for (int i = 0; i < kWBlk; ++i) {
    const uint32_t row_any = 16u * (wave * kWBlk + i) + lane / 4u, row = row_any < BN ? row_any : BN - 1u;
    w_src[i] = (n0 + row < n ? row : n - 1u - n0) * (k * 2u) + (((lane % 4u) ^ ((row >> 2) & 3u)) * 16u);
  }
  auto issue = [&](uint32_t slice_any) {
    const uint32_t slice = __builtin_amdgcn_readfirstlane(slice_any < slices ? slice_any : slices - 1u), stage = slice_any & 3u;
#pragma unroll
    for (int i = 0; i < kABlk; ++i)
      direct_load16(a_tile + slice * 64u, a_src[i], lds_base + stage * kStage + (wave * kABlk + i) * 1024u);
#pragma unroll
    for (int i = 0; i < kWBlk; ++i)
      direct_load16(w_tile + slice * 64u, w_src[i], lds_base + stage * kStage + kAStage + (wave * kWBlk + i) * 1024u);
  };

#pragma unroll
  for (int i = 0; i < kTI; ++i)
#pragma unroll
    for (int j = 0; j < kTJ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  uint32_t a_fr[2], w_fr[2];   // fragment offsets: MFMA step tt takes chunk 2tt + kg
#pragma unroll
  for (int tt = 0; tt < 2; ++tt) {
    const uint32_t in = l32 * 64u + (((tt * 2u + kg) ^ ((l32 >> 2) & 3u)) * 16u);
    a_fr[tt] = wave_m * (WM * 64u) + in, w_fr[tt] = kAStage + wave_n * (WN * 64u) + in;
  }
  struct Frag {
    half8_t a[kTI], b[kTJ];
  };
  auto read = [&](uint32_t slice, int tt, Frag& f) {
    const uint8_t* stage = lds + (slice & 3u) * kStage;
#pragma unroll
    for (int j = 0; j < kTJ; ++j) f.b[j] = *reinterpret_cast<const half8_t*>(stage + w_fr[tt] + j * 32 * 64);
#pragma unroll
    for (int i = 0; i < kTI; ++i) f.a[i] = *reinterpret_cast<const half8_t*>(stage + a_fr[tt] + i * 32 * 64);
  };
  // The matrix instructions of `f`, the reads of `g` spread among them.
  auto multiply_reading = [&](const Frag& f, uint32_t slice, int tt, Frag& g) {
    read(slice, tt, g);
#pragma unroll
    for (int i = 0; i < kTI; ++i)
#pragma unroll
      for (int j = 0; j < kTJ; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.a[i], f.b[j], acc[i][j], 0, 0, 0);
    constexpr int kMost = kTI * kTJ > kTI + kTJ ? kTI * kTJ : kTI + kTJ;
#pragma unroll
    for (int q = 0; q < kMost; ++q) {
      if (q < kTI * kTJ) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (q < kTI + kTJ) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  };

  issue(0);
  issue(1);
  issue(2);
  issue(3);
  Frag f0, f1;
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(3 * kDma) : "memory");
  read(0, 0, f0);
  for (uint32_t slice = 0; slice < slices; ++slice) {
    multiply_reading(f0, slice, 1, f1);
    if constexpr (kWaves == 8) {       // keeps these matrix instructions on this side of the barrier
#pragma unroll
      for (int i = 0; i < kTI; ++i)
#pragma unroll
        for (int j = 0; j < kTJ; ++j) asm volatile("" : "+v"(acc[i][j]));
    }
    // slice + 1 has landed; every wavefront has read all of `slice`, whose stage takes slice + 4
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * kDma) : "memory");
    issue(slice + 4u);
    multiply_reading(f1, slice + 1u, 0, f0);    // (after the last slice: a stage that nobody needs)
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no direct load may outlive the workgroup
}

template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64) void f16w_gemm_kernel(
    const _Float16* __restrict__ a16, const float* __restrict__ a_scale, const _Float16* __restrict__ w16,
    float* __restrict__ c, uint32_t m, uint32_t n, uint32_t k, uint32_t n_begin, uint32_t n_end, bool as_decoded) {
  const uint32_t tiles_n = (n_end - n_begin + BN - 1) / BN;
  const TileAt at = as_decoded ? TileAt{blockIdx.x / tiles_n, blockIdx.x % tiles_n} : xcd_tile(blockIdx.x, (m + BM - 1) / BM, tiles_n);
  const uint32_t m0 = at.m * BM, n0 = n_begin + at.n * BN;
  TileSums<WM, WN> acc;
  f16w_tile_sums<BM, BN, WM, WN>(acc, a16, w16, m, n, k, m0, n0, 0u, k / 32u);
  q4k_tile_store<BM, BN, WM, WN>(acc, a_scale, c, m, n, m0, n0, n_end);
}

template <int BM, int BN, int WM, int WN>
void launch_f16w_range(const _Float16* a16, const float* a_scale, const _Float16* w16, float* c, uint32_t m, uint32_t n, uint32_t k,
                       uint32_t n_begin, uint32_t n_end, hipStream_t stream) {
  const uint32_t tiles = ((m + BM - 1) / BM) * ((n_end - n_begin + BN - 1) / BN);
  hipLaunchKernelGGL((f16w_gemm_kernel<BM, BN, WM, WN>), dim3(tiles), dim3((BM / WM) * (BN / WN) * 64), 0, stream, a16, a_scale,
                     w16, c, m, n, k, n_begin, n_end, f16w_tiles_as_decoded(m, n, k, static_cast<uint32_t>(num_cus()), BM == 128));
}

// ---- tiles whose steps of K workgroups share --------------------------------------------------------------------------
// A (tile, super-block) unit is 256 of K.  The tiles' units, tile after tile down the columns, are dealt out evenly:
// workgroup g takes those from unit_bound(g) on.  A tile that several share has its sums in `parts`, block g + t for
// workgroup g's piece of tile t, each in the order in which the registers lie (a float4 of a lane is four rows of a
// column), for piece_sums_kernel to add up in the workgroups' order.  512 rows of 1024 x 5120: Q4_K 44 -> 26 us (the tiles
// 37 -> 14, the sums 5), Q6_K 46 -> 28; of 6144 x 5120 Q4_K 64 -> 59.
// CUT: no room for `parts`, but the same bits.  A workgroup has a whole tile (within one of the plan's, of as many rows) and adds
// its pieces in registers, in that order.  us, tiles that are not cut / cut / with room: Q4_K 64 x 1024 x 5120 37 / 71 / 18, 1000 x
// 2040 x 5120 48 / 56 / 43, 1024 x 5120 x 5120 103 / 112 / 95, 512 x 6144 x 5120 64 / 63 / 59, Q6_K 512 x 1024 x 5120 46 / 51 / 28.
struct Q4KWeights {
  using Type = uint8_t;
  static constexpr int kCutWN = 64;
  template <int BM, int BN, int WM, int WN>
  static __device__ __forceinline__ void sums(TileSums<WM, WN>& acc, const _Float16* a16, const Type* w, uint32_t m, uint32_t n,
                                              uint32_t k, uint32_t m0, uint32_t n0, uint32_t from, uint32_t to) {
    q4k_tile_sums<BM, BN, 2 * WM, WN, false, 2>(acc, a16, w, m, n, k, m0, n0, from, to - from);
  }
};
struct F16Weights {
  using Type = _Float16;
  static constexpr int kCutWN = 32;
  template <int BM, int BN, int WM, int WN>
  static __device__ __forceinline__ void sums(TileSums<WM, WN>& acc, const _Float16* a16, const Type* w, uint32_t m, uint32_t n,
                                              uint32_t k, uint32_t m0, uint32_t n0, uint32_t from, uint32_t to) {
    f16w_tile_sums<BM, BN, WM, WN>(acc, a16, w, m, n, k, m0, n0, from * 8u, (to - from) * 8u);
  }
};

template <class W, int BM, int BN, int WM, int WN, bool CUT>
__global__ __launch_bounds__((BM / WM) * (BN / WN) * 64, CUT ? 1 : 2) void shared_tiles_kernel(
    const _Float16* __restrict__ a16, const float* __restrict__ a_scale, const typename W::Type* __restrict__ w,
    float* __restrict__ c, uint32_t m, uint32_t n, uint32_t k, float* __restrict__ parts, SharedTiles plan) {
  constexpr int kTI = WM / 32, kTJ = WN / 32;
  const uint32_t steps = k / 256u, tiles_m = (m + BM - 1) / BM;
  TileSums<WM, WN> acc;
  if constexpr (CUT) {
    const uint32_t m0 = blockIdx.x % tiles_m * BM, n0 = blockIdx.x / tiles_m * BN;
    const uint64_t first = static_cast<uint64_t>(n0 / plan.columns * tiles_m + m0 / plan.rows) * steps;
    uint32_t owner = unit_owner(first, plan, steps), from = 0;
    TileSums<WM, WN> total = {};
    while (from < steps) {
      const uint64_t cut = unit_bound(++owner, plan.groups, plan.tiles, steps) - first;
      const uint32_t to = cut < steps ? static_cast<uint32_t>(cut) : steps;
      W::template sums<BM, BN, WM, WN>(acc, a16, w, m, n, k, m0, n0, from, to);
      const bool whole = from == 0u && to == steps;
#pragma unroll
      for (int i = 0; i < kTI; ++i)
#pragma unroll
        for (int j = 0; j < kTJ; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) total[i][j][e] = whole ? acc[i][j][e] : total[i][j][e] + acc[i][j][e];
      from = to;
      if (from < steps) __syncthreads();      // every wavefront has read the last slice
    }
    q4k_tile_store<BM, BN, WM, WN>(total, a_scale, c, m, n, m0, n0, n);
  } else {
    const uint32_t lane = threadIdx.x & 63u, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Workgroups go round the eight XCDs: neighbours in the units' order, which read the same weights, stay on one.
    const uint32_t group = gridDim.x % 8u == 0u ? blockIdx.x % 8u * (gridDim.x / 8u) + blockIdx.x / 8u : blockIdx.x;
    uint64_t v = unit_bound(group, plan.groups, plan.tiles, steps);
    const uint64_t end = unit_bound(group + 1u, plan.groups, plan.tiles, steps);
    while (v < end) {
      const uint32_t tile = static_cast<uint32_t>(v / steps), from = static_cast<uint32_t>(v % steps);
      const uint32_t to = end - v < steps - from ? from + static_cast<uint32_t>(end - v) : steps;
      const uint32_t m0 = tile % tiles_m * BM, n0 = tile / tiles_m * BN;
      W::template sums<BM, BN, WM, WN>(acc, a16, w, m, n, k, m0, n0, from, to);
      if (from == 0u && to == steps) {
        q4k_tile_store<BM, BN, WM, WN>(acc, a_scale, c, m, n, m0, n0, n);
      } else {
        float4_t* block = reinterpret_cast<float4_t*>(parts + static_cast<size_t>(group + tile) * (BM * BN));
#pragma unroll
        for (int i = 0; i < kTI; ++i) {
          if (m0 + (wave / (BN / WN)) * WM + i * 32u >= m) continue;
#pragma unroll
          for (int j = 0; j < kTJ; ++j)
#pragma unroll
            for (int q = 0; q < 4; ++q)
              block[(((wave * kTI + i) * kTJ + j) * 4u + q) * 64u + lane] =
                  float4_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
        }
      }
      v += to - from;
      if (v < end) __syncthreads();           // every wavefront has read the last slice
    }
  }
}

// Adds the pieces of the tiles that several workgroups shared and scales: a workgroup a 32 x 32 matrix tile, a float4 a thread.
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(256) void piece_sums_kernel(const float* __restrict__ parts, const float* __restrict__ a_scale,
                                                         float* __restrict__ c, uint32_t m, uint32_t n, uint32_t steps,
                                                         SharedTiles plan) {
  constexpr uint32_t kTI = WM / 32, kTJ = WN / 32, kPer = BM * BN / 1024;
  const uint32_t tile = blockIdx.x / kPer, at = blockIdx.x % kPer, tiles_m = (m + BM - 1) / BM;
  const uint64_t v0 = static_cast<uint64_t>(tile) * steps, v1 = v0 + steps;
  const uint32_t first = unit_owner(v0, plan, steps), last = unit_owner(v1 - 1u, plan, steps);
  const uint32_t wave = at / (kTI * kTJ), i = at / kTJ % kTI, j = at % kTJ, lane = threadIdx.x & 63u;
  const uint32_t row0 = tile % tiles_m * BM + wave / (BN / WN) * WM + i * 32u;
  if (first == last || row0 >= m) return;
  const float4_t* block = reinterpret_cast<const float4_t*>(parts + static_cast<size_t>(first + tile) * (BM * BN)) + at * 256u + threadIdx.x;
  float4_t sum = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  for (uint32_t g = first; g <= last; ++g, block += BM * BN / 4) sum += *block;
  const uint32_t col = tile / tiles_m * BN + wave % (BN / WN) * WN + j * 32u + (lane & 31u);
  const uint32_t row = row0 + (threadIdx.x >> 6) * 8u + (lane >> 5) * 4u;
  if (col >= n) return;
#pragma unroll
  for (uint32_t e = 0; e < 4; ++e) {
    if (row + e < m) c[static_cast<size_t>(row + e) * n + col] = sum[e] * a_scale[row + e];
  }
}

template <class W>
hipError_t launch_shared(const _Float16* a16, const float* a_scale, const typename W::Type* w, float* c, float* parts, uint32_t m,
                         uint32_t n, uint32_t k, const SharedTiles& plan, hipStream_t stream) {
  if (parts == nullptr) {
    constexpr int WN = W::kCutWN;
    hipLaunchKernelGGL((shared_tiles_kernel<W, 128, 64, 64, WN, true>), dim3((m + 127u) / 128u * ((n + 63u) / 64u)),
                       dim3(2 * 64 / WN * 64), 0, stream, a16, a_scale, w, c, m, n, k, parts, plan);
    return hipGetLastError();
  }
  hipLaunchKernelGGL((shared_tiles_kernel<W, 128, 128, 64, 64, false>), dim3(plan.groups), dim3(256), 0, stream, a16, a_scale, w, c, m,
                     n, k, parts, plan);
  hipLaunchKernelGGL((piece_sums_kernel<128, 128, 64, 64>), dim3(plan.tiles * 16u), dim3(256), 0, stream, parts, a_scale, c, m, n,
                     k / 256u, plan);
  return hipGetLastError();
}

}  // namespace

// The bulk of C goes to 256 x 256 tiles, whole rounds of one tile per CU; columns left over
// when the tile count is not a multiple of the CU count are cut into 128 x 64 tiles that
// spread over every CU instead of keeping a few CUs busy for a whole extra round.
hipError_t launch_q4k_gemm(const float* a, const uint8_t* w, float* c, void* workspace, float* parts, uint32_t m,
                           uint32_t n, uint32_t k, hipStream_t stream) {
  _Float16* a16 = static_cast<_Float16*>(workspace);
  float* a_scale = reinterpret_cast<float*>(a16 + static_cast<size_t>(m) * k);
  launch_rows_to_f16(a, a16, a_scale, m, k, nullptr, 1u, stream);
  const uint32_t cus = static_cast<uint32_t>(num_cus());
  const SharedTiles plan = shared_f16_tiles(m, n, k / 256u, cus, true);
  if (plan.groups != 0u) return launch_shared<Q4KWeights>(a16, a_scale, w, c, parts, m, n, k, plan, stream);
  const uint32_t tiles_m = (m + 255u) / 256u, tiles_n = (n + 255u) / 256u;
  const uint32_t tiles = tiles_m * tiles_n;
  uint32_t main_tn = tiles_n;
  if (tiles > cus && tiles % cus != 0 && tiles % cus <= cus / 2) {
    main_tn = (tiles / cus) * cus / tiles_m;
  } else if (tiles < cus / 2) {
    main_tn = 0;
  }
  if (m <= 64) {
    // A short stack of rows is bound by the weight stream: narrow tiles (one wavefront, 32
    // columns) give every CU several workgroups' worth of super-blocks in flight.
    if (m <= 32) {
      launch_range<32, 32>(a16, a_scale, w, c, m, n, k, 0u, n, stream);
    } else {
      launch_range<64, 32>(a16, a_scale, w, c, m, n, k, 0u, n, stream);
    }
    return hipGetLastError();
  }
  const uint32_t n_split = main_tn * 256u < n ? main_tn * 256u : n;
  if (n_split > 0) launch_range<256, 256, 128, 64>(a16, a_scale, w, c, m, n, k, 0u, n_split, stream);
  if (n_split < n) launch_range<128, 64, 64, 32>(a16, a_scale, w, c, m, n, k, n_split, n, stream);
  return hipGetLastError();
}

size_t gemm_f16_parts_bytes(uint64_t m, uint64_t n, uint64_t k, bool q4k) {
  return shared_tiles_bytes(shared_f16_tiles(m, n, k / 256, static_cast<uint64_t>(num_cus()), q4k));
}

bool gemm_kquant_f16_supported(uint64_t m, uint64_t n, uint64_t k) {
  return k % 256 == 0 && k <= (1u << 20) && m * k < (1ull << 31) && n * k < (1ull << 31);
}

// fp16 copy of A, its row scales (padded by a tile of rows), then the fp16 copy of W.
size_t gemm_kquant_f16_workspace_bytes(uint64_t m, uint64_t n, uint64_t k) {
  return static_cast<size_t>(m) * k * 2 + (static_cast<size_t>(m) + 256) * 4 + static_cast<size_t>(n) * k * 2;
}

// block_bytes selects the format: 176 = Q5_K, 210 = Q6_K.
hipError_t launch_kquant_f16_gemm(const float* a, const uint8_t* w, uint32_t block_bytes, float* c, void* workspace,
                                  float* parts, uint32_t m, uint32_t n, uint32_t k, hipStream_t stream) {
  _Float16* a16 = static_cast<_Float16*>(workspace);
  float* a_scale = reinterpret_cast<float*>(a16 + static_cast<size_t>(m) * k);
  _Float16* w16 = reinterpret_cast<_Float16*>(a_scale + m + 256);
  if (block_bytes != 210 && block_bytes != 176) return hipErrorInvalidValue;
  if (block_bytes == 210) launch_operands_to_f16<6>(a, a16, a_scale, m, n, k, w, w16, stream);
  else launch_operands_to_f16<5>(a, a16, a_scale, m, n, k, w, w16, stream);
  const SharedTiles plan = shared_f16_tiles(m, n, k / 256u, static_cast<uint64_t>(num_cus()), false);
  if (plan.groups != 0u) return launch_shared<F16Weights>(a16, a_scale, w16, c, parts, m, n, k, plan, stream);
  const F16wTiles tiles = f16w_tiles(m, n, k, static_cast<uint32_t>(num_cus()));
  const uint32_t n_split = tiles.large * tiles.columns < n ? tiles.large * tiles.columns : n;
  if (n_split > 0) {
    switch (tiles.columns) {
      case 128: launch_f16w_range<256, 128, 64, 64>(a16, a_scale, w16, c, m, n, k, 0u, n_split, stream); break;
      case 192: launch_f16w_range<256, 192, 64, 96>(a16, a_scale, w16, c, m, n, k, 0u, n_split, stream); break;
      default: launch_f16w_range<256, 256, 128, 64>(a16, a_scale, w16, c, m, n, k, 0u, n_split, stream); break;
    }
  }
  if (n_split < n) launch_f16w_range<128, 64, 64, 32>(a16, a_scale, w16, c, m, n, k, n_split, n, stream);
  return hipGetLastError();
}

}  // namespace qmm
