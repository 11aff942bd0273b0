// The non-matmul pieces of a transformer block that sit between the projections, as plain correct
// kernels so that a trunk can run on this backend end to end: rotary embeddings, the quantizers of a
// key/value cache, the query/gate split of gated attention (attention itself: attention.hip).  Contracts:
// include/tessera/backend.hpp:162-179,378-390; CPU statements src/core/numerics/attention.cpp.
// None of them is tuned: they move kilobytes where the projections move megabytes.

#include "qmm_device.hpp"
#include "qmm_kernels.hpp"
#include "launch_rules.hpp"

namespace qmm {
namespace {

// (x[j], x[j + pairs]) rotated by pos * theta^(-2j / rope_dim), one thread for pair j of HEADS heads of a row.
// The angle, its cosine and sine are formed in double and rounded to fp32 once, as RopeRef does
// (src/core/numerics/attention.cpp:11-44); `pos3` non-null selects the multimodal form, where pair
// j takes the temporal, height or width position of its row (MropeRef, attention.cpp:227-264).
// That arithmetic is the kernel's time (512 rows of 24 heads of 256: 23 us at a thread a pair, 7.5 at eight heads), so
// many rows share it among heads; with few there is one head a thread, and the elements are under way meanwhile.
template <int HEADS>
__global__ __launch_bounds__(256) void rope_kernel(float* __restrict__ data, const uint64_t* __restrict__ pos3, uint64_t rows,
                                                   uint64_t heads, uint64_t head_dim, uint64_t rope_dim, uint64_t pos_base,
                                                   float theta, uint64_t sec_t, uint64_t sec_h) {
  const uint64_t pairs = rope_dim / 2, groups = (heads + HEADS - 1) / HEADS, total = rows * groups * pairs;
  const uint64_t t = static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x;
  if (t >= total) return;
  uint64_t row, rem, group, j;
  if (total <= 0xFFFFFFFFull) {        // uniform: 32-bit divisions where they do
    const uint32_t t32 = static_cast<uint32_t>(t), per_row = static_cast<uint32_t>(groups * pairs), p32 = static_cast<uint32_t>(pairs);
    row = t32 / per_row, rem = t32 % per_row;
    group = static_cast<uint32_t>(rem) / p32, j = static_cast<uint32_t>(rem) % p32;
  } else {
    row = t / (groups * pairs), rem = t % (groups * pairs), group = rem / pairs, j = rem % pairs;
  }
  float* base = data + (row * heads + group * HEADS) * head_dim;
  const uint64_t left = heads - group * HEADS;
  const uint32_t here = left < HEADS ? static_cast<uint32_t>(left) : HEADS;
  float x1[HEADS], x2[HEADS];
#pragma unroll
  for (uint32_t h = 0; h < HEADS; ++h) {
    const float* x = base + (h < here ? h : 0u) * head_dim;
    x1[h] = x[j], x2[h] = x[j + pairs];
  }
  uint64_t p = pos_base + row;
  if (pos3 != nullptr) p = pos3[row * 3 + (j < sec_t ? 0 : (j < sec_t + sec_h ? 1 : 2))];
  const double angle = static_cast<double>(p) * pow(static_cast<double>(theta), -2.0 * static_cast<double>(j) / static_cast<double>(rope_dim));
  const float c = static_cast<float>(cos(angle)), s = static_cast<float>(sin(angle));
#pragma unroll
  for (uint32_t h = 0; h < HEADS; ++h) {
    if (h >= here) break;
    float* x = base + h * head_dim;
    x[j] = fmaf(x1[h], c, -(x2[h] * s));         // written out: the same bits from either instance
    x[j + pairs] = fmaf(x2[h], c, x1[h] * s);
  }
}

__global__ __launch_bounds__(256) void qgate_split_kernel(const float* __restrict__ fused, float* __restrict__ q,
                                                          float* __restrict__ gate, uint64_t head_dim, uint64_t total) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x;
  if (i >= total) return;
  const uint64_t rh = i / head_dim, e = i % head_dim;
  q[i] = fused[rh * 2 * head_dim + e];
  gate[i] = fused[rh * 2 * head_dim + head_dim + e];
}

// Per-row symmetric quantizer of the quantized key/value caches (QuantizeQ8Ref / QuantizeQ4Ref,
// src/core/numerics/quant.cpp:123-178): scale = amax / QMAX (1 for an all-zero row), code =
// x / scale rounded half away from zero and clamped to +-QMAX; int8 codes a byte each, 4-bit codes
// two a byte, low nibble first.  One workgroup per row.
template <int BITS>
__global__ __launch_bounds__(256) void quantize_kv_kernel(const float* __restrict__ in, uint8_t* __restrict__ out,
                                                          float* __restrict__ scale, uint64_t cols) {
  constexpr float kMax = BITS == 8 ? 127.0f : 7.0f;
  __shared__ float red[4];
  const uint32_t t = threadIdx.x;
  const float* row = in + static_cast<size_t>(blockIdx.x) * cols;
  float amax = 0.0f;
  for (uint64_t c = t; c < cols; c += 256u) amax = fmaxf(amax, fabsf(row[c]));
  amax = wave_max(amax);
  if ((t & 63u) == 0) red[t >> 6] = amax;
  __syncthreads();
  amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  const float s = amax > 0.0f ? amax / kMax : 1.0f;
  if (t == 0) scale[blockIdx.x] = s;
  auto code = [&](float x) {
    const float r = roundf(x / s);                       // half away from zero, as lround
    return static_cast<int>(fminf(fmaxf(r, -kMax), kMax));
  };
  if constexpr (BITS == 8) {
    uint8_t* dst = out + static_cast<size_t>(blockIdx.x) * cols;
    for (uint64_t c = t; c < cols; c += 256u) dst[c] = static_cast<uint8_t>(static_cast<int8_t>(code(row[c])));
  } else {
    uint8_t* dst = out + static_cast<size_t>(blockIdx.x) * (cols / 2);
    for (uint64_t c = t; c < cols / 2; c += 256u) {
      dst[c] = static_cast<uint8_t>((code(row[2 * c]) & 0xF) | ((code(row[2 * c + 1]) & 0xF) << 4));
    }
  }
}

// fp32 -> binary16 with the significand cut toward zero, magnitudes from 2^16 up (and NaN) to
// infinity, below 2^-24 to zero: the conversion of the "cast_f32_f16" built-in
// (src/backends/rocm/rocm_kernels.hpp:26-45), not the hardware's round-to-nearest.
__device__ __forceinline__ uint32_t float_to_fp16_cut(float value) {
  const uint32_t bits = bit_cast<uint32_t>(value);
  const uint32_t sign = (bits >> 16) & 0x8000u;
  const int exponent = static_cast<int>((bits >> 23) & 0xFFu) - 127;
  const uint32_t mantissa = bits & 0x7FFFFFu;
  if (exponent > 15) return sign | 0x7C00u;
  if (exponent < -24) return sign;
  if (exponent < -14) return sign | ((mantissa | 0x800000u) >> static_cast<uint32_t>(-exponent - 1));
  return sign | (static_cast<uint32_t>(exponent + 15) << 10) | (mantissa >> 13);
}

__global__ __launch_bounds__(256) void cast_f32_f16_kernel(const float* __restrict__ in, uint32_t* __restrict__ out, uint64_t pairs) {
  const uint64_t i = static_cast<uint64_t>(blockIdx.x) * 256u + threadIdx.x;
  if (i >= pairs) return;
  const float2 v = reinterpret_cast<const float2*>(in)[i];
  out[i] = float_to_fp16_cut(v.x) | (float_to_fp16_cut(v.y) << 16);
}

dim3 blocks_for(uint64_t count) { return dim3(static_cast<uint32_t>((count + 255) / 256)); }

}  // namespace

hipError_t launch_rope(float* data, const uint64_t* pos3, uint64_t rows, uint64_t heads, uint64_t head_dim, uint64_t rope_dim,
                       uint64_t pos_base, float theta, uint64_t sec_t, uint64_t sec_h, hipStream_t stream) {
  const uint64_t pairs = rope_dim / 2;
  auto go = [&](auto kernel, uint64_t per_thread) {
    hipLaunchKernelGGL(kernel, blocks_for(rows * ((heads + per_thread - 1) / per_thread) * pairs), dim3(256), 0, stream, data, pos3,
                       rows, heads, head_dim, rope_dim, pos_base, theta, sec_t, sec_h);
  };
  rope_heads_a_thread(rows, heads, pairs) == 8u ? go(rope_kernel<8>, 8) : go(rope_kernel<1>, 1);
  return hipGetLastError();
}

hipError_t launch_quantize_kv(const float* in, uint8_t* out, float* scale, uint64_t rows, uint64_t cols, uint32_t bits,
                              hipStream_t stream) {
  if (bits == 8) {
    hipLaunchKernelGGL(quantize_kv_kernel<8>, dim3(static_cast<uint32_t>(rows)), dim3(256), 0, stream, in, out, scale, cols);
  } else {
    hipLaunchKernelGGL(quantize_kv_kernel<4>, dim3(static_cast<uint32_t>(rows)), dim3(256), 0, stream, in, out, scale, cols);
  }
  return hipGetLastError();
}

hipError_t launch_cast_f32_f16(const float* in, void* out, uint64_t n, hipStream_t stream) {
  hipLaunchKernelGGL(cast_f32_f16_kernel, blocks_for(n / 2), dim3(256), 0, stream, in, static_cast<uint32_t*>(out), n / 2);
  return hipGetLastError();
}

hipError_t launch_qgate_split(const float* fused, float* q, float* gate, uint64_t heads, uint64_t head_dim, uint64_t rows,
                              hipStream_t stream) {
  const uint64_t total = rows * heads * head_dim;
  hipLaunchKernelGGL(qgate_split_kernel, blocks_for(total), dim3(256), 0, stream, fused, q, gate, head_dim, total);
  return hipGetLastError();
}

}  // namespace qmm
