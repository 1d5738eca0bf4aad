// Merge of the source pieces of split sink-attention rows, shared by the drop-in attention kernels.
#pragma once

#include "aekv_common.h"

namespace aekv {
namespace sinkc {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kNegInf = -__builtin_inff();
// One piece of one (target, head): max, sum, 2 pad, O[D].
template <int D>
constexpr int kPartStride = D + 4;

// Value i of an array of element type DT, as fp32.
template <int DT>
__device__ __forceinline__ float load_elem(const void* p, int64_t i) {
  if constexpr (DT == AEKV_F32) return static_cast<const float*>(p)[i];
  else if constexpr (DT == AEKV_BF16) return bf16_to_f32(static_cast<const uint16_t*>(p)[i]);
  else return f16_to_f32(static_cast<const uint16_t*>(p)[i]);
}

// Four consecutive values from element i, rounded to DT (one 8- or 16-byte store).
template <int DT>
__device__ __forceinline__ void store4(void* p, int64_t i, float x, float y, float z, float w) {
  if constexpr (DT == AEKV_F32)
    *reinterpret_cast<float4*>(static_cast<float*>(p) + i) = make_float4(x, y, z, w);
  else if constexpr (DT == AEKV_BF16)
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p) + i) = make_uint2(pack_bf16x2(x, y), pack_bf16x2(z, w));
  else
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(p) + i) =
        make_uint2(f32_to_f16_bits(x) | (f32_to_f16_bits(y) << 16), f32_to_f16_bits(z) | (f32_to_f16_bits(w) << 16));
}

// Merges the source pieces of each (target, head) row: M = max(sink, piece maxima),
// L = 2^(sink - M) + sum_p 2^(m_p - M) l_p, out = sum_p 2^(m_p - M) O_p / L (log2 units), as an
// online merge over chunks of 8 pieces whose loads are all issued together.  D / 4 threads per
// row, 4 dims each, NT / (D / 4) rows per workgroup (NT = 256, or 64 when that would leave CUs
// without a workgroup, so that a call of few rows spreads its loads over as many CUs).
template <int DT, int D, int NT>
__global__ __launch_bounds__(NT) void sink_attn_combine_kernel(const float* __restrict__ part, int n_split,
                                                               const void* __restrict__ sink, int sink_scalar,
                                                               int H, int rows, void* __restrict__ out) {
  constexpr int kChunk = 8, kPer = D / 4, kStride = kPartStride<D>;
  const int row = static_cast<int>(blockIdx.x) * (NT / kPer) + static_cast<int>(threadIdx.x) / kPer;
  if (row >= rows) return;
  const int j = threadIdx.x % kPer;
  const float* p = part + static_cast<int64_t>(row) * n_split * kStride;
  float m[kChunk], l[kChunk];
  f32x4_t o[kChunk];
  // A chunk's loads (and the sink's, with the first) all precede the empty asm that takes their
  // values, so every load is issued before the first wait (the compiler would otherwise wait for
  // the sink first, and move loads into the branches that use them, each with its own wait).  A
  // piece past n_split reads piece 0 and is replaced by the empty state.
  auto load_chunk = [&](const int s0, float* sk) {
    float2 ml[kChunk];
#pragma unroll
    for (int i = 0; i < kChunk; ++i) {
      const float* ps = p + (s0 + i < n_split ? s0 + i : 0) * kStride;
      ml[i] = *reinterpret_cast<const float2*>(ps);
      o[i] = *reinterpret_cast<const f32x4_t*>(ps + 4 + 4 * j);
    }
    if (sk) *sk = load_elem<DT>(sink, sink_scalar ? 0 : row % H);
#pragma unroll
    for (int i = 0; i < kChunk; ++i) asm volatile("" : "+v"(ml[i].x), "+v"(ml[i].y), "+v"(o[i]));
    if (sk) asm volatile("" : "+v"(*sk));
#pragma unroll
    for (int i = 0; i < kChunk; ++i) {
      const bool in = s0 + i < n_split;
      m[i] = in ? ml[i].x : kNegInf;
      l[i] = in ? ml[i].y : 0.0f;
      o[i] = in ? o[i] : f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
  float skv;
  load_chunk(0, &skv);
  const float sk = skv * kLog2e;
  float M = sk, den = sk == kNegInf ? 0.0f : 1.0f;
  f32x4_t acc = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  for (int s0 = 0; s0 < n_split; s0 += kChunk) {
    if (s0 > 0) load_chunk(s0, nullptr);
    float cm = M;
#pragma unroll
    for (int i = 0; i < kChunk; ++i) cm = fmaxf(cm, m[i]);
    // (nothing yet, no sink and no source: the sums stay zero, or NaN where a piece's are)
    const float r = M == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(M - cm);
    den *= r;
    acc *= r;
    M = cm;
#pragma unroll
    for (int i = 0; i < kChunk; ++i) {
      const float f = m[i] == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(m[i] - M);
      den = fmaf(f, l[i], den);
      acc = f32x4_t{fmaf(f, o[i][0], acc[0]), fmaf(f, o[i][1], acc[1]), fmaf(f, o[i][2], acc[2]), fmaf(f, o[i][3], acc[3])};
    }
  }
  const float r = den > 0.0f ? 1.0f / den : 0.0f;
  store4<DT>(out, static_cast<int64_t>(row) * D + 4 * j, acc[0] * r, acc[1] * r, acc[2] * r, acc[3] * r);
}

// Enqueues the combine of `rows` (target, head) rows of n_split pieces each.
template <int DT, int D>
void launch_combine(const float* part, int n_split, const void* sink, int sink_scalar, int H, int64_t rows, void* out,
                    hipStream_t st) {
  constexpr int kPer = D / 4;
  const bool wide = ceil_div(rows, static_cast<int64_t>(256 / kPer)) >= 256;
  const int nt = wide ? 256 : 64;
  const dim3 grid(static_cast<uint32_t>(ceil_div(rows, static_cast<int64_t>(nt / kPer))));
  auto fn = wide ? sink_attn_combine_kernel<DT, D, 256> : sink_attn_combine_kernel<DT, D, 64>;
  hipLaunchKernelGGL(fn, grid, dim3(nt), 0, st, part, n_split, sink, sink_scalar, H, static_cast<int>(rows), out);
}

}  // namespace sinkc
}  // namespace aekv
