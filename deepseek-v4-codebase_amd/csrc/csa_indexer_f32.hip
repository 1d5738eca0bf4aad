// CSA indexer scores over fp32 keys (the drop-in csa_indexer_topk, aether_kernels/sparse_attention.py:
// 45-67, aether_kernels/csrc/csa_indexer_cuda.cu:21-110) on the fp32 matrix instruction; the top-k is
// the select of idx_mfma_device.h, over the same order keys and 16-key slot maxima.
//
// Bound by HBM (4 IC bytes per key): the products of 16 keys x 64 dims take 512 cycles of a SIMD, a
// quarter of the time their 4 KB take at the chip's rate.  A wave scores groups of 64 keys as four
// blocks of 16 (v_mfma_f32_16x16x4_f32, A = the row's queries, rows = heads; B = keys):
//   lane (g = l / 16, c = l % 16) loads dims 16 j + 4 g .. + 3 of key c with one 16-byte load per j
//   (four lanes read 64 consecutive bytes of a key), element e of which is k = g of product
//   4 j + e; the queries are loaded in the same order, so no data moves between lanes.  Each lane
//   gets the dots of heads 4 g + v (v < 4) with key c: weights, relu, and a sum over the lane groups
//   that leaves lane l the key of block l / 16 (row_sums_scatter).
// A block's registers are requested again for the next group as soon as they are consumed, through a
// buffer resource that ends at the wave's last key (no branch, exact wait counts).
// Measured with 4 heads x 64 dims: 8 x 16384 keys 8.2 us (33.5 MB, 4.1 TB/s, read while the caches
// hold part of them) and 7.6 us of select, 498 + 23 us with one lane per key and 4096 keys per
// workgroup; 16 x 65536 keys 42 us (268 MB, 6.4 TB/s), 560 + 134 us before.
#include "idx_mfma_device.h"

namespace aekv {
namespace idx {

typedef __attribute__((ext_vector_type(4))) float f32x4_t;

template <int IC>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void idx_f32_score_kernel(MfmaIdxArgs a) {
  touch_kernargs<sizeof(a)>();
  constexpr int NJ = IC / 16;
  constexpr int kGroupKeys = 64;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int row = blockIdx.y;
  const int64_t S = a.S;
  const int64_t wave_base = (static_cast<int64_t>(blockIdx.x) * 4 + wv) * a.gpw * kGroupKeys;
  const int64_t wkeys = max<int64_t>(0, min<int64_t>(wave_base + static_cast<int64_t>(a.gpw) * kGroupKeys, S) - wave_base);
  const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<uint8_t*>(a.codes + (row * S + (wkeys > 0 ? wave_base : 0)) * (IC * 4)), 0,
      static_cast<int>(wkeys * (IC * 4)), 0x00020000);
  f32x4_t kr[4][NJ];  // one group: block, 16-dim step
  auto fetch = [&](const int gi, const int tq) {  // past the wave's keys: zeros, no access
    const uint32_t off = static_cast<uint32_t>(gi * kGroupKeys + 16 * tq + c) * (IC * 4) + 16 * g;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
      kr[tq][j] = __builtin_bit_cast(f32x4_t, static_cast<u32x4_t>(__builtin_amdgcn_raw_buffer_load_b128(krs, off + 64 * j, 0, 0)));
  };
  // one memory round: the row's count, query and head weight, then the first group's keys
  int64_t nv = S;
  if (a.valid) {
    const int32_t v = a.valid[row];
    nv = v <= 0 ? 0 : (v < S ? v : S);
  }
  f32x4_t qf[NJ];  // row c of A: head c
  {
    const float* qp = a.q + (static_cast<int64_t>(row) * a.IH + (c < a.IH ? c : 0)) * IC + 4 * g;
#pragma unroll
    for (int j = 0; j < NJ; ++j) qf[j] = *reinterpret_cast<const f32x4_t*>(qp + 16 * j);
  }
  const float wr = a.w[static_cast<int64_t>(row) * a.IH + (c < a.IH ? c : 0)];
#pragma unroll
  for (int tq = 0; tq < 4; ++tq) fetch(0, tq);
  __builtin_amdgcn_sched_barrier(0);
  // the weight of head c, then of the lane's output heads 4 g + v; heads past IH: dot and weight 0
  const float wc = a.mode == AEKV_IDX_SOFTPLUS ? softplus_f32(wr) : (a.mode == AEKV_IDX_RELU_W ? fmaxf(wr, 0.0f) : wr);
  float wa[4];
  bool real[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    real[v] = 4 * g + v < a.IH;
    const float w = __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute((4 * g + v) * 4, __builtin_bit_cast(int, wc)));
    wa[v] = real[v] ? w : 0.0f;
  }
  const float floor = a.mode == AEKV_IDX_RELU_W ? -__builtin_inff() : 0.0f;  // relu on the dots, or none
  uint8_t* const krow = reinterpret_cast<uint8_t*>(a.keys + static_cast<int64_t>(row) * a.ks);
  uint8_t* const mrow = reinterpret_cast<uint8_t*>(a.smax + static_cast<int64_t>(row) * a.ms);
  const int nvi = static_cast<int>(nv);
#pragma unroll 1
  for (int gi = 0; gi < a.gpw; ++gi) {
    const int64_t kb64 = wave_base + static_cast<int64_t>(gi) * kGroupKeys;
    if (kb64 >= nv) break;  // wave-uniform
    float t[4];
#pragma unroll
    for (int tq = 0; tq < 4; ++tq) {
      f32x4_t acc[2] = {f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[j][e], kr[tq][j][e], acc[e & 1], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      fetch(gi + 1, tq);
      __builtin_amdgcn_sched_barrier(0);
      acc[0] += acc[1];
      float s = 0.0f;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const float dot = real[v] ? acc[0][v] : 0.0f;
        s = fmaf(wa[v], a.mode == AEKV_IDX_RELU_W ? dot : fmaxf(dot, floor), s);
      }
      t[tq] = s;
    }
    const float score = row_sums_scatter(t) + 0.0f;  // (+ 0: one order key for both zeros)
    const int jo = static_cast<int>(kb64) + lane;
    const bool ok = jo < nvi;
    const uint32_t key = ok ? order_key(score) : 0u;
    if (ok) *reinterpret_cast<uint32_t*>(krow + static_cast<uint32_t>(jo) * 4u) = key;
    // the 16-key slot's maximum in its last lane (a prefix maximum along the row of 16 lanes)
    uint32_t mx = key;
    mx = max(mx, dpp_or_zero<0x111>(mx));
    mx = max(mx, dpp_or_zero<0x112>(mx));
    mx = max(mx, dpp_or_zero<0x114>(mx));
    mx = max(mx, dpp_or_zero<0x118>(mx));
    if ((lane & 15) == 15 && jo - 15 < nvi) *reinterpret_cast<uint32_t*>(mrow + static_cast<uint32_t>(jo >> 4) * 4u) = mx;
  }
}

}  // namespace idx

using namespace idx;

int launch_f32_indexer(const float* q, const float* w, const float* keys, const int32_t* valid, int64_t B, int64_t S,
                       int IH, int IC, int k, int mode, void* ws, int64_t* out_idx, float* out_score, hipStream_t st,
                       const char* who) {
  MfmaIdxArgs a{};
  a.q = q;
  a.w = w;
  a.codes = reinterpret_cast<const uint8_t*>(keys);
  a.valid = valid;
  a.T = 1;
  a.IH = IH;
  a.k = k;
  a.mode = mode;
  bind_workspace(a, B, S, ws);
  // one group of 64 keys per wave until the launch has 2048 workgroups, then more (at most 16)
  const int64_t groups = ceil_div(S, int64_t(64));
  a.gpw = static_cast<int>(std::min<int64_t>(16, std::max<int64_t>(1, B * groups / (4 * kScoreTargetWG))));
  const dim3 grid(static_cast<uint32_t>(ceil_div(groups, int64_t(4) * a.gpw)), static_cast<uint32_t>(B));
  auto fn = IC == 64 ? idx_f32_score_kernel<64> : idx_f32_score_kernel<128>;
  hipLaunchKernelGGL(fn, grid, dim3(kThreads), 0, st, a);
  if (int rc = check_launch(who)) return rc;
  return launch_select(a, B, out_idx, out_score, st, who);
}

}  // namespace aekv
