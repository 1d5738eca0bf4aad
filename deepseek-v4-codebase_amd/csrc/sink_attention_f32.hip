// Drop-in sink attention in fp32 arithmetic on the matrix cores: fp32 inputs at head_dim 64 and 128,
// and bf16 / fp16 inputs at head_dim 64 (16-bit inputs at 128 take the 16-bit products of
// sink_attention_mfma.hip and prefill_flash.hip; every other head dim the VALU kernel).
//
// Reference: sparse_sink_attention (aether_kernels/sparse_attention.py:8-16; semantics
// aether_kernels/csrc/sparse_sink_attention_cuda.cu:47-114) and tiled_prefill_attention
// (aether_kernels/sparse_attention.py:19-42), the sink counted once (aether_2b/modeling.py:158-178).
//
// What bounds it: the fp32 matrix rate (v_mfma_f32_16x16x4_f32: 1024 multiply-adds in 32 cycles, 32 per
// cycle and SIMD) on dense calls with many rows, memory latency on the others.  A workgroup owns 16 NQ query rows that
// attend the same sources (consecutive (target, head) rows of a dense call, the heads of one target
// of a sparse one); its NW waves take every NW-th group of 16 sources straight from global memory
// into registers, in layouts that need no LDS and no lane exchange:
//   S^T = K Q^T   A: lane (g = l / 16, c = l % 16) holds dims 16 j + 4 g .. + 3 of source c (one
//                 16-byte load per j), element e of it is product 4 j + e's k = g; B: the same dims
//                 of query row c, so any order of the dims serves.  Lane (g, c) gets the scores of
//                 sources 4 g + v (v < 4) for row c.
//   O^T += V^T P^T  product v takes source 4 g + v as k = g, so B is the lane's own weight v; A: lane
//                 (g, c) holds dims 64 i + 4 c .. + 3 of that source (16 lanes read 256 consecutive
//                 bytes), element e of load i is row c of the product whose rows are dims
//                 64 i + 4 c + e: register r of lane (g, c) is dim 64 i + 16 g + 4 r + e of row c.
// The values and weights stay fp32 throughout (the products are fp32 fused multiply-adds), with an
// online softmax in base 2.  A wave computes the next group's scores before this group's softmax, and
// requests the keys after next and the next values once their registers are free, so both are in
// flight under matrix work.  (fp32 products do not overlap vector instructions on gfx950: one vector
// instruction after each product costs 6 to 10 cycles of 32, so the softmax stands in one block.)  The waves merge through
// LDS; launches with few row blocks and many sources also split the sources over workgroups
// (sink_combine.h).
//
// Measured (256 targets x 12 heads over 2176 fp32 sources, 128 dims): 46 us and a 4.5 us combine, where
// the VALU kernel took 1.1 to 1.7 ms (22x to 34x); the matrix cores are busy for 24 us of it (the loop runs 84% busy
// with two waves per SIMD, the rest is the first and last memory rounds and the waves' merge).
// 128 targets x 16 heads over 64 picked sources: 6.4 us (40.7); one target over 2176: 12 + 4 us (677).
#include <algorithm>

#include "sink_combine.h"

namespace aekv {
namespace {

using sinkc::f32x4_t;
using sinkc::kLog2e;
using sinkc::kNegInf;

constexpr int kSrc = 16;  // sources per wave step

struct SinkF32Args {
  const void* q;     // [B, T, H, D]
  const void* kv;    // [B, S, 2, D]: K then V of each source
  const void* idx;   // [B, T, K] int32 / int64 (null: dense, source j = j)
  const void* sink;  // [H] or [1]
  int sink_scalar, H, T, S, K;
  uint32_t n_blk;    // row blocks per sequence (dense) or per target (sparse)
  float scale2;      // softmax scale * log2(e)
  int n_split;       // source pieces per row block (grid y)
  int gps;           // 16-source groups per piece
  float* part;       // [B * T * H, n_split, D + 4] when n_split > 1
  void* out;         // [B, T, H, D]
};

// Four consecutive elements as loaded, and as fp32.
template <int DT>
struct Quad {
  typedef uint2 raw;
  __device__ static f32x4_t cvt(const raw& r) {
    const uint32_t w[4] = {r.x & 0xFFFFu, r.x >> 16, r.y & 0xFFFFu, r.y >> 16};
    f32x4_t f;
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = DT == AEKV_BF16 ? bf16_to_f32(w[e]) : f16_to_f32(w[e]);
    return f;
  }
  __device__ static raw zero() { return make_uint2(0u, 0u); }
};
template <>
struct Quad<AEKV_F32> {
  typedef f32x4_t raw;
  __device__ static f32x4_t cvt(const raw& r) { return r; }
  __device__ static raw zero() { return f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}; }
};

// IDX: 0 dense, 4 int32 indices, 8 int64 indices.  Two waves per SIMD (256 registers) hold the
// queries, the accumulators and one group's keys and values at NQ = 2, D = 128 without spills.
template <int DT, int D, int IDX, int NQ, int NW>
__global__ __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) void sink_attn_f32_kernel(SinkF32Args a) {
  using E = Quad<DT>;
  using raw = typename E::raw;
  constexpr int ES = DT == AEKV_F32 ? 4 : 2;
  constexpr int NK = D / 16, NV = D / 64, R = 16 * NQ;
  constexpr int kObStride = D + 4;  // merge rows: row r at bank 4 r
  constexpr int kPart = sinkc::kPartStride<D>;
  __shared__ __align__(16) float s_ob[NW * R * kObStride];
  __shared__ float s_ml[NW][R][2];
  __shared__ float s_inv[R];
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wv = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  // the block's rows: base_row .. base_row + n_rows - 1 of (b, t, h) order, attending sequence b
  const uint32_t blk = blockIdx.x / a.n_blk, sub = blockIdx.x - blk * a.n_blk;
  const int seq_rows = IDX == 0 ? a.T * a.H : a.H;  // rows that share the sources
  const int r0 = static_cast<int>(sub) * R;         // first row within them
  const int n_rows = min(R, seq_rows - r0);
  const int64_t base_row = static_cast<int64_t>(blk) * seq_rows + r0;
  const int64_t b = IDX == 0 ? blk : blk / static_cast<uint32_t>(a.T);
  const char* const kvb = static_cast<const char*>(a.kv) + b * a.S * (2 * D * ES);
  const int K = a.K;

  const int split = blockIdx.y;
  const int g_end = min((K + kSrc - 1) / kSrc, (split + 1) * a.gps);
  int G = split * a.gps + wv;

  // Source of position j of the row block's list: validity and a readable row (0 when skipped).
  // Positions past the list read its last entry and are not valid.
  const int64_t ibase = static_cast<int64_t>(blk) * K;
  auto read_idx = [&](int gr) -> int64_t {
    const int j = min(kSrc * gr + c, K - 1);
    if constexpr (IDX == 0) return j;
    else if constexpr (IDX == 4) return static_cast<const int32_t*>(a.idx)[ibase + j];
    else return static_cast<const int64_t*>(a.idx)[ibase + j];
  };
  raw kr[NK], vr[4][NV];
  auto load_k = [&](int src) {
    const char* p = kvb + static_cast<int64_t>(src) * (2 * D * ES) + 4 * g * ES;
#pragma unroll
    for (int j = 0; j < NK; ++j) kr[j] = *reinterpret_cast<const raw*>(p + 16 * j * ES);
  };
  // the values of group gr, whose sources are `src` (lane c: source c; dense positions are computed)
  auto load_v = [&](int gr, int src) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      int vs;
      if constexpr (IDX == 0) vs = min(kSrc * gr + 4 * g + v, K - 1);
      else vs = __builtin_amdgcn_ds_bpermute((4 * g + v) * 4, src);
      const char* p = kvb + (static_cast<int64_t>(vs) * 2 + 1) * (D * ES) + 4 * c * ES;
#pragma unroll
      for (int i = 0; i < NV; ++i) vr[v][i] = *reinterpret_cast<const raw*>(p + 64 * i * ES);
    }
  };

  float m_run[NQ], l_run[NQ];  // l_run: this lane's weights only (its four sources of each group)
  f32x4_t O[NQ][4 * NV];
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    m_run[n] = kNegInf;
    l_run[n] = 0.0f;
#pragma unroll
    for (int i = 0; i < 4 * NV; ++i) O[n][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  }
  if (G < g_end) {  // wave-uniform
    f32x4_t qf[NQ][NK];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const int r = 16 * n + c;
      const char* p = static_cast<const char*>(a.q) + ((base_row + (r < n_rows ? r : 0)) * D + 4 * g) * ES;
#pragma unroll
      for (int j = 0; j < NK; ++j) qf[n][j] = E::cvt(*reinterpret_cast<const raw*>(p + 16 * j * ES));
    }
    // scores of the keys in kr; one row group keeps two partial sums so that consecutive products
    // do not depend on each other
    constexpr int NS = NQ == 1 ? 2 : 1;
    auto scores = [&](f32x4_t (&st)[NQ]) {
      f32x4_t acc[NQ][NS];
#pragma unroll
      for (int n = 0; n < NQ; ++n)
#pragma unroll
        for (int s = 0; s < NS; ++s) acc[n][s] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int j = 0; j < NK; ++j) {
        const f32x4_t k4 = E::cvt(kr[j]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int n = 0; n < NQ; ++n)
            acc[n][(4 * j + e) % NS] =
                __builtin_amdgcn_mfma_f32_16x16x4f32(k4[e], qf[n][j][e], acc[n][(4 * j + e) % NS], 0, 0, 0);
      }
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        st[n] = acc[n][0];
        if constexpr (NS == 2) st[n] += acc[n][1];
      }
    };
    // a group's weights from its scores (bit i of okm: source i), and the rescale of the sums
    float p[NQ][4];
    auto softmax = [&](const f32x4_t (&st)[NQ], const uint32_t okm) {
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        float tm = kNegInf;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          p[n][v] = ((okm >> (4 * g + v)) & 1u) ? st[n][v] * a.scale2 : kNegInf;
          tm = fmaxf(tm, p[n][v]);
        }
        tm = fmaxf(tm, xor_lane<16>(tm));
        tm = fmaxf(tm, xor_lane<32>(tm));
        const float mnew = fmaxf(m_run[n], tm);
        // (first group: 2^-inf = 0; no source yet: 1)
        const float corr = mnew == m_run[n] ? 1.0f : __builtin_amdgcn_exp2f(m_run[n] - mnew);
        m_run[n] = mnew;
        l_run[n] *= corr;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          p[n][v] = p[n][v] == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(p[n][v] - mnew);
          l_run[n] += p[n][v];
        }
#pragma unroll
        for (int i = 0; i < 4 * NV; ++i) O[n][i] *= corr;
      }
    };
    auto weigh = [&](const uint32_t okm) {
      if (okm != 0xFFFFu) {  // skipped sources: a zero weight must not meet an infinity or NaN
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (!((okm >> (4 * g + v)) & 1u)) {
#pragma unroll
            for (int i = 0; i < NV; ++i) vr[v][i] = E::zero();
          }
      }
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int i = 0; i < NV; ++i) {
          const f32x4_t v4 = E::cvt(vr[v][i]);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int n = 0; n < NQ; ++n)
              O[n][4 * i + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v4[e], p[n][v], O[n][4 * i + e], 0, 0, 0);
        }
    };
    auto check = [&](int gr, int64_t si, bool& ok) {
      ok = kSrc * gr + c < K && si >= 0 && si < a.S;
      return ok ? static_cast<int>(si) : 0;
    };
    auto mask = [](bool ok) { return static_cast<uint32_t>(__builtin_amdgcn_ballot_w64(ok)) & 0xFFFFu; };

    // group G's scores, then per step: the next group's scores, this group's softmax and values
    bool ok;
    int src_v = check(G, read_idx(G), ok);
    load_k(src_v);
    int64_t si = read_idx(G + 2 * NW);
    bool ok_next;
    int src = check(G + NW, read_idx(G + NW), ok_next);
    uint32_t okm = mask(ok);
    f32x4_t st[NQ];
    scores(st);
    __builtin_amdgcn_sched_barrier(0);
    load_k(src);
    __builtin_amdgcn_sched_barrier(0);
    load_v(G, src_v);  // (keys, then values, as the loop requests them: its waits count in that order)
#pragma unroll 1
    for (; G + NW < g_end; G += NW) {
      __builtin_amdgcn_sched_barrier(0);
      f32x4_t st_next[NQ];
      scores(st_next);
      softmax(st, okm);
      // (kept here: the compiler would sink the rescale to the products below)
#pragma unroll
      for (int n = 0; n < NQ; ++n)
#pragma unroll
        for (int i = 0; i < 4 * NV; ++i) asm volatile("" : "+v"(O[n][i]));
      __builtin_amdgcn_sched_barrier(0);
      // the keys after next (positions past the end read the list's last entries, unused)
      const int src_next = check(G + 2 * NW, si, ok);
      load_k(src_next);
      if constexpr (IDX != 0) si = read_idx(G + 3 * NW);
      else si = min(kSrc * (G + 3 * NW) + c, K - 1);
      __builtin_amdgcn_sched_barrier(0);
      weigh(okm);
      __builtin_amdgcn_sched_barrier(0);
      load_v(G + NW, src);
      okm = mask(ok_next);
      ok_next = ok;
      src = src_next;
#pragma unroll
      for (int n = 0; n < NQ; ++n) st[n] = st_next[n];
    }
    softmax(st, okm);
    weigh(okm);
  }

  // ---- merge the waves; the sink joins the normaliser once (in the combine for a split) ----
#pragma unroll
  for (int n = 0; n < NQ; ++n) {
    const int r = 16 * n + c;
    float l = l_run[n];
    l += xor_lane<16>(l);
    l += xor_lane<32>(l);
    float* ob = s_ob + (wv * R + r) * kObStride;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4_t*>(ob + 64 * i + 16 * g + 4 * q) =
            f32x4_t{O[n][4 * i][q], O[n][4 * i + 1][q], O[n][4 * i + 2][q], O[n][4 * i + 3][q]};
    if (g == 0) {
      s_ml[wv][r][0] = m_run[n];
      s_ml[wv][r][1] = l;
    }
  }
  __syncthreads();
  const bool whole = a.n_split == 1;
  if (static_cast<int>(threadIdx.x) < n_rows) {
    const int r = threadIdx.x;
    const int h = (r0 + r) % a.H;
    const float sk = whole ? sinkc::load_elem<DT>(a.sink, a.sink_scalar ? 0 : h) * kLog2e : kNegInf;
    float M = sk;
#pragma unroll
    for (int w = 0; w < NW; ++w) M = fmaxf(M, s_ml[w][r][0]);
    float den = whole ? __builtin_amdgcn_exp2f(sk - M) : 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float mw = s_ml[w][r][0];
      const float f = mw == kNegInf ? 0.0f : __builtin_amdgcn_exp2f(mw - M);
      den = fmaf(f, s_ml[w][r][1], den);
      s_ml[w][r][0] = f;
    }
    if (whole) {
      s_inv[r] = M == kNegInf ? 0.0f : 1.0f / den;  // no valid source and sink -inf: 0
    } else {
      float* dst = a.part + ((base_row + r) * a.n_split + split) * kPart;
      dst[0] = M;
      dst[1] = den;
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < n_rows * (D / 4); t += 64 * NW) {
    const int r = t / (D / 4), d4 = 4 * (t % (D / 4));
    f32x4_t acc = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float f = s_ml[w][r][0];
      const f32x4_t o = *reinterpret_cast<const f32x4_t*>(s_ob + (w * R + r) * kObStride + d4);
      acc = f32x4_t{fmaf(f, o[0], acc[0]), fmaf(f, o[1], acc[1]), fmaf(f, o[2], acc[2]), fmaf(f, o[3], acc[3])};
    }
    if (whole) {
      const float i = s_inv[r];
      sinkc::store4<DT>(a.out, (base_row + r) * D + d4, acc[0] * i, acc[1] * i, acc[2] * i, acc[3] * i);
    } else {
      *reinterpret_cast<f32x4_t*>(a.part + ((base_row + r) * a.n_split + split) * kPart + 4 + d4) = acc;
    }
  }
}

struct F32Plan {
  int nq, nw, n_split, gps;
  int64_t n_blk, wgs;  // row blocks per sequence / target; workgroups per piece
  size_t ws;
};

// Rows of a workgroup, its waves, and the source pieces.  One row group of 8 waves against two of 4 (which
// read each source half as often, and leave more pieces to split into), 12 heads, kernel and combine.  Split
// calls take two from 65 blocks of 32 rows, where one group's blocks are more than 128 and no longer split:
// over 2176 sources, fp32, 128 dims, 57 blocks 31.6 / 33.4 us, 65 50 / 35.6, 96 50 / 45.5 (113 50 / 54, 150 96
// / 67: the rounds of a full chip alternate); 64 dims 57 blocks 18.3 / 20.3, 65 27.6 / 21.4; bf16 19.9 / 21.1
// and 30.7 / 22.3; over 1003 sources 20.3 / 24.5 and 27.3 / 25.4 (fp32, 128 dims).  Below 56 groups the line
// is 36: over 700 sources 41 blocks 17.7 / 16.0, 48 18.0 / 16.4 (57 to 128 blocks 19 to 21 / 23 to 28, 150 40
// / 32.5).  Calls that are not split take two from 256 blocks: over 300 sources 96 blocks 13.4 / 17.9, 257 34
// / 28, 64 dims 257 16.4 / 16.7, 512 22.1 / 18.1 (at 128 dims two are ahead from 150 blocks already, 24.5 /
// 18.1; over 600 sources x 64 dims 257 blocks take 25 / 29). Splits start above 40 groups (640 sources) when
// the workgroups leave CUs idle: one target over 656 sources takes 11.4 us and a 4 us combine instead of 18.8
// us; pieces fill the chip (512 four-wave workgroups or 256 of eight) and keep at least two groups per wave.
// Sparse calls of at most eight groups and six heads take one wave per workgroup once those fill half the chip:
// with so few of a product's 16 rows in use, the merge of four waves' 16 rows (one to three of them without a
// group at few sources) left the VALU kernel ahead.  VALU / four waves / one, fp32: 4096 targets x 4 heads x 128
// dims over 16 sources 51 / 35 / 14.7 us, over one 19.5 / 27.9 / 12.4; 16384 targets of one head x 128 dims over 64
// 129 / 173 / 104, x 64 dims over 16 26.0 / 39.4 / 20.8; 1024 targets of one head x 64 dims over 64 21 / 7.0 / 6.6;
// 512 over 64 20.8 / 5.1 / 6.1.  One wave sums its groups in sequence: fp32 error against 64 bits over 64 / 128
// sources 2.2e-7 / 2.8e-7, four waves 1.9e-7 / 2.1e-7, the VALU kernel 2.8e-7 / 3.3e-7 (64 dims).
F32Plan f32_plan(bool dense, int64_t D, int64_t B, int64_t T, int64_t H, int64_t K, bool may_split) {
  F32Plan p{};
  const int64_t shared = dense ? T * H : H, units = dense ? B : B * T;
  const int64_t groups = ceil_div(K, static_cast<int64_t>(kSrc));
  const bool split = may_split && groups > 40;
  const int64_t blocks2 = units * ceil_div(shared, int64_t(32));
  p.nq = dense && blocks2 >= (!split ? 256 : groups < 56 ? 36 : 65) ? 2 : 1;
  p.n_blk = ceil_div(shared, static_cast<int64_t>(16 * p.nq));
  p.wgs = units * p.n_blk;
  p.nw = p.nq == 1 && groups >= 16 ? 8 : !dense && H <= 6 && groups <= 8 && p.wgs >= 1024 ? 1 : 4;
  p.n_split = 1;
  const int64_t fill = p.nw == 8 ? 256 : 512;
  if (split && p.wgs > 0)
    p.n_split = static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(fill / p.wgs, groups / (2 * p.nw))));
  p.gps = static_cast<int>(std::max<int64_t>(1, ceil_div(groups, p.n_split)));
  if (p.n_split > 1) p.n_split = static_cast<int>(ceil_div(groups, p.gps));  // no empty pieces
  p.ws = p.n_split > 1 ? align_up(static_cast<size_t>(B * T * H) * p.n_split * (D + 4) * sizeof(float), 256) : 0;
  return p;
}

template <int DT, int D, int IDX>
void launch_f32(const SinkF32Args& a, const F32Plan& p, hipStream_t st) {
  const dim3 grid(static_cast<uint32_t>(p.wgs), static_cast<uint32_t>(p.n_split));
  if constexpr (IDX == 0) {
    if (p.nq == 2) {
      hipLaunchKernelGGL((sink_attn_f32_kernel<DT, D, 0, 2, 4>), grid, dim3(256), 0, st, a);
      return;
    }
  }
  if constexpr (IDX != 0) {
    if (p.nw == 1) {
      hipLaunchKernelGGL((sink_attn_f32_kernel<DT, D, IDX, 1, 1>), grid, dim3(64), 0, st, a);
      return;
    }
  }
  if (p.nw == 8) hipLaunchKernelGGL((sink_attn_f32_kernel<DT, D, IDX, 1, 8>), grid, dim3(512), 0, st, a);
  else hipLaunchKernelGGL((sink_attn_f32_kernel<DT, D, IDX, 1, 4>), grid, dim3(256), 0, st, a);
}

template <int DT, int D>
void launch_f32_idx(const SinkF32Args& a, const F32Plan& p, int64_t rows, int idx_kind, hipStream_t st) {
  if (idx_kind == 0) launch_f32<DT, D, 0>(a, p, st);
  else if (idx_kind == 4) launch_f32<DT, D, 4>(a, p, st);
  else launch_f32<DT, D, 8>(a, p, st);
  if (p.n_split > 1)
    sinkc::launch_combine<DT, D>(a.part, p.n_split, a.sink, a.sink_scalar, a.H, rows, a.out, st);
}

}  // namespace

bool sink_attention_f32_supported(int32_t dtype, int64_t D) {
  return dtype == AEKV_F32 ? (D == 64 || D == 128) : D == 64;
}

bool sink_attention_f32_takes(bool dense, int64_t D, int64_t B, int64_t T, int64_t H, int64_t S, int64_t K) {
  // Many targets of one or two heads over a few sources: 15 or 14 of the 16 rows of a product are empty, and
  // the VALU kernel's wave per row is the faster one.  VALU / this kernel, fp32, one head: 4096 targets x 64 dims
  // over one source 5.2 / 6.9 us, over 16 10.6 / 7.3; x 128 dims 7.4 / 11.0 and 20 / 13; 16384 targets x 64 dims 11.7 /
  // 19.9 and 26 / 20.8, x 128 dims 22 / 38 and 50 / 45; 2048 x 128 dims over one 5.5 / 6.4; 1024 targets equal.
  if (!dense && H <= 2 && H * H * K <= 12 && B * T >= 2048 && H * H * K * 512 <= B * T) return false;
  const int64_t lim = 0x7fffffff - 4096;  // (32-bit positions, a few groups past the end among them)
  if (S > lim || K > lim || B * T * H > lim || T * H > lim) return false;
  // (256 or 512 threads per 16 or 32 rows, where the VALU kernel takes 64 per row: sparse calls of many
  // targets with few heads reach the launch's limit first here)
  for (const bool split : {false, true}) {
    const F32Plan p = f32_plan(dense, D, B, T, H, K, split);
    if (p.wgs * 64 * p.nw > kMaxGridThreads) return false;
  }
  return true;
}

size_t sink_attention_f32_workspace(bool dense, int64_t D, int64_t B, int64_t T, int64_t H, int64_t K) {
  return f32_plan(dense, D, B, T, H, K, true).ws;
}

int sink_attention_f32(const void* q, const void* kv, const void* idx, int idx_kind, const void* sink, int sink_scalar,
                       int32_t dtype, int64_t B, int64_t T, int64_t H, int64_t D, int64_t S, int64_t K, float scale,
                       void* ws, size_t ws_bytes, void* out, hipStream_t st, const char* who) {
  if (S == 0) K = 0;  // every index is out of range
  F32Plan p = f32_plan(idx_kind == 0, D, B, T, H, K, ws != nullptr);
  // the split is only a faster order: a workspace too small for it runs the call unsplit
  if (p.ws > 0 && (ws_bytes < p.ws || !is_aligned(ws, 16))) p = f32_plan(idx_kind == 0, D, B, T, H, K, false);
  SinkF32Args a{};
  a.q = q;
  a.kv = kv;
  a.idx = idx;
  a.sink = sink;
  a.sink_scalar = sink_scalar;
  a.H = static_cast<int>(H);
  a.T = static_cast<int>(T);
  a.S = static_cast<int>(S);
  a.K = static_cast<int>(K);
  a.n_blk = static_cast<uint32_t>(p.n_blk);
  a.scale2 = scale * kLog2e;
  a.n_split = p.n_split;
  a.gps = p.gps;
  a.part = p.n_split > 1 ? static_cast<float*>(ws) : nullptr;
  a.out = out;
  if (dtype == AEKV_F32) {
    if (D == 128) launch_f32_idx<AEKV_F32, 128>(a, p, B * T * H, idx_kind, st);
    else launch_f32_idx<AEKV_F32, 64>(a, p, B * T * H, idx_kind, st);
  } else if (dtype == AEKV_F16) {
    launch_f32_idx<AEKV_F16, 64>(a, p, B * T * H, idx_kind, st);
  } else {
    launch_f32_idx<AEKV_BF16, 64>(a, p, B * T * H, idx_kind, st);
  }
  return check_launch(who);
}

}  // namespace aekv
