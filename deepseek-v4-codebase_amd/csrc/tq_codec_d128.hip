// Fast TurboQuant encode and decode for the production shapes (gfx950): the 4-bit D = 128 bf16 KV
// layer (encode and decode), and the encode of the other 16-bit blocks of D = 128 and index keys of D = 64.
//
// ENCODE
// Same result, bit for bit, as tq_forward_kernel<BF16, 128, ENC4> and as
// aether_2b/turbo_quant.py:127-166 (rot = _wht(x*diag); m = max(max|rot|, 1e-8); scale = m/7;
// q = clamp(rne(rot/m*7)); nibble pack), with about half the VALU work:
//
// * Layout.  A wave handles 16 vectors; lane l = 4v + g holds elements [32g, 32g+32) of vector v
//   of its group: a wave reads 4 KiB and writes 1 KiB of codes, contiguous, 64 and 16 bytes per
//   lane.  Butterfly stages h = 1..16 run in registers; stage h = 32 pairs lanes g ^ 1 and stage
//   h = 64 lanes g ^ 2 of the same quad.
// * Cross-lane stages.  Each is one v_fmac_f32 per element whose src0 reads the partner through
//   DPP quad_perm: own + s * partner with s = -1 on the upper lane, i.e. x + y on the lower lane
//   and y - x = -(x - y) on the upper one (an exact product and one rounding; RNE is symmetric, so
//   the magnitude is the reference's x - y bit for bit).  After both stages lane g holds its
//   elements times sigma = (-1)^(g0 + g1); the sign is folded into the quantiser's factor.
// * x * diag and the first butterfly stage: per packed bf16 word w and its diag sign mask M (bit
//   31: the high element's diag is negative, bit 15: the low one's), lo*diag = (w + M) << 16 (one
//   v_add_lshl_u32: adding 0x8000 flips bit 15 and the carry out of it is shifted away),
//   hi*diag = (w ^ M) & 0xFFFF0000 (one v_bitop3), and the reference's fp32 add and sub of the
//   two.  (v_dot2_f32_bf16 computes the same sum but does not round it like an fp32 add when the
//   two halves are more than 2^16 apart, so it is not used.)
// * Scale folding.  max|rot| = RN(c * max|raw|) because rounding is monotonic (raw = butterfly
//   output before the * c, c = fp32(128^-0.5)), so the per-element work uses the exact products
//   raw * K-, raw * K+ with K+- = K (1 +- 2^-20), K = RN(RN(7c) * rcp(m)) (v_rcp_f32, relative
//   error <= 2^-23), instead of t = RN(RN(RN(raw*c)/m)*7).  |K / (7c/m) - 1| <= 2^-22 and
//   |t / (raw*7c/m) - 1| <= 3 * 2^-24, so t lies between raw*K- and raw*K+, and since rne is
//   monotonic, rne(raw*K-) == rne(raw*K+) implies rne(t) equals both.  A wave in which any element
//   has the two apart (a tie within ~7 * 2^-19 of the product) re-encodes its 16 vectors with the
//   reference's exact operation sequence (about 1e-5 of the elements on Gaussian data).
// * rne and the nibble come from one FMA with the magic constant M8 = 1.5 * 2^23 + 8:
//   RN(p + M8) = M8 + rne(p) for |p| <= 2^22, whose low byte is rne(p) + 8 (offset binary); a
//   nibble pair is one shift-or and one XOR with 0x88888888 per dword restores two's complement.
// * The next group's 4 KiB are requested before the current group is transformed, so every wave
//   keeps one group of loads in flight while it computes.
#include <atomic>
#include <cstdlib>
#include <cstring>

#include "tq_device.h"

namespace aekv {
namespace {

constexpr int kThreads = 256;
constexpr int kEncThreads = 256;  // encode workgroup size (each workgroup builds the diag-mask table once)
constexpr int kEncMinWaves = 4;   // waves per SIMD the encode's register allocation must allow
constexpr int kDecPasses = 8;     // 4-vector passes per decode wave on large inputs
constexpr int64_t kDecMaxBlocks = 2048;  // the grid-stride decode (smaller inputs): at most this many workgroups
typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
constexpr float kMagic8 = 12582920.0f;  // 1.5 * 2^23 + 8: RN(t + kMagic8) = kMagic8 + rne(t), ulp 1

// Stages h = 32 and h = 64 on eight registers: a += s * a(partner), the partner's value read by
// v_fmac_f32 through DPP quad_perm [1,0,3,2] (lane ^ 1), then [2,3,0,1] (lane ^ 2).  Written as
// inline asm because the compiler only forms v_fmac from its VOP3 FMA after the pass that folds
// DPP moves, and VOP3 has no DPP form on gfx950.  A DPP read of a VGPR needs two wait states after
// the VALU write of it: s_nop 1 covers the code before the block, and inside it every register is
// read through DPP eight instructions after its write.
__device__ __forceinline__ void quad_stages8(float& a0, float& a1, float& a2, float& a3, float& a4, float& a5,
                                             float& a6, float& a7, float s32, float s64) {
  asm("s_nop 1\n"
      "v_fmac_f32_dpp %0, %0, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %1, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %2, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %3, %3, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %4, %4, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %5, %5, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %6, %6, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %7, %7, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %0, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %1, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %2, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %3, %3, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %4, %4, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %5, %5, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %6, %6, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %7, %7, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf"
      : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5), "+v"(a6), "+v"(a7)
      : "v"(s32), "v"(s64));
}

// ue, uo: bit patterns of M8 + n (n in [-7, 7]), whose low byte is n + 8 in [1, 15].
// Returns a word whose low byte is (n_odd + 8) << 4 | (n_even + 8); bits 8.. are garbage.
__device__ __forceinline__ uint32_t nib_pair(uint32_t ue, uint32_t uo) { return (uo << 4) | ue; }

// Low bytes of four nib_pair words -> one dword of two's-complement nibbles (xor 8 per nibble
// turns the offset-binary n + 8 into n & 15).
__device__ __forceinline__ uint32_t pack4(uint32_t b0, uint32_t b1, uint32_t b2, uint32_t b3) {
  const uint32_t lo = __builtin_amdgcn_perm(b1, b0, 0x0c0c0400u);  // [b0.0, b1.0, 0, 0]
  const uint32_t hi = __builtin_amdgcn_perm(b3, b2, 0x04000c0cu);  // [0, 0, b2.0, b3.0]
  return (lo | hi) ^ 0x88888888u;
}

// max(acc, |x|, |y|) as one v_max3_f32 with abs source modifiers.
__device__ __forceinline__ float max3_abs(float acc, float x, float y) {
  float r;
  asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(acc), "v"(x), "v"(y));
  return r;
}

// Loads the lane's 64 bytes of group `grp`: a wave-uniform base (scalar registers) plus a 32-bit
// lane offset.  Lanes past the end of a partial last group re-read its last vector (never stored),
// so every lane runs the same code.
__device__ __forceinline__ void load_group(const uint4* __restrict__ x, int64_t grp, int64_t n_vec, int v, int g,
                                           uint4 (&t)[4]) {
  const char* base = reinterpret_cast<const char*>(x + grp * 256);
  const int64_t rem = n_vec - grp * 16;
  const uint32_t vv = static_cast<uint32_t>(v < rem ? v : rem - 1);
  const uint32_t off = vv * 256u + static_cast<uint32_t>(g) * 64u;  // bytes
#pragma unroll
  for (int i = 0; i < 4; ++i) t[i] = *reinterpret_cast<const uint4*>(base + (off + 16u * i));
  __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the transform that follows
}

// The reference's exact operation sequence for the 16 vectors of group `grp`, re-read from x:
// tq_forward_kernel's per-lane code (16 lanes x 8 elements per vector, four passes of four
// vectors).  Used when the fast quantiser cannot decide a rounding; it needs few registers, so it
// does not raise the kernel's register budget.
__device__ __forceinline__ void encode_group_exact(const uint4* __restrict__ x, int64_t grp, int64_t n_vec,
                                                             const float* __restrict__ diag, float c,
                                                             uint8_t* __restrict__ codes, float* __restrict__ scale) {
  constexpr int D = 128, EPL = 8, LPV = 16;
  const int lane = threadIdx.x & 63;
  const int sub = lane % LPV, slot = lane / LPV;
  float dg[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) dg[e] = diag[sub * EPL + e];
#pragma unroll 1
  for (int pass = 0; pass < 4; ++pass) {
    const int64_t v = grp * 16 + pass * 4 + slot;
    const bool ok = v < n_vec;
    float a[EPL];
    load_elems<AEKV_BF16, EPL>(x, v * D + sub * EPL, ok, a);
#pragma unroll
    for (int e = 0; e < EPL; ++e) a[e] = a[e] * dg[e];
    wht_butterflies<D, EPL, true>(a, sub);
#pragma unroll
    for (int e = 0; e < EPL; ++e) a[e] = a[e] * c;
    const float m = fmaxf(group_absmax<D, EPL, true>(a), 1e-8f);
    uint32_t w = 0u;
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      float t = a[e] / m;  // correctly rounded division (-fhip-fp32-correctly-rounded-divide-sqrt)
      t = fminf(fmaxf(rintf(t * 7.0f), -7.0f), 7.0f);
      w |= (static_cast<uint32_t>(static_cast<int>(t)) & 15u) << (4 * e);
    }
    if (ok) {
      if (sub == 0) scale[v] = m / 7.0f;
      *reinterpret_cast<uint32_t*>(codes + v * (D / 2) + sub * (EPL / 2)) = w;
    }
  }
}

// Encodes the 16 vectors of group `grp` from the lane's 64 loaded bytes `t`.
__device__ __forceinline__ void encode_group(const uint4 (&t)[4], const uint4* __restrict__ x, int64_t grp,
                                             int64_t n_vec, int v, int g, const uint4* dm_lds, float s32,
                                             float s64, float sigma, const float* __restrict__ diag, float c,
                                             float c7, uint4* __restrict__ codes, float* __restrict__ scale) {
  uint32_t w[16];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    w[4 * i] = t[i].x;
    w[4 * i + 1] = t[i].y;
    w[4 * i + 2] = t[i].z;
    w[4 * i + 3] = t[i].w;
  }
  // the lane's diag sign masks, read from LDS each group (keeping them in registers would cost 16)
  uint32_t dm[16];
  asm volatile("" ::: "memory");  // not hoisted out of the group loop
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint4 d = dm_lds[i];
    dm[4 * i] = d.x;
    dm[4 * i + 1] = d.y;
    dm[4 * i + 2] = d.z;
    dm[4 * i + 3] = d.w;
  }
  float a[32];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    // stage h = 1 on x * diag: lo + hi, lo - hi
    const float lo = __builtin_bit_cast(float, (w[k] + dm[k]) << 16);
    const float hi = __builtin_bit_cast(float, __builtin_amdgcn_bitop3_b32(w[k], 0xFFFF0000u, dm[k], 0x48));
    a[2 * k] = lo + hi;
    a[2 * k + 1] = lo - hi;
  }
  // stages h = 2, 4, 8, 16 in registers
#pragma unroll
  for (int h = 2; h < 32; h <<= 1) {
#pragma unroll
    for (int blk = 0; blk < 32; blk += 2 * h) {
#pragma unroll
      for (int i = 0; i < h; ++i) {
        const float p = a[blk + i], q = a[blk + h + i];
        a[blk + i] = p + q;
        a[blk + h + i] = p - q;
      }
    }
  }
  // stages h = 32 and h = 64 across the quad
#pragma unroll
  for (int r = 0; r < 32; r += 8)
    quad_stages8(a[r], a[r + 1], a[r + 2], a[r + 3], a[r + 4], a[r + 5], a[r + 6], a[r + 7], s32, s64);

  // m = max(RN(c * max|raw|), 1e-8) over the 4 lanes of the vector
  float mr = 0.0f;
#pragma unroll
  for (int r = 0; r < 32; r += 2) mr = max3_abs(mr, a[r], a[r + 1]);
  mr = fmaxf(mr, xor_lane<1>(mr));
  mr = fmaxf(mr, xor_lane<2>(mr));
  const float m = fmaxf(mr * c, 1e-8f);
  const float K = c7 * __builtin_amdgcn_rcpf(m);  // v_rcp_f32: 1 ulp; only feeds the checked fast path
  const float klo = (K - K * 0x1p-20f) * sigma, khi = (K + K * 0x1p-20f) * sigma;

  // fast path: u = RN(a*K- + M8) = M8 + rne(a*K-); any bit of u(K-) ^ u(K+) flags a tie in reach
  uint32_t o[4];
  uint32_t diff = 0u;
#pragma unroll
  for (int dw = 0; dw < 4; ++dw) {
    uint32_t b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float x0 = a[8 * dw + 2 * j], x1 = a[8 * dw + 2 * j + 1];
      const uint32_t u0 = __builtin_bit_cast(uint32_t, fmaf(x0, klo, kMagic8));
      const uint32_t u1 = __builtin_bit_cast(uint32_t, fmaf(x1, klo, kMagic8));
      // diff | (u ^ u(K+)) as one v_bitop3 (truth table 0xF0 | (0xCC ^ 0xAA))
      diff = __builtin_amdgcn_bitop3_b32(diff, u0, __builtin_bit_cast(uint32_t, fmaf(x0, khi, kMagic8)), 0xF6);
      diff = __builtin_amdgcn_bitop3_b32(diff, u1, __builtin_bit_cast(uint32_t, fmaf(x1, khi, kMagic8)), 0xF6);
      b[j] = nib_pair(u0, u1);
    }
    o[dw] = pack4(b[0], b[1], b[2], b[3]);
  }
  if (__builtin_amdgcn_ballot_w64(diff != 0u) != 0) {  // a tie is within reach of the fast path's error
    encode_group_exact(x, grp, n_vec, diag, c, reinterpret_cast<uint8_t*>(codes), scale);
    return;
  }
  if (v < n_vec - grp * 16) {  // streaming stores: the outputs are not read again by this kernel
    if (g == 0)
      __builtin_nontemporal_store(m / 7.0f, reinterpret_cast<float*>(reinterpret_cast<char*>(scale + grp * 16) +
                                                                     4u * static_cast<uint32_t>(v)));
    const u32x4_t ov = {o[0], o[1], o[2], o[3]};
    __builtin_nontemporal_store(ov, reinterpret_cast<u32x4_t*>(reinterpret_cast<char*>(codes + grp * 64) +
                                                              16u * static_cast<uint32_t>(4 * v + g)));
  }
}

__global__ __launch_bounds__(kEncThreads, kEncMinWaves) void tq_encode4_d128_bf16_kernel(
    const uint4* __restrict__ x, int64_t n_vec, const float* __restrict__ diag, float c, float c7,
    uint4* __restrict__ codes, float* __restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int v = lane >> 2, g = lane & 3;

  // diag signs of the packed words lane part g loads: bit 15 for diag[32g + 2k], bit 31 for the next
  __shared__ uint4 dm_tab[4][4];  // [g][i]: masks of words 4i .. 4i+3 of lane part g
  if (threadIdx.x < 64) {
    const int gg = threadIdx.x >> 4, k = threadIdx.x & 15;
    reinterpret_cast<uint32_t*>(dm_tab[gg])[k] = (diag[32 * gg + 2 * k] < 0.0f ? 0x8000u : 0u) |
                                                (diag[32 * gg + 2 * k + 1] < 0.0f ? 0x80000000u : 0u);
  }
  __syncthreads();
  const uint4* dm = dm_tab[g];
  const float s32 = (g & 1) ? -1.0f : 1.0f;  // stage 32: upper lane of the pair
  const float s64 = (g & 2) ? -1.0f : 1.0f;  // stage 64
  const float sigma = s32 * s64;             // the lane holds its elements times sigma afterwards

  const int64_t n_groups = (n_vec + 15) >> 4;
  // wave index in a scalar register: the code below is wave-uniform
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * (kEncThreads / 64) +
                       __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int64_t grp = wave;
  if (grp >= n_groups) return;
  // One group per wave (the launch covers every group): the hardware's turnover of short waves
  // overlaps one wave's loads with other waves' transforms, with no loop whose wait counts the
  // compiler has to merge over the rare paths (measured 8% faster on cfg2 than a grid-stride loop
  // with a two-group register prefetch).
  uint4 ta[4];
  load_group(x, grp, n_vec, v, g, ta);
  encode_group(ta, x, grp, n_vec, v, g, dm, s32, s64, sigma, diag, c, c7, codes, scale);
}

// ---- encode of the other shapes: D = 64 and 128, 4 and 8 bits, from bf16 and fp16 -------------------
// The 4-bit D = 128 design with these changes.
// * Layout: 32 elements per lane as above, LPV = D / 32 lanes per vector (4 at D = 128: stages h =
//   32, 64 across the quad; 2 at D = 64: stage h = 32 across the lane pair), 64 / LPV vectors per
//   wave.  A wave reads 4 KiB and writes 64 / LPV vectors' codes (1 or 2 KiB), contiguous.
// * fp16 elements take their diag sign on the packed word, before the conversion.
// * Quantiser interval.  K = RN(RN(Qc) v_rcp_f32(m)) is within 4 2^-24 relative of Qc/m (the product
//   Qc and K round once each, the reciprocal is within 2 2^-24); the reference's three roundings keep t =
//   RN(RN(RN(raw c) / m) Q) within 3 2^-24 of raw c Q / m; so t lies between raw K- and raw K+ for K+- =
//   K (1 +- 10 2^-24) (their own rounding takes one 2^-24 of the ten), and, rne being monotonic, equal
//   roundings of the two decide rne(t).
// * Undecided elements (within ~10 2^-24 |t| of a half-integer: ~8% of 8-bit D = 128 waves hold one on
//   Gaussian data) get the reference's exact sequence in place: the wave walks its 32 elements per lane and
//   divides only where some lane is undecided.
// * A vector with an infinite or NaN element, or beyond the range where K and its margin are normal
//   numbers, sends its wave through the generic kernel's sequence, re-read from x.
// Measured: 100 M fp16 elements, 4-bit / 8-bit D = 128 114 / 134 us, D = 64 115 / 132 us, 190 / 186 and 190 /
// 209 us by the generic kernel (8 divisions per lane); 49152 bf16 vectors 8-bit D = 128 6.8 us, 9.4 us with
// undecided waves re-encoded from memory and K in fp64 to have fewer of them; 100 M bf16 elements 136 us
// either way, at the rate of their reads and writes.  fp32 inputs stay with the generic kernel, which is
// bound by its bytes (110 us here and 111 there for 4-bit, 110 against 119 us for 8-bit D = 128).
// * 8-bit codes: RN(p + 1.5 2^23 + 128) = 1.5 2^23 + 128 + rne(p) for |p| <= 2^22, whose low
//   byte is rne(p) + 128; xor 0x80 gives the two's-complement int8.
constexpr float kMagic128 = 12583040.0f;  // 1.5 * 2^23 + 128

template <int BITS, int D>
struct FastEnc {
  static constexpr int LPV = D / 32;               // lanes per vector
  static constexpr int VPW = 64 / LPV;             // vectors per wave (one group)
  static constexpr int RB = BITS == 8 ? D : D / 2; // code bytes per vector
  static constexpr int LB = RB / LPV;              // code bytes per lane (16 or 32)
  static constexpr float Q = BITS == 8 ? 127.0f : 7.0f;
};

// Stage h = 32 alone (lane ^ 1 through DPP quad_perm [1,0,3,2]) on eight registers, as in
// quad_stages8.
__device__ __forceinline__ void pair_stage8(float& a0, float& a1, float& a2, float& a3, float& a4, float& a5,
                                            float& a6, float& a7, float s32) {
  asm("s_nop 1\n"
      "v_fmac_f32_dpp %0, %0, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %1, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %2, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %3, %3, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %4, %4, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %5, %5, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %6, %6, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %7, %7, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
      : "+v"(a0), "+v"(a1), "+v"(a2), "+v"(a3), "+v"(a4), "+v"(a5), "+v"(a6), "+v"(a7)
      : "v"(s32));
}

// The reference's exact sequence for the group's vectors, re-read from x (the generic kernel's
// per-lane code: 8 elements per lane, D / 8 lanes per vector).
template <int DT, int BITS, int D>
__device__ __forceinline__ void encode_group_exact_g(const void* __restrict__ x, int64_t grp, int64_t n_vec,
                                                     const float* __restrict__ diag, float c,
                                                     uint8_t* __restrict__ codes, float* __restrict__ scale) {
  using F = FastEnc<BITS, D>;
  constexpr int EPL = 8, LPV8 = D / EPL, VPP = 64 / LPV8, NB = BITS == 8 ? EPL : EPL / 2;
  const int lane = threadIdx.x & 63;
  const int sub = lane % LPV8, slot = lane / LPV8;
  float dg[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) dg[e] = diag[sub * EPL + e];
#pragma unroll 1
  for (int pass = 0; pass < F::VPW / VPP; ++pass) {
    const int64_t v = grp * F::VPW + pass * VPP + slot;
    const bool ok = v < n_vec;
    float a[EPL];
    load_elems<DT, EPL>(x, v * D + sub * EPL, ok, a);
#pragma unroll
    for (int e = 0; e < EPL; ++e) a[e] = a[e] * dg[e];
    float m;
    const Bytes<NB> w = encode_lane<BITS, D, false>(a, sub, c, &m);
    if (ok) {
      if (sub == 0) scale[v] = m / F::Q;
      *reinterpret_cast<Bytes<NB>*>(codes + v * F::RB + sub * NB) = w;
    }
  }
}

template <int DT, int BITS, int D>
__global__ __launch_bounds__(kEncThreads, kEncMinWaves) void tq_encode_fast_kernel(
    const void* __restrict__ x, int64_t n_vec, const float* __restrict__ diag, float c, float cq,
    uint8_t* __restrict__ codes, float* __restrict__ scale) {
  using F = FastEnc<BITS, D>;
  constexpr int LPV = F::LPV, VPW = F::VPW;
  static_assert(DT == AEKV_BF16 || DT == AEKV_F16, "16-bit elements");
  const int lane = threadIdx.x & 63;
  const int v = lane / LPV, g = lane % LPV;
  // diag sign masks of the lane part's 16 packed words (bit 15: low element, bit 31: high)
  __shared__ uint4 dm_tab[LPV][4];
  if (threadIdx.x < 16 * LPV) {
    const int gg = threadIdx.x >> 4, k = threadIdx.x & 15;
    reinterpret_cast<uint32_t*>(dm_tab[gg])[k] = (diag[32 * gg + 2 * k] < 0.0f ? 0x8000u : 0u) |
                                                (diag[32 * gg + 2 * k + 1] < 0.0f ? 0x80000000u : 0u);
  }
  __syncthreads();
  const int64_t n_groups = (n_vec + VPW - 1) / VPW;
  const int64_t grp = static_cast<int64_t>(blockIdx.x) * (kEncThreads / 64) +
                      __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  if (grp >= n_groups) return;
  // the lane's 64 bytes (lanes past a partial last group re-read its last vector, never stored)
  uint32_t w[16];
  {
    const char* base = static_cast<const char*>(x) + grp * VPW * D * 2;
    const int64_t rem = n_vec - grp * VPW;
    const uint32_t vv = static_cast<uint32_t>(v < rem ? v : rem - 1);
    const uint32_t off = vv * (2u * D) + static_cast<uint32_t>(g) * 64u;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint4 t = *reinterpret_cast<const uint4*>(base + (off + 16u * i));
      w[4 * i] = t.x;
      w[4 * i + 1] = t.y;
      w[4 * i + 2] = t.z;
      w[4 * i + 3] = t.w;
    }
  }
  uint32_t dm[16];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint4 d = dm_tab[g][i];
    dm[4 * i] = d.x;
    dm[4 * i + 1] = d.y;
    dm[4 * i + 2] = d.z;
    dm[4 * i + 3] = d.w;
  }
  float a[32];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    // stage h = 1 on x * diag: lo + hi, lo - hi
    float lo, hi;
    if constexpr (DT == AEKV_BF16) {
      lo = __builtin_bit_cast(float, (w[k] + dm[k]) << 16);
      hi = __builtin_bit_cast(float, __builtin_amdgcn_bitop3_b32(w[k], 0xFFFF0000u, dm[k], 0x48));
    } else {
      const uint32_t s = w[k] ^ dm[k];
      lo = f16_to_f32(s & 0xFFFFu);
      hi = f16_to_f32(s >> 16);
    }
    a[2 * k] = lo + hi;
    a[2 * k + 1] = lo - hi;
  }
#pragma unroll
  for (int h = 2; h < 32; h <<= 1) {
#pragma unroll
    for (int blk = 0; blk < 32; blk += 2 * h) {
#pragma unroll
      for (int i = 0; i < h; ++i) {
        const float p = a[blk + i], q = a[blk + h + i];
        a[blk + i] = p + q;
        a[blk + h + i] = p - q;
      }
    }
  }
  const float s32 = (g & 1) ? -1.0f : 1.0f;
  float sigma = s32;
  if constexpr (LPV == 4) {
    const float s64 = (g & 2) ? -1.0f : 1.0f;
    sigma = s32 * s64;
#pragma unroll
    for (int r = 0; r < 32; r += 8)
      quad_stages8(a[r], a[r + 1], a[r + 2], a[r + 3], a[r + 4], a[r + 5], a[r + 6], a[r + 7], s32, s64);
  } else {
#pragma unroll
    for (int r = 0; r < 32; r += 8)
      pair_stage8(a[r], a[r + 1], a[r + 2], a[r + 3], a[r + 4], a[r + 5], a[r + 6], a[r + 7], s32);
  }
  // m = max(RN(c max|raw|), 1e-8) over the LPV lanes of the vector
  float mr = 0.0f;
#pragma unroll
  for (int r = 0; r < 32; r += 2) mr = max3_abs(mr, a[r], a[r + 1]);
  mr = fmaxf(mr, xor_lane<1>(mr));
  if constexpr (LPV == 4) mr = fmaxf(mr, xor_lane<2>(mr));
  const float m = fmaxf(mr * c, 1e-8f);
  const float K = cq * __builtin_amdgcn_rcpf(m);
  const float klo = (K - K * 0x1.4p-21f) * sigma, khi = (K + K * 0x1.4p-21f) * sigma;
  constexpr float kMag = BITS == 8 ? kMagic128 : kMagic8;
  constexpr int NW = F::LB / 4;  // code dwords per lane
  constexpr int EPW = BITS == 8 ? 4 : 8;  // elements per code dword
  uint32_t o[NW];
  uint32_t diff = 0u;
#pragma unroll
  for (int dw = 0; dw < NW; ++dw) {
    uint32_t b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if constexpr (BITS == 8) {
        const float x0 = a[EPW * dw + j];
        const uint32_t u0 = __builtin_bit_cast(uint32_t, fmaf(x0, klo, kMag));
        diff = __builtin_amdgcn_bitop3_b32(diff, u0, __builtin_bit_cast(uint32_t, fmaf(x0, khi, kMag)), 0xF6);
        b[j] = u0;
      } else {
        const float x0 = a[EPW * dw + 2 * j], x1 = a[EPW * dw + 2 * j + 1];
        const uint32_t u0 = __builtin_bit_cast(uint32_t, fmaf(x0, klo, kMag));
        const uint32_t u1 = __builtin_bit_cast(uint32_t, fmaf(x1, klo, kMag));
        diff = __builtin_amdgcn_bitop3_b32(diff, u0, __builtin_bit_cast(uint32_t, fmaf(x0, khi, kMag)), 0xF6);
        diff = __builtin_amdgcn_bitop3_b32(diff, u1, __builtin_bit_cast(uint32_t, fmaf(x1, khi, kMag)), 0xF6);
        b[j] = nib_pair(u0, u1);
      }
    }
    if constexpr (BITS == 8) {
      const uint32_t lo = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u);  // [b0.0, b1.0, 0, 0]
      const uint32_t hi = __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);  // [0, 0, b2.0, b3.0]
      o[dw] = (lo | hi) ^ 0x80808080u;
    } else {
      o[dw] = pack4(b[0], b[1], b[2], b[3]);
    }
  }
  // (every output sums every input, so a lane's first output shows an infinite or NaN input)
  // (2^100: K and its margin stay normal numbers)
  const bool odd = !(mr < 0x1p100f) || !(fabsf(a[0]) < __builtin_inff());
  if (__builtin_amdgcn_ballot_w64(odd) != 0) {
    encode_group_exact_g<DT, BITS, D>(x, grp, n_vec, diag, c, codes, scale);
    return;
  }
  if (__builtin_amdgcn_ballot_w64(diff != 0u) != 0) {  // some rounding the interval cannot decide
    float rlo = klo, rhi = khi;
    asm volatile("" : "+v"(rlo), "+v"(rhi));  // (the 64 products are formed again here, not kept in registers)
#pragma unroll
    for (int e = 0; e < 32; ++e) {
      const bool open = fmaf(a[e], rlo, kMag) != fmaf(a[e], rhi, kMag);
      if (__builtin_amdgcn_ballot_w64(open) == 0) continue;  // wave-uniform
      float t = ((a[e] * sigma) * c) / m;  // correctly rounded division, then * Q, rne
      t = fminf(fmaxf(rintf(t * F::Q), -F::Q), F::Q);
      constexpr int kBits = 32 / EPW;
      constexpr uint32_t kMask = BITS == 8 ? 0xFFu : 0xFu;
      const int sh = kBits * (e % EPW);
      const uint32_t code = (static_cast<uint32_t>(static_cast<int>(t)) & kMask) << sh;
      o[e / EPW] = open ? (o[e / EPW] & ~(kMask << sh)) | code : o[e / EPW];
    }
  }
  if (v < n_vec - grp * VPW) {  // streaming stores: the outputs are not read again by this kernel
    if (g == 0)
      __builtin_nontemporal_store(m / F::Q, reinterpret_cast<float*>(reinterpret_cast<char*>(scale + grp * VPW) +
                                                                      4u * static_cast<uint32_t>(v)));
    char* cb = reinterpret_cast<char*>(codes + grp * VPW * F::RB) + static_cast<uint32_t>(lane) * F::LB;
#pragma unroll
    for (int i = 0; i < NW / 4; ++i) {
      const u32x4_t ov = {o[4 * i], o[4 * i + 1], o[4 * i + 2], o[4 * i + 3]};
      __builtin_nontemporal_store(ov, reinterpret_cast<u32x4_t*>(cb + 16 * i));
    }
  }
}

// ---- decode: 4-bit codes -> bf16, D = 128 ------------------------------------------------------
// Same result, bit for bit, as tq_decode_kernel<4, 128, BF16> and aether_2b/turbo_quant.py:187-211
// (rot = code * scale; x = _wht(rot) * diag; bf16 RNE).
//  * Layout: 16 lanes per vector, four vectors per wave and pass; lane l of a vector's row holds
//    the 8 elements of chunk pi(l) = l ^ f(l bit 2, l bit 3) with f = 0, 3, 4, 7.  Its code dword
//    and its 16 output bytes are where chunk pi(l) lives, so a load instruction covers 256
//    contiguous bytes and a store 1 KiB.  Butterfly stages h = 1, 2, 4 run in the lane; stages
//    8 / 16 / 32 / 64 act on chunk bits 0 / 1 / 2 / 3, which pi turns into the DPP patterns
//    quad_perm [1,0,3,2] (l ^ 1), quad_perm [2,3,0,1] (l ^ 2), row_half_mirror (l ^ 7) and
//    row_mirror (l ^ 15), each one v_fmac_f32_dpp per element (own + s * partner, s = -1 on the
//    lane whose chunk has the stage's bit set).
//  * Unpack: (w ^ 0x88888888) & 0x0F0F0F0F (one v_bitop3) turns the nibbles of a word into n + 8
//    in bytes (low nibbles; the high ones after a shift), v_cvt_f32_ubyte converts, and
//    rot = fma(n + 8, s, -8s) = RN(n*s) exactly (8s is exact, so the fma's one rounding is the
//    reference's product rounding).
//  * After the cross stages a lane holds sigma * raw (sigma = -1 per stage in which it was the
//    upper lane; RNE is sign-symmetric), and fma(sigma*raw, sigma*c, +0) = RN(raw * c): the +0
//    addend turns a zero of either sign into +0, which is what the reference's butterflies give
//    for a zero when every scale is positive (its zeros come from exact cancellation or 0 * s).
//    The sign of diag is then XORed into the packed bf16 pair.
//  * A pass with any scale outside (0, 2^124) (zero, negative, NaN, or too large for -8s to be
//    exact) decodes its vectors with the generic per-lane sequence instead.

// Stages h = 8, 16, 32, 64 on the lane's eight elements: a += s * a(partner) with the partner read
// by v_fmac_f32 through DPP (inline asm for the reason given at quad_stages8; s_nop 1 covers the
// DPP read-after-VALU-write hazard of the code before the block, and inside it each register is
// read through DPP eight instructions after its write).
__device__ __forceinline__ void row_stages8(float (&a)[8], float s8, float s16, float s32, float s64) {
  asm("s_nop 1\n"
      "v_fmac_f32_dpp %0, %0, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %1, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %2, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %3, %3, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %4, %4, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %5, %5, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %6, %6, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %7, %7, %8 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %0, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %1, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %2, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %3, %3, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %4, %4, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %5, %5, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %6, %6, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %7, %7, %9 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %0, %10 row_half_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %1, %10 row_half_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %2, %10 row_half_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %3, %3, %10 row_half_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %4, %4, %10 row_half_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %5, %5, %10 row_half_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %6, %6, %10 row_half_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %7, %7, %10 row_half_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %0, %0, %11 row_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %1, %1, %11 row_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %2, %2, %11 row_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %3, %3, %11 row_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %4, %4, %11 row_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %5, %5, %11 row_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %6, %6, %11 row_mirror row_mask:0xf bank_mask:0xf\n"
      "v_fmac_f32_dpp %7, %7, %11 row_mirror row_mask:0xf bank_mask:0xf"
      : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(a[4]), "+v"(a[5]), "+v"(a[6]), "+v"(a[7])
      : "v"(s8), "v"(s16), "v"(s32), "v"(s64));
}

// Decodes the four vectors of pass `pv` (vectors 4pv .. 4pv+3) from the lane's code dword `w` and
// its vector's scale `s`.
template <bool NT>
__device__ __forceinline__ void decode_pass(uint32_t w, float s, int64_t pv, int64_t n_vec, int row, int chunk,
                                            const float (&sg)[4], float sc, uint32_t dsig0, uint32_t dsig1,
                                            uint32_t dsig2, uint32_t dsig3, const uint8_t* __restrict__ codes,
                                            const float* __restrict__ scale, const float* __restrict__ diag,
                                            float c, uint16_t* __restrict__ out) {
  const int64_t v = pv * 4 + row;
  if (__builtin_amdgcn_ballot_w64(!(s > 0.0f && s < 0x1p124f)) != 0) {  // wave-uniform, rare
    // the generic kernel's per-lane sequence: lane l of the row holds elements 8l .. 8l+7
    const int sub = threadIdx.x & 15;
    float dg[8], a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) dg[e] = diag[8 * sub + e];
    const int64_t vr = v < n_vec ? v : n_vec - 1;
    decode_lane<4, 128, true>(codes + vr * 64, scale[vr], sub, dg, c, a);
    if (v < n_vec)
      *reinterpret_cast<uint4*>(out + v * 128 + 8 * sub) =
          make_uint4(pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(a[4], a[5]), pack_bf16x2(a[6], a[7]));
    return;
  }
  const uint32_t lo = __builtin_amdgcn_bitop3_b32(w, 0x88888888u, 0x0F0F0F0Fu, 0x28);  // (x ^ y) & z
  const uint32_t hi = __builtin_amdgcn_bitop3_b32(w >> 4, 0x88888888u, 0x0F0F0F0Fu, 0x28);
  const float m8s = -8.0f * s;
  float a[8];
#pragma unroll
  for (int k = 0; k < 4; ++k) {  // n + 8 converts exactly
    a[2 * k] = fmaf(static_cast<float>((lo >> (8 * k)) & 0xFFu), s, m8s);
    a[2 * k + 1] = fmaf(static_cast<float>((hi >> (8 * k)) & 0xFFu), s, m8s);
  }
#pragma unroll
  for (int h = 1; h < 8; h <<= 1) {
#pragma unroll
    for (int blk = 0; blk < 8; blk += 2 * h) {
#pragma unroll
      for (int i = 0; i < h; ++i) {
        const float p = a[blk + i], q = a[blk + h + i];
        a[blk + i] = p + q;
        a[blk + h + i] = p - q;
      }
    }
  }
  row_stages8(a, sg[0], sg[1], sg[2], sg[3]);
  const uint32_t o0 = pack_bf16x2(fmaf(a[0], sc, 0.0f), fmaf(a[1], sc, 0.0f)) ^ dsig0;
  const uint32_t o1 = pack_bf16x2(fmaf(a[2], sc, 0.0f), fmaf(a[3], sc, 0.0f)) ^ dsig1;
  const uint32_t o2 = pack_bf16x2(fmaf(a[4], sc, 0.0f), fmaf(a[5], sc, 0.0f)) ^ dsig2;
  const uint32_t o3 = pack_bf16x2(fmaf(a[6], sc, 0.0f), fmaf(a[7], sc, 0.0f)) ^ dsig3;
  if (v < n_vec) {
    if constexpr (NT)  // a layer-sized output streams past the caches
      __builtin_nontemporal_store(u32x4_t{o0, o1, o2, o3}, reinterpret_cast<u32x4_t*>(out + v * 128 + 8 * chunk));
    else
      *reinterpret_cast<uint4*>(out + v * 128 + 8 * chunk) = make_uint4(o0, o1, o2, o3);
  }
}

// PP > 0: PP consecutive 4-vector passes per wave, all loads issued first, no loop (the launch
// covers every pass; short waves whose turnover overlaps loads with other waves' transforms).
// PP == 0: a grid-stride loop with a one-pass prefetch, for inputs too small to fill the chip.
template <int PP>
__global__ __launch_bounds__(kThreads) void tq_decode4_d128_bf16_kernel(const uint32_t* __restrict__ codes,
                                                                        const float* __restrict__ scale,
                                                                        int64_t n_vec, const float* __restrict__ diag,
                                                                        float c, uint16_t* __restrict__ out) {
  const int l = threadIdx.x & 15, row = (threadIdx.x >> 4) & 3;
  const int chunk = l ^ (((l >> 2) & 1) ? 3 : 0) ^ (((l >> 3) & 1) ? 4 : 0);  // pi(l)
  float sg[4];  // stage factors: -1 on the lane whose chunk has the stage's bit set
#pragma unroll
  for (int k = 0; k < 4; ++k) sg[k] = ((chunk >> k) & 1) ? -1.0f : 1.0f;
  const float sc = ((__builtin_popcount(static_cast<unsigned>(chunk)) & 1) ? -c : c);  // sigma * c
  uint32_t dsig[4];  // diag sign bits of the packed output pairs
#pragma unroll
  for (int k = 0; k < 4; ++k)
    dsig[k] = (diag[8 * chunk + 2 * k] < 0.0f ? 0x8000u : 0u) | (diag[8 * chunk + 2 * k + 1] < 0.0f ? 0x80000000u : 0u);

  const int64_t n_pass = (n_vec + 3) >> 2;
  const int64_t wave = static_cast<int64_t>(blockIdx.x) * (kThreads / 64) +
                       __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const uint8_t* cb = reinterpret_cast<const uint8_t*>(codes);
  // lanes past the end read the last vector (never stored)
  auto load = [&](int64_t p, uint32_t& w, float& s) {
    const int64_t v = p * 4 + row;
    const int64_t vr = v < n_vec ? v : n_vec - 1;
    w = codes[vr * 16 + chunk];
    s = scale[vr];
  };
  if constexpr (PP > 0) {
    const int64_t p0 = wave * PP;
    if (p0 >= n_pass) return;
    uint32_t wq[PP];
    float sq[PP];
#pragma unroll
    for (int i = 0; i < PP; ++i) load(p0 + i < n_pass ? p0 + i : p0, wq[i], sq[i]);
#pragma unroll
    for (int i = 0; i < PP; ++i)
      if (p0 + i < n_pass)
        decode_pass<true>(wq[i], sq[i], p0 + i, n_vec, row, chunk, sg, sc, dsig[0], dsig[1], dsig[2], dsig[3], cb, scale,
                    diag, c, out);
    return;
  }
  const int64_t n_waves = static_cast<int64_t>(gridDim.x) * (kThreads / 64);
  int64_t pv = wave;
  if (pv >= n_pass) return;
  // the next pass's codes and scales are requested before the current pass is transformed
  uint32_t w;
  float s;
  load(pv, w, s);
  while (true) {
    uint32_t wn;
    float sn;
    load(pv + n_waves < n_pass ? pv + n_waves : pv, wn, sn);
    __builtin_amdgcn_sched_barrier(0);
    decode_pass<false>(w, s, pv, n_vec, row, chunk, sg, sc, dsig[0], dsig[1], dsig[2], dsig[3], cb, scale, diag, c, out);
    pv += n_waves;
    if (pv >= n_pass) break;
    w = wn;
    s = sn;
  }
}

}  // namespace

namespace {
std::atomic<int> g_generic_only{-1};  // -1: not yet read from the environment
}

bool use_specialised_codec() {
  int v = g_generic_only.load(std::memory_order_relaxed);
  if (v < 0) {
    const char* e = std::getenv("AETHERKV_CODEC");
    v = (e && std::strcmp(e, "generic") == 0) ? 1 : 0;
    g_generic_only.store(v, std::memory_order_relaxed);
  }
  return v == 0;
}

}  // namespace aekv

extern "C" int aekv_set_generic_kernels(int generic_only) {
  (void)aekv::use_specialised_codec();
  return aekv::g_generic_only.exchange(generic_only ? 1 : 0);
}

namespace aekv {

// Launches the specialised kernel; returns false when the shape is not the specialised one.
bool launch_encode4_d128_bf16(const void* x, int64_t n_vec, const float* diag, float c, void* codes, float* scale,
                              hipStream_t st) {
  if ((reinterpret_cast<uintptr_t>(x) & 15) || (reinterpret_cast<uintptr_t>(codes) & 15)) return false;
  if (n_vec <= 0) return true;
  const int64_t n_groups = (n_vec + 15) / 16;
  const int64_t blocks = ceil_div(n_groups, kEncThreads / 64);
  if (blocks > 0x7fffffff) return false;
  const float c7 = c * 7.0f;
  hipLaunchKernelGGL(tq_encode4_d128_bf16_kernel, dim3(static_cast<uint32_t>(blocks)), dim3(kEncThreads), 0, st,
                     static_cast<const uint4*>(x), n_vec, diag, c, c7, static_cast<uint4*>(codes), scale);
  return true;
}


namespace {

typedef void (*fast_enc_fn)(const void*, int64_t, const float*, float, float, uint8_t*, float*);

template <int DT>
fast_enc_fn pick_fast(int bits, int d, int& vpw) {
  vpw = d == 128 ? FastEnc<8, 128>::VPW : FastEnc<8, 64>::VPW;
  if (bits == 8) return d == 128 ? tq_encode_fast_kernel<DT, 8, 128> : tq_encode_fast_kernel<DT, 8, 64>;
  if (d == 64) return tq_encode_fast_kernel<DT, 4, 64>;
  if constexpr (DT == AEKV_BF16) return nullptr;  // tq_encode4_d128_bf16_kernel
  else return tq_encode_fast_kernel<DT, 4, 128>;
}

}  // namespace

// fp16 elements from which the fast encode is the faster one: a wave takes 16 or 32 vectors where the generic
// kernel's takes 4 or 8, so that a small call leaves most of the chip idle and waits for one wave's chain.
// Generic / fast, 8-bit D = 128: 100 vectors 2.45 / 3.2 us, 8192 3.5 / 4.4, 16384 4.6 / 4.7, 32768 6.2 / 5.8, 65536
// 10.2 / 7.5; 4-bit D = 64: 100 vectors 2.3 / 2.6, 16384 3.4 / 4.1, 32768 4.3 / 4.4, 65536 6.0 / 5.2.
// (bf16, whose fast kernel needs no conversion, takes it at every size.)
constexpr int64_t kFastF16Elements = int64_t(3) << 20;

// Launches the fast encode; false when the shape, the type, the size or the alignment is not one of its own.
bool launch_encode_fast(const void* x, int x_dtype, int64_t n_vec, int bits, int d, const float* diag, float c,
                        void* codes, float* scale, hipStream_t st) {
  if (!is_aligned(x, 16) || !is_aligned(codes, 16) || (d != 64 && d != 128)) return false;
  if (x_dtype == AEKV_F16 && n_vec * d < kFastF16Elements) return false;
  int vpw = 0;
  const fast_enc_fn kern = x_dtype == AEKV_BF16  ? pick_fast<AEKV_BF16>(bits, d, vpw)
                           : x_dtype == AEKV_F16 ? pick_fast<AEKV_F16>(bits, d, vpw)
                                                 : nullptr;
  if (!kern) return false;
  if (n_vec <= 0) return true;
  const int64_t blocks = ceil_div(ceil_div(n_vec, static_cast<int64_t>(vpw)), kEncThreads / 64);
  if (blocks > 0x7fffffff) return false;
  hipLaunchKernelGGL(kern, dim3(static_cast<uint32_t>(blocks)), dim3(kEncThreads), 0, st, x, n_vec, diag, c,
                     (bits == 8 ? 127.0f : 7.0f) * c, static_cast<uint8_t*>(codes), scale);
  return true;
}

// Launches the specialised decode; returns false when the shape or alignment is not the specialised one.
bool launch_decode4_d128_bf16(const void* codes, const float* scale, int64_t n_vec, const float* diag, float c,
                              void* out, hipStream_t st) {
  if ((reinterpret_cast<uintptr_t>(codes) & 15) || (reinterpret_cast<uintptr_t>(out) & 15) ||
      (reinterpret_cast<uintptr_t>(scale) & 3))
    return false;
  if (n_vec <= 0) return true;
  const int64_t n_pass = (n_vec + 3) / 4;
  // 8 passes per wave once that still gives >= 2048 workgroups (measured 0.64 of HBM peak on cfg2
  // against 0.59 for the loop); smaller inputs keep the loop's wider grid
  const bool per_wave = n_pass >= int64_t(kDecPasses) * (kThreads / 64) * 2048;
  int64_t blocks = ceil_div(per_wave ? ceil_div(n_pass, int64_t(kDecPasses)) : n_pass, kThreads / 64);
  if (!per_wave && blocks > kDecMaxBlocks) blocks = kDecMaxBlocks;
  if (blocks > 0x7fffffff) return false;
  auto kern = per_wave ? tq_decode4_d128_bf16_kernel<kDecPasses> : tq_decode4_d128_bf16_kernel<0>;
  hipLaunchKernelGGL(kern, dim3(static_cast<uint32_t>(blocks)), dim3(kThreads), 0, st,
                     static_cast<const uint32_t*>(codes), scale, n_vec, diag, c, static_cast<uint16_t*>(out));
  return true;
}

}  // namespace aekv
