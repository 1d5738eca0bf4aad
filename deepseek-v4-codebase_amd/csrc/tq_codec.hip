// TurboQuant ("PolarQuant") codec for gfx950: normalised Walsh-Hadamard transform, absmax
// 8/4-bit quantisation with nibble packing, and the inverse.
//
// Reference: aether_2b/turbo_quant.py:49-76 (_wht), :127-166 (encode), :168-211 (decode).
// Bit-exact with the reference: every fp32 operation of the reference is performed once, in the
// same order, with the same rounding (the library is built with -ffp-contract=off; the only FMAs
// are the explicit fmaf(a, +-1, b) below, whose product is exact).
//
// Layout: a vector of D elements is spread over LPV = D/EPL lanes, EPL = min(D, 8) consecutive
// elements per lane, so one lane's load is one 16-byte access for bf16 and a wave reads 64*16
// contiguous bytes.  Butterfly stages h = 1..EPL/2 run inside the lane; stages h = EPL..D/2 pair
// lane l with lane l ^ (h/EPL) (DPP for 1/2, ds_swizzle for 4/8/16, ds_bpermute for 32).  The
// butterfly result for the lane holding the upper element is partner - mine, for the lower one
// mine + partner; both are one fmaf(mine, +-1, partner).
#include "tq_device.h"

namespace aekv {
namespace {

constexpr int kThreads = 256;
enum { kModeWht = 0, kModeEnc4 = 4, kModeEnc8 = 8 };

// Elements per lane of a decode: 8, but 4 for fp32 outputs of 16 to 256 elements, one 16-byte store per
// lane and 1 KB contiguous per wave (with 8 the two halves of a lane's store are 32 bytes apart in each
// instruction).  Measured on 100 M elements, 8-bit D = 64 / 4-bit D = 64 / 8-bit D = 128: 95 / 108 / 101 us
// against 100 / 114 / 108 with 8; 131072 vectors of 64 9.1 against 11.2 us.  (The same split of an
// encode's loads is slower, 112 to 131 us against 108 to 111: one more lane exchange per element.)
template <int ODT, int D>
constexpr int kDecEpl = ODT == AEKV_F32 && D >= 16 && D <= 256 ? 4 : (D < 8 ? D : 8);

// Forward kernel: WHT (fp32 out), or encode to 8/4-bit codes + fp32 scale.
template <int DT, int D, int MODE>
__global__ __launch_bounds__(kThreads) void tq_forward_kernel(const void* __restrict__ x, int64_t n_vec,
                                                              const float* __restrict__ diag, float c,
                                                              void* __restrict__ out,
                                                              float* __restrict__ out_scale) {
  constexpr int EPL = D < 8 ? D : 8;
  constexpr int LPV = D / EPL;
  constexpr int VPW = 64 / LPV;
  const int lane = threadIdx.x & 63;
  const int sub = lane % LPV;
  const int slot = lane / LPV;

  float dg[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) dg[e] = MODE == kModeWht ? 1.0f : diag[sub * EPL + e];

  const int64_t wave = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) >> 6;
  const int64_t n_waves = (static_cast<int64_t>(gridDim.x) * kThreads) >> 6;
  for (int64_t base = wave * VPW; base < n_vec; base += n_waves * VPW) {
    const int64_t v = base + slot;
    const bool ok = v < n_vec;
    float a[EPL];
    load_elems<DT, EPL>(x, v * D + sub * EPL, ok, a);
    if constexpr (MODE == kModeWht) {
      wht_butterflies<D, EPL, true>(a, sub);
      if (ok) {
        float* o = static_cast<float*>(out) + v * D + sub * EPL;
#pragma unroll
        for (int e = 0; e < EPL; ++e) o[e] = a[e] * c;  // * fp32(d ** -0.5)
      }
    } else {
#pragma unroll
      for (int e = 0; e < EPL; ++e) a[e] = a[e] * dg[e];  // x.float() * diag (exact sign flip)
      constexpr int BITS = MODE == kModeEnc8 ? 8 : 4;
      constexpr int NB = BITS == 8 ? EPL : EPL / 2;
      float m;
      const Bytes<NB> w = encode_lane<BITS, D, true>(a, sub, c, &m);
      if (ok) {
        if (sub == 0) out_scale[v] = m / (BITS == 8 ? 127.0f : 7.0f);
        *reinterpret_cast<Bytes<NB>*>(static_cast<uint8_t*>(out) + v * (BITS == 8 ? D : D / 2) + sub * NB) = w;
      }
    }
  }
}

// Stores a lane's EPL decoded elements at o, rounded to ODT; NT: past the caches.
template <int ODT, int EPL, bool NT>
__device__ __forceinline__ void store_decoded(uint8_t* o, const float (&a)[EPL]) {
  constexpr int NB = EPL * (ODT == AEKV_F32 ? 4 : 2);
  Bytes<NB> w;
  if constexpr (ODT == AEKV_F32) {
    __builtin_memcpy(w.b, a, NB);
  } else if constexpr (ODT == AEKV_BF16 && EPL >= 2) {
    uint32_t wv[EPL / 2];
#pragma unroll
    for (int i = 0; i < EPL / 2; ++i) wv[i] = pack_bf16x2(a[2 * i], a[2 * i + 1]);
    __builtin_memcpy(w.b, wv, NB);
  } else {
#pragma unroll
    for (int e = 0; e < EPL; ++e) {
      const uint16_t h = static_cast<uint16_t>(ODT == AEKV_BF16 ? pack_bf16x2(a[e], 0.0f) & 0xffffu : f32_to_f16_bits(a[e]));
      __builtin_memcpy(w.b + 2 * e, &h, 2);
    }
  }
  if constexpr (NT) {
    static_assert(NB == 16, "one 16-byte store per lane");
    typedef __attribute__((ext_vector_type(4))) uint32_t u32x4_t;
    __builtin_nontemporal_store(__builtin_bit_cast(u32x4_t, w), reinterpret_cast<u32x4_t*>(o));
  } else if constexpr (NB <= 16) {
    *reinterpret_cast<Bytes<NB>*>(o) = w;
  } else {
    reinterpret_cast<Bytes<16>*>(o)[0] = *reinterpret_cast<Bytes<16>*>(w.b);
    reinterpret_cast<Bytes<16>*>(o)[1] = *reinterpret_cast<Bytes<16>*>(w.b + 16);
  }
}

// Decode kernel: codes * scale -> WHT -> * diag -> out dtype.  PP == 0: a grid-stride loop.  PP > 0: PP
// consecutive groups of 64 / LPV vectors per wave, all their loads issued first, no loop (the launch covers
// every group); NT: with stores past the caches.
template <int BITS, int D, int ODT, int PP, bool NT>
__global__ __launch_bounds__(kThreads) void tq_decode_kernel(const void* __restrict__ codes,
                                                             const float* __restrict__ scale, int64_t n_vec,
                                                             const float* __restrict__ diag, float c,
                                                             void* __restrict__ out) {
  constexpr int EPL = kDecEpl<ODT, D>;
  constexpr int LPV = D / EPL;
  constexpr int VPW = 64 / LPV;
  constexpr int RB = BITS == 8 ? D : D / 2, OB = D * (ODT == AEKV_F32 ? 4 : 2);  // bytes of a vector
  const int lane = threadIdx.x & 63;
  const int sub = lane % LPV;
  const int slot = lane / LPV;
  const uint8_t* cb = static_cast<const uint8_t*>(codes);
  uint8_t* ob = static_cast<uint8_t*>(out) + sub * (OB / LPV);

  float dg[EPL];
#pragma unroll
  for (int e = 0; e < EPL; ++e) dg[e] = diag[sub * EPL + e];

  const int64_t wave = (static_cast<int64_t>(blockIdx.x) * kThreads + threadIdx.x) >> 6;
  if constexpr (PP > 0) {
    using LC = LaneCodes<BITS, EPL>;
    const int64_t v0 = wave * (PP * VPW) + slot;
    typename LC::type w[PP];
    float s[PP];
#pragma unroll
    for (int i = 0; i < PP; ++i) {  // (lanes past the end decode row 0, never stored)
      const int64_t v = v0 + i * VPW, vr = v < n_vec ? v : 0;
      w[i] = *reinterpret_cast<const typename LC::type*>(cb + vr * RB + sub * LC::NB);
      s[i] = scale[vr];
    }
#pragma unroll
    for (int i = 0; i < PP; ++i) {
      float a[EPL];
      decode_lane_bytes<BITS, D, true, EPL>(w[i], s[i], sub, dg, c, a);
      if (v0 + i * VPW < n_vec) store_decoded<ODT, EPL, NT>(ob + (v0 + i * VPW) * OB, a);
    }
    return;
  }
  const int64_t n_waves = (static_cast<int64_t>(gridDim.x) * kThreads) >> 6;
  for (int64_t base = wave * VPW; base < n_vec; base += n_waves * VPW) {
    const int64_t v = base + slot;
    const bool ok = v < n_vec;
    float a[EPL];
    // inactive lanes decode row 0 so every lane joins the cross-lane butterflies
    const int64_t vr = ok ? v : 0;
    decode_lane<BITS, D, true, EPL>(cb + vr * RB, scale[vr], sub, dg, c, a);
    if (ok) store_decoded<ODT, EPL, false>(ob + v * OB, a);
  }
}

int64_t grid_for(int64_t n_vec, int d, int epl) {
  const int vpb = (64 / (d / epl)) * (kThreads / 64);  // vectors per block per iteration
  int64_t g = ceil_div(n_vec, vpb);
  if (g > 65536) g = 65536;
  return g < 1 ? 1 : g;
}

typedef void (*fwd_fn)(const void*, int64_t, const float*, float, void*, float*);
typedef void (*dec_fn)(const void*, const float*, int64_t, const float*, float, void*);

template <int DT, int MODE>
fwd_fn pick_fwd(int d) {
  switch (d) {
    case 1: return MODE == kModeEnc4 ? nullptr : tq_forward_kernel<DT, 1, MODE>;
    case 2: return tq_forward_kernel<DT, 2, MODE>;
    case 4: return tq_forward_kernel<DT, 4, MODE>;
    case 8: return tq_forward_kernel<DT, 8, MODE>;
    case 16: return tq_forward_kernel<DT, 16, MODE>;
    case 32: return tq_forward_kernel<DT, 32, MODE>;
    case 64: return tq_forward_kernel<DT, 64, MODE>;
    case 128: return tq_forward_kernel<DT, 128, MODE>;
    case 256: return tq_forward_kernel<DT, 256, MODE>;
    case 512: return tq_forward_kernel<DT, 512, MODE>;
    default: return nullptr;
  }
}

template <int MODE>
fwd_fn pick_fwd_dt(int dt, int d) {
  if (dt == AEKV_F32) return pick_fwd<AEKV_F32, MODE>(d);
  if (dt == AEKV_F16) return pick_fwd<AEKV_F16, MODE>(d);
  return pick_fwd<AEKV_BF16, MODE>(d);
}

template <int BITS, int ODT>
dec_fn pick_dec(int d) {
  switch (d) {
    case 1: return BITS == 4 ? nullptr : tq_decode_kernel<BITS, 1, ODT, 0, false>;
    case 2: return tq_decode_kernel<BITS, 2, ODT, 0, false>;
    case 4: return tq_decode_kernel<BITS, 4, ODT, 0, false>;
    case 8: return tq_decode_kernel<BITS, 8, ODT, 0, false>;
    case 16: return tq_decode_kernel<BITS, 16, ODT, 0, false>;
    case 32: return tq_decode_kernel<BITS, 32, ODT, 0, false>;
    case 64: return tq_decode_kernel<BITS, 64, ODT, 0, false>;
    case 128: return tq_decode_kernel<BITS, 128, ODT, 0, false>;
    case 256: return tq_decode_kernel<BITS, 256, ODT, 0, false>;
    case 512: return tq_decode_kernel<BITS, 512, ODT, 0, false>;
    default: return nullptr;
  }
}

constexpr int kDecPasses = 4;
// Codes and output together from which a decode streams (D = 64 and 128), and from which its stores go past
// the caches.  Measured on codes coming round from two sets, loop / streamed / streamed past the caches, the
// decode alone and with a caller's pass that reads the decoded tensor (a product with four columns):
//   fp32, 8-bit D = 128   170 MB 29 / 27 / 26 and 69 / 66 / 74 us    300 MB 60 / 47 / 44 and 121 / 108 / 118
//                         400 MB 82 / 71 / 57 and 181 / 167 / 157    600 MB 120 / 105 / 86 and 261 / 239 / 227
//   bf16, 8-bit D = 128   170 MB 30 / 27 / 27 and 71 / 70 / 78 us    300 MB 59 / 50 / 46 and 115 / 107 / 123
//                         400 MB 80 / 70 / 67 and 162 / 153 / 150    600 MB 113 / 103 / 101 and 249 / 240 / 238
// Up to about 1.5 times the Infinity Cache a reader gains more from an output that is still there than the
// decode loses by it.  Below 160 MB the loop and the streams are within the noise of each other.
constexpr int64_t kDecStreamBytes = 160000000;
constexpr int64_t kDecPastCachesBytes = 400000000;

template <int BITS, int ODT, bool NT>
dec_fn pick_dec_stream(int d) {
  return d == 128 ? tq_decode_kernel<BITS, 128, ODT, kDecPasses, NT> : tq_decode_kernel<BITS, 64, ODT, kDecPasses, NT>;
}

template <int BITS, bool NT>
dec_fn pick_dec_stream_dt(int odt, int d) {
  if (odt == AEKV_F32) return pick_dec_stream<BITS, AEKV_F32, NT>(d);
  if (odt == AEKV_F16) return pick_dec_stream<BITS, AEKV_F16, NT>(d);
  return pick_dec_stream<BITS, AEKV_BF16, NT>(d);
}

template <int BITS>
dec_fn pick_dec_dt(int odt, int d) {
  if (odt == AEKV_F32) return pick_dec<BITS, AEKV_F32>(d);
  if (odt == AEKV_F16) return pick_dec<BITS, AEKV_F16>(d);
  return pick_dec<BITS, AEKV_BF16>(d);
}

int check_vec_dim(int32_t d) {
  if (!is_pow2(d)) return fail(AEKV_ERR_VALUE, "WHT requires last dim to be a power of 2, got %d", d);
  if (d > 512) return fail(AEKV_ERR_UNSUPPORTED, "vector length %d exceeds the supported maximum 512", d);
  return AEKV_OK;
}

}  // namespace
}  // namespace aekv

using namespace aekv;

extern "C" int aekv_wht(const void* x, int32_t x_dtype, int64_t n_vec, int32_t d, float* out, void* stream) {
  if (int rc = check_vec_dim(d)) return rc;
  if (!is_float_dtype(x_dtype)) return fail(AEKV_ERR_DTYPE, "aekv_wht: x_dtype %d is not f32/f16/bf16", x_dtype);
  if (n_vec < 0) return fail(AEKV_ERR_SHAPE, "aekv_wht: n_vec %lld < 0", (long long)n_vec);
  if (n_vec == 0) return AEKV_OK;
  if (!x || !out) return fail(AEKV_ERR_VALUE, "aekv_wht: null pointer");
  const int epl = d < 8 ? d : 8;
  if (!is_aligned(x, epl * dtype_size(x_dtype) > 16 ? 16 : epl * dtype_size(x_dtype)) || !is_aligned(out, 4))
    return fail(AEKV_ERR_ALIGN, "aekv_wht: misaligned pointer");
  fwd_fn fn = pick_fwd_dt<kModeWht>(x_dtype, d);
  hipLaunchKernelGGL(fn, dim3(static_cast<uint32_t>(grid_for(n_vec, d, d < 8 ? d : 8))), dim3(kThreads), 0, as_stream(stream), x,
                     n_vec, nullptr, wht_scale(d), static_cast<void*>(out), nullptr);
  return check_launch("aekv_wht");
}

extern "C" int aekv_tq_encode(const void* x, int32_t x_dtype, int64_t n_vec, int32_t d, int32_t bits,
                              const float* diag, void* codes, float* scale, void* stream) {
  if (bits != 4 && bits != 8) return fail(AEKV_ERR_VALUE, "bits must be 4 or 8, got %d", bits);
  if (int rc = check_vec_dim(d)) return rc;
  if (bits == 4 && d < 2) return fail(AEKV_ERR_VALUE, "4-bit packing needs an even last dim, got %d", d);
  if (!is_float_dtype(x_dtype)) return fail(AEKV_ERR_DTYPE, "aekv_tq_encode: x_dtype %d is not f32/f16/bf16", x_dtype);
  if (n_vec < 0) return fail(AEKV_ERR_SHAPE, "aekv_tq_encode: n_vec %lld < 0", (long long)n_vec);
  if (n_vec == 0) return AEKV_OK;
  if (!x || !diag || !codes || !scale) return fail(AEKV_ERR_VALUE, "aekv_tq_encode: null pointer");
  const int epl = d < 8 ? d : 8;
  const size_t in_al = epl * dtype_size(x_dtype) > 16 ? 16 : epl * dtype_size(x_dtype);
  const size_t out_al = bits == 8 ? epl : epl / 2;
  if (!is_aligned(x, in_al) || !is_aligned(codes, out_al) || !is_aligned(scale, 4) || !is_aligned(diag, 4))
    return fail(AEKV_ERR_ALIGN, "aekv_tq_encode: misaligned pointer (x needs %zu, codes %zu bytes)", in_al, out_al);
  if (bits == 4 && d == 128 && x_dtype == AEKV_BF16 && use_specialised_codec() &&
      launch_encode4_d128_bf16(x, n_vec, diag, wht_scale(d), codes, scale, as_stream(stream)))
    return check_launch("aekv_tq_encode");
  if (use_specialised_codec() &&
      launch_encode_fast(x, x_dtype, n_vec, bits, d, diag, wht_scale(d), codes, scale, as_stream(stream)))
    return check_launch("aekv_tq_encode");
  fwd_fn fn = bits == 8 ? pick_fwd_dt<kModeEnc8>(x_dtype, d) : pick_fwd_dt<kModeEnc4>(x_dtype, d);
  hipLaunchKernelGGL(fn, dim3(static_cast<uint32_t>(grid_for(n_vec, d, d < 8 ? d : 8))), dim3(kThreads), 0, as_stream(stream), x,
                     n_vec, diag, wht_scale(d), codes, scale);
  return check_launch("aekv_tq_encode");
}

extern "C" int aekv_tq_decode(const void* codes, const float* scale, int64_t n_vec, int32_t d, int32_t bits,
                              const float* diag, void* out, int32_t out_dtype, void* stream) {
  if (bits != 4 && bits != 8) return fail(AEKV_ERR_VALUE, "bits must be 4 or 8, got %d", bits);
  if (int rc = check_vec_dim(d)) return rc;
  if (bits == 4 && d < 2) return fail(AEKV_ERR_VALUE, "4-bit packing needs an even last dim, got %d", d);
  if (!is_float_dtype(out_dtype)) return fail(AEKV_ERR_DTYPE, "aekv_tq_decode: out_dtype %d is not f32/f16/bf16", out_dtype);
  if (n_vec < 0) return fail(AEKV_ERR_SHAPE, "aekv_tq_decode: n_vec %lld < 0", (long long)n_vec);
  if (n_vec == 0) return AEKV_OK;
  if (!codes || !scale || !diag || !out) return fail(AEKV_ERR_VALUE, "aekv_tq_decode: null pointer");
  const int epl = d < 8 ? d : 8;
  const size_t in_al = bits == 8 ? epl : epl / 2;
  const size_t out_al = epl * dtype_size(out_dtype) > 16 ? 16 : epl * dtype_size(out_dtype);
  if (!is_aligned(codes, in_al) || !is_aligned(out, out_al) || !is_aligned(scale, 4) || !is_aligned(diag, 4))
    return fail(AEKV_ERR_ALIGN, "aekv_tq_decode: misaligned pointer (codes needs %zu, out %zu bytes)", in_al, out_al);
  if (bits == 4 && d == 128 && out_dtype == AEKV_BF16 && use_specialised_codec() &&
      launch_decode4_d128_bf16(codes, scale, n_vec, diag, wht_scale(d), out, as_stream(stream)))
    return check_launch("aekv_tq_decode");
  const int lane_el = out_dtype == AEKV_F32 && d >= 16 && d <= 256 ? 4 : epl;  // kDecEpl
  const int64_t blocks = ceil_div(n_vec, static_cast<int64_t>(kDecPasses) * (kThreads / 64) * (64 / (d / lane_el)));
  const int64_t bytes = n_vec * d * static_cast<int64_t>(dtype_size(out_dtype)) + n_vec * d * bits / 8;
  if (use_specialised_codec() && (d == 64 || d == 128) && bytes >= kDecStreamBytes && blocks <= 0x7fffffff) {
    const bool past = bytes >= kDecPastCachesBytes;
    dec_fn fn = bits == 8 ? (past ? pick_dec_stream_dt<8, true>(out_dtype, d) : pick_dec_stream_dt<8, false>(out_dtype, d))
                          : (past ? pick_dec_stream_dt<4, true>(out_dtype, d) : pick_dec_stream_dt<4, false>(out_dtype, d));
    hipLaunchKernelGGL(fn, dim3(static_cast<uint32_t>(blocks)), dim3(kThreads), 0, as_stream(stream), codes, scale, n_vec,
                       diag, wht_scale(d), out);
    return check_launch("aekv_tq_decode");
  }
  dec_fn fn = bits == 8 ? pick_dec_dt<8>(out_dtype, d) : pick_dec_dt<4>(out_dtype, d);
  hipLaunchKernelGGL(fn, dim3(static_cast<uint32_t>(grid_for(n_vec, d, lane_el))), dim3(kThreads), 0, as_stream(stream),
                     codes, scale, n_vec, diag, wht_scale(d), out);
  return check_launch("aekv_tq_decode");
}
