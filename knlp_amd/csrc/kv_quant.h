// Row quantisers shared by the append kernel and the decode kernels' fused
// append (gfx950).  One (token, head) row of D elements is handled by D/8
// consecutive lanes, eight elements per lane (one 16-byte load, one 4-byte
// store of INT4 codes); a scale group of GS elements spans GS/8 aligned lanes.
// Maxima and minima are taken in-lane first; the symmetric trimmed mean adds
// in a fixed order that the CPU oracle restates (element i adds element
// i + GS/2, then + GS/4, ...), so its wide strides cross lanes first and the
// strides 4, 2, 1 end in-lane.
//
// All quantisation arithmetic is IEEE fp32 without contraction: floor/ceil
// rounding of F:198-202, and round-to-nearest-even fp32 -> fp16 for the stored
// scale / zero-point.  The codes are computed from the fp32 scale; the fp16
// scale is what is stored.  F = fused-quant/fused_int4.v0.1.0.py.
//
// Divisions.  An element's x / scale is a reciprocal y of the scale (v_rcp and
// one Newton step, once per lane) and one residual step, q0 = x y, q = q0 +
// (x - q0 scale) y; amax / 7 and the like take 1 / 7 the same way.  Compared
// with IEEE division on the CPU: every mantissa of the scale, v_rcp results up
// to 2 ulp off, every rounding threshold k - 1/2 (k = 1 .. 128) and x within
// 4 ulps of it (4.8e10 cases) give the same code, and the constant divisors
// the same quotient for every mantissa (a sample of it: test_quotients.py).  Both are exact in the exponent while
// nothing over- or underflows, which `safe` tests for (else the wave divides).
// An IEEE division is about 11 VALU operations, the step 3.
#pragma once

#include "kv_common.h"

namespace knlp {

struct RowDst {
  uint8_t* codes;       // start of this (block, offset, head) row of codes
  uint16_t* scales;     // start of its scale row
  uint16_t* zeros;      // start of its zero-point row (asymmetric only)
};

__device__ __forceinline__ RowDst row_dst(const knlp_kv_plane& P, int64_t blk, int64_t off,
                                          int head) {
  RowDst r;
  const int64_t eb = P.format == KNLP_KV_FP16 ? 2 : 1;   // strides are in elements
  r.codes = static_cast<uint8_t*>(P.data) +
            eb * (blk * P.stride_block + off * P.stride_page + head * P.stride_head);
  r.scales = static_cast<uint16_t*>(P.scales) + blk * P.s_stride_block +
             off * P.s_stride_page + head * P.s_stride_head;
  r.zeros = static_cast<uint16_t*>(P.zeros) + blk * P.z_stride_block + off * P.z_stride_page +
            head * P.z_stride_head;
  return r;
}

template <int CTRL>
__device__ __forceinline__ float dpp_row(float x) {
  return __builtin_bit_cast(
      float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xF, 0xF, false));
}

// Formats and group sizes are compile-time constants (Fixed) in the append
// kernel and uniform run-time values in the decode kernels, where one row per
// sequence is quantised and a copy of the code for each would only be larger.
template <int N>
struct Fixed {
  __device__ constexpr operator int() const { return N; }
};

// OP over the gs/8 lanes of a scale group (any order of the lanes).  Each step
// reads a lane of the other half of a group of 2, 4, 8, 16, whose lanes all
// hold that half's result, so mirrors serve as well as xors.
template <class GS, class OP>
__device__ __forceinline__ float group_reduce(float x, GS gs, OP op) {
  x = op(x, dpp_row<0xB1>(x));                   // quad_perm [1,0,3,2]
  if (gs >= 32) x = op(x, dpp_row<0x4E>(x));     // quad_perm [2,3,0,1]
  if (gs >= 64) x = op(x, dpp_row<0x141>(x));    // row_half_mirror
  if (gs >= 128) x = op(x, dpp_row<0x140>(x));   // row_mirror
  return x;
}

// The trimmed mean's sum, strides GS/2 .. 8 across lanes, then 4, 2, 1.
template <class GS>
__device__ __forceinline__ float group_tree_sum(float (&b)[8], GS gs) {
#pragma clang fp contract(off)
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    if (gs >= 128) b[e] = b[e] + shfl_xor(b[e], 8);
    if (gs >= 64) b[e] = b[e] + shfl_xor(b[e], 4);
    if (gs >= 32) b[e] = b[e] + dpp_row<0x4E>(b[e]);
    b[e] = b[e] + dpp_row<0xB1>(b[e]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) b[e] = b[e] + b[e + 4];
  b[0] = b[0] + b[2];
  b[1] = b[1] + b[3];
  return b[0] + b[1];
}

// x / C, correctly rounded for finite x in the ranges that `safe` admits.
template <int C>
__device__ __forceinline__ float div_const(float x) {
#pragma clang fp contract(off)
  constexpr float c = C, rc = 1.0f / C;
  const float q0 = x * rc;
  return __builtin_fmaf(__builtin_fmaf(-q0, c, x), rc, q0);
}

// The scale range / C of a group, and x[e] / scale rounded half away from zero
// (F:198-202) and cut to lo .. hi in place.  `top`: no |x| of the group is
// larger.
template <int C, bool SIGNED>
__device__ __forceinline__ float scale_and_round(float (&x)[8], float range, float top, float lo,
                                                 float hi) {
#pragma clang fp contract(off)
  float scale = div_const<C>(range);
  const float y0 = __builtin_amdgcn_rcpf(scale);
  const float y = __builtin_fmaf(__builtin_fmaf(-scale, y0, 1.0f), y0, y0);
  const bool safe = scale > 0x1p-60f && scale < 0x1p60f && top * y < 0x1p60f;
  if (__all(safe)) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float q0 = x[e] * y;
      const float t = __builtin_fmaf(__builtin_fmaf(-q0, scale, x[e]), y, q0);
      x[e] = SIGNED ? __builtin_copysignf(floorf(fabsf(t) + 0.5f), t) : floorf(t + 0.5f);
    }
  } else {
    scale = range / static_cast<float>(C);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = round_half_away(x[e] / scale);
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = fmaxf(fminf(x[e], hi), lo);   // a NaN becomes hi
  return scale;
}

// What a lane's 8 elements become: the codes (INT4: w[0], INT8: w[0 .. 1],
// fp16: the source words) and its group's scale and zero-point.  Separate
// from the stores so that the slot's load, which only the stores need, is in
// flight under the row's load and its arithmetic.
struct Quantised {
  uint32_t w[4];
  uint16_t scale, zero;
};

// n0 .. n7 (whole values 0 .. 15) as 8 nibbles, element 0 lowest.
__device__ __forceinline__ uint32_t pack_nibbles(const float (&n)[8]) {
  uint32_t w = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    w |= static_cast<uint32_t>(__builtin_fmaf(n[2 * i + 1], 16.0f, n[2 * i])) << (8 * i);
  return w;
}

template <class GS>
__device__ __forceinline__ void quant_int4_asym(float (&x)[8], GS gs, Quantised& o) {
#pragma clang fp contract(off)
  float mn = x[0], mx = x[0];
#pragma unroll
  for (int e = 1; e < 8; ++e) {
    mn = fminf(mn, x[e]);
    mx = fmaxf(mx, x[e]);
  }
  mn = group_reduce(mn, gs, [](float a, float b) { return fminf(a, b); });
  mx = group_reduce(mx, gs, [](float a, float b) { return fmaxf(a, b); });
  const float rng = fmaxf(mx - mn, 1e-8f);          // F:314
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = x[e] - mn;
  const float scale = scale_and_round<15, false>(x, rng, rng, 0.0f, 15.0f);   // F:315
  o.w[0] = pack_nibbles(x);
  o.scale = float_to_half_bits(scale);
  o.zero = float_to_half_bits(mn);
}

template <class GS>
__device__ __forceinline__ void quant_int4_sym(float (&x)[8], GS gs, float clip_ratio,
                                               Quantised& o) {
#pragma clang fp contract(off)
  float amax = fabsf(x[0]);
#pragma unroll
  for (int e = 1; e < 8; ++e) amax = fmaxf(amax, fabsf(x[e]));
  amax = group_reduce(amax, gs, [](float a, float b) { return fmaxf(a, b); });
  const float top = amax;
  amax = fmaxf(amax, 1e-8f);                         // F:336
  if (clip_ratio > 0.0f) {                           // F:342-347
    float b[8];
    int below = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const bool lt = fabsf(x[e]) < amax;
      b[e] = lt ? fabsf(x[e]) : 0.0f;
      below += lt;                                   // the compare's carry: one operation
    }
    // (a whole number, at most 128: exact as a float in any order)
    const float c = group_reduce(static_cast<float>(below), gs,
                                 [](float u, float v) { return u + v; });
    const float sum = group_tree_sum(b, gs);
    const float cnt = fmaxf(c, 1.0f);
    const float tmean = sum / cnt;
    const float clip = tmean * clip_ratio;
    amax = fminf(amax, fmaxf(clip, 1e-8f));
  }
  const float scale = scale_and_round<7, true>(x, amax, top, -8.0f, 7.0f);    // F:348
#pragma unroll
  for (int e = 0; e < 8; ++e) x[e] = x[e] + 8.0f;
  o.w[0] = pack_nibbles(x);
  o.scale = float_to_half_bits(scale);
}

template <class GS>
__device__ __forceinline__ void quant_int8(float (&x)[8], GS gs, Quantised& o) {
#pragma clang fp contract(off)
  float amax = fabsf(x[0]);
#pragma unroll
  for (int e = 1; e < 8; ++e) amax = fmaxf(amax, fabsf(x[e]));
  amax = group_reduce(amax, gs, [](float a, float b) { return fmaxf(a, b); });
  const float top = amax;
  amax = fmaxf(amax, 1e-8f);                         // F:1276
  const float scale = scale_and_round<127, true>(x, amax, top, -128.0f, 127.0f);   // F:1277
  o.w[0] = o.w[1] = 0;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    o.w[e / 4] |= (static_cast<uint32_t>(static_cast<int>(x[e])) & 0xFFu) << (8 * (e % 4));
  o.scale = float_to_half_bits(scale);
}

// This lane's 8 elements of a source row (a: the row's elements start on 16
// bytes, uniform; else on 4).
__device__ __forceinline__ uint4 load_row8(const uint16_t* src, int lane, bool a) {
  const uint16_t* p = src + 8 * lane;
  if (a) return *reinterpret_cast<const uint4*>(p);
  const uint32_t* d = reinterpret_cast<const uint32_t*>(p);
  return make_uint4(d[0], d[1], d[2], d[3]);
}

__device__ __forceinline__ bool src_aligned(const uint16_t* src, int64_t st, int64_t sh) {
  return ((reinterpret_cast<uintptr_t>(src) | static_cast<uintptr_t>(2 * (st | sh))) & 15) == 0;
}

// Quantise this lane's 8 elements `w` (raw 16-bit) of one row to `format` with
// group size gs; the row's lanes call it together.
template <class F, class GS>
__device__ __forceinline__ Quantised quant_row(const uint4& w, bool bf16, F format, GS gs,
                                               float clip_ratio) {
  Quantised o{{w.x, w.y, w.z, w.w}, 0, 0};
  if (format == KNLP_KV_FP16) return o;              // plain copy (fp16 source only)
  float x[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (bf16) {
      x[2 * i] = __builtin_bit_cast(float, o.w[i] << 16);
      x[2 * i + 1] = __builtin_bit_cast(float, o.w[i] & 0xFFFF0000u);
    } else {
      x[2 * i] = half_bits_to_float(static_cast<uint16_t>(o.w[i]));
      x[2 * i + 1] = half_bits_to_float(static_cast<uint16_t>(o.w[i] >> 16));
    }
  }
  if (format == KNLP_KV_INT4_ASYM)
    quant_int4_asym(x, gs, o);
  else if (format == KNLP_KV_INT4_SYM)
    quant_int4_sym(x, gs, clip_ratio, o);
  else
    quant_int8(x, gs, o);
  return o;
}

// Whether a plane's rows of codes start on a multiple of `a` bytes (uniform);
// they may start at any byte (INT4), 2 (INT8) or 4 bytes (fp16).
__device__ __forceinline__ bool rows_aligned(const knlp_kv_plane& P, int eb, uintptr_t a) {
  const uintptr_t m = reinterpret_cast<uintptr_t>(P.data) |
                      static_cast<uintptr_t>(eb * (P.stride_block | P.stride_page | P.stride_head));
  return (m & (a - 1)) == 0;
}

// Store lane `lane`'s part of the row at `r`.
template <class F, class GS>
__device__ __forceinline__ void store_row(const Quantised& o, const knlp_kv_plane& P, F format,
                                          GS gs, const RowDst& r, int lane) {
  if (format == KNLP_KV_FP16) {
    if (rows_aligned(P, 2, 16)) {
      reinterpret_cast<uint4*>(r.codes)[lane] = make_uint4(o.w[0], o.w[1], o.w[2], o.w[3]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) reinterpret_cast<uint32_t*>(r.codes)[4 * lane + i] = o.w[i];
    }
    return;
  }
  if (format == KNLP_KV_INT8_SYM) {
    if (rows_aligned(P, 1, 8)) {
      reinterpret_cast<uint2*>(r.codes)[lane] = make_uint2(o.w[0], o.w[1]);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        reinterpret_cast<uint16_t*>(r.codes)[4 * lane + i] =
            static_cast<uint16_t>(o.w[i / 2] >> (16 * (i % 2)));
    }
  } else if (rows_aligned(P, 1, 4)) {
    reinterpret_cast<uint32_t*>(r.codes)[lane] = o.w[0];
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) r.codes[4 * lane + i] = static_cast<uint8_t>(o.w[0] >> (8 * i));
  }
  const int per = gs / 8;                            // lanes of a group
  if ((lane & (per - 1)) == 0) {
    const int g = lane >> __builtin_ctz(per);
    r.scales[g] = o.scale;
    if (format == KNLP_KV_INT4_ASYM) r.zeros[g] = o.zero;
  }
}

}  // namespace knlp
