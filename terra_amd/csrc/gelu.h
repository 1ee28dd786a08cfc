// Exact GELU of bf16 values by table, shared by the MLP kernels:
// nn.GELU() (0.5 x (1 + erf(x / sqrt 2)), models/mlp.py:152-172) applied to a
// bf16 tensor, i.e. computed in fp32 and rounded to bf16.
#pragma once

#include "common.h"

namespace terra {
namespace {

// GELU of a bf16 input by table.  The fc1 output is rounded to bf16 before
// the activation, so GELU sees one of 2^16 inputs; for 2^-22 <= |x| < 32 the
// bf16 result is read from a table that each workgroup fills at start with
// the module's formula, 0.5 x (1 + erf(x / sqrt 2)) in fp32 rounded to bf16
// (the value PyTorch's GPU kernel computes for a bf16 input).  Outside that
// range the bf16 result has a closed form: 0.5 x for |x| < 2^-22 (the fp32
// value is 0.5 x (1 + d) with |d| < 2^-22, and 0.5 x is a bf16 value, so it
// rounds to 0.5 x); x for x >= 32 (erf = 1 in fp32); -0 for x <= -32 (erf =
// -1 in fp32); -inf gives NaN (-inf * 0) and NaN stays NaN.
constexpr uint32_t kGeluLo = 0x3480;   // bf16 bits of 2^-22
constexpr uint32_t kGeluHi = 0x4200;   // bf16 bits of 32
constexpr int kGeluSpan = (int)(kGeluHi - kGeluLo);  // 3456 entries per sign
constexpr int kGeluBytes = 2 * kGeluSpan * 2;

// Fills the GELU table (see kGeluLo): entry sign * kGeluSpan + (mag - kGeluLo).
__device__ __forceinline__ void gelu_table_fill(uint16_t* table, int tid, int nthreads) {
  for (int e = tid; e < 2 * kGeluSpan; e += nthreads) {
    const uint32_t sign = e >= kGeluSpan ? 0x8000u : 0u;
    const uint32_t bits = sign | (kGeluLo + (uint32_t)(e - (sign ? kGeluSpan : 0)));
    const float x = bf16_bits_to_f32((uint16_t)bits);
    table[e] = f32_to_bf16_bits(x * 0.5f * (1.f + erff(x * 0.70710678118654752f)));
  }
}

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));

// Table lookups for the two bf16 values of `p` (two GELU results, packed the
// same way), with packed 16-bit index arithmetic.  `dmax` collects mag - kGeluLo
// per half (wrapping below kGeluLo): a value >= kGeluSpan marks an input
// outside the table, whose lookup here is clamped and wrong.
__device__ __forceinline__ uint32_t gelu_pair_table(uint32_t p, const uint16_t* table, u16x2& dmax) {
  const u16x2 v = __builtin_bit_cast(u16x2, p);
  const u16x2 d = (v & (u16x2)0x7fff) - (u16x2)(uint16_t)kGeluLo;
  dmax = __builtin_elementwise_max(dmax, d);
  const u16x2 idx = __builtin_elementwise_min(d, (u16x2)(uint16_t)(kGeluSpan - 1)) + (v >> 15) * (u16x2)(uint16_t)kGeluSpan;
  const u16x2 off = idx << 1;  // byte offsets (< 2^15)
  const uint8_t* t = reinterpret_cast<const uint8_t*>(table);
  return (uint32_t)*reinterpret_cast<const uint16_t*>(t + off.x) |
         ((uint32_t)*reinterpret_cast<const uint16_t*>(t + off.y) << 16);
}

// bf16 bits of GELU(x) for the bf16 bits of any x (the table or the closed forms).
__device__ __forceinline__ uint32_t gelu_bf16(uint32_t b, const uint16_t* table) {
  const uint32_t mag = b & 0x7fffu;
  const uint32_t sign = b >> 15;
  const uint32_t d = mag - kGeluLo;  // wraps below kGeluLo
  const uint32_t idx = (d < (uint32_t)kGeluSpan ? d : 0u) + (sign ? kGeluSpan : 0);
  const uint32_t tab = table[idx];
  const uint32_t half = __builtin_bit_cast(uint16_t, (__bf16)(0.5f * bf16_bits_to_f32((uint16_t)b)));
  const uint32_t big = b == 0xff80u ? 0x7fc0u : ((sign && mag <= 0x7f80u) ? 0x8000u : b);
  return mag < kGeluLo ? half : (mag < kGeluHi ? tab : big);
}

// d/dh GELU(h) in fp32 (the erf form's exact derivative, before the
// multiplication by the incoming gradient).
__device__ __forceinline__ float gelu_slope(float h) {
  constexpr float kAlpha = 0.70710678118654752f;  // 1 / sqrt(2)
  constexpr float kBeta = 0.39894228040143268f;   // 1 / sqrt(2 pi)
  const float cdf = 0.5f * (1.f + erff(h * kAlpha));
  const float pdf = expf(-0.5f * h * h) * kBeta;
  return cdf + h * pdf;
}

// The GELU's slope Phi(h) + h phi(h) of a bf16 h: an fp32 table for 2^-12 <=
// |h| < 16 filled with gelu_slope; from 16 on the last entries (1, and 0 for
// negative h: exp(-127) is 0 in fp32) are the limits; below 2^-12 the slope is
// 1/2 + 2 phi(0) h to fp32 rounding (the next term, -2/3 phi(0) h^3, is below
// 2^-37).  The table ends where the slope does: with 2^-13 .. 8 in the same
// 16 KB (all that the linear kernel's LDS leaves) every h <= -8 kept the slope
// of -7.97, -5e-14.  +-inf and NaN give NaN (inf * 0).
constexpr uint32_t kSlopeTabLo = 0x3980;  // bf16 bits of 2^-12
constexpr uint32_t kSlopeTabHi = 0x4180;  // bf16 bits of 16
constexpr int kSlopeTabSpan = (int)(kSlopeTabHi - kSlopeTabLo);
constexpr int kSlopeTabBytes = 2 * kSlopeTabSpan * 4;

typedef uint32_t gelu_u32x4 __attribute__((ext_vector_type(4)));

// Slope of any bf16 value (bits b): the table or the closed forms.
__device__ __forceinline__ float slope_any(uint32_t b, const uint8_t* table) {
  const uint32_t mag = b & 0x7fffu, sign = b >> 15;
  const uint32_t d = mag - kSlopeTabLo;  // wraps below kSlopeTabLo
  const uint32_t idx = (d < (uint32_t)kSlopeTabSpan ? d : (uint32_t)kSlopeTabSpan - 1u) + sign * (uint32_t)kSlopeTabSpan;
  const float tab = *reinterpret_cast<const float*>(table + 4u * idx);
  const float small = fmaf(0.79788456080286536f, __uint_as_float(b << 16), 0.5f);
  return mag >= 0x7f80u ? __uint_as_float(0x7fc00000u) : (mag < kSlopeTabLo ? small : tab);
}

__device__ __forceinline__ void slope_table_fill(float* table, int tid, int nthreads) {
  for (int e = tid; e < 2 * kSlopeTabSpan; e += nthreads) {
    const uint32_t bits = e < kSlopeTabSpan ? kSlopeTabLo + e : 0x8000u + kSlopeTabLo + (e - kSlopeTabSpan);
    table[e] = gelu_slope(__uint_as_float(bits << 16));
  }
}

// Slopes of the two bf16 values of `p` by table; `dmax`
// collects mag - kSlopeTabLo per half (wrapping below it): from kSlopeRare on
// a value is tiny, infinite or NaN and its lookup is wrong.
constexpr uint32_t kSlopeRare = 0x7f80u - kSlopeTabLo;
__device__ __forceinline__ void slope_pair(uint32_t p, const uint8_t* table, u16x2& dmax, float& lo, float& hi) {
  const u16x2 v = __builtin_bit_cast(u16x2, p);
  const u16x2 d = (v & (u16x2)0x7fff) - (u16x2)(uint16_t)kSlopeTabLo;
  dmax = __builtin_elementwise_max(dmax, d);
  const u16x2 off = (__builtin_elementwise_min(d, (u16x2)(uint16_t)(kSlopeTabSpan - 1)) +
                     (v >> 15) * (u16x2)(uint16_t)kSlopeTabSpan) << 2;  // < 2^14
  lo = *reinterpret_cast<const float*>(table + off.x);
  hi = *reinterpret_cast<const float*>(table + off.y);
}

// Slopes of the eight bf16 values of a 16-byte chunk.  A wave holding a value
// whose lookup is wrong redoes the chunk with the closed forms.
__device__ __forceinline__ void slope_chunk(gelu_u32x4 h, const uint8_t* table, float (&sl)[8]) {
  u16x2 dmax = {0, 0};
#pragma unroll
  for (int e = 0; e < 4; ++e) slope_pair(h[e], table, dmax, sl[2 * e], sl[2 * e + 1]);
  const uint32_t dm = dmax.x > dmax.y ? dmax.x : dmax.y;
  if (__builtin_amdgcn_ballot_w64(dm >= kSlopeRare) != 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      sl[2 * e] = slope_any(h[e] & 0xffffu, table);
      sl[2 * e + 1] = slope_any(h[e] >> 16, table);
    }
  }
}

// GELU of four packed bf16 pairs in place: table lookups; a wave holding a
// value outside the table (|x| < 2^-22 or >= 32) redoes the chunk exactly.
__device__ __forceinline__ void gelu_chunk(uint32_t (&v)[4], const uint16_t* table) {
  u16x2 dmax = {0, 0};
  uint32_t r[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    asm volatile("" : "+v"(v[e]));
    r[e] = gelu_pair_table(v[e], table, dmax);
  }
  const uint32_t dm = dmax.x > dmax.y ? dmax.x : dmax.y;
  if (__builtin_amdgcn_ballot_w64(dm >= (uint32_t)kGeluSpan) != 0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) r[e] = gelu_bf16(v[e] & 0xffffu, table) | (gelu_bf16(v[e] >> 16, table) << 16);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = r[e];
}

}  // namespace
}  // namespace terra
