// F32 products on the f16 matrix cores.
//
// An f32 value is taken as two f16 values, x = x0 + x1 / 2^11: x0 is x rounded
// to f16, x1 the remainder times 2^11 rounded to f16.  Two 11-bit significands
// and the remainder's sign leave an error of at most 2^-23 |x| (rms about
// 2^-25 |x|), with a floor of 2^-36 where x1 is a subnormal.  Of the four
// products of two such values three are taken, in two f32 accumulators,
//   main += x0 y0,   corr += x0 y1 + x1 y0,   sum = main + corr / 2^11;
// the one left out is at most 2^-22 |x y| (rms about 2^-25).  The products are
// exact, and main rounds once per 32 of k where the F32 matrix instruction
// rounds once per 4: sums come out closer to the 64-bit values than from F32
// products (K = 768: 2.0e-7 against 3.5-5.0e-7 relative), and
// v_mfma_f32_16x16x32_f16 runs 16 times the F32 rate for three products.
//
// What the split holds less well than F32, and who answers for it:
//  * values beyond f16's largest, infinities and NaN: x0 is an infinity or a
//    NaN, and so is every sum that x enters (is_finite below);
//  * values below 2^-13: held to 2^-36, not to 2^-23 of themselves.  The
//    linear counts them and proves, output by output, that the floor is below
//    one F32 rounding of the sum's terms (linear.hip); the attention scales
//    the columns of V and looks at every query's result (attention.hip).
#pragma once

#include "common.h"

namespace vks {

typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kUp = 2048.0f;          // 2^11
constexpr float kDown = 1.0f / 2048.0f;
// Both parts of two values, packed (a in the low half).
__device__ __forceinline__ void split2(float a, float b, uint32_t* p0, uint32_t* p1) {
  const f16x2 h = __builtin_convertvector((f32x2{a, b}), f16x2);
  const f32x2 r = {__builtin_fmaf(static_cast<float>(h[0]), -kUp, a * kUp),
                   __builtin_fmaf(static_cast<float>(h[1]), -kUp, b * kUp)};
  *p0 = __builtin_bit_cast(uint32_t, h);
  *p1 = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, f16x2));
}

// Both parts of eight values, in the order of the values.
__device__ __forceinline__ void split8(const float4& x, const float4& y, u32x4* p0, u32x4* p1) {
  uint32_t h[4], l[4];
  split2(x.x, x.y, &h[0], &l[0]);
  split2(x.z, x.w, &h[1], &l[1]);
  split2(y.x, y.y, &h[2], &l[2]);
  split2(y.z, y.w, &h[3], &l[3]);
  *p0 = u32x4{h[0], h[1], h[2], h[3]};
  *p1 = u32x4{l[0], l[1], l[2], l[3]};
}

// Both parts with the remainder left at its own scale, x = x0 + x1: for values
// scaled up beforehand (the floor is 2^-25 of the scaled value), summed in one
// accumulator.
__device__ __forceinline__ void split2_plain(float a, float b, uint32_t* p0, uint32_t* p1) {
  const f16x2 h = __builtin_convertvector((f32x2{a, b}), f16x2);
  const f32x2 r = {a - static_cast<float>(h[0]), b - static_cast<float>(h[1])};
  *p0 = __builtin_bit_cast(uint32_t, h);
  *p1 = __builtin_bit_cast(uint32_t, __builtin_convertvector(r, f16x2));
}

// The largest and the smallest |x| of eight values (NaN left out).
__device__ __forceinline__ float max_abs8(const float4& x, const float4& y) {
  float m = fmaxf(fmaxf(fabsf(x.x), fabsf(x.y)), fabsf(x.z));
  m = fmaxf(fmaxf(m, fabsf(x.w)), fabsf(y.x));
  m = fmaxf(fmaxf(m, fabsf(y.y)), fabsf(y.z));
  return fmaxf(m, fabsf(y.w));
}

__device__ __forceinline__ float min_abs8(const float4& x, const float4& y) {
  float m = fminf(fminf(fabsf(x.x), fabsf(x.y)), fabsf(x.z));
  m = fminf(fminf(m, fabsf(x.w)), fabsf(y.x));
  m = fminf(fminf(m, fabsf(y.y)), fabsf(y.z));
  return fminf(m, fabsf(y.w));
}

__device__ __forceinline__ float4 scale4(const float4& x, float s) {
  return make_float4(x.x * s, x.y * s, x.z * s, x.w * s);
}

__device__ __forceinline__ f32x4 mfma(const u32x4& a, const u32x4& b, const f32x4& c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ bool is_finite(float v) {
  return (__float_as_uint(v) & 0x7f800000u) != 0x7f800000u;
}

}  // namespace vks
