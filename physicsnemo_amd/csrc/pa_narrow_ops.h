// What the float32 kernels of narrow heads share: tiles of 16 points on v_mfma_f32_16x16x4_f32.
//
// A lane is (i, g) = 16 g + i.  A operand (16 x 4): row i, k = g.  B operand (4 x 16): column i, k = g.  C/D (16 x 16): column i,
// register r = row 4 g + r.  Values held as four registers at channels (or slices) 4 g + r of point i are an accumulator's layout
// and, one register per step, an operand whose reduction index runs over them in the order 4 g + r, g = 0 .. 3.
#pragma once

#include <float.h>

#include "pa_mfma_ops.h"

namespace pa {
namespace narrow {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kS = 32, kTilePts = 16;

__device__ __forceinline__ f32x4 mma16(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
// over the four lanes that hold a point's (or a slice's) registers
__device__ __forceinline__ float group_sum(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return mfma::half_sum(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}
__device__ __forceinline__ float group_max(float v) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return mfma::half_max(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}
// a value that is the same in all lanes, in a scalar register
__device__ __forceinline__ float uniform(float v) { return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v))); }

// keeps the LDS reads of a later section from being hoisted into registers here
__device__ __forceinline__ void section() { asm volatile("" ::: "memory"); }

// exp(z / T) = 2^(z sc), sc = log2(e) / T as the sum of two floats: nothing is lost to the rounding of z / T or of its product
__device__ __forceinline__ void exponent_scale(float temp, float &sc, float &sc_low) {
  const float hi = kLog2e / temp;
  sc = uniform(hi);
  sc_low = uniform((fmaf(-hi, temp, kLog2e) + 1.92596299e-8f) / temp);  // log2(e) = kLog2e + 1.93e-8
}
// z <= 0 or NaN.  Where the power is a normal number, low is below 1e-4; from z sc = -FLT_MAX down it is +inf or, at z = -inf, NaN, and e
// is 0: fminf makes 1 of either, so that a slice switched off by a bias of -inf or the lowest float has weight 0.
__device__ __forceinline__ float exponential(float z, float sc, float sc_low) {
  const float hi = z * sc, low = fminf(fmaf(z, sc_low, fmaf(z, sc, -hi)), 1.f), e = __builtin_amdgcn_exp2f(hi);
  return fmaf(e * 0.69314718f, low, e);
}

}  // namespace narrow
}  // namespace pa
