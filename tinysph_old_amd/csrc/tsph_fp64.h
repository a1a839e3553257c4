// Division and square root of the FP64 pair loops, correctly rounded like the
// operators they stand for, in the parts that a pair term can share.
//
// A general FP64 division on gfx950 is eleven instructions: two that scale the
// operands' exponents, a reciprocal estimate (v_rcp_f64, quarter rate), four
// FMAs of Newton iterations, the quotient, its residual and correction, and
// the handling of special values.  In the pair loops the operands' exponents
// are moderate (lengths, densities, pressures), which leaves
//   y = recip64(b)      estimate and two Newton iterations: 1/b to below an ulp
//   quot64(a, b, y)     q = a y, then q + (a - b q) y: with the residual exact
//                       in one FMA this is the correctly rounded a/b
//                       (Markstein 1990)
// and y serves every quotient with the denominator b: a constant of the case,
// a particle's density, or the pair's r^2 + eps h^2, which two terms divide
// by.  quot64_any adds the special values (zero, infinite or NaN operands) as
// the operator gives them, for whatever holds a velocity, a density or a
// pressure.  Quotients of a pair's distances and the case's constants go without:
// both are finite, and the denominators positive (with it three more quotients
// per pair: 740k particles 498 us per step and 501).  Denormal operands are not
// provided for: a density of 1e-310 may give NaN where the operator overflows.
//
// sqrt64 runs the coupled iteration for sqrt(x) and 1/(2 sqrt(x)) (Goldschmidt
// 1964) from the reciprocal square root estimate and corrects the root with
// two exact residuals; recip_of_root64 makes 1/sqrt(x) of the second value.
//
// The 740k-particle dam break's pair pass takes 199 us with these, 251 with the
// operators.
#pragma once

#include <hip/hip_runtime.h>

namespace tsph {

__device__ __forceinline__ double recip64(double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
  return __builtin_fma(y, __builtin_fma(-b, y, 1.0), y);
}

// a / b for y = recip64(b) (or the rounded 1/b)
__device__ __forceinline__ double quot64(double a, double b, double y) {
  const double q = a * y;
  return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}

__device__ __forceinline__ double quot64_any(double a, double b, double y) {
  return __builtin_amdgcn_div_fixup(quot64(a, b, y), b, a);
}

struct Root64 {
  double s;     // sqrt(x)
  double half;  // 1 / (2 sqrt(x)), to a few ulp
};
// for x = 0 or normal, finite
__device__ __forceinline__ Root64 sqrt64(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  double h = 0.5 * y, s = x * y;
  const double e = __builtin_fma(-h, s, 0.5);
  s = __builtin_fma(s, e, s);
  h = __builtin_fma(h, e, h);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  s = __builtin_fma(__builtin_fma(-s, s, x), h, s);
  return {x == 0.0 ? 0.0 : s, h};
}

// 1 / r.s to below an ulp
__device__ __forceinline__ double recip_of_root64(const Root64 &r) {
  const double y = r.half + r.half;
  return __builtin_fma(y, __builtin_fma(-r.s, y, 1.0), y);
}

}  // namespace tsph
