// Correctly rounded square roots and quotients without range handling, for
// operands far inside the FP64 range (fast64 RVEs): the scaling and special cases
// of the compiler's IEEE sequences fall away, and a reciprocal that is at hand
// replaces the one each division computes.  No fused or contracted operation but
// the ones written here: compile with -ffp-contract=off.
#pragma once
#ifdef __HIP__
#define MF_ROOT64_FN __device__ inline
#else
#define MF_ROOT64_FN inline  // the host check of the arithmetic
#endif

namespace mf {
namespace kern {

// a / b from a reciprocal rb of b that is good to 1.25 ulp (an ulp: 2^-52 of the
// value): the quotient of the first product is within 2 ulp, its remainder is
// formed by an FMA (exact but for a few bits below its own precision) and
// corrects it.  What is rounded last differs from a / b by at most about 2^-50
// ulp, and quotients that close to a rounding boundary are as rare.
MF_ROOT64_FN double div64(double a, double b, double rb) {
  const double q = a * rb;
  return __builtin_fma(__builtin_fma(-q, b, a), rb, q);
}
// l = sqrt(x) and rl = 1 / l from a seed y of 1 / sqrt(x) that is off by at most
// 2^-23 (the hardware's is within 2^-24.1: 2^33 arguments evenly over [1, 4)).
// With r = (1 - x y^2) / 2, 1 / sqrt(x) = y (1 + r + 3/2 r^2 + 5/2 r^3 ..); the
// term left out is below 2^-67, so g and h are off by their roundings, 0.75 ulp,
// h as a reciprocal of the rounded root by 1.25.  One Newton correction of g with
// an exact remainder then leaves l 2^-50 ulp before its rounding.  Goldschmidt's
// second-order step and two corrections take as many operations, but leave h
// 1.5 e^2 off for a seed off by e: 37 ulp for the hardware's.  x = 0 gives NaN
// (its quotient by l would be one as well).
MF_ROOT64_FN void root64(double x, double y, double &l, double &rl) {
  double g = x * y, h = 0.5 * y;
  const double r = __builtin_fma(-h, g, 0.5);
  const double p = __builtin_fma(__builtin_fma(0.5, r, r), r, r);  // 0.5: an inline constant
  g = __builtin_fma(g, p, g);
  h = __builtin_fma(h, p, h);
  l = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  rl = h + h;
}

}  // namespace kern
}  // namespace mf
