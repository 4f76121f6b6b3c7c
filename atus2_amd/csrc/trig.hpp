// trig.hpp -- sine and cosine of the V steps' phases.
#pragma once

namespace atus {

// sin and cos: Taylor series (to x^11 and x^10) for |x| < 2^-5, where the
// truncation error is below 1e-27 relative; the library routine otherwise.
// The phases of the potential and Bragg steps are dt*E, usually small.
__device__ __forceinline__ void sincos_fast(double x, double* s, double* c) {
  if (fabs(x) < 0.03125) {
    const double x2 = x * x;
    *s = x * (1.0 + x2 * (-1.0 / 6.0 + x2 * (1.0 / 120.0 + x2 * (-1.0 / 5040.0 + x2 * (1.0 / 362880.0 +
                                                                                  x2 * (-1.0 / 39916800.0))))));
    *c = 1.0 + x2 * (-0.5 + x2 * (1.0 / 24.0 + x2 * (-1.0 / 720.0 + x2 * (1.0 / 40320.0 + x2 * (-1.0 / 3628800.0)))));
  } else {
    sincos(x, s, c);
  }
}

// any argument by the library's routine, out of line: the callers' points
// are unrolled, and a copy of its reduction of large arguments for each cost
// 2-4% of the kernels that use sincos_mid
__device__ __attribute__((noinline)) double2 sincos_large(double x) {
  double s, c;
  sincos(x, &s, &c);
  return make_double2(s, c);
}

// r + rl = x - n pi/2 with n = rint(x 2/pi), |x| < 10^6 (Cody-Waite): pi/2 =
// h1 + h2 + h3 with h1 of 33 bits, so n h1 is exact and x - n h1 too; t is a
// multiple of the last bit of n h2, so what t - p rounds off is (t - r) - p
// exactly, also where x is next to a multiple of pi/2 and r is tiny.  No
// contraction: r has to be the difference from the rounded product.  The
// order of rl's terms is the one whose code costs the resident blocks nothing
// (4096 points, 1000 steps: 9.4 ms; with the two tails added first 9.6).
__device__ __forceinline__ double reduce_half_pi(double x, double* r, double* rl) {
#pragma clang fp contract(off)
  const double n = rint(x * 0.6366197723675814);
  const double t = fma(-n, 1.5707963267341256, x);
  const double p = n * 6.077100506506192e-11;
  const double d = t - p;
  *r = d;
  *rl = fma(n, -3.5215598651832e-27, ((t - d) - p) - fma(n, 6.077100506506192e-11, -p));
  return n;
}

// The same where larger phases are common (kernels whose V step bounds them:
// the 1D resident blocks, whose potential reaches far from the origin, and
// the coupled steps of multi.hpp): for |x| < 10^6 the reduction above, then
// Taylor series to x^19 and x^18 on |r| <= pi/4 (truncation 2e-19 and 2e-18),
// the cosine's 1 - r^2/2 compensated as in the kernel cosine of fdlibm (Sun
// Microsystems, 1993).  At most 0.76 ulp off, over random arguments and over
// the doubles next to the multiples of pi/2.  In the passes that stream
// (k_vfuse) its code costs more than it saves: 2% of the 2048^2 step, 3% of
// the 32x64x32 one.
__device__ __forceinline__ void sincos_mid(double x, double* s, double* c) {
  if (fabs(x) < 0.03125) {
    const double x2 = x * x;
    const double sx = fma(x * x2, -1.0 / 6.0 + x2 * (1.0 / 120.0 + x2 * (-1.0 / 5040.0 +
                                                     x2 * (1.0 / 362880.0 + x2 * (-1.0 / 39916800.0)))), x);
    *s = __builtin_copysign(sx, x);  // the sum loses the sign of zero
    *c = 1.0 + x2 * (-0.5 + x2 * (1.0 / 24.0 + x2 * (-1.0 / 720.0 + x2 * (1.0 / 40320.0 + x2 * (-1.0 / 3628800.0)))));
  } else if (fabs(x) < 1e6) {
    double r, rl;
    const double n = reduce_half_pi(x, &r, &rl);
    const double x2 = r * r;
    double p = -1.0 / 121645100408832000.0;
    p = fma(p, x2, 1.0 / 355687428096000.0);
    p = fma(p, x2, -1.0 / 1307674368000.0);
    p = fma(p, x2, 1.0 / 6227020800.0);
    p = fma(p, x2, -1.0 / 39916800.0);
    p = fma(p, x2, 1.0 / 362880.0);
    p = fma(p, x2, -1.0 / 5040.0);
    p = fma(p, x2, 1.0 / 120.0);
    p = fma(p, x2, -1.0 / 6.0);
    double q = -1.0 / 6402373705728000.0;
    q = fma(q, x2, 1.0 / 20922789888000.0);
    q = fma(q, x2, -1.0 / 87178291200.0);
    q = fma(q, x2, 1.0 / 479001600.0);
    q = fma(q, x2, -1.0 / 3628800.0);
    q = fma(q, x2, 1.0 / 40320.0);
    q = fma(q, x2, -1.0 / 720.0);
    q = fma(q, x2, 1.0 / 24.0);
    // sin(r + rl) = r + (r^3 p + rl cos r), cos(r + rl) = (1 - r^2/2) +
    // (r^4 q - r rl) with the rounding of 1 - r^2/2 added back
    const double hz = 0.5 * x2, w = 1.0 - hz;
    const double sr = r + fma(r * x2, p, rl * w);
    const double cr = w + (((1.0 - w) - hz) + fma(x2 * x2, q, -r * rl));
    const int k = (int)n;
    const double a = (k & 1) ? cr : sr, b = (k & 1) ? sr : cr;
    *s = (k & 2) ? -a : a;
    *c = ((k + 1) & 2) ? -b : b;
  } else {
    const double2 v = sincos_large(x);
    *s = v.x;
    *c = v.y;
  }
}

}  // namespace atus
