// FP64 real-space Ewald terms shared by the pair, energy, point and adjoint
// kernels.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace cav {

// alpha and its square to twice double precision (a2 + a2lo), so that
// exp(-alpha^2 r^2) does not carry the rounding of alpha^2 times x^2.
struct EwaldAlpha {
  double alpha, a2, a2lo;
};

inline EwaldAlpha ewald_alpha(double alpha)
{
  const double a2 = alpha * alpha;
  return {alpha, a2, std::fma(alpha, alpha, -a2)};
}

// a b + c with the constant c in scalar registers.  (The compiler takes the
// two-address fmac for a Horner step and copies each constant into its
// accumulator first: a third of the instructions of the code below.)
__device__ __forceinline__ double fma_k(double a, double b, double c)
{
  double r;
  asm("v_fma_f64 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
  return r;
}

// exp(-(x + lo)), x >= 0, |lo| far below x: 2^n times the Taylor series of the
// remainder (|r| <= 0.347, degree 13: 4e-18 of the value).
__device__ __forceinline__ double exp_neg(double x, double lo)
{
  const double y = fmin(x, 800.0);  // exp(-800) is 0 in FP64
  const double n = rint(y * -1.44269504088896339e+00);
  double r = fma(n, -6.93147180485539138e-01, -y);  // ln 2 in two parts: 33 bits, so that n times it is exact, and the rest
  r = fma(n, -7.44061711001239685e-11, r) - lo;
  double p = 1.60590438368216133e-10;
  p = fma_k(p, r, 2.08767569878681002e-09);
  p = fma_k(p, r, 2.50521083854417202e-08);
  p = fma_k(p, r, 2.75573192239858883e-07);
  p = fma_k(p, r, 2.75573192239858925e-06);
  p = fma_k(p, r, 2.48015873015873016e-05);
  p = fma_k(p, r, 1.98412698412698413e-04);
  p = fma_k(p, r, 1.38888888888888894e-03);
  p = fma_k(p, r, 8.33333333333333322e-03);
  p = fma_k(p, r, 4.16666666666666644e-02);
  p = fma_k(p, r, 1.66666666666666657e-01);
  p = fma(p, r, 0.5);
  p = fma(p, r, 1.0);
  p = fma(p, r, 1.0);
  return ldexp(p, (int)n);
}

// For r^2 > 0: e = exp(-alpha^2 r^2), ec = erfc(alpha r) / r, ri2 = 1 / r^2.
//
// erfc(x) = exp(-x^2) erfcx(x), and erfcx is smooth on [0, inf): with
// t = 1 / (1 + x/4) (the form of Hastings' approximations, Abramowitz & Stegun
// 7.1.26) erfcx(x) = t P(2t - 1), P of degree 22, its Chebyshev fit in 40-digit
// arithmetic truncated at 3e-17 relative.  The exponential is shared with the
// Gaussian term of the force, 1/r comes from v_rsq_f64 and a Newton step, and
// no lane branches; sqrt, two divisions, exp and the library's erfc, whose
// ranges all run in a wave of mixed distances, take more instructions.  FP64
// issue bounds the kernels that are not bound by their
// gathers: real-space energy at N = 100003 395 -> 267 us, adjoint pairs of 64
// replicas 327 -> 310, the pair kernel at N = 65536 56 -> 37 (in order).
//
// The quantities that the terms are most sensitive to (1/r, its square, 2t - 1)
// each take a last correction from their residual.  Without these the kernels
// took 256, 306 and 34 us, but the forces of 100 ions (alpha 0.9) were 2.7e-16
// off 64-bit exact (2-norm) where the library's functions gave 2.4e-16; now
// 2.3e-16, point potentials 2.1e-16 (library 3.2e-16), their fields 2.7e-16
// (4.2e-16).  A term's own error is 1.6e-16 root mean square and 7e-16 at most.
__device__ __forceinline__ void ewald_real(double r2, const EwaldAlpha &al, double &e, double &ec,
                                           double &ri2)
{
  double y = __builtin_amdgcn_rsq(r2);
  y = fma(y, fma(-0.5 * r2 * y, y, 0.5), y);
  // r = r2 y and 1 / r from the residual 1 - r2 y^2 of the unrounded product
  double rn = r2 * y;
  const double f = fma(-fma(r2, y, -rn), y, fma(-rn, y, 1.0));
  rn = fma(0.5 * rn, f, rn);
  y = fma(0.5 * y, f, y);
  // s = 2t - 1 = (1 - w) / (1 + w), w = x / 4: a rounding of 1 + w alone would
  // count four times in x
  const double w = 0.25 * (al.alpha * rn);
  const double d = 1.0 + w;
  double t = __builtin_amdgcn_rcp(d);
  t = fma(t, fma(-d, t, 1.0), t);
  double s = fma(2.0, t, -1.0);
  s = fma(fma(-w, s, (1.0 - s) - w), t, s);
  t = fma(0.5, s, 0.5);
  double p = 3.01845414851638119e-10;
  p = fma_k(p, s, -6.63613627087004204e-11);
  p = fma_k(p, s, -3.81882222497661988e-09);
  p = fma_k(p, s, -2.05956021403690043e-10);
  p = fma_k(p, s, 3.06322051766131277e-08);
  p = fma_k(p, s, 1.89922483216737570e-08);
  p = fma_k(p, s, -2.10912903014044835e-07);
  p = fma_k(p, s, -3.56236604332617538e-07);
  p = fma_k(p, s, 1.17309597843865979e-06);
  p = fma_k(p, s, 4.71536834474533832e-06);
  p = fma_k(p, s, -9.08550953736742834e-07);
  p = fma_k(p, s, -4.42032701640101717e-05);
  p = fma_k(p, s, -1.13763242914232012e-04);
  p = fma_k(p, s, 7.02397339847800215e-05);
  p = fma_k(p, s, 1.52801392709659800e-03);
  p = fma_k(p, s, 6.59251333229525591e-03);
  p = fma_k(p, s, 1.90953787259277030e-02);
  p = fma_k(p, s, 4.35027343102230776e-02);
  p = fma_k(p, s, 8.27128969695789668e-02);
  p = fma_k(p, s, 1.35213457828299410e-01);
  p = fma_k(p, s, 1.93302175566307660e-01);
  p = fma_k(p, s, 2.44137182270220604e-01);
  p = fma_k(p, s, 2.73998915250122765e-01);
  const double xx = al.a2 * r2;
  e = exp_neg(xx, fma(al.a2, r2, -xx) + al.a2lo * r2);
  ec = e * ((t * p) * y);
  ri2 = y * y;
  ri2 = fma(ri2, fma(-r2, ri2, 1.0), ri2);
}

}  // namespace cav
