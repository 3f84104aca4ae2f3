// hg_device.hpp -- device-side arithmetic shared by the forward and adjoint
// kernels of libhgswe (gfx950).
//
// Every expression keeps Hydrograd.jl's evaluation order (left-to-right, no
// fused multiply-add: the library is compiled with -ffp-contract=off), so a
// forward evaluation is bit-identical to the reference's Float64 arithmetic
// except for pow(), whose last bit may differ between math libraries.
// Multiplications by 0.5 replace the reference's divisions by 2.0 (exact).
#pragma once
#include <hip/hip_runtime.h>

namespace hg {

constexpr double EPS = 2.220446049250313e-16;  // eps(Float64)

// ---- FP64 division and square root with shared parts.  The compiler's own
// sequences cost 11 (division) and 16 (square root) vector instructions
// each and cannot share work between two quotients of one denominator.
// These keep the correctly rounded result on the ranges the solver forms
// them on (tests/test_gpu_rounding_parts.py compares 2^24 pairs from 1e-100 to
// 1e100 and the mantissas next to powers of two with IEEE quotients and roots),
// from the textbook iterations (P. Markstein, "Software division
// and square root using Goldschmidt's algorithms", RNC 2004): 9 and 10
// instructions, and 4 for a further quotient of the same denominator (the
// step kernel: 596 -> 502 FP64 instructions).  1,000 steps of the 1M-triangle
// channel went from 43.0 to 41.5 ms, 200 of a 96k-cell batch from 2.03 to
// 1.89 ms, the same bits.

// 1 / b to within an ulp: the hardware estimate and two Newton steps.
__device__ __forceinline__ double rcp_est(double b) {
  double y = __builtin_amdgcn_rcp(b);
  y = __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
  return __builtin_fma(__builtin_fma(-b, y, 1.0), y, y);
}

// a / b given y = rcp_est(b): the quotient's residual corrects its last bit;
// zeros, infinities and NaN as a division gives them.
__device__ __forceinline__ double div_est(double a, double b, double y) {
  const double q = a * y;
  return __builtin_amdgcn_div_fixup(__builtin_fma(__builtin_fma(-b, q, a), y, q), b, a);
}

// 1 / sqrt(x) for normal finite x > 0, within about an ulp: the hardware's
// estimate y and, with e = 1 - x y^2, the series y (1 + e / 2 + 3 e^2 / 8).
__device__ __forceinline__ double rsq_est(double x) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = __builtin_fma(-x * y, y, 1.0);
  return __builtin_fma(y * e, __builtin_fma(e, 0.375, 0.5), y);
}

// sqrt(x) for normal finite x > 0 (every caller adds eps to a square or a
// depth, so x >= 2^-52); r2 = 0.5 / sqrt(x) to about 2^-46.
__device__ __forceinline__ double sqrt_est(double x, double& r2) {
  const double y = __builtin_amdgcn_rsq(x);
  double g = x * y, h = 0.5 * y;
  const double e = __builtin_fma(-h, g, 0.5);
  g = __builtin_fma(g, e, g);
  r2 = h = __builtin_fma(h, e, h);
  g = __builtin_fma(__builtin_fma(-g, g, x), h, g);
  return __builtin_fma(__builtin_fma(-g, g, x), h, g);
}
__device__ __forceinline__ double sqrt_pos(double x) {
  double r2;
  return sqrt_est(x, r2);
}
// s = sqrt(x) and o = 0.5 / s.
__device__ __forceinline__ double sqrt_half_rcp(double x, double& o) {
  double r2;
  const double s = sqrt_est(x, r2);
  o = __builtin_fma(__builtin_fma(-s, r2, 0.5), 2.0 * r2, r2);
  return s;
}
__device__ __forceinline__ double cbrt_of(double x) { return cbrt(x); }

// x^(7/3) for the Manning term as (x * x) * cbrt(x): within a few ulp of
// the correctly rounded power (the reference's pow(x, 7.0/3.0) carries an
// exponent 1.5e-16 off 7/3, a relative 1.5e-16 * |ln x| on its own), at a
// sixth of the instruction count of a general double pow.
template <class T>
__device__ __forceinline__ T pow_7_3(const T& x) { return (x * x) * cbrt_of(x); }

// Manning friction (semi_discretize_swe_2D.jl:544-547); h is the clamped
// depth, q the masked discharge.  Dividing by k_n^2 = 1 is exact and skipped.
// T: double, or a dual number for the JVP.
template <class T>
__device__ __forceinline__ void friction(double g, double kn2, double hsmall, const T& h, const T& qx, const T& qy,
                                         const T& n, T& fx, T& fy) {
  T c = g * (n * n);
  if (kn2 != 1.0) c = c / kn2;
  const T p = pow_7_3(h + hsmall);
  c = div_est(c, p, rcp_est(p));
  const T s = sqrt_pos(qx * qx + qy * qy + EPS);
  fx = c * s * qx;
  fy = c * s * qy;
}

// FlowResistance friction (semi_discretize_swe_2D.jl:521-531): the UDE's
// friction magnitude m along the discharge, m q / sqrt(q_x^2 + q_y^2 + eps).
template <class T>
__device__ __forceinline__ void friction_mag(const T& m, const T& qx, const T& qy, T& fx, T& fy) {
  const T s = sqrt_pos(qx * qx + qy * qy + EPS);
  const double y = rcp_est(s);
  fx = div_est(m * qx, s, y);
  fy = div_est(m * qy, s, y);
}

}  // namespace hg
