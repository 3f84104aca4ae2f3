// hg_dual.hpp -- forward-mode dual numbers (one tangent direction) for the
// device JVP of the step: value v and derivative d, with the product,
// quotient and chain rules of ForwardDiff.Dual.  Comparisons look at values
// only, so branches follow the primal path (the semantics ForwardDiff gives
// the reference).
#pragma once
#include <hip/hip_runtime.h>

#include "hg_device.hpp"

namespace hg {

struct Dual1 {
  double v, d;
  __host__ __device__ Dual1() : v(0.0), d(0.0) {}
  __host__ __device__ Dual1(double x) : v(x), d(0.0) {}  // NOLINT: constants carry no tangent
  __host__ __device__ Dual1(double x, double dx) : v(x), d(dx) {}
};

__host__ __device__ __forceinline__ double val(double x) { return x; }
__host__ __device__ __forceinline__ double val(const Dual1& x) { return x.v; }

__host__ __device__ __forceinline__ Dual1 operator-(const Dual1& a) { return Dual1(-a.v, -a.d); }
__host__ __device__ __forceinline__ Dual1 operator+(const Dual1& a, const Dual1& b) {
  return Dual1(a.v + b.v, a.d + b.d);
}
__host__ __device__ __forceinline__ Dual1 operator-(const Dual1& a, const Dual1& b) {
  return Dual1(a.v - b.v, a.d - b.d);
}
__host__ __device__ __forceinline__ Dual1 operator*(const Dual1& a, const Dual1& b) {
  return Dual1(a.v * b.v, a.d * b.v + a.v * b.d);
}
__host__ __device__ __forceinline__ Dual1 operator/(const Dual1& a, const Dual1& b) {
  return Dual1(a.v / b.v, (a.d * b.v - a.v * b.d) / (b.v * b.v));
}
// A constant carries no tangent.
__host__ __device__ __forceinline__ Dual1 operator+(const Dual1& a, double b) { return Dual1(a.v + b, a.d); }
__host__ __device__ __forceinline__ Dual1 operator+(double a, const Dual1& b) { return Dual1(a + b.v, b.d); }
__host__ __device__ __forceinline__ Dual1 operator-(const Dual1& a, double b) { return Dual1(a.v - b, a.d); }
__host__ __device__ __forceinline__ Dual1 operator-(double a, const Dual1& b) { return Dual1(a - b.v, -b.d); }
__host__ __device__ __forceinline__ Dual1 operator*(const Dual1& a, double b) { return Dual1(a.v * b, a.d * b); }
__host__ __device__ __forceinline__ Dual1 operator*(double a, const Dual1& b) { return Dual1(a * b.v, a * b.d); }
__host__ __device__ __forceinline__ Dual1 operator/(const Dual1& a, double b) { return Dual1(a.v / b, a.d / b); }
__host__ __device__ __forceinline__ Dual1 operator/(double a, const Dual1& b) { return Dual1(a) / b; }

__host__ __device__ __forceinline__ bool operator<(const Dual1& a, const Dual1& b) { return a.v < b.v; }
__host__ __device__ __forceinline__ bool operator<=(const Dual1& a, const Dual1& b) { return a.v <= b.v; }
__host__ __device__ __forceinline__ bool operator>(const Dual1& a, const Dual1& b) { return a.v > b.v; }
__host__ __device__ __forceinline__ bool operator<(const Dual1& a, double b) { return a.v < b; }
__host__ __device__ __forceinline__ bool operator<=(const Dual1& a, double b) { return a.v <= b; }
__host__ __device__ __forceinline__ bool operator>(const Dual1& a, double b) { return a.v > b; }

// The shared-part quotients and roots of hg_device.hpp: y = 1 / b.v, and the
// root's derivative from the same 0.5 / sqrt.
__device__ __forceinline__ double rcp_est(const Dual1& b) { return rcp_est(b.v); }
__device__ __forceinline__ Dual1 div_est(const Dual1& a, const Dual1& b, double y) {
  const double v = div_est(a.v, b.v, y);
  return Dual1(v, (a.d - v * b.d) * y);
}
__device__ __forceinline__ Dual1 div_est(const Dual1& a, double b, double y) {
  return Dual1(div_est(a.v, b, y), div_est(a.d, b, y));  // both as a / b gives them
}
__device__ __forceinline__ Dual1 sqrt_half_rcp(const Dual1& x, Dual1& o) {
  double ov;
  const double s = sqrt_half_rcp(x.v, ov);
  const double sd = x.d * ov;
  o = Dual1(ov, -2.0 * (ov * ov) * sd);
  return Dual1(s, sd);
}
__device__ __forceinline__ Dual1 sqrt_pos(const Dual1& x) {
  double ov;
  const double s = sqrt_half_rcp(x.v, ov);
  return Dual1(s, x.d * ov);
}
__device__ __forceinline__ Dual1 cbrt_of(const Dual1& a) {
  const double r = ::cbrt(a.v);
  return Dual1(r, a.d * (r / (3.0 * a.v)));
}

}  // namespace hg
