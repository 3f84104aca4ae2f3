// hg_roe_pair.hpp -- face-once Roe flux that returns the flux seen from
// BOTH cells of an internal face, each bit-identical to the reference's
// per-cell evaluation (Riemann_2D_Roe, swe_2D_solvers.jl:4-164, called
// once from each side by compute_inviscid_fluxes, semi_discretize_swe_2D.jl:286-419).
//
// Why two values from one evaluation are exact: evaluating the face from
// cell B (left = B, right = A, normal -n) negates n and dQ exactly, so
// unRoe, w0 and every physical flux negate exactly, w1 <-> -w2 and
// lambda1 <-> lambda2 swap exactly, and uRoe / vRoe / cRoe are unchanged
// (IEEE addition is commutative, multiplication and subtraction are
// sign-symmetric).  Only the final rows of R * (Lambda * w) for the two
// momentum components are summed in a different order:
//   A side: (T0 + T1) + T2,  B side: -((T0 + T2) + T1).
// Both sums are formed here, so each side receives exactly the value the
// reference computes for it.  The branch tests are mirror images of each
// other (branches 2/3 and 4/5 swap), so the same holds on wet/dry faces.
#pragma once
#include "hg_device.hpp"
#include "hg_dual.hpp"

namespace hg {

// Cell state as the flux reads it, plus per-cell derived quantities that
// the reference recomputes identically for every face of the cell:
// u = hu / h, v = hv / h, s = sqrt(h + eps), p = 0.5 g (xi^2 + 2 xi h_still)
// with the eps-smoothed square of smooth_pow.
// T: double, or a dual number for the JVP (h_still is a constant there).
template <class T>
struct CellQT {
  T xi;
  double hs;
  T h, hu, hv, zb, u, v, s, p;
};
using CellQ = CellQT<double>;

template <class T>
__device__ __forceinline__ CellQT<T> make_cellq(const T& xi, double hs, const T& qx, const T& qy, const T& zb,
                                                double half_g, double hsmall) {
  CellQT<T> c;
  c.xi = xi;
  c.hs = hs;
  T h = xi + hs, hu = qx, hv = qy;
  if (h <= hsmall) {  // semi_discretize_swe_2D.jl:101-106
    h = T(hsmall);
    hu = T(0.0);
    hv = T(0.0);
  }
  c.h = h;
  c.hu = hu;
  c.hv = hv;
  c.zb = zb;
  const double rh = rcp_est(h);
  c.u = div_est(hu, h, rh);
  c.v = div_est(hv, h, rh);
  c.s = sqrt_pos(h + EPS);
  c.p = half_g * ((xi + EPS) * (xi + EPS) + 2.0 * xi * hs);
  return c;
}

__device__ __forceinline__ double pick(bool c, double x, double y) { return c ? x : y; }
__device__ __forceinline__ Dual1 pick(bool c, const Dual1& x, const Dual1& y) {
  return Dual1(c ? x.v : y.v, c ? x.d : y.d);
}

// Flux through the face (A | B), normal n pointing from A to B.
// fa = flux seen from A; when BOTH, fb = flux seen from B (normal -n).
template <bool BOTH, class T>
__device__ __forceinline__ void roe_pair(const CellQT<T>& A, const CellQT<T>& B, double nx, double ny, double g,
                                         double half_g, double hmin, T fa[3], T fb[3]) {
  if (A.h <= hmin && B.h <= hmin) {  // :16-22
    fa[0] = fa[1] = fa[2] = T(0.0);
    if (BOTH) fb[0] = fb[1] = fb[2] = T(0.0);
    return;
  }
  // :23-36, B := mirror of A, and :39-51, A := mirror of B (xi and h_still are kept)
  const bool mB = (B.h <= hmin) && (A.h + A.zb) < (B.zb + hmin);
  const bool mA = !mB && (A.h <= hmin) && (B.h + B.zb) < (A.zb + hmin);
  T hA = A.h, huA = A.hu, hvA = A.hv, uA = A.u, vA = A.v, sA = A.s;
  T hB = B.h, huB = B.hu, hvB = B.hv, uB = B.u, vB = B.v, sB = B.s;
  if constexpr (sizeof(T) == sizeof(double)) {
    if (mB) {
      hB = A.h; huB = -A.hu; hvB = -A.hv; uB = -A.u; vB = -A.v; sB = A.s;
    } else if (mA) {
      hA = B.h; huA = -B.hu; hvA = -B.hv; uA = -B.u; vA = -B.v; sA = B.s;
    }
  } else {  // value by value: assigned as pairs in a branch, the compiler lost the negations
    hB = pick(mB, A.h, B.h); huB = pick(mB, -A.hu, B.hu); hvB = pick(mB, -A.hv, B.hv);
    uB = pick(mB, -A.u, B.u); vB = pick(mB, -A.v, B.v); sB = pick(mB, A.s, B.s);
    hA = pick(mA, B.h, A.h); huA = pick(mA, -B.hu, A.hu); hvA = pick(mA, -B.hv, A.hv);
    uA = pick(mA, -B.u, A.u); vA = pick(mA, -B.v, A.v); sA = pick(mA, B.s, A.s);
  }
  if (!mA && !mB && (A.h <= hmin || B.h <= hmin)) {  // :54-75, physical flux of the wet side, h^2 pressure
    const bool left_dry = A.h <= hmin;
    const T hw = left_dry ? B.h : A.h;
    const T huw = left_dry ? B.hu : A.hu, hvw = left_dry ? B.hv : A.hv;
    const T uw = left_dry ? B.u : A.u, vw = left_dry ? B.v : A.v;
    const T pr = half_g * ((hw + EPS) * (hw + EPS));
    const T f0 = huw * nx + hvw * ny;
    const T f1 = (huw * uw + pr) * nx + huw * vw * ny;
    const T f2 = (hvw * uw) * nx + (hvw * vw + pr) * ny;
    fa[0] = f0; fa[1] = f1; fa[2] = f2;
    if (BOTH) { fb[0] = -f0; fb[1] = -f1; fb[2] = -f2; }
    return;
  }
  const T hRoe = (hA + hB) * 0.5;
  const T sAB = sA + sB;
  const double ys = rcp_est(sAB);
  const T uRoe = div_est(sA * uA + sB * uB, sAB, ys);
  const T vRoe = div_est(sA * vA + sB * vB, sAB, ys);
  const T unRoe = uRoe * nx + vRoe * ny;
  T o;  // 0.5 / cRoe
  const T cRoe = sqrt_half_rcp(g * hRoe + EPS, o);
  const T d0 = B.xi - A.xi, d1 = huB - huA, d2 = hvB - hvA;
  const T w0 = (-(uRoe * ny - vRoe * nx)) * d0 + ny * d1 + (-nx) * d2;
  const T w1 = (unRoe * o + 0.5) * d0 + (-nx * o) * d1 + (-ny * o) * d2;
  const T w2 = (-unRoe * o + 0.5) * d0 + (nx * o) * d1 + (ny * o) * d2;
  const T a0 = sqrt_pos(unRoe * unRoe + EPS) * w0;
  const T um = unRoe - cRoe, up = unRoe + cRoe;
  const T a1 = sqrt_pos(um * um + EPS) * w1;
  const T a2 = sqrt_pos(up * up + EPS) * w2;
  const T r0 = a1 + a2;
  const T T0 = ny * a0, T1 = (uRoe - cRoe * nx) * a1, T2 = (uRoe + cRoe * nx) * a2;
  const T U0 = (-nx) * a0, U1 = (vRoe - cRoe * ny) * a1, U2 = (vRoe + cRoe * ny) * a2;
  // physical fluxes (the pressures of both sides are unchanged by the
  // mirror branches: they depend on xi and h_still only)
  const T fA0 = huA * nx + hvA * ny;
  const T fA1 = (huA * uA + A.p) * nx + huA * vA * ny;
  const T fA2 = (hvA * uA) * nx + (hvA * vA + A.p) * ny;
  const T fB0 = huB * nx + hvB * ny;
  const T fB1 = (huB * uB + B.p) * nx + huB * vB * ny;
  const T fB2 = (hvB * uB) * nx + (hvB * vB + B.p) * ny;
  const T s0 = fA0 + fB0, s1 = fA1 + fB1, s2 = fA2 + fB2;
  fa[0] = (s0 - r0) * 0.5;
  fa[1] = (s1 - ((T0 + T1) + T2)) * 0.5;
  fa[2] = (s2 - ((U0 + U1) + U2)) * 0.5;
  if (BOTH) {
    fb[0] = -fa[0];
    fb[1] = -((s1 - ((T0 + T2) + T1)) * 0.5);
    fb[2] = -((s2 - ((U0 + U2) + U1)) * 0.5);
  }
}

}  // namespace hg
