// hg_adj_tile.hpp -- device functions of the tiled reverse step: ghost states
// and the routing of their cotangents, a tile's cells in LDS, and the VJP of
// one work item.
#pragma once
#include <hip/hip_runtime.h>

#include "hg_adjoint.hpp"
#include "hg_tile.hpp"

namespace hg {

// A boundary face's ghost state (bc_2D.jl:640-834) formed from its cell's
// flux inputs `me`, and what the routing of its cotangent back to the cell
// needs (the ghost's kind; inlet-Q: the ghost velocity v and wet flag w).
struct GhostAdj {
  int kind, bc;
  double v, w;
};

__device__ __forceinline__ CellQ adj_ghost_state(const AdjArgs& a, const CellQ& me, double n_i, int gi,
                                                     double nx, double ny, GhostAdj& gs, double& rh, double& r2s) {
#pragma clang fp contract(on)
  const double hsmall = a.hsmall;
  gs.kind = a.g_kind[gi];
  gs.bc = a.g_bc[gi];
  gs.v = 0.0;
  gs.w = 0.0;
  double hgh, qxg, qyg;
  switch (gs.kind) {
    case HG_BC_INLETQ: {
      gs.w = (me.h > hsmall) ? 1.0 : 0.0;
      gs.v = a.inletQ[gs.bc] / a.totalA[gs.bc] * a.g_L23[gi] / n_i;
      hgh = me.h;
      qxg = -me.h * gs.v * nx * gs.w;
      qyg = -me.h * gs.v * ny * gs.w;
      break;
    }
    case HG_BC_EXITH: {
      const double hx = a.exitWSE[gs.bc] - me.zb;
      hgh = (hx > hsmall) ? hx : hsmall;
      qxg = me.hu;
      qyg = me.hv;
      break;
    }
    case HG_BC_WALL:
      hgh = me.h;
      qxg = -me.hu;
      qyg = -me.hv;
      break;
    default: {
      const double vdn = me.hu * nx + me.hv * ny;
      hgh = me.h;
      qxg = me.hu - 2.0 * vdn * nx;
      qyg = me.hv - 2.0 * vdn * ny;
      break;
    }
  }
  CellQ B;
  B.hs = a.g_hstill[gi];
  B.xi = hgh - B.hs;
  B.h = hgh;
  B.hu = qxg;
  B.hv = qyg;
  B.zb = a.g_zb[gi];
  rh = rcp_est(hgh);
  const double he = hgh + EPS, rs = rsq_est(he);
  B.u = qxg * rh;
  B.v = qyg * rh;
  B.s = he * rs;
  r2s = 0.5 * rs;
  B.p = a.half_g * ((B.xi + EPS) * (B.xi + EPS) + 2.0 * B.xi * B.hs);
  return B;
}

// Routes the ghost's cotangent Bb back through its boundary rule: adds to
// the cell's U, and its n / exit-H bed cotangents; writes the inlet ghost's
// velocity cotangent for the inlet conveyance adjoint.
__device__ __forceinline__ void adj_ghost_route(const AdjArgs& a, const CellQ& me, double n_i, int gi,
                                                const GhostAdj& gs, const SideBar& Bb, double nx, double ny,
                                                SideBar& U, double& nb, double& zbb) {
#pragma clang fp contract(on)
  const double hgb = Bb.h + Bb.xi;  // xi_g = h_g - hstill_g
  switch (gs.kind) {
    case HG_BC_INLETQ: {  // h_g = h, q_g = -h v n w, v = (Q / A) L^(2/3) / n
      const double v = gs.v, w = gs.w;
      U.h += hgb + Bb.hu * (-v * nx * w) + Bb.hv * (-v * ny * w);
      const double vb = Bb.hu * (-me.h * nx * w) + Bb.hv * (-me.h * ny * w);
      nb += vb * (-v / n_i);
      store_state(a.vbar + gi, vb);  // at device scope: other tiles of a resident run poll it
      break;
    }
    case HG_BC_EXITH: {  // h_g = max(h_small, WSE - zb_cell), q_g = q
      if (a.exitWSE[gs.bc] - me.zb > a.hsmall) zbb -= hgb;
      U.hu += Bb.hu;
      U.hv += Bb.hv;
      break;
    }
    case HG_BC_WALL:
      U.h += hgb;
      U.hu -= Bb.hu;
      U.hv -= Bb.hv;
      break;
    default: {
      const double vdnb = -2.0 * (Bb.hu * nx + Bb.hv * ny);
      U.h += hgb;
      U.hu += Bb.hu + vdnb * nx;
      U.hv += Bb.hv + vdnb * ny;
      break;
    }
  }
}

constexpr int kAdjRows = 13;  // CellQ without h and p (8), z (3), 1 / h, 0.5 / s

// Rows: 0 xi, 1 h_still, 2 hu, 3 hv, 4 zb, 5 u, 6 v, 7 s, 8-10 z, 11 1 / h,
// 12 0.5 / s.  The depth and the pressure are re-formed where read, with
// make_cellq's operations.
template <int T>
__device__ __forceinline__ CellQ lds_cellq(const double* C, int r, double half_g, double hsmall) {
#pragma clang fp contract(on)
  CellQ q;
  q.xi = C[0 * T + r]; q.hs = C[1 * T + r]; q.hu = C[2 * T + r]; q.hv = C[3 * T + r];
  q.zb = C[4 * T + r]; q.u = C[5 * T + r]; q.v = C[6 * T + r]; q.s = C[7 * T + r];
  double h = q.xi + q.hs;
  if (h <= hsmall) h = hsmall;
  q.h = h;
  q.p = half_g * ((q.xi + EPS) * (q.xi + EPS) + 2.0 * q.xi * q.hs);
  return q;
}

// A cell's flux inputs as the tiled reverse step forms them, for the tile's
// own cells and for cross-tile neighbours alike (so a face's VJP has the same
// bits whichever work-group evaluates it): make_cellq's clamp and pressure,
// with u and v from one reciprocal of h and sqrt(h + eps) and its reciprocal
// from one rsqrt.  rh = 1 / h, r2s = 0.5 / sqrt(h + eps).
__device__ __forceinline__ CellQ adj_cellq(double xi, double hs, double qx, double qy, double zb, double half_g,
                                               double hsmall, double& rh, double& r2s) {
#pragma clang fp contract(on)
  CellQ c;
  c.xi = xi;
  c.hs = hs;
  double h = xi + hs, hu = qx, hv = qy;
  if (h <= hsmall) {
    h = hsmall;
    hu = 0.0;
    hv = 0.0;
  }
  c.h = h;
  c.hu = hu;
  c.hv = hv;
  c.zb = zb;
  rh = rcp_est(h);
  c.u = hu * rh;
  c.v = hv * rh;
  const double he = h + EPS;
  const double rs = rsq_est(he);
  c.s = he * rs;
  r2s = 0.5 * rs;
  c.p = half_g * ((xi + EPS) * (xi + EPS) + 2.0 * xi * hs);
  return c;
}

// A cross-tile neighbour's raw data as a work item of the tiled reverse step
// reads it.
struct NbrRaw {
  double xi, hs, qx, qy, zb, m0, m1, m2, dt, area;
  uint8_t clamped;
};

template <bool STEP>
__device__ __forceinline__ NbrRaw nbr_load(const AdjArgs& a, int j) {
  NbrRaw r;
  r.xi = a.xi[j]; r.hs = a.hstill[j]; r.qx = a.qx[j]; r.qy = a.qy[j]; r.zb = a.zb[j];
  r.m0 = a.lx[j]; r.m1 = a.lqx[j]; r.m2 = a.lqy[j];
  r.clamped = (STEP && a.mask) ? a.mask[j] : uint8_t(0);
  r.dt = a.dtc ? a.dtc[j] : a.dt;
  r.area = a.area[j];
  return r;
}

// One work item of the tiled reverse step (see k_adj_tile); nr is the
// neighbour of a cross-tile item.
template <bool STEP, int T, int MD>
__device__ __forceinline__ void adj_item(const AdjArgs& a, int t, const double* C, double* S, int32_t* Xm,
                                         const ItemRec& rec, const NbrRaw& nr) {
#pragma clang fp contract(on)
  const double hsmall = a.hsmall, half_g = a.half_g;
  const int code = rec.code;
  const int ia = code & 1023, ka = (code >> 10) & 15;
  const int ib = (code >> 14) & 1023, kb = (code >> 24) & 15;
  const int type = (code >> 28) & 3;
  const double nx = rec.nx, ny = rec.ny, L = rec.len;
  // P / Q: the evaluation's first / second side (normal from P)
  const bool sw = type != 2 && !(nx > 0.0 || (nx == 0.0 && ny > 0.0));
  const double ex = sw ? -nx : nx, ey = sw ? -ny : ny;
  CellQ P, Q;
  double zP0, zP1, zP2, zQ0, zQ1, zQ2, rhP, rhQ, r2P, r2Q;
  int ip = ia, kp = ka, iq = ia, kq = ka;  // LDS slots of P and Q (type 0); the tile's cell otherwise
  GhostAdj gs{};
  double n_a = 0.0;
  if (type == 0) {
    if (sw) { ip = ib; kp = kb; } else { iq = ib; kq = kb; }
    P = lds_cellq<T>(C, ip, half_g, hsmall);
    Q = lds_cellq<T>(C, iq, half_g, hsmall);
    zP0 = C[8 * T + ip]; zP1 = C[9 * T + ip]; zP2 = C[10 * T + ip];
    zQ0 = C[8 * T + iq]; zQ1 = C[9 * T + iq]; zQ2 = C[10 * T + iq];
    rhP = C[11 * T + ip]; r2P = C[12 * T + ip];
    rhQ = C[11 * T + iq]; r2Q = C[12 * T + iq];
  } else {
    const CellQ Lc = lds_cellq<T>(C, ia, half_g, hsmall);
    const double zL0 = C[8 * T + ia], zL1 = C[9 * T + ia], zL2 = C[10 * T + ia];
    const double rhL = C[11 * T + ia], r2L = C[12 * T + ia];
    CellQ G;
    double zG0 = 0.0, zG1 = 0.0, zG2 = 0.0;
    double rhG, r2G;
    if (type == 1) {  // cross-tile neighbour
      G = adj_cellq(nr.xi, nr.hs, nr.qx, nr.qy, nr.zb, half_g, hsmall, rhG, r2G);
      double m0 = nr.m0, m1 = nr.m1, m2 = nr.m2;
      if (nr.clamped) m0 = m1 = m2 = 0.0;
      const double rAj = rcp_est(nr.area);
      zG0 = (STEP ? nr.dt * m0 : m0) * rAj;
      zG1 = (STEP ? nr.dt * m1 : m1) * rAj;
      zG2 = (STEP ? nr.dt * m2 : m2) * rAj;
    } else {  // ghost (no cotangent of its own)
      n_a = a.n[t * T + ia];
      G = adj_ghost_state(a, Lc, n_a, rec.ref, nx, ny, gs, rhG, r2G);
    }
    P = sw ? G : Lc;
    Q = sw ? Lc : G;
    zP0 = sw ? zG0 : zL0; zP1 = sw ? zG1 : zL1; zP2 = sw ? zG2 : zL2;
    zQ0 = sw ? zL0 : zG0; zQ1 = sw ? zL1 : zG1; zQ2 = sw ? zL2 : zG2;
    rhP = sw ? rhG : rhL; r2P = sw ? r2G : r2L;
    rhQ = sw ? rhL : rhG; r2Q = sw ? r2L : r2G;
  }
  const double c[3] = {L * zQ0 - L * zP0, L * zQ1 - L * zP1, L * zQ2 - L * zP2};
  ExtBar eP, eQ;
  roe_vjp_ext(P, Q, ex, ey, a.g, half_g, hsmall, c, eP, eQ);
  SideBar sP = ext_to_side_r(eP, P, rhP, r2P, half_g);
  const SideBar sQ = ext_to_side_r(eQ, Q, rhQ, r2Q, half_g);
  if (type == 2) {
    double nb = 0.0, zbb = 0.0;
    adj_ghost_route(a, P, n_a, rec.ref, gs, sQ, nx, ny, sP, nb, zbb);
    if (gs.kind == HG_BC_EXITH) {
      S[(3 * MD + ka) * T + ia] = zbb;
      atomicOr(&Xm[ia], 1 << ka);
    } else {
      S[(3 * MD + ka) * T + ia] = nb;
    }
  }
  if (type == 0 || !sw) {
    S[(0 * MD + kp) * T + ip] = (P.h > hsmall) ? sP.xi + sP.h : sP.xi;
    S[(1 * MD + kp) * T + ip] = sP.hu;
    S[(2 * MD + kp) * T + ip] = sP.hv;
  }
  if (type == 0 || sw) {
    S[(0 * MD + kq) * T + iq] = (Q.h > hsmall) ? sQ.xi + sQ.h : sQ.xi;
    S[(1 * MD + kq) * T + iq] = sQ.hu;
    S[(2 * MD + kq) * T + iq] = sQ.hv;
  }
}

}  // namespace hg
