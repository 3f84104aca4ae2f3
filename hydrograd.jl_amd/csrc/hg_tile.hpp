// hg_tile.hpp -- device functions shared by the step kernels: the inlet fold,
// ghost states, work items and the state store.
#pragma once
#include <hip/hip_runtime.h>

#include "hg_ctx.hpp"
#include "hg_roe_pair.hpp"

namespace hg {

constexpr int kTileInlets = 64;  // inlet boundaries one tile may touch when the conveyance is fused

// acc + the first cnt lanes' terms of this wave, one after the other (lanes
// from cnt on hold +0.0; the terms are not negative, so the zeros that fill
// the last group of eight change nothing).  A lane read costs two scalar
// moves; a lane exchange through LDS per term instead took 8.8 us, not 6.9, for
// a resident step of a 96k-cell channel whose inlet has 69 faces.
__device__ __forceinline__ double wave_left_fold(double acc, double term, int cnt) {
  const long long v = __double_as_longlong(term);
  const int lo = int(v), hi = int(v >> 32);
  for (int k = 0; k < cnt; k += 8)
#pragma unroll
    for (int u = 0; u < 8; ++u)
      acc = acc + __hiloint2double(__builtin_amdgcn_readlane(hi, k + u), __builtin_amdgcn_readlane(lo, k + u));
  return acc;
}

// The new state of a step, stored as a relaxed store at device (agent)
// scope: the same vector store with the device-scope cache policy bit
// (sc1).  The next step's kernel reads these values, from any XCD; on the
// 1M-cell channel the step kernel measured about 1 % faster with it than
// with plain stores (the stored values are the same).
__device__ __forceinline__ void store_state(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// What a boundary face's ghost state reads besides its cell and the inlet's
// conveyance: p is the inlet's discharge or the outlet's stage.
template <class T>
struct GhostFaceT {
  int kind, bc;
  double hs, L23;
  T zb, p;
};
using GhostFace = GhostFaceT<double>;
template <class T = double, class Args>
__device__ __forceinline__ GhostFaceT<T> ghost_face(const Args& a, int gi) {
  GhostFaceT<T> g;
  g.kind = a.g_kind[gi];
  g.bc = a.g_bc[gi];
  g.hs = a.g_hstill[gi];
  g.zb = T(a.g_zb[gi]);
  g.L23 = a.g_L23[gi];
  g.p = T(g.kind == HG_BC_INLETQ ? a.inletQ[g.bc] : g.kind == HG_BC_EXITH ? a.exitWSE[g.bc] : 0.0);
  return g;
}

// A boundary face's ghost state (bc_2D.jl:640-834) as the flux reads it,
// formed from its internal cell's flux inputs A (Manning n: n_i); tot: the
// conveyance of an inlet-Q ghost's inlet.
template <class T>
__device__ __forceinline__ CellQT<T> ghost_cellq(const GhostFaceT<T>& g, const CellQT<T>& A, const T& n_i,
                                                     double nx, double ny, const T& tot, double half_g,
                                                     double hsmall) {
  // chosen value by value, as in roe_pair
  const bool inlet = g.kind == HG_BC_INLETQ, exit = g.kind == HG_BC_EXITH, wall = g.kind == HG_BC_WALL;
  T qn(0.0);  // inlet: the discharge into the domain (per width)
  if (inlet) qn = A.h * (g.p / tot * g.L23 / n_i) * ((A.h > hsmall) ? 1.0 : 0.0);
  const T hx = g.p - A.zb;
  const T h = pick(exit, pick(hx > hsmall, hx, T(hsmall)), A.h);
  const T vdn = A.hu * nx + A.hv * ny;
  T qx = pick(inlet, -qn * nx, pick(exit, A.hu, pick(wall, -A.hu, A.hu - 2.0 * vdn * nx)));
  T qy = pick(inlet, -qn * ny, pick(exit, A.hv, pick(wall, -A.hv, A.hv - 2.0 * vdn * ny)));
  CellQT<T> B;
  B.hs = g.hs;
  B.xi = h - B.hs;
  B.h = h;
  B.hu = qx;
  B.hv = qy;
  B.zb = g.zb;
  const double rh = rcp_est(h);
  B.u = div_est(qx, h, rh);
  B.v = div_est(qy, h, rh);
  B.s = sqrt_pos(h + EPS);
  B.p = half_g * ((B.xi + EPS) * (B.xi + EPS) + 2.0 * B.xi * B.hs);
  return B;
}

// Work item it of a tile whose items before ix0 carry a ref (see ItemTable).
__device__ __forceinline__ ItemRec load_item(const ItemTable& tb, int it, int ix0) {
  ItemRec r;
  r.code = tb.code[it];
  r.ref = it < ix0 ? tb.ref[it] : 0;
  const ItemGeo g = tb.geo[it];
  r.nx = g.nx;
  r.ny = g.ny;
  r.len = g.len;
  return r;
}

}  // namespace hg
