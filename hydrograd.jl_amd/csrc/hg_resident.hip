// hg_resident.hip -- resident runs (see hg_resident.hpp): the tile of
// k_swe_tile held on the device over many right-hand sides, as Euler steps
// (on doubles, or dual numbers for forward mode), as an adaptive Tsit5
// integration, and in reverse.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "hg_adj_tile.hpp"
#include "hg_ctx.hpp"
#include "hg_dual.hpp"
#include "hg_lux.hpp"
#include "hg_nlaw.hpp"
#include "hg_resident.hpp"
#include "hg_tile.hpp"
#include "hg_tsit5.hpp"
#include "hgswe.h"

namespace hg {
namespace {

constexpr int kBlock = 256;

// ---- resident run: many steps of a small mesh in one launch.
// A step of a mesh of up to about 130,000 cells is one dependent chain --
// launch, cell loads, items, neighbours, two barriers -- of 7 us and more,
// however few cells it has; the chip is mostly idle.  Here every tile keeps
// its cells, their constants and its work items in registers for the whole
// run, and only the cells that another tile reads travel through memory.
// Per step: 1,000 quads 7.4 -> 2.5 us; a closed 59k-triangle mesh about 7 ->
// 3.7 us; channels, whose inlet tiles also wait for all of the inlet's cells
// and fold their conveyance, 3.5 us at 1,300 cells, 4.0 at 20k, 6.5 at 96k
// (8.7 us with one launch per step) and 6.8 at 126k.  Larger meshes do not fit
// on the chip in this form.
//
// Exchange: a published cell's new state goes to slot (s + 1) % 4 of a ring of
// four states, whose entries hold kResEmpty (a signalling NaN no arithmetic
// produces) until then; a reader polls the values themselves, each a relaxed
// agent-scope access, so one memory trip carries data and readiness.  When a
// tile publishes state s + 1 it has read its neighbours' state s, hence they
// have read its state s - 1 (face and inlet neighbours are mutual): it resets
// that slot, which state s + 3 takes, and the wait before publishing s + 2
// completes the reset before any reader can poll for s + 3.
//
// All tiles must be on the device together: the host launches no more
// work-groups than fit, and every wait is bounded (kResTicks); a wait that
// runs out raises ctl[0], every tile then leaves, and the host repeats the
// steps with one launch each (the input state is not written).
//
// The first T work-items own the cells; the cross-tile items go to others, so
// a poll is not queued behind the publishing stores; the last wave forms the
// inlet conveyances; the cells' friction is formed while the faces are
// waited for.  Each work-item takes at most one item: tiles of triangles hold
// up to 256, others up to 320 (fuller tiles are not run this way).  SPLIT
// (few tiles): the cells' work-items take no items, so the friction is off the
// step's critical path; else they take the items that the rest leave.
constexpr unsigned long long kResEmpty = 0x7ff4c0de5ea1ed01ull;
// wall_clock64 ticks (100 MHz) that a wait may take: 1 s.  A constant: from memory or scalar registers the bound cost 2
// to 3 % of a step of 1,000 cells, through the code around the polling loop.
constexpr long long kResTicks = 100000000;
constexpr int kResIn = 128;                 // inlet faces whose constants a tile keeps in LDS
constexpr int res_threads(int MD, bool split) { return res_items(MD) + (split ? kResT : 0); }

__device__ __forceinline__ unsigned long long res_peek(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void res_put(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The NC values p, p + stride, ...: waits until none is empty.  False when
// the wait ran out here or elsewhere.
template <int NC>
__device__ __forceinline__ bool res_poll(const unsigned long long* p, int64_t stride, int32_t* ctl, double (&v)[NC]) {
  long long t0 = 0;
  for (int n = 0;; ++n) {
    unsigned long long u[NC];
    bool ready = true;
    for (int c = 0; c < NC; ++c) u[c] = res_peek(p + c * stride);
    for (int c = 0; c < NC; ++c) ready = ready && u[c] != kResEmpty;
    if (ready) {
      for (int c = 0; c < NC; ++c) v[c] = __longlong_as_double((long long)u[c]);
      return true;
    }
    if ((n & 63) == 63) {
      const long long t = wall_clock64();
      if (n == 63) t0 = t;
      if (t - t0 > kResTicks) __hip_atomic_store(ctl, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (__hip_atomic_load(ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
        for (int c = 0; c < NC; ++c) v[c] = 0.0;
        return false;
      }
    }
  }
}

__global__ __launch_bounds__(kBlock) void k_res_init(int64_t n, unsigned long long* ring, int32_t* ctl) {
  const int64_t i = int64_t(blockIdx.x) * kBlock + threadIdx.x;
  if (i < n) ring[i] = kResEmpty;
  if (i == 0) *ctl = 0;
}

// ---- scalars: double, or Dual1 (value and tangent)
template <class T>
struct Words {
  static constexpr int W = 1;
};
template <>
struct Words<Dual1> {
  static constexpr int W = 2;
};
__device__ __forceinline__ double from_words(double, const double* v) { return v[0]; }
__device__ __forceinline__ Dual1 from_words(Dual1, const double* v) { return Dual1(v[0], v[1]); }
__device__ __forceinline__ double with_tangent(double v, const double*, int) { return v; }
__device__ __forceinline__ Dual1 with_tangent(Dual1 v, const double* d, int i) { return Dual1(v.v, d ? d[i] : 0.0); }
__device__ __forceinline__ double word(double v, int) { return v; }
__device__ __forceinline__ double word(const Dual1& v, int w) { return w ? v.d : v.v; }
__device__ __forceinline__ double left_fold(double acc, double term, int cnt) { return wave_left_fold(acc, term, cnt); }
__device__ __forceinline__ Dual1 left_fold(const Dual1& acc, const Dual1& term, int cnt) {
  return Dual1(wave_left_fold(acc.v, term.v, cnt), wave_left_fold(acc.d, term.d, cnt));
}

// One tile of a resident run: the constants of this work-item's cell and work
// item in registers, and one RHS evaluation (k_swe_tile<false>'s values).
template <class T, int MD, bool SPLIT, int NM>
struct ResTile {
  static constexpr int TT = kResT, NT = res_threads(MD, SPLIT), W = Words<T>::W, NC = 3 * W;
  static constexpr int kRows = NM ? 10 : 9;  // xi, h, hu, hv, zb, u, v, s, p and, when it changes, n
  static constexpr int kNet = NM == RES_N_NET ? W * kLuxPadN : 0;  // the network's weights (and tangents)

  static constexpr size_t lds_bytes() {
    return size_t((kRows + 3 * MD) * W * TT + W * kTileInlets + (2 + W) * kResIn + kNet) * sizeof(double) +
           (kResIn + 1) * sizeof(int32_t);
  }

  const TileArgs& a;
  const ResArgs& R;
  double *C, *FL, *tA, *net, *in_c;
  int32_t *in_i, *stop;
  int t, tid, i, d, it_code, type, ref, in0, in1, bl0, fl0, fl1;
  bool own, pub, has;
  double hs, A, dti, ks, nx, ny, len;
  T zb, n, S0x, S0y, gn;
  GhostFaceT<T> gf;  // the other side's constants: a cross-tile neighbour's h_still and zb, or the ghost's

  __device__ __forceinline__ ResTile(const TileArgs& a_, const ResArgs& R_) : a(a_), R(R_) {}

  __device__ __forceinline__ T get(const double* B, int row, int x) const {
    double v[W];
    for (int w = 0; w < W; ++w) v[w] = B[(row * W + w) * TT + x];
    return from_words(T(), v);
  }
  __device__ __forceinline__ void put(double* B, int row, int x, const T& q) const {
    for (int w = 0; w < W; ++w) B[(row * W + w) * TT + x] = word(q, w);
  }
  __device__ __forceinline__ CellQT<T> cell(int x) const {
    CellQT<T> q;
    q.xi = get(C, 0, x); q.h = get(C, 1, x); q.hu = get(C, 2, x); q.hv = get(C, 3, x); q.zb = get(C, 4, x);
    q.u = get(C, 5, x); q.v = get(C, 6, x); q.s = get(C, 7, x); q.p = get(C, 8, x);
    q.hs = 0.0;  // the flux takes it through p
    return q;
  }
  // The law's n, or the network's output, at one cell's state.
  __device__ __forceinline__ T closure(const T& xi, const T& qx, const T& qy, double hsc, double ksc) const {
    if (NM == RES_N_LAW) {
      T h, U;
      nlaw_features<T>(R.law, xi, qx, qy, hsc, a.hsmall, h, U);
      return nlaw_eval<T, false>(R.law, h, U, ksc, nullptr, nullptr, nullptr);
    }
    T f[3];
    lux_features<T>(R.net, xi, qx, qy, hsc, a.hsmall, ksc, f);
    return lux_eval<4, T>(R.net, LuxPad{net, net + kLuxPadN, R.net.n_hidden}, f);
  }
  __device__ __forceinline__ bool gives_n() const { return NM == RES_N_LAW || R.net.choice != LUX_FLOW_RESISTANCE; }

  __device__ __forceinline__ void setup(double* lds, T& xi, T& qx, T& qy) {
    C = lds;
    FL = C + kRows * W * TT;
    tA = FL + 3 * MD * W * TT;
    net = tA + W * kTileInlets;
    in_c = net + kNet;
    in_i = reinterpret_cast<int32_t*>(in_c + (2 + W) * kResIn);
    stop = in_i + kResIn;
    t = blockIdx.x;
    tid = threadIdx.x;
    i = t * TT + tid;
    own = tid < TT && i < a.N;
    hs = 0.0; A = 1.0; dti = a.dt; ks = 1.0;
    xi = qx = qy = zb = n = S0x = S0y = T(0.0);
    d = 0;
    pub = false;  // read by another tile, or an inlet cell
    if (own) {
      xi = with_tangent(T(a.xi[i]), R.dxi, i);
      qx = with_tangent(T(a.qx[i]), R.dqx, i);
      qy = with_tangent(T(a.qy[i]), R.dqy, i);
      hs = a.hstill[i];
      zb = with_tangent(T(a.zb[i]), R.dzb, i);
      n = with_tangent(T(a.n[i]), R.dn, i);
      S0x = with_tangent(T(a.S0x[i]), R.dS0x, i);
      S0y = with_tangent(T(a.S0y[i]), R.dS0y, i);
      A = a.area[i];
      if (NM && R.ks) ks = R.ks[i];
      d = a.deg ? a.deg[i] : MD;
      if (a.dtc) dti = a.dtc[i];
      for (int k = 0; k < d; ++k) {
        const int j = R.nbr[int64_t(k) * a.N + i];
        pub = pub || (j >= 0 ? j / TT != t : a.g_kind[~j] == HG_BC_INLETQ);
      }
    }
    // this work-item's item (the cross-tile ones are the first of the list)
    const int it = a.items.off[t] + (SPLIT ? tid - TT : (tid + NT - TT) % NT);
    has = it >= a.items.off[t] && it < a.items.off[t + 1];
    ItemRec rec{};
    if (has) rec = load_item(a.items, it, a.items.x0[t]);
    it_code = rec.code;
    ref = rec.ref;
    nx = rec.nx; ny = rec.ny; len = rec.len;
    type = has ? (it_code >> 28) & 3 : 3;
    gf = GhostFaceT<T>{};
    gn = T(1.0);
    if (type == 1) {
      gf.hs = a.hstill[ref];
      gf.zb = with_tangent(T(a.zb[ref]), R.dzb, ref);
    } else if (type == 2) {
      gf = ghost_face<T>(a, ref);
      gf.zb = with_tangent(gf.zb, R.dg_zb, ref);
      if (gf.kind == HG_BC_INLETQ) gf.p = with_tangent(gf.p, R.dinletQ, gf.bc);
      const int c = t * TT + (it_code & 1023);
      gn = with_tangent(T(a.n[c]), R.dn, c);
    }
    in0 = a.n_inlet > 0 ? a.tile_in_off[t] : 0;
    in1 = a.n_inlet > 0 ? a.tile_in_off[t + 1] : 0;
    bl0 = fl0 = fl1 = 0;  // the tile's first inlet
    if (in1 > in0) {
      bl0 = a.tile_in_list[in0];
      fl0 = a.in_off[bl0];
      fl1 = a.in_off[bl0 + 1];
      for (int f = tid; f < min(kResIn, fl1 - fl0); f += NT) {
        const int c = a.in_cell[fl0 + f];
        const T nc = with_tangent(T(a.n[c]), R.dn, c);
        in_i[f] = c;
        in_c[f] = a.in_L53[fl0 + f];
        in_c[kResIn + f] = a.hstill[c];
        for (int w = 0; w < W; ++w) in_c[(2 + w) * kResIn + f] = word(nc, w);
      }
    }
    if (NM == RES_N_NET) {
      lux_pad_fill(R.net, R.net_w, net, tid, NT);
      if (W > 1) lux_pad_fill(R.net, R.net_dw, net + kLuxPadN, tid, NT);
    }
    if (tid == 0) *stop = 0;
    __syncthreads();
  }

  // Inlet face f (the k-th of its inlet): the conveyance term of evaluation s.
  __device__ __forceinline__ T conveyance_term(int64_t s, int f, int k, bool kept, bool& ok) const {
    const unsigned long long* slot = R.ring + (s & 3) * NC * a.N;
    const int c = kept ? in_i[k] : a.in_cell[f];
    T x[3];
    constexpr int M = NM ? 3 : 1;  // a law or network may read the discharge too
    if (s == 0) {
      x[0] = with_tangent(T(a.xi[c]), R.dxi, c);
      x[1] = with_tangent(T(a.qx[c]), R.dqx, c);
      x[2] = with_tangent(T(a.qy[c]), R.dqy, c);
    } else {
      double v[M * W];
      bool got = true;
      if (W == 1) {
        got = res_poll<M>(slot + c, a.N, R.ctl, reinterpret_cast<double(&)[M]>(v));
      } else {  // values are the first three components, tangents the others
        double lo[M], hi[M];
        got = res_poll<M>(slot + c, a.N, R.ctl, lo);
        got = res_poll<M>(slot + 3 * int64_t(a.N) + c, a.N, R.ctl, hi) && got;
        for (int m = 0; m < M; ++m) {
          v[m * W] = lo[m];
          v[m * W + W - 1] = hi[m];
        }
      }
      for (int m = 0; m < M; ++m) x[m] = from_words(T(), v + m * W);
      ok = ok && got;
    }
    const double hsc = kept ? in_c[kResIn + k] : a.hstill[c];
    T h = x[0] + hsc;
    if (h <= a.hsmall) h = T(a.hsmall);
    const double w = (h > a.hsmall) ? 1.0 : 0.0;
    T nc;
    if (NM && gives_n()) {
      nc = closure(x[0], x[1], x[2], hsc, R.ks ? R.ks[c] : 1.0);
    } else if (kept) {
      double v[W];
      for (int m = 0; m < W; ++m) v[m] = in_c[(2 + m) * kResIn + k];
      nc = from_words(T(), v);
    } else {
      nc = with_tangent(T(a.n[c]), R.dn, c);
    }
    return (kept ? in_c[k] : a.in_L53[f]) * h / nc * w;
  }

  // dQ/dt of this work-item's cell at its state (evaluation s: the border
  // cells' states are in slot s % 4, or the input arrays for s = 0).  False
  // when a wait ran out; the whole tile then leaves.
  __device__ __forceinline__ bool eval(int64_t s, const T& xi, const T& qx, const T& qy, T (&dq)[3]) {
    const double hsmall = a.hsmall;
    CellQT<T> me{};
    T nv = n, mag(0.0);
    if (own) {
      me = make_cellq(xi, hs, qx, qy, zb, a.half_g, hsmall);
      put(C, 0, tid, me.xi); put(C, 1, tid, me.h); put(C, 2, tid, me.hu); put(C, 3, tid, me.hv); put(C, 4, tid, me.zb);
      put(C, 5, tid, me.u); put(C, 6, tid, me.v); put(C, 7, tid, me.s); put(C, 8, tid, me.p);
      if (NM) {
        const T o = closure(xi, qx, qy, hs, ks);
        if (gives_n())
          nv = o;
        else
          mag = o;
        put(C, 9, tid, nv);
        if (R.rec_n) R.rec_n[s * a.N + i] = word(o, 0);
      }
    }
    if (in1 > in0 && tid >= NT - 64) {  // inlet conveyances (as in k_swe_tile)
      const int l = tid & 63;
      for (int sl = in0; sl < in1; ++sl) {
        const int b = sl == in0 ? bl0 : a.tile_in_list[sl];
        const int f0 = sl == in0 ? fl0 : a.in_off[b], f1 = sl == in0 ? fl1 : a.in_off[b + 1];
        T acc(0.0);
        bool ok = true;
        constexpr int P = NM || W > 1 ? 1 : 2;  // faces per lane in flight
        for (int base = f0; base < f1; base += 64 * P) {
          T term[P];
#pragma unroll
          for (int r = 0; r < P; ++r) {
            const int f = base + 64 * r + l;
            term[r] = T(0.0);
            if (f < f1) term[r] = conveyance_term(s, f, f - f0, sl == in0 && base - f0 + 64 * P <= kResIn, ok);
          }
#pragma unroll
          for (int r = 0; r < P; ++r)
            if (f1 - base > 64 * r) acc = left_fold(acc, term[r], min(64, f1 - base - 64 * r));
        }
        if (__ballot(!ok)) {
          *stop = 1;
        } else if (l == 0) {
          for (int w = 0; w < W; ++w) tA[(sl - in0) * W + w] = word(acc, w);
          if (R.rec_totalA) R.rec_totalA[s * R.n_inlet + b] = word(acc, 0);  // every tile of inlet b writes the same value
          if (!(word(acc, 0) > 1e-10)) a.flag[0] = 1;
        }
      }
    }
    __syncthreads();
    if (has) {
      const int ia = it_code & 1023, ka = (it_code >> 10) & 15, ib = (it_code >> 14) & 1023, kb = (it_code >> 24) & 15;
      const CellQT<T> P = cell(ia);
      CellQT<T> Q;
      if (type == 0) {
        Q = cell(ib);
      } else if (type == 1) {
        T x[3];
        if (s == 0) {
          x[0] = with_tangent(T(a.xi[ref]), R.dxi, ref);
          x[1] = with_tangent(T(a.qx[ref]), R.dqx, ref);
          x[2] = with_tangent(T(a.qy[ref]), R.dqy, ref);
        } else {
          double v[NC];
          if (!res_poll<NC>(R.ring + (s & 3) * NC * a.N + ref, a.N, R.ctl, v)) *stop = 1;
          for (int c = 0; c < 3; ++c) {
            const double q[2] = {v[c], v[NC - 3 + c]};
            x[c] = from_words(T(), q);
          }
        }
        Q = make_cellq(x[0], gf.hs, x[1], x[2], gf.zb, a.half_g, hsmall);
      } else {
        T tot(0.0);
        if (gf.kind == HG_BC_INLETQ) {
          double v[W];
          for (int w = 0; w < W; ++w) v[w] = tA[((it_code >> 14) & (kTileInlets - 1)) * W + w];
          tot = from_words(T(), v);
        }
        Q = ghost_cellq(gf, P, NM ? get(C, NM ? 9 : 0, ia) : gn, nx, ny, tot, a.half_g, hsmall);
      }
      T fa[3], fb[3];
      roe_pair<true>(P, Q, nx, ny, a.g, a.half_g, hsmall, fa, fb);
      if (type == 0)
        for (int c = 0; c < 3; ++c) put(FL, c * MD + kb, ib, fb[c] * len);
      for (int c = 0; c < 3; ++c) put(FL, c * MD + ka, ia, fa[c] * len);
    }
    T s1(0.0), s2(0.0);
    if (own && me.h > hsmall) {
      T fx, fy;
      if (NM == RES_N_NET && !gives_n())
        friction_mag(mag, me.hu, me.hv, fx, fy);
      else
        friction(a.g, a.kn2, hsmall, me.h, me.hu, me.hv, nv, fx, fy);
      s1 = a.g * xi * S0x - fx;
      s2 = a.g * xi * S0y - fy;
    }
    const double rA = rcp_est(A);
    __syncthreads();
    if (*stop) {  // the same for the whole tile: set before the barrier only
      if (tid == 0) a.flag[2] = 1;
      return false;
    }
    if (!own) return true;
    T acc0(0.0), acc1(0.0), acc2(0.0);
    for (int k = 0; k < MD; ++k) {  // local face order
      if (k < d) {
        acc0 = acc0 + get(FL, 0 * MD + k, tid);
        acc1 = acc1 + get(FL, 1 * MD + k, tid);
        acc2 = acc2 + get(FL, 2 * MD + k, tid);
      }
    }
    dq[0] = div_est(-acc0, A, rA) + 0.0;
    dq[1] = div_est(-acc1, A, rA) + s1;
    dq[2] = div_est(-acc2, A, rA) + s2;
    return true;
  }

  // Makes a border cell's state of evaluation s known to the other tiles, and
  // empties the slot that evaluation s + 2 takes.
  __device__ __forceinline__ void publish(int64_t s, const T& xi, const T& qx, const T& qy) {
    if (!(own && pub)) return;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last reset is done (lgkmcnt, expcnt not waited on)
    const int64_t N = a.N;
    unsigned long long* o = R.ring + (s & 3) * NC * N + i;
    unsigned long long* e = R.ring + ((s + 2) & 3) * NC * N + i;
    for (int w = 0; w < W; ++w) {
      res_put(o + (3 * w + 0) * N, __double_as_longlong(word(xi, w)));
      res_put(o + (3 * w + 1) * N, __double_as_longlong(word(qx, w)));
      res_put(o + (3 * w + 2) * N, __double_as_longlong(word(qy, w)));
    }
    for (int c = 0; c < NC; ++c) res_put(e + c * N, kResEmpty);
  }
};

// Registers: two waves per SIMD (one tile per CU) except the field-n variants.
constexpr int res_waves(bool split, int nmode, bool dual) { return nmode || dual ? 2 : split ? 3 : 4; }

template <class T, int MD, bool SPLIT, int NM>
__global__ __launch_bounds__(res_threads(MD, SPLIT), res_waves(SPLIT, NM, Words<T>::W == 2)) void k_swe_run(TileArgs a,
                                                                                                     ResArgs R) {
  extern __shared__ double lds[];
  ResTile<T, MD, SPLIT, NM> rt(a, R);
  T xi, qx, qy;
  rt.setup(lds, xi, qx, qy);
  const int64_t N = a.N;
  const int i = rt.i;
  for (int64_t s = 0; s < R.ns; ++s) {
    T dq[3];
    if (!rt.eval(s, xi, qx, qy, dq)) return;
    if (!rt.own) continue;
    xi = xi + rt.dti * dq[0];
    qx = qx + rt.dti * dq[1];
    qy = qy + rt.dti * dq[2];
    const bool dry = xi < a.hsmall;
    if (dry) {
      xi = T(a.hsmall);
      qx = T(0.0);
      qy = T(0.0);
    }
    if (s + 1 < R.ns) rt.publish(s + 1, xi, qx, qy);
    const double x = word(xi, 0), u = word(qx, 0), v = word(qy, 0);
    // checked after the stepping call (a forward-mode run does not report it)
    if (Words<T>::W == 1 && !(isfinite(x) && isfinite(u) && isfinite(v))) a.flag[1] = 1;
    if (R.rec) {
      double* q = R.rec + (s + 1) * 3 * N + i;
      q[0] = x;
      q[N] = u;
      q[2 * N] = v;
      R.rec_clamp[s * N + i] = dry ? 1 : 0;
    }
  }
  if (rt.own) {
    a.xo[i] = word(xi, 0);
    a.qxo[i] = word(qx, 0);
    a.qyo[i] = word(qy, 0);
    if (Words<T>::W == 2) {
      R.dxo[i] = word(xi, 1);
      R.dqxo[i] = word(qx, 1);
      R.dqyo[i] = word(qy, 1);
    }
  }
}

// Adaptive Tsit5 (hg_tsit5_solve's steps) resident: the stages of a cell stay
// in its tile's LDS; every right-hand side exchanges the border cells, and every
// trial step the tiles' error sums (each tile adds them in the same order, so
// all take the same decision).  Leaves after P.trials trial steps, or when the
// integration is done or fails; the next launch goes on from P.out.
__constant__ double kTsitA[7][6] = {
    {tsit5::a[0][0], tsit5::a[0][1], tsit5::a[0][2], tsit5::a[0][3], tsit5::a[0][4], tsit5::a[0][5]},
    {tsit5::a[1][0], tsit5::a[1][1], tsit5::a[1][2], tsit5::a[1][3], tsit5::a[1][4], tsit5::a[1][5]},
    {tsit5::a[2][0], tsit5::a[2][1], tsit5::a[2][2], tsit5::a[2][3], tsit5::a[2][4], tsit5::a[2][5]},
    {tsit5::a[3][0], tsit5::a[3][1], tsit5::a[3][2], tsit5::a[3][3], tsit5::a[3][4], tsit5::a[3][5]},
    {tsit5::a[4][0], tsit5::a[4][1], tsit5::a[4][2], tsit5::a[4][3], tsit5::a[4][4], tsit5::a[4][5]},
    {tsit5::a[5][0], tsit5::a[5][1], tsit5::a[5][2], tsit5::a[5][3], tsit5::a[5][4], tsit5::a[5][5]},
    {tsit5::a[6][0], tsit5::a[6][1], tsit5::a[6][2], tsit5::a[6][3], tsit5::a[6][4], tsit5::a[6][5]}};

template <int MD, int NM>
__global__ __launch_bounds__(res_threads(MD, true), 2) void k_tsit5_run(TileArgs a, ResArgs R, Tsit5Args P) {
  extern __shared__ double lds[];
  __shared__ double red[kResRed];
  using Tile = ResTile<double, MD, true, NM>;
  Tile rt(a, R);
  double y[3];
  rt.setup(lds, y[0], y[1], y[2]);
  double* K = lds + Tile::lds_bytes() / sizeof(double) + 1 + rt.tid;  // [7][3] of this cell, kResT apart
  auto k_of = [&](int g, int c) -> double& { return K[(3 * g + c) * kResT]; };
  const int64_t N = a.N, n3 = 3 * N;
  const int tid = rt.tid, i = rt.i, nt = gridDim.x;
  Tsit5State st{P.t0, P.dt0, 1, 0, 0, 1, HG_OK, 0, 0};
  auto save = [&](int64_t k) {
    if (rt.own)
      for (int c = 0; c < 3; ++c) P.frames[k * n3 + c * N + P.perm[i]] = y[c];
  };
  int64_t ev = 0;  // evaluation 0 reads the input arrays; a launch that goes on has none and starts at 4
  if (P.in) {
    st = *P.in;
    if (rt.own)
      for (int c = 0; c < 3; ++c) k_of(0, c) = P.k0[c * N + i];
    ev = 4;
  } else {
    save(0);
    double k0[3] = {0.0, 0.0, 0.0};
    if (!rt.eval(0, y[0], y[1], y[2], k0)) return;
    if (rt.own)
      for (int c = 0; c < 3; ++c) k_of(0, c) = k0[c];
    ev = 1;
  }
  for (int64_t trial = 0; trial < P.trials && !st.done; ++trial) {
    if (st.accepted + st.rejected >= P.max_steps) {
      st.code = HG_ERR_STATE;
      st.sub = 2;
      break;
    }
    const double tt = (st.frame == P.n_save) ? P.t1 : P.t0 + (P.t1 - P.t0) * double(st.frame) / double(P.n_save);
    const bool last = st.dt >= (tt - st.t) * (1.0 - 1e-12);
    const double h = last ? tt - st.t : st.dt;
    double x[3] = {0.0, 0.0, 0.0};
#pragma unroll 1
    for (int g = 1; g < 7; ++g) {  // stages 2..7; stage 7's input is the new solution
      if (rt.own)
        for (int c = 0; c < 3; ++c) {
          double s = 0.0;
          for (int j = 0; j < g; ++j) s += (h * kTsitA[g][j]) * k_of(j, c);
          x[c] = y[c] + s;
        }
      rt.publish(ev, x[0], x[1], x[2]);
      double kg[3] = {0.0, 0.0, 0.0};
      if (!rt.eval(ev, x[0], x[1], x[2], kg)) return;
      ++ev;
      if (rt.own)
        for (int c = 0; c < 3; ++c) k_of(g, c) = kg[c];
    }
    st.nrhs += 6;
    double v = 0.0;
    if (rt.own) {
      for (int c = 0; c < 3; ++c) {
        double e = 0.0;
#pragma unroll
        for (int j = 0; j < 7; ++j) e += (h * tsit5::btilde[j]) * k_of(j, c);
        const double sc = P.abstol + P.reltol * fmax(fabs(y[c]), fabs(x[c]));
        v += (e / sc) * (e / sc);
      }
    }
    for (int w = 32; w > 0; w >>= 1) v += __shfl_xor(v, w, 64);
    if ((tid & 63) == 0) red[tid >> 6] = v;
    __syncthreads();
    const int64_t q = st.accepted + st.rejected;  // this trial step's slot
    if (tid == 0) {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last reset is done
      res_put(P.red + (q & 3) * kResRed + rt.t, __double_as_longlong(red[0] + red[1]));
      res_put(P.red + ((q + 2) & 3) * kResRed + rt.t, kResEmpty);
    }
    __syncthreads();
    double part[1] = {0.0};
    if (tid < nt && !res_poll<1>(P.red + (q & 3) * kResRed + tid, 0, R.ctl, part)) *rt.stop = 1;
    if (tid < kResRed) red[tid] = part[0];
    __syncthreads();
    if (*rt.stop) {
      if (tid == 0) a.flag[2] = 1;
      return;
    }
    double ss = 0.0;
    for (int w = 0; w < kResRed; w += 64) ss += red[w + (tid & 63)];
    for (int w = 32; w > 0; w >>= 1) ss += __shfl_xor(ss, w, 64);
    __syncthreads();  // red is reused
    const double err = ::sqrt(ss / double(n3));
    if (!isfinite(err)) {
      st.code = HG_ERR_NONFINITE;
      break;
    }
    const double fac = tsit5::step_factor(err);
    if (err <= 1.0) {  // accept: the new solution and its derivative (first same as last)
      st.t = last ? tt : st.t + h;
      for (int c = 0; c < 3; ++c) {
        y[c] = x[c];
        if (rt.own) k_of(0, c) = k_of(6, c);
      }
      ++st.accepted;
      const double hn = h * fmin(10.0, fmax(0.2, fac));
      if (!last || hn < st.dt) st.dt = hn;
    } else {
      ++st.rejected;
      st.dt = h * fmax(0.2, fac);
    }
    if (st.dt < 1e-14 * (P.t1 - P.t0)) {
      st.code = HG_ERR_STATE;
      st.sub = 1;
      break;
    }
    if (!(st.t < tt)) {
      save(st.frame);
      st.done = st.frame == P.n_save;
      ++st.frame;
    }
  }
  if (rt.own)
    for (int c = 0; c < 3; ++c) {
      P.y[c * N + i] = y[c];
      P.k0[c * N + i] = k_of(0, c);
    }
  if (rt.t == 0 && tid == 0) *P.out = st;
}

// Reverse mode of a resident run: R.ns steps of k_adj_tile and k_inlet_adj in
// one launch over tiles of 128 cells, with the values they form, in their
// order (same bits).  A tile keeps its cells' cotangents and sums in
// registers and reads ahead the recorded state of the next step; the border
// cells' cotangents and the inlet ghosts' velocity cotangents travel through
// rings as the forward run's states do (see k_swe_run).  Sums are written to
// arrays of their own (o_*), which the host takes over when the run is done.
// One launch per step took 8.5 us for the tiles and 2.6 us for the inlets, of
// which about 3 us and 1 us were launch and first loads; a step takes 4.6 us
// here on 1,000 quads, 5.8 on a 1,300-cell channel (its inlet tiles exchange
// twice per step) and 6.4 on 59k triangles.  Up to 512 tiles: the registers
// that hold the cells allow two tiles per CU.
constexpr int adj_run_base_doubles(int MD) {  // without the network's values
  return (kAdjRows + 4 * MD) * kResT + 512 + kTileInlets + (kResT + 2) / 2;
}
template <int MD>
__device__ __forceinline__ int32_t* adj_run_stop(double* lds) {
  return reinterpret_cast<int32_t*>(lds + (kAdjRows + 4 * MD) * kResT + 512 + kTileInlets) + kResT;
}
// The network's derivatives are formed by a work-item of their own for each
// cell, one step ahead of the cells' and faces' (adj_run_net).
constexpr int adj_run_threads(int MD, int NM) { return res_items(MD) + (NM == RES_N_NET ? kResT : 0); }
// LDS of the network: two values per weight and cell, four per cell, the padded weights.
constexpr int adj_run_net_doubles(int P) { return 2 * P * kResT + 4 * kResT + kLuxPadN; }

// The network's part of a resident reverse run, by the tile's last kResT
// work-items (cell c): for every step, the derivatives of the network's output
// by the weights (J, one value per weight and cell) and by the cell's state
// (Cs), from the recorded state alone; then the sums over the steps of J times
// the output's cotangent, which the cell's work-item leaves in Ob.  The forward
// pass of the next step runs while the cells finish theirs.  Takes every
// barrier that the tile's other work-items take.  A step of the [3, 3] network
// on 180 cells takes 10.1 us, and took 12.9 with the derivatives formed by the
// cells' own work-items between the faces and the sums.
template <int NH>
__device__ __forceinline__ bool adj_run_net(const AdjArgs& a, const AdjRunArgs& R, const LuxPad& pad, double* J,
                                            double* Wsum, double* Cs, const double* Ob, const int32_t* stop, int i,
                                            bool own, int n_in) {
  constexpr int T = kResT;
  const int64_t N = a.N;
  const int ns = lux_state_inputs(R.net), P = R.net.P;
  const double hs = own ? a.hstill[i] : 0.0, ksc = R.ks && own ? R.ks[i] : 1.0;
  double q[3] = {0.0, 0.0, 0.0}, nx[3] = {0.0, 0.0, 0.0};  // the step's recorded state, and the next one's
  auto read_ahead = [&](int64_t k) {
    if (own)
      for (int c = 0; c < 3; ++c) nx[c] = R.rec[(k * 3 + c) * N + i];
  };
  LuxPass<4, NH> pass;
  auto forward = [&] {
    double f[3];
    lux_features<double>(R.net, q[0], q[1], q[2], hs, a.hsmall, ksc, f);
    lux_pass<4, NH>(R.net, pad, f, pass);
  };
  auto add = [&] {
    const double ob = Ob[0];
#pragma unroll 8
    for (int p = 0; p < P; ++p) Wsum[p * T] += ob * J[p * T];
  };
  if (own)
    for (int p = 0; p < P; ++p) Wsum[p * T] = 0.0;
  __syncthreads();  // the padded weights
  read_ahead(R.ns - 1);
  for (int64_t r = -1; r < R.ns; ++r) {
    if (r >= 0) __syncthreads();  // the last step's Ob is there, its Cs has been read
    if (r >= 0 && own) {
      if (r > 0) add();
      double df[3];
      lux_jacobian<4, NH>(R.net, pad, pass, J, T, df);
      lux_state_derivatives(R.net, ns, q, hs, a.hsmall, ksc, df, Cs, T);
    }
    if (r >= 0) {
      __syncthreads();
      if (*stop) return false;
    }
    if (r + 1 < R.ns) {  // the next step's state and forward pass
      for (int c = 0; c < 3; ++c) q[c] = nx[c];
      if (r + 2 < R.ns) read_ahead(R.ns - 3 - r);
      if (own) forward();
    }
    for (int k = 0; r >= 0 && k < n_in; ++k) {
      __syncthreads();
      if (*stop) return false;
      for (int b = 0; b < 3; ++b) __syncthreads();
    }
  }
  __syncthreads();  // the last Ob
  if (own) add();
  return true;
}

// The cells and faces of a tile, by its first res_items(MD) work-items; false
// when a wait ran out.
template <int MD, int NM>
__device__ __forceinline__ bool adj_run_cells(AdjArgs a, const AdjRunArgs& R, double* lds) {
  constexpr int T = kResT, NT = res_items(MD);
  double* C = lds;                                         // kAdjRows x T
  double* S = lds + kAdjRows * T;                          // 4 x MD x T
  double* sA = S + 4 * MD * T;                             // 256
  double* sQ = sA + 256;                                   // 256
  double* qa = sQ + 256;                                   // kTileInlets: the inlets' discharge cotangents
  int32_t* Xm = reinterpret_cast<int32_t*>(qa + kTileInlets);  // T
  int32_t* stop = adj_run_stop<MD>(lds);
  const int t = blockIdx.x, tid = threadIdx.x, i = t * T + tid;
  const bool own = tid < T && i < a.N;
  const int64_t N = a.N;
  const double hsmall = a.hsmall;
  const bool mag = NM == RES_N_NET && R.net.choice == LUX_FLOW_RESISTANCE;  // the output is the friction magnitude
  double* const Cs = lds + adj_run_base_doubles(MD) + 2 * (NM == RES_N_NET ? R.net.P : 0) * T + tid;  // see adj_run_net
  const double ksc = NM == RES_N_LAW && R.ks && own ? R.ks[i] : 1.0;
  double hs = 0.0, zb = 0.0, n = 0.0, S0x = 0.0, S0y = 0.0, A = 1.0, dti = a.dt;
  double l0 = 0.0, l1 = 0.0, l2 = 0.0, nbar = 0.0, zbbar = 0.0, S0bx = 0.0, S0by = 0.0;
  int d = 0;
  bool pub = false;  // read by another tile
  if (own) {
    hs = a.hstill[i]; zb = a.zb[i]; n = a.n[i]; S0x = a.S0x[i]; S0y = a.S0y[i]; A = a.area[i];
    d = a.deg ? a.deg[i] : MD;
    if (a.dtc) dti = a.dtc[i];
    l0 = a.lx[i]; l1 = a.lqx[i]; l2 = a.lqy[i];
    if (a.nbar) nbar = a.nbar[i];
    if (a.zbbar) {
      zbbar = a.zbbar[i];
      S0bx = a.S0bar[i];
      S0by = a.S0bar[N + i];
    }
    for (int k = 0; k < d; ++k) {
      const int j = a.nbr[k * N + i];
      pub = pub || (j >= 0 && j / T != t);
    }
  }
  const int it = a.items.off[t] + (tid + NT - T) % NT;
  const bool has = it < a.items.off[t + 1];
  ItemRec rec{};
  if (has) rec = load_item(a.items, it, a.items.x0[t]);
  const int type = has ? (rec.code >> 28) & 3 : 3;
  NbrRaw nr{};
  if (type == 1) {
    nr.hs = a.hstill[rec.ref]; nr.zb = a.zb[rec.ref]; nr.area = a.area[rec.ref];
    nr.dt = a.dtc ? a.dtc[rec.ref] : a.dt;
  }
  const bool in_ghost = type == 2 && a.g_kind[rec.ref] == HG_BC_INLETQ;
  const int in0 = R.n_inlet > 0 ? R.tile_in_off[t] : 0, in1 = R.n_inlet > 0 ? R.tile_in_off[t + 1] : 0;
  int my_sl = -1, my_f = -1;  // an inlet cell's inlet and first face there
  for (int sl = in0; sl < in1; ++sl) {
    const int b = R.tile_in_list[sl];
    for (int f = R.in_off[b]; f < R.in_off[b + 1]; ++f)
      if (own && R.in_rec[f].cell == i && R.in_rec[f].first) {
        my_sl = sl;
        my_f = f;
      }
    if (tid == 0) qa[sl - in0] = R.Qbar[b];
  }
  if (tid == 0) *stop = 0;
  // the recorded state of the step (own cell, and a cross-tile neighbour's), read one step ahead
  double px = 0.0, pqx = 0.0, pqy = 0.0, jx = 0.0, jqx = 0.0, jqy = 0.0, pn = 0.0;
  uint8_t pm = 0, jm = 0;
  auto read_ahead = [&](int64_t k) {
    const double* q = R.rec + k * 3 * N;
    const uint8_t* m = R.rec_clamp + k * N;
    if (own) {
      px = q[i]; pqx = q[N + i]; pqy = q[2 * N + i];
      pm = m[i];
      if (NM) pn = R.rec_n[k * N + i];
    }
    if (type == 1) {
      jx = q[rec.ref]; jqx = q[N + rec.ref]; jqy = q[2 * N + rec.ref];
      jm = m[rec.ref];
    }
  };
  read_ahead(R.ns - 1);
  if (NM == RES_N_NET) __syncthreads();

  for (int64_t r = 0; r < R.ns; ++r) {
    const int64_t k = R.ns - 1 - r;  // the step that is reversed
    const unsigned long long* slot = R.ring + (r & 3) * 3 * N;
    a.totalA = R.rec_totalA ? R.rec_totalA + k * R.n_inlet : nullptr;
    a.vbar = reinterpret_cast<double*>(R.vring + (r & 3) * R.G);
    CellQ me{};
    double y0 = 0.0, y1 = 0.0, y2 = 0.0;
    const double sx1 = pqx, sx2 = pqy;  // the raw discharge of the step's state
    double ncl = 0.0;  // the law's or network's value of this step
    if (NM) {
      ncl = pn;
      if (!mag) {
        n = pn;
        a.n = R.rec_n + k * N;
      }
    }
    if (pm) l0 = l1 = l2 = 0.0;
    nr.xi = jx; nr.qx = jqx; nr.qy = jqy;
    nr.clamped = jm;
    if (own) {
      double rh, r2s;
      me = adj_cellq(px, hs, pqx, pqy, zb, a.half_g, hsmall, rh, r2s);
      const double rA = rcp_est(A);
      y0 = dti * l0;
      y1 = dti * l1;
      y2 = dti * l2;
      C[0 * T + tid] = me.xi; C[1 * T + tid] = me.hs; C[2 * T + tid] = me.hu; C[3 * T + tid] = me.hv;
      C[4 * T + tid] = me.zb; C[5 * T + tid] = me.u; C[6 * T + tid] = me.v; C[7 * T + tid] = me.s;
      C[8 * T + tid] = y0 * rA;
      C[9 * T + tid] = y1 * rA;
      C[10 * T + tid] = y2 * rA;
      C[11 * T + tid] = rh;
      C[12 * T + tid] = r2s;
      for (int c = 0; c < MD; ++c) S[(3 * MD + c) * T + tid] = 0.0;
      Xm[tid] = 0;
    }
    if (k > 0) read_ahead(k - 1);
    __syncthreads();
    if (has) {
      if (type == 1) {
        const int j = rec.ref;
        double v[3];
        if (r == 0) {
          v[0] = a.lx[j]; v[1] = a.lqx[j]; v[2] = a.lqy[j];
        } else if (!res_poll<3>(slot + j, N, R.ctl, v)) {
          *stop = 1;
        }
        nr.m0 = v[0]; nr.m1 = v[1]; nr.m2 = v[2];
      }
      if (in_ghost) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): its last reset is done before it publishes again
      adj_item<true, T, MD>(a, t, C, S, Xm, rec, nr);
      if (in_ghost) res_put(R.vring + ((r + 2) & 3) * R.G + rec.ref, kResEmpty);
    }
    // the source term's cotangents, while the faces are waited for
    double sxi = 0.0, sh = 0.0, sqx = 0.0, sqy = 0.0, sn = 0.0, sS0x = 0.0, sS0y = 0.0;
    const bool wet = me.h > hsmall;
    if (own && wet) {
      if (NM == RES_N_NET && mag)
        source_vjp_mag(a.g, me.xi, me.hu, me.hv, ncl, S0x, S0y, y1, y2, sxi, sqx, sqy, sn, sS0x, sS0y);
      else
        source_vjp(a.g, a.kn2, hsmall, me.xi, me.h, me.hu, me.hv, n, S0x, S0y, y1, y2, sxi, sh, sqx, sqy, sn, sS0x,
                   sS0y);
    }
    // the law's derivatives by the cell's state
    double cs[3] = {0.0, 0.0, 0.0};
    if (NM == RES_N_LAW && own) {
      const double q[3] = {me.xi, sx1, sx2};
      const int ns = R.law.kind == NLAW_H_UMAG_KS ? 3 : 1;
      for (int c = 0; c < ns; ++c) {
        const Dual1 x0(q[0], c == 0 ? 1.0 : 0.0), x1(q[1], c == 1 ? 1.0 : 0.0), x2(q[2], c == 2 ? 1.0 : 0.0);
        Dual1 h, U;
        nlaw_features<Dual1>(R.law, x0, x1, x2, hs, hsmall, h, U);
        const double v = nlaw_eval<Dual1, false>(R.law, h, U, ksc, nullptr, nullptr, nullptr).d;
        if (c == 0)
          cs[0] = v;
        else if (c == 1)
          cs[1] = v;
        else
          cs[2] = v;
      }
    }
    __syncthreads();
    if (*stop) {
      if (tid == 0) R.flag[2] = 1;
      return false;
    }
    double ob = 0.0;
    if (own) {
      double uxh = 0.0, uqx = 0.0, uqy = 0.0, nb = 0.0, zbb = 0.0;
      const int xm = Xm[tid];
      for (int c = 0; c < MD; ++c) {  // local face order
        if (c < d) {
          uxh += S[(0 * MD + c) * T + tid];
          uqx += S[(1 * MD + c) * T + tid];
          uqy += S[(2 * MD + c) * T + tid];
          const double e = S[(3 * MD + c) * T + tid];
          if ((xm >> c) & 1)
            zbb += e;
          else
            nb += e;
        }
      }
      double mb = 0.0;
      if (NM == RES_N_NET && mag)
        mb = sn;
      else
        nb += sn;
      double ox = uxh + sxi, oqx = 0.0, oqy = 0.0;
      if (wet) {
        ox += sh;
        oqx = uqx + sqx;
        oqy = uqy + sqy;
      }
      l0 = ox + l0;
      l1 = oqx + l1;
      l2 = oqy + l2;
      ob = mag ? mb : nb;  // this step's cotangent of the closure's output
      if (!NM || mag) nbar = nbar + nb;
      zbbar = zbbar + zbb;
      S0bx = S0bx + sS0x;
      S0by = S0by + sS0y;
    }
    // inlet conveyance adjoint (as k_inlet_adj)
    for (int sl = in0; sl < in1; ++sl) {
      const int b = R.tile_in_list[sl];
      const int f0 = R.in_off[b], f1 = R.in_off[b + 1];
      const double Ai = a.totalA[b], Qb = a.inletQ[b];
      if (tid < 256) {
        double pa = 0.0, pq = 0.0;
        for (int f = f0 + tid; f < f1; f += 256) {
          const InletFaceRec fr = R.in_rec[f];
          double vb[1];
          if (!res_poll<1>(R.vring + (r & 3) * R.G + fr.ghost, 0, R.ctl, vb)) *stop = 1;
          const double nc = a.n[fr.cell];
          const double v = Qb / Ai * fr.L23 / nc;
          pa += vb[0] * (-v / Ai);
          pq += vb[0] * (fr.L23 / (Ai * nc));
        }
        sA[tid] = pa;
        sQ[tid] = pq;
      }
      __syncthreads();
      if (*stop) {
        if (tid == 0) R.flag[2] = 1;
        return false;
      }
      if (tid < 128) {
        sA[tid] += sA[tid + 128];
        sQ[tid] += sQ[tid + 128];
      }
      __syncthreads();
      if (tid < 64) {
        double xa = sA[tid] + sA[tid + 64], xq = sQ[tid] + sQ[tid + 64];
        for (int w = 32; w > 0; w >>= 1) {
          xa = xa + __shfl_xor(xa, w, 64);
          xq = xq + __shfl_xor(xq, w, 64);
        }
        if (tid == 0) {
          sA[0] = xa;
          qa[sl - in0] = qa[sl - in0] + xq;
        }
      }
      __syncthreads();
      if (my_sl == sl) {
        const double h0 = me.xi + hs;
        if (h0 > hsmall) {
          const double Ab = sA[0];
          for (int f = my_f; f >= 0;) {
            const InletFaceRec fr = R.in_rec[f];
            l0 += Ab * fr.L53 / n;
            ob += (NM && !mag) ? Ab * (-fr.L53 * h0 / (n * n)) : 0.0;
            if (!NM || mag) nbar += Ab * (-fr.L53 * h0 / (n * n));
            f = fr.next;
          }
        }
      }
      __syncthreads();  // sA / sQ reuse
    }
    if (NM == RES_N_NET && own) {
      for (int c = 0; c < 3; ++c) cs[c] = Cs[c * T];
      Cs[3 * T] = ob;
    }
    if (NM && own && ob != 0.0) {
      l0 += ob * cs[0];
      l1 += ob * cs[1];
      l2 += ob * cs[2];
    }
    if (own && pub && r + 1 < R.ns) {
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the last step's reset is done
      unsigned long long* o = R.ring + ((r + 1) & 3) * 3 * N + i;
      unsigned long long* e = R.ring + ((r + 3) & 3) * 3 * N + i;
      res_put(o, __double_as_longlong(l0));
      res_put(o + N, __double_as_longlong(l1));
      res_put(o + 2 * N, __double_as_longlong(l2));
      for (int c = 0; c < 3; ++c) res_put(e + c * N, kResEmpty);
    }
  }
  if (own) {
    a.ox[i] = l0;
    a.oqx[i] = l1;
    a.oqy[i] = l2;
    if (R.o_nbar) R.o_nbar[i] = nbar;
    if (R.o_zbbar) {
      R.o_zbbar[i] = zbbar;
      R.o_S0bar[i] = S0bx;
      R.o_S0bar[N + i] = S0by;
    }
  }
  for (int sl = in0 + tid; sl < in1; sl += NT) {  // by the tile of the inlet's first face
    const int b = R.tile_in_list[sl];
    if (R.in_rec[R.in_off[b]].cell / T == t) R.o_Qbar[b] = qa[sl - in0];
  }
  if (NM == RES_N_NET) __syncthreads();
  return true;
}

template <int MD, int NM>
__global__ __launch_bounds__(adj_run_threads(MD, NM), 2) void k_adj_run(AdjArgs a, AdjRunArgs R) {
  extern __shared__ double lds[];
  if constexpr (NM != RES_N_NET) {
    (void)adj_run_cells<MD, NM>(a, R, lds);
  } else {
    constexpr int T = kResT, NT = res_items(MD);
    const int t = blockIdx.x, tid = threadIdx.x, P = R.net.P;
    double* const J = lds + adj_run_base_doubles(MD);
    double* const Wsum = J + P * T;
    double* const Cs = Wsum + P * T;
    double* const net = Cs + 4 * T;
    lux_pad_fill(R.net, R.net_w, net, tid, adj_run_threads(MD, NM));
    if (tid >= NT) {
      const int c = tid - NT, i = t * T + c;
      const LuxPad pad{net, nullptr, R.net.n_hidden};
      const int n_in = R.n_inlet > 0 ? R.tile_in_off[t + 1] - R.tile_in_off[t] : 0;
      const int32_t* stop = adj_run_stop<MD>(lds);
      const bool done = R.net.n_hidden == 1
                            ? adj_run_net<1>(a, R, pad, J + c, Wsum + c, Cs + c, Cs + 3 * T + c, stop, i, i < a.N, n_in)
                            : adj_run_net<2>(a, R, pad, J + c, Wsum + c, Cs + c, Cs + 3 * T + c, stop, i, i < a.N, n_in);
      if (!done) return;
    } else if (!adj_run_cells<MD, NM>(a, R, lds)) {
      return;
    }
    __syncthreads();
    for (int p = tid / 64; p < P; p += adj_run_threads(MD, NM) / 64) {  // the tile's sum per weight, by a fixed tree
      const int l = tid & 63;
      const double v = lux_tile_sum(Wsum + p * T, t * T, a.N, l);
      if (l == 0) R.o_wpart[int64_t(p) * gridDim.x + t] = v;
    }
  }
}

size_t adj_run_lds_bytes(int MD, int P) {
  return (size_t(adj_run_base_doubles(MD)) + (P ? adj_run_net_doubles(P) : 0)) * sizeof(double);
}

// Tiles per CU: a tile's waves need not spread evenly over the four SIMDs (two
// tiles of six waves each were not resident together where three waves fit
// per SIMD), so each tile counts with its fullest SIMD.
template <class F>
int capacity(F* kernel, int threads, size_t lds, int waves_per_simd, int ncu) {
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, threads, lds) != hipSuccess) return 0;
  return std::min(per_cu, waves_per_simd / ((threads / 64 + 3) / 4)) * ncu;
}

template <class T, int MD, bool SPLIT, int NM>
struct RunVariant {
  using Tile = ResTile<T, MD, SPLIT, NM>;
  static int cap(int ncu) {
    return capacity(k_swe_run<T, MD, SPLIT, NM>, Tile::NT, Tile::lds_bytes(), res_waves(SPLIT, NM, Words<T>::W == 2),
                    ncu);
  }
  static void launch(hipStream_t st, int ntiles, const TileArgs& a, const ResArgs& R) {
    hipLaunchKernelGGL((k_swe_run<T, MD, SPLIT, NM>), dim3(ntiles), dim3(Tile::NT), Tile::lds_bytes(), st, a, R);
  }
};

// Calls f(RunVariant) for the variant k; false when there is none.
template <class F>
bool with_variant(const ResKind& k, F&& f) {
  if (!k.split) {
    if (k.nmode || k.dual) return false;
    k.md == 3 ? f(RunVariant<double, 3, false, 0>()) : f(RunVariant<double, 4, false, 0>());
    return true;
  }
#define HG_RUN_MD(T, NM) (k.md == 3 ? f(RunVariant<T, 3, true, NM>()) : f(RunVariant<T, 4, true, NM>()))
  if (k.dual)
    k.nmode == 0 ? HG_RUN_MD(Dual1, 0) : k.nmode == 1 ? HG_RUN_MD(Dual1, 1) : HG_RUN_MD(Dual1, 2);
  else
    k.nmode == 0 ? HG_RUN_MD(double, 0) : k.nmode == 1 ? HG_RUN_MD(double, 1) : HG_RUN_MD(double, 2);
#undef HG_RUN_MD
  return true;
}

template <int MD, int NM>
struct Tsit5Variant {
  using Tile = ResTile<double, MD, true, NM>;
  static constexpr size_t lds = Tile::lds_bytes() + (21 * kResT + 2) * sizeof(double);
  static int cap(int ncu) { return std::min(kResRed, capacity(k_tsit5_run<MD, NM>, Tile::NT, lds, 2, ncu)); }
  static void launch(hipStream_t st, int ntiles, const TileArgs& a, const ResArgs& R, const Tsit5Args& P) {
    hipLaunchKernelGGL((k_tsit5_run<MD, NM>), dim3(ntiles), dim3(Tile::NT), lds, st, a, R, P);
  }
};
template <class F>
void with_tsit5(int md, int nm, F&& f) {
#define HG_TSIT5_MD(NM) (md == 3 ? f(Tsit5Variant<3, NM>()) : f(Tsit5Variant<4, NM>()))
  nm == 0 ? HG_TSIT5_MD(0) : nm == 1 ? HG_TSIT5_MD(1) : HG_TSIT5_MD(2);
#undef HG_TSIT5_MD
}

template <int MD, int NM>
struct AdjVariant {
  static int cap(int P, int ncu) {
    return capacity(k_adj_run<MD, NM>, adj_run_threads(MD, NM), adj_run_lds_bytes(MD, P), 2, ncu);
  }
  static void launch(hipStream_t st, int P, int ntiles, const AdjArgs& a, const AdjRunArgs& R) {
    hipLaunchKernelGGL((k_adj_run<MD, NM>), dim3(ntiles), dim3(adj_run_threads(MD, NM)), adj_run_lds_bytes(MD, P), st, a, R);
  }
};
template <class F>
void with_adj_run(int md, int nm, F&& f) {
#define HG_ADJ_MD(NM) (md == 3 ? f(AdjVariant<3, NM>()) : f(AdjVariant<4, NM>()))
  nm == 0 ? HG_ADJ_MD(0) : nm == 1 ? HG_ADJ_MD(1) : HG_ADJ_MD(2);
#undef HG_ADJ_MD
}

}  // namespace

int res_capacity(const ResKind& k, int ncu) {
  int c = 0;
  with_variant(k, [&](auto v) { c = v.cap(ncu); });
  return c;
}

int adj_run_capacity(int md, int nmode, int net_P, int ncu) {
  int c = 0;
  with_adj_run(md, nmode, [&](auto v) { c = v.cap(nmode == RES_N_NET ? net_P : 0, ncu); });
  return c;
}

int tsit5_capacity(int md, int nmode, int ncu) {
  int c = 0;
  with_tsit5(md, nmode, [&](auto v) { c = v.cap(ncu); });
  return c;
}

hipError_t res_init(hipStream_t stream, int64_t n, unsigned long long* ring, int32_t* ctl) {
  hipLaunchKernelGGL(k_res_init, dim3(unsigned((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, stream, n, ring, ctl);
  return hipGetLastError();
}

hipError_t launch_run(hipStream_t stream, const ResKind& k, int ntiles, const TileArgs& a, const ResArgs& R) {
  if (!with_variant(k, [&](auto v) { v.launch(stream, ntiles, a, R); })) return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_adj_run(hipStream_t stream, int md, int nmode, int ntiles, const AdjArgs& a, const AdjRunArgs& R) {
  with_adj_run(md, nmode, [&](auto v) { v.launch(stream, nmode == RES_N_NET ? R.net.P : 0, ntiles, a, R); });
  return hipGetLastError();
}

hipError_t launch_tsit5(hipStream_t stream, int md, int nmode, int ntiles, const TileArgs& a, const ResArgs& R,
                        const Tsit5Args& P) {
  with_tsit5(md, nmode, [&](auto v) { v.launch(stream, ntiles, a, R, P); });
  return hipGetLastError();
}

}  // namespace hg
