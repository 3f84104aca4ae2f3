// hg_lux.hpp -- the reference's UDE network on the device, in FP64.
//
// create_NN_model (process_UDE.jl:2-65) builds a Lux chain
//   [Dense(in, w_l, act_l) -> LayerNorm(w_l)] per hidden layer l,
//   Dense(w_L, 1), then x -> lo + (hi - lo) sigmoid(x)  (output bounds),
// and the RHS feeds it inputs normalised to [-1, 1] by bounds,
//   x_norm = 2 (x - x_lo) / (x_hi - x_lo) - 1,
// per UDE_choice:
//   ManningN_h          h                     -> n   (process_ManningN_2D.jl:216-273)
//   ManningN_h_Umag_ks  h, |U| = |q| / h, ks  -> n
//   FlowResistance      h, |q|_eps            -> friction magnitude
//                       (process_FlowResistance_UDE.jl:3-46, |q| bounds
//                        h_lo U_lo .. h_hi U_hi; semi_discretize_swe_2D.jl:521-531)
// with h the clamped depth and q the masked discharge of the RHS.
//
// Layer semantics are Lux's and NNlib's published ones: Dense y = act(W x + b)
// with W (out x in); LayerNorm over the units of one cell, uncorrected
// variance, y = (a - mean) / sqrt(var + eps) * scale + bias, eps = 1f-5 (as
// Float64); NNlib's relu, leakyrelu (slope 0.01), sigmoid
// (exp(-|x|) form), tanh and softplus (log1p(exp(-|x|)) + relu(x)).
//
// One cell per lane, every layer in registers (widths up to MW, a compile-
// time bound; runtime widths are predicates).  Reverse mode recomputes each
// layer's input from the cell's features instead of storing activations, and
// sums weight cotangents per wave (fixed xor tree) into per-block slots.
#pragma once
#include <hip/hip_runtime.h>

#include "hg_ctx.hpp"
#include "hg_dual.hpp"
#include "hg_nlaw.hpp"
#include "hg_roe_pair.hpp"

namespace hg {

// The weights as the device functions read them: uniform over a wave and
// constant while a kernel runs, through the scalar cache.  As plain pointers
// they were vector loads beside the stores of a resident run (24.0 ms instead
// of 21.3 for the training iteration below).
using LuxW = const __attribute__((address_space(4))) double*;
__device__ __forceinline__ LuxW lux_const(const double* w) { return (LuxW)(reinterpret_cast<uintptr_t>(w)); }

constexpr double kLuxLayerNormEps = 9.999999747378752e-06;  // Float64(1f-5), Lux's LayerNorm default

__device__ __forceinline__ double nn_sigmoid(double x) {  // NNlib.sigmoid
  const double t = ::exp(-::fabs(x)), d = 1.0 + t;
  return div_est(x >= 0.0 ? 1.0 : t, d, rcp_est(d));
}

// tanh(x) = e / (e + 2), e = expm1(2 |x|) = 2^k (expm1(r)) + (2^k - 1) with
// 2 |x| = k ln 2 + r, expm1(r) from its Taylor series to r^14 (|r| <= ln(2)/2:
// the next term is below 2^-61 of r), and the rounding errors of r, e and e + 2
// carried through the quotient.  Below 0.8 ulp from |x| = 1e-300 to 700 on an
// emulation of its operations (tests/test_tanh64_host.py), in 60 instructions;
// the math library's takes 165, and the two hidden layers of the reference's
// networks call it for every unit: 1,000 steps forward and back of a 180-cell
// channel with a [3, 3] network went from 26.8 to 24.3 ms.
__device__ __forceinline__ double tanh64(double x) {
  double y = 2.0 * ::fabs(x);
  y = y > 80.0 ? 80.0 : y;  // 1 - 2 e^-80 is 1; NaN stays NaN
  const double k = __builtin_rint(y * 1.4426950408889634);
  const double r0 = __builtin_fma(-k, 0x1.62e42feep-1, y);  // exact
  const double r = __builtin_fma(-k, 0x1.a39ef35793c76p-33, r0);
  const double rl = __builtin_fma(-k, 0x1.a39ef35793c76p-33, r0 - r);
  double p = 1.0 / 87178291200.0;
  p = __builtin_fma(p, r, 1.0 / 6227020800.0);
  p = __builtin_fma(p, r, 1.0 / 479001600.0);
  p = __builtin_fma(p, r, 1.0 / 39916800.0);
  p = __builtin_fma(p, r, 1.0 / 3628800.0);
  p = __builtin_fma(p, r, 1.0 / 362880.0);
  p = __builtin_fma(p, r, 1.0 / 40320.0);
  p = __builtin_fma(p, r, 1.0 / 5040.0);
  p = __builtin_fma(p, r, 1.0 / 720.0);
  p = __builtin_fma(p, r, 1.0 / 120.0);
  p = __builtin_fma(p, r, 1.0 / 24.0);
  p = __builtin_fma(p, r, 1.0 / 6.0);
  p = __builtin_fma(p, r, 0.5);
  const double c = p * r * r;
  const double ph = r + c, pl = ((r - ph) + c) + __builtin_fma(rl, ph, rl);
  const double s = __builtin_ldexp(1.0, int(k));
  const double a = s * ph, b = s - 1.0;
  const double e = b + a, el = __builtin_fma(s, pl, (b - e) + a);
  const double d = e + 2.0, t = d - e, dl = (e - (d - t)) + (2.0 - t) + el;
  const double yd = rcp_est(d), q = e * yd;
  const double res = __builtin_fma(-q, dl, __builtin_fma(-d, q, e)) + el;
  return __builtin_copysign(__builtin_fma(res, yd, q), x);
}

__device__ __forceinline__ double act_f(int k, double x) {
  switch (k) {
    case ACT_RELU: return x < 0.0 ? 0.0 : x;
    case ACT_LEAKYRELU: return x > 0.0 ? x : 0.01 * x;
    case ACT_SIGMOID: return nn_sigmoid(x);
    case ACT_TANH: return tanh64(x);
    default: return ::log1p(::exp(-::fabs(x))) + (x < 0.0 ? 0.0 : x);  // softplus
  }
}

// d act / dz at z, given a = act(z) (NNlib's derivative rules).
__device__ __forceinline__ double act_d(int k, double z, double a) {
  switch (k) {
    case ACT_RELU: return z > 0.0 ? 1.0 : 0.0;
    case ACT_LEAKYRELU: return z > 0.0 ? 1.0 : 0.01;
    case ACT_SIGMOID: return a * (1.0 - a);
    case ACT_TANH: return 1.0 - a * a;
    default: return nn_sigmoid(z);
  }
}

// Input i normalised to [-1, 1] by its bounds.
template <class T>
__device__ __forceinline__ T lux_normalised(const T& x, const LuxNet& L, int i) {
  const double span = L.in_hi[i] - L.in_lo[i];
  return div_est(2.0 * (x - L.in_lo[i]), span, rcp_est(span)) - 1.0;
}

// Normalised inputs of one cell (features f[0..n_in-1]).
template <class T>
__device__ __forceinline__ void lux_features(const LuxNet& L, const T& xi, const T& qx, const T& qy, double hs,
                                             double hsmall, double ks, T f[3]) {
  T h = xi + hs;
  T hu = qx, hv = qy;
  if (h <= hsmall) {
    h = T(hsmall);
    hu = T(0.0);
    hv = T(0.0);
  }
  f[0] = lux_normalised(h, L, 0);
  f[1] = T(0.0);
  f[2] = T(0.0);
  if (L.choice == LUX_MANNING_H_UMAG_KS) {
    const T u = hu / h, v = hv / h;
    const T U = l_sqrt(u * u + v * v);
    f[1] = lux_normalised(U, L, 1);
    f[2] = T(lux_normalised(ks, L, 2));
  } else if (L.choice == LUX_FLOW_RESISTANCE) {
    const T qm = l_sqrt(hu * hu + hv * hv + EPS);
    f[1] = lux_normalised(qm, L, 1);
  }
}

// Scalars of the forward pass: double, or Dual1 for forward mode (value and
// one tangent; the tangents of the weights may be absent).  The value part of
// a Dual1 pass is computed by the same operations in the same order as the
// double pass, so both give the same bits.
__device__ __forceinline__ double lux_scalar(double, double v, double) { return v; }
__device__ __forceinline__ Dual1 lux_scalar(Dual1, double v, double d) { return Dual1(v, d); }

// The weights where they are: layer widths are predicates.
struct LuxRaw {
  static constexpr bool kPad = false;
  const LuxNet& L;
  LuxW P, dP;
  template <class T>
  __device__ __forceinline__ T at(int k) const {
    return lux_scalar(T(), P[k], sizeof(T) > sizeof(double) && dP ? dP[k] : 0.0);
  }
  template <class T> __device__ __forceinline__ T W(int l, int j, int k) const { return at<T>(L.off_W[l] + j + k * L.width[l]); }
  template <class T> __device__ __forceinline__ T b(int l, int j) const { return at<T>(L.off_b[l] + j); }
  template <class T> __device__ __forceinline__ T g(int l, int j) const { return at<T>(L.off_g[l] + j); }
  template <class T> __device__ __forceinline__ T be(int l, int j) const { return at<T>(L.off_be[l] + j); }
  template <class T> __device__ __forceinline__ T Wo(int k) const { return at<T>(L.off_Wo + k); }
  template <class T> __device__ __forceinline__ T bo() const { return at<T>(L.off_bo); }
};

// A network of at most four units per layer laid out in LDS for a run of many
// steps, every layer padded with zeros to 4 x 4: all offsets are constants and
// no load waits for a predicate.  The zeros leave every sum as it is (units
// beyond the width are masked after the activation).  The small network's
// training iteration (1,000 steps on 180 cells): 21.3 -> 18.9 ms.
constexpr int kLuxPadLayer = 28, kLuxPadN = kLuxMaxLayers * kLuxPadLayer + 6;
struct LuxPad {
  static constexpr bool kPad = true;
  const double *s, *ds;  // values; tangents (Dual1)
  int nh;
  template <class T>
  __device__ __forceinline__ T at(int k) const {
    return lux_scalar(T(), s[k], sizeof(T) > sizeof(double) ? ds[k] : 0.0);
  }
  template <class T> __device__ __forceinline__ T W(int l, int j, int k) const { return at<T>(kLuxPadLayer * l + j + 4 * k); }
  template <class T> __device__ __forceinline__ T b(int l, int j) const { return at<T>(kLuxPadLayer * l + 16 + j); }
  template <class T> __device__ __forceinline__ T g(int l, int j) const { return at<T>(kLuxPadLayer * l + 20 + j); }
  template <class T> __device__ __forceinline__ T be(int l, int j) const { return at<T>(kLuxPadLayer * l + 24 + j); }
  template <class T> __device__ __forceinline__ T Wo(int k) const { return at<T>(kLuxPadLayer * nh + k); }
  template <class T> __device__ __forceinline__ T bo() const { return at<T>(kLuxPadLayer * nh + 4); }
};
// Fills out[0 .. kLuxPadN) from the weights P (zeros without them), by work-item tid of nt.
__device__ __forceinline__ void lux_pad_fill(const LuxNet& L, const double* P, double* out, int tid, int nt) {
  for (int x = tid; x < kLuxPadN; x += nt) {
    const int l = x / kLuxPadLayer, r = x - l * kLuxPadLayer, j = r & 3, q = r >> 2;
    int k = -1;
    if (l < L.n_hidden) {
      const int w = L.width[l], win = l ? L.width[l - 1] : L.n_in;
      if (j < w) k = q < 4 ? (q < win ? L.off_W[l] + j + q * w : -1) : (q == 4 ? L.off_b : q == 5 ? L.off_g : L.off_be)[l] + j;
    } else if (l == L.n_hidden) {
      k = r == 4 ? L.off_bo : r < L.width[L.n_hidden - 1] ? L.off_Wo + r : -1;
    }
    out[x] = P && k >= 0 ? P[k] : 0.0;
  }
}
__device__ __forceinline__ double act_t(int k, double z) { return act_f(k, z); }
__device__ __forceinline__ Dual1 act_t(int k, const Dual1& z) {
  const double a = act_f(k, z.v);
  return Dual1(a, act_d(k, z.v, a) * z.d);
}
__device__ __forceinline__ double sigmoid_t(double x) { return nn_sigmoid(x); }
__device__ __forceinline__ Dual1 sigmoid_t(const Dual1& x) {
  const double s = nn_sigmoid(x.v);
  return Dual1(s, s * (1.0 - s) * x.d);
}
// a = act(z) over one layer.  One activation kind per branch, its units side by
// side in groups of four, so that the tanh or exp chains of a group overlap
// (chosen unit by unit they run one after the other).
template <int K, int MW, class T>
__device__ __forceinline__ void act_units(int w, const T (&z)[MW], T (&a)[MW]) {
#pragma unroll
  for (int j0 = 0; j0 < MW; j0 += 4)
    if (j0 < w) {
#pragma unroll
      for (int j = j0; j < j0 + 4; ++j) a[j] = act_t(K, z[j]);
    }
}
template <int MW, class T>
__device__ __forceinline__ void act_layer(int k, int w, const T (&z)[MW], T (&a)[MW]) {
  switch (k) {
    case ACT_RELU: act_units<ACT_RELU>(w, z, a); break;
    case ACT_LEAKYRELU: act_units<ACT_LEAKYRELU>(w, z, a); break;
    case ACT_SIGMOID: act_units<ACT_SIGMOID>(w, z, a); break;
    case ACT_TANH: act_units<ACT_TANH>(w, z, a); break;
    default: act_units<ACT_SOFTPLUS>(w, z, a); break;
  }
}

// Hidden layer l on input x (width win): pre-activation z, activation a,
// normalised xh = (a - mean) / s.
template <int MW, class T = double, class A>
__device__ __forceinline__ void lux_layer(const LuxNet& L, const A& P, int l, const T (&x)[MW], int win, T (&z)[MW],
                                          T (&a)[MW], T (&xh)[MW], T& s) {
  const int w = L.width[l];
#pragma unroll
  for (int j = 0; j < MW; ++j) {
    z[j] = T(0.0);
    if (A::kPad || j < w) {
      T acc = 0.0;
#pragma unroll
      for (int k = 0; k < MW; ++k)
        if (A::kPad || k < win)
          acc = (k == 0) ? P.template W<T>(l, j, 0) * x[0] : acc + P.template W<T>(l, j, k) * x[k];
      z[j] = acc + P.template b<T>(l, j);
    }
  }
  act_layer<MW, T>(L.act[l], w, z, a);
  if (A::kPad) {
#pragma unroll
    for (int j = 1; j < MW; ++j) a[j] = pick(j < w, a[j], T(0.0));
  }
  const double rw = rcp_est(double(w));
  T mu = a[0];
#pragma unroll
  for (int j = 1; j < MW; ++j)
    if (A::kPad || j < w) mu = mu + a[j];
  mu = div_est(mu, double(w), rw);
  T var = 0.0;
#pragma unroll
  for (int j = 0; j < MW; ++j) {
    if (A::kPad || j < w) {
      T d = a[j] - mu;
      if (A::kPad && j) d = pick(j < w, d, T(0.0));
      var = (j == 0) ? d * d : var + d * d;
    }
  }
  var = div_est(var, double(w), rw);
  s = sqrt_pos(var + L.eps);
  const double rs = rcp_est(s);
#pragma unroll
  for (int j = 0; j < MW; ++j)
    if (A::kPad || j < w) xh[j] = div_est(a[j] - mu, s, rs);
}

// Input of hidden layer `upto` (the last hidden output when upto == n_hidden).
template <int MW, class T = double, class A>
__device__ __forceinline__ int lux_forward_to(const LuxNet& L, const A& P, const T (&f)[3], int upto, T (&x)[MW]) {
#pragma unroll
  for (int k = 0; k < MW; ++k) x[k] = k < 3 ? f[k < 3 ? k : 0] : T(0.0);
  int win = L.n_in;
  for (int l = 0; l < upto; ++l) {
    T z[MW], a[MW], xh[MW], s;
    lux_layer<MW, T>(L, P, l, x, win, z, a, xh, s);
    const int w = L.width[l];
#pragma unroll
    for (int j = 0; j < MW; ++j)
      if (A::kPad || j < w) x[j] = xh[j] * P.template g<T>(l, j) + P.template be<T>(l, j);
    win = w;
  }
  return win;
}

// Output layer and bounds: returns lo + (hi - lo) sigmoid(Wo x + bo).
template <int MW, class T = double, class A>
__device__ __forceinline__ T lux_output(const LuxNet& L, const A& P, const T (&x)[MW], int win, T& sg) {
  T acc = 0.0;
#pragma unroll
  for (int k = 0; k < MW; ++k)
    if (A::kPad || k < win)
      acc = (k == 0) ? P.template Wo<T>(0) * x[0] : acc + P.template Wo<T>(k) * x[k];
  sg = sigmoid_t(acc + P.template bo<T>());
  return L.lo + (L.hi - L.lo) * sg;
}

template <int MW, class T = double, class A>
__device__ __forceinline__ T lux_eval(const LuxNet& L, const A& P, const T (&f)[3]) {
  T x[MW];
  const int win = lux_forward_to<MW, T>(L, P, f, L.n_hidden, x);
  T sg;
  return lux_output<MW, T>(L, P, x, win, sg);
}

// Sum over the 64 lanes of a wave (fixed xor tree: every lane gets the total).
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) v += __shfl_xor(v, m, 64);
  return v;
}

// Reverse mode of one cell: given the output cotangent ob, adds the weight
// cotangents (summed over the wave; lane 0 adds into acc) and returns the
// feature cotangents fb.  Every lane of the wave must call it (lanes without
// a cell pass ob = 0).
template <int MW>
__device__ __forceinline__ void lux_backward(const LuxNet& L, LuxW weights, const double (&f)[3],
                                             double ob, double* acc, int lane, double (&fb)[3]) {
  const LuxRaw P{L, weights, nullptr};
  auto add = [&](int k, double v) {
    v = wave_sum(v);
    if (lane == 0) acc[k] += v;
  };
  double x[MW];
  const int wL = lux_forward_to<MW>(L, P, f, L.n_hidden, x);
  double sg;
  lux_output<MW>(L, P, x, wL, sg);
  const double oo = ob * (L.hi - L.lo) * (sg * (1.0 - sg));
  const LuxW Wo = weights + L.off_Wo;
  double xb[MW];
#pragma unroll
  for (int k = 0; k < MW; ++k) {
    if (k < wL) add(L.off_Wo + k, oo * x[k]);
    xb[k] = k < wL ? oo * Wo[k < wL ? k : 0] : 0.0;
  }
  add(L.off_bo, oo);
  for (int l = L.n_hidden - 1; l >= 0; --l) {
    double xin[MW];
    const int wi = lux_forward_to<MW>(L, P, f, l, xin);
    double z[MW], a[MW], xh[MW], s;
    lux_layer<MW>(L, P, l, xin, wi, z, a, xh, s);
    const int w = L.width[l];
    const LuxW g = weights + L.off_g[l];
    const LuxW W = weights + L.off_W[l];
    double gg[MW];
    double m1 = 0.0, m2 = 0.0;
#pragma unroll
    for (int j = 0; j < MW; ++j) {
      if (j < w) {
        add(L.off_g[l] + j, xb[j] * xh[j]);
        add(L.off_be[l] + j, xb[j]);
        gg[j] = xb[j] * g[j];
        m1 += gg[j];
        m2 += gg[j] * xh[j];
      }
    }
    m1 = m1 / double(w);
    m2 = m2 / double(w);
    double zb[MW];
#pragma unroll
    for (int j = 0; j < MW; ++j) {
      zb[j] = 0.0;
      if (j < w) {
        zb[j] = (gg[j] - m1 - xh[j] * m2) / s * act_d(L.act[l], z[j], a[j]);
#pragma unroll
        for (int k = 0; k < MW; ++k)
          if (k < wi) add(L.off_W[l] + j + k * w, zb[j] * xin[k]);
        add(L.off_b[l] + j, zb[j]);
      }
    }
#pragma unroll
    for (int k = 0; k < MW; ++k) {
      double t = 0.0;
      if (k < wi) {
#pragma unroll
        for (int j = 0; j < MW; ++j)
          if (j < w) t += W[j + k * w] * zb[j];
      }
      xb[k] = t;
    }
  }
  fb[0] = xb[0];
  fb[1] = MW > 1 ? xb[MW > 1 ? 1 : 0] : 0.0;
  fb[2] = MW > 2 ? xb[MW > 2 ? 2 : 0] : 0.0;
}

// The network's derivatives at features f, by the features and by every
// weight, of NH hidden layers of at most MW units, in two halves: the forward
// pass, whose values stay in LuxPass ...
template <int MW, int NHM>
struct LuxPass {
  double xin[NHM][MW], xh[NHM][MW], ad[NHM][MW], s[NHM], x[MW], oo;
};
template <int MW, int NH, int NHM>
__device__ __forceinline__ void lux_pass(const LuxNet& L, const LuxPad& P, const double (&f)[3], LuxPass<MW, NHM>& v) {
#pragma unroll
  for (int k = 0; k < MW; ++k) v.x[k] = k < 3 ? f[k < 3 ? k : 0] : 0.0;
#pragma unroll
  for (int l = 0; l < NH; ++l) {
    double z[MW], a[MW];
    lux_layer<MW>(L, P, l, v.x, 0, z, a, v.xh[l], v.s[l]);
#pragma unroll
    for (int j = 0; j < MW; ++j) {
      v.xin[l][j] = v.x[j];
      v.ad[l][j] = j < L.width[l] ? act_d(L.act[l], z[j], a[j]) : 0.0;
      v.x[j] = v.xh[l][j] * P.g<double>(l, j) + P.be<double>(l, j);
    }
  }
  double sg;
  (void)lux_output<MW>(L, P, v.x, 0, sg);
  v.oo = (L.hi - L.lo) * (sg * (1.0 - sg));
}

// ... and the reverse pass: df, and J[k * stride] for weight k.
template <int MW, int NH, int NHM>
__device__ __forceinline__ void lux_jacobian(const LuxNet& L, const LuxPad& P, const LuxPass<MW, NHM>& v, double* J,
                                             int stride, double (&df)[3]) {
  double xb[MW];
#pragma unroll
  for (int k = 0; k < MW; ++k) {
    if (k < L.width[NH - 1]) J[(L.off_Wo + k) * stride] = v.oo * v.x[k];
    xb[k] = v.oo * P.Wo<double>(k);
  }
  J[L.off_bo * stride] = v.oo;
#pragma unroll
  for (int l = NH - 1; l >= 0; --l) {
    const int w = L.width[l], wi = l ? L.width[l - 1] : L.n_in;
    const double rw = rcp_est(double(w)), rs = rcp_est(v.s[l]);
    double gg[MW], m1 = 0.0, m2 = 0.0;
#pragma unroll
    for (int j = 0; j < MW; ++j) {
      if (j < w) {
        J[(L.off_g[l] + j) * stride] = xb[j] * v.xh[l][j];
        J[(L.off_be[l] + j) * stride] = xb[j];
      }
      gg[j] = xb[j] * P.g<double>(l, j);
      m1 += gg[j];
      m2 += gg[j] * v.xh[l][j];
    }
    m1 = div_est(m1, double(w), rw);
    m2 = div_est(m2, double(w), rw);
    double zb[MW];
#pragma unroll
    for (int j = 0; j < MW; ++j) {
      zb[j] = div_est(gg[j] - m1 - v.xh[l][j] * m2, v.s[l], rs) * v.ad[l][j];
      if (j < w) {
#pragma unroll
        for (int k = 0; k < MW; ++k)
          if (k < wi) J[(L.off_W[l] + j + k * w) * stride] = zb[j] * v.xin[l][k];
        J[(L.off_b[l] + j) * stride] = zb[j];
      }
    }
#pragma unroll
    for (int k = 0; k < MW; ++k) {
      double t = 0.0;
#pragma unroll
      for (int j = 0; j < MW; ++j) t += P.W<double>(l, j, k) * zb[j];
      xb[k] = t;
    }
  }
  df[0] = xb[0];
  df[1] = MW > 1 ? xb[MW > 1 ? 1 : 0] : 0.0;
  df[2] = MW > 2 ? xb[MW > 2 ? 2 : 0] : 0.0;
}

// State components that the features read: ManningN_h takes the depth only.
__device__ __forceinline__ int lux_state_inputs(const LuxNet& L) { return L.choice == LUX_MANNING_H ? 1 : 3; }

// The output's derivatives cs by the cell's state (xi, q_x, q_y), from those
// by the features: one dual pass for each of the ns components they read.
__device__ __forceinline__ void lux_state_derivatives(const LuxNet& L, int ns, const double (&q)[3], double hs,
                                                      double hsmall, double ks, const double (&df)[3], double* cs,
                                                      int stride) {
  for (int c = 0; c < ns; ++c) {
    const Dual1 x0(q[0], c == 0 ? 1.0 : 0.0), x1(q[1], c == 1 ? 1.0 : 0.0), x2(q[2], c == 2 ? 1.0 : 0.0);
    Dual1 fd[3];
    lux_features<Dual1>(L, x0, x1, x2, hs, hsmall, ks, fd);
    cs[c * stride] = df[0] * fd[0].d + df[1] * fd[1].d + df[2] * fd[2].d;
  }
  for (int c = ns; c < 3; ++c) cs[c * stride] = 0.0;
}

// The sum over a tile of 2 x 64 cells of v[cell], by one wave and a fixed
// tree; N: cells of the mesh, c0: the tile's first.
__device__ __forceinline__ double lux_tile_sum(const double* v, int c0, int N, int lane) {
  double s = (c0 + lane < N ? v[lane] : 0.0) + (c0 + 64 + lane < N ? v[64 + lane] : 0.0);
  for (int w = 32; w > 0; w >>= 1) s += __shfl_xor(s, w, 64);
  return s;
}

struct LuxArgs {
  LuxNet net;
  int32_t N;
  const double* w;       // P weights
  const double* xi;      // state (lib order)
  const double* qx;
  const double* qy;
  const double* hstill;
  const double* ks;      // per cell (ManningN_h_Umag_ks), else unused
  double hsmall;
  double* out;           // forward: n or friction magnitude per cell
  const double* obar;    // reverse: cotangent of the output per cell
  double* ox;            // += state cotangent
  double* oqx;
  double* oqy;
  double* wpart;         // [P][blocks] per-block weight cotangents
  double* wcell;         // [P][N] per-cell ones (k_lux_vjp_cells)
};

__device__ __forceinline__ double lux_ks(const LuxArgs& a, int i) {
  return a.net.choice == LUX_MANNING_H_UMAG_KS ? a.ks[i] : 0.0;
}

}  // namespace hg
