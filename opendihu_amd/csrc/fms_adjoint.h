// Discrete adjoint of the split step (Hodgkin-Huxley fibres, current-pulse
// stimulation): reverse Heun steps with the transposed reaction Jacobian and a
// reverse tridiagonal solve, parameter gradients for g_Na, g_K, g_L per fibre
// and for the diffusion prefactor sigma/(Am Cm) per fibre.
//
// Forward split step (fast_monodomain_solver_compute.tpp:110-126):
//   y^a = H_{n0D}(y, t)  ->  V^b = A^{-1} B V^a  ->  y' = H_{n0D}(y^b, t + dt/2)
// Heun step y' = y + dt/2 (f(y) + f(y*)), y* = y + dt f(y). With lambda' the
// adjoint of y', mu = J(y*)^T lambda':
//   lambda = lambda' + dt/2 mu + dt/2 J(y)^T (lambda' + dt mu)
//   theta_bar += dt/2 [ f_theta(y)^T (lambda' + dt mu) + f_theta(y*)^T lambda' ]
// Diffusion: A and B are symmetric (consistent P1 mass and stiffness), so with
// w = A^{-1} lambda_b:  lambda_a = B w,  pf_bar += w^T (dB/dpf V^a - dA/dpf V^b),
// dA/dpf = K1 (IE) or K1/2 (CN), dB/dpf = 0 (IE) or -K1/2 (CN), K1 the stiffness
// matrix for prefactor 1.
// The derivatives are those of the implemented forward (discrete adjoint): for
// the approximate exponential E(x) = (1 + x/1024)^1024, E'(x) = E(x)/(1 + x/1024).
#pragma once

#include "fms_fibre.h"

namespace fms {

template <class E> struct ExpDeriv;
template <> struct ExpDeriv<ExpApprox> {
  // power-series coefficients of E(x) - 1 = sum_k c_k x^k, c_k = binom(1024, k) / 1024^k
  static FMS_HD constexpr double c(int k) {
    double v = 1.0;
    for (int j = 1; j < k; j++) v = v * (1024.0 - j) / ((j + 1) * 1024.0);
    return v;
  }
};
template <> struct ExpDeriv<ExpLibm> {
  static FMS_HD constexpr double c(int k) {   // 1 / k!
    double v = 1.0;
    for (int j = 2; j <= k; j++) v /= j;
    return v;
  }
};
template <> struct ExpDeriv<ExpApproxFma> : ExpDeriv<ExpApprox> {};
template <> struct ExpDeriv<ExpLibmFma> : ExpDeriv<ExpLibm> {};

// u(x) = x / (E(x) - 1) has a removable singularity at x = 0: the HH rates
// alpha_m = u(-(V+50)/10) and alpha_n = u(-(V+65)/10) / 10. The quotient rule
// u' = (E - 1 - x E') / (E - 1)^2 loses its accuracy near 0: the numerator is
// about -x^2/2, while E - 1 and x E' each carry ~1e-13 absolute rounding error
// (the approximate exponential raises a rounded 1 + x/1024 to the 1024th
// power), so the relative error is ~2e-13 / x^2 - O(1) a few hundredths of a
// millivolt from the singular voltage, a point every action potential's
// upstroke passes. For |x| < 0.05, u' is taken from its own power series
// u'(x) = sum_j d_j x^j, degree 7 (truncation ~1e-18 relative at |x| = 0.05;
// the quotient rule's error there is 1e-10). The coefficients follow at
// compile time from the series of E: with s(x) = (E(x) - 1)/x = sum_k c_{k+1} x^k,
// u = 1/s term by term, d_j = (j+1) u_{j+1}.
template <class E>
constexpr double du_coeff(int j) {
  double s[9] = {}, u[9] = {};
  for (int k = 0; k < 9; k++) s[k] = ExpDeriv<E>::c(k + 1);
  u[0] = 1.0 / s[0];
  for (int m = 1; m < 9; m++) {
    double acc = 0.0;
    for (int k = 1; k <= m; k++) acc += s[k] * u[m - k];
    u[m] = -acc / s[0];
  }
  return (j + 1) * u[j + 1];
}

// against the exact rational coefficients (binomial series inverted in fractions)
static_assert(du_coeff<ExpApprox>(0) == -0.49951171875, "d0 = -binom(1024,2)/1024^2");
static_assert(du_coeff<ExpApprox>(1) - 0.16666650772094727 < 1e-17 &&
                  du_coeff<ExpApprox>(1) - 0.16666650772094727 > -1e-17, "d1");
static_assert(du_coeff<ExpApprox>(3) - -0.0055554495918386237 < 1e-18 &&
                  du_coeff<ExpApprox>(3) - -0.0055554495918386237 > -1e-18, "d3");
static_assert(du_coeff<ExpApprox>(7) - -6.6127054049909082e-06 < 1e-20 &&
                  du_coeff<ExpApprox>(7) - -6.6127054049909082e-06 > -1e-20, "d7");
static_assert(du_coeff<ExpLibm>(0) == -0.5, "Bernoulli: B1 = -1/2");
static_assert(du_coeff<ExpLibm>(2) < 1e-16 && du_coeff<ExpLibm>(2) > -1e-16, "B3 = 0 (to the rounding of the inversion)");
static_assert(du_coeff<ExpLibm>(5) - 1.0 / 5040 < 1e-17 && du_coeff<ExpLibm>(5) - 1.0 / 5040 > -1e-17, "B6 / 5! = 1/5040");

template <class E>
__device__ __forceinline__ double du_near_zero(double x) {
  constexpr double d0 = du_coeff<E>(0), d1 = du_coeff<E>(1), d2 = du_coeff<E>(2), d3 = du_coeff<E>(3);
  constexpr double d4 = du_coeff<E>(4), d5 = du_coeff<E>(5), d6 = du_coeff<E>(6), d7 = du_coeff<E>(7);
  return d0 + x * (d1 + x * (d2 + x * (d3 + x * (d4 + x * (d5 + x * (d6 + x * d7))))));
}

__device__ __forceinline__ bool near_removable(double x) { return x < 0.05 && x > -0.05; }

// Linearisation of the HH right-hand side at y: the rates r(y), in the operations
// of hh_rates_fused (so y* = y + dt r(y) has the forward's bits), and the partial
// derivatives that J(y)^T w and f_theta(y)^T w need, from the same exponentials.
// dE/dV = slope E / base: the six bases share one reciprocal. About 190
// instructions instead of the 340 of an evaluation with a division per quotient
// and without fused multiply-adds.
struct HHLin {
  double r[4];
  double f0V, f0m, f0h, f0n;       // d f0 / d(V, m, h, n)
  double f1V, f1m, f2V, f2h, f3V, f3n;
  double gna, gk, gl;              // d f0 / d(g_Na, g_K, g_L)
  FMS_HD void jt(const double *w, double *out) const {
    out[0] = __builtin_fma(w[0], f0V, __builtin_fma(w[1], f1V, __builtin_fma(w[2], f2V, w[3] * f3V)));
    out[1] = __builtin_fma(w[0], f0m, w[1] * f1m);
    out[2] = __builtin_fma(w[0], f0h, w[2] * f2h);
    out[3] = __builtin_fma(w[0], f0n, w[3] * f3n);
  }
};

template <class E>
__device__ __forceinline__ HHLin hh_linearize(const double *y, const double *p) {
  HHLin L;
  const double V = y[0], m = y[1], h = y[2], n = y[3];
  HHBases b;
  const HHExps e = hh_exps<E>(V, &b);
  double im, in, ih;
  hh_inverses(e, im, in, ih);
  const HHQuotients qu = hh_quotients<E>(e, im, in, ih);
  const double am = qu.am, an = qu.an, bh = qu.bh;
  const double ah = 0.07 * e.eah, bm = 4.0 * e.ebm, bn = 0.125 * e.ebn;
  const double sm = __builtin_fma(4.0, e.ebm, am), sh = ah + bh, sn = __builtin_fma(0.125, e.ebn, an);
  L.r[1] = hh_gate_rate<E>(am, 4.0, e.ebm, sm, m);
  L.r[2] = hh_gate_rate<E>(ah, 1.0, bh, sh, h);
  L.r[3] = hh_gate_rate<E>(an, 0.125, e.ebn, sn, n);
  const double m2 = m * m, m3 = m2 * m, m3h = m3 * h, n2 = n * n, n4 = n2 * n2;
  const double gm3h = p[1] * m3h, gn4 = p[2] * n4;
  const double vna = V - 40.0, vk = V + 87.0, vl = V + (75.0 - 10.6130);
  L.r[0] = __builtin_fma(-gm3h, vna, __builtin_fma(-gn4, vk, -(p[3] * vl))) + p[0];
  // E'(x) of the exponential used, divided by it: 1/base (approximate), 1 (exact)
  HHBases ib{1.0, 1.0, 1.0, 1.0, 1.0, 1.0};
  if constexpr (std::is_base_of<ExpApprox, E>::value) ib = hh_inverse_bases(b);
  // alpha_m = u(xm), alpha_n = u(xn) / 10 (u above): u' = (1 - u E') / (E - 1) by the
  // quotient rule, and the series within |x| < 0.05 of a singular voltage. A lane is
  // near at most one of the two singular voltages (1.5 apart in x). The polynomial is
  // evaluated on every lane and selected: a branch would split the nodes' code into
  // blocks that the scheduler cannot interleave.
  const double xn = 10.0 * e.xn01;
  const bool near_m = near_removable(e.xm), near_n = near_removable(xn);
  const double dus = du_near_zero<E>(near_m ? e.xm : xn);
  const double dum = near_m ? dus : im * __builtin_fma(-am, e.em * ib.m, 1.0);
  const double dun = near_n ? dus : in * __builtin_fma(-10.0 * an, e.en * ib.n, 1.0);
  const double dam = -0.1 * dum, dan = -0.01 * dun;
  const double dbm = bm * ib.bm * (-1.0 / 18.0), dah = ah * ib.ah * (-1.0 / 20.0);
  const double dbh = bh * bh * (e.ebh * ib.bh) * 0.1, dbn = bn * ib.bn * (1.0 / 80.0);
  L.f0V = -(gm3h + gn4 + p[3]);
  const double gv = -p[1] * vna;
  L.f0m = 3.0 * m2 * h * gv;
  L.f0h = m3 * gv;
  L.f0n = -4.0 * (p[2] * vk) * (n2 * n);
  L.f1V = __builtin_fma(-(dam + dbm), m, dam);
  L.f1m = -sm;
  L.f2V = __builtin_fma(-(dah + dbh), h, dah);
  L.f2h = -sh;
  L.f3V = __builtin_fma(-(dan + dbn), n, dan);
  L.f3n = -sn;
  L.gna = -(m3h * vna);
  L.gk = -(n4 * vk);
  L.gl = -vl;
  return L;
}

// reverse of one Heun step from its input y (no clamp):
// lam[4] in: adjoint of the output, out: adjoint of y; gacc[3] += parameter gradient
template <class E>
__device__ __forceinline__ void hh_heun_step_reverse(const double *y, const double *p, double dt, double *lam, double *gacc) {
  const double hdt = 0.5 * dt;
  const HHLin Ly = hh_linearize<E>(y, p);
  double ys[4];
#pragma unroll
  for (int k = 0; k < 4; k++) ys[k] = __builtin_fma(dt, Ly.r[k], y[k]);
  double mu[4], nu[4], jy[4], gs[3];
  {
    const HHLin Ls = hh_linearize<E>(ys, p);
    Ls.jt(lam, mu);
    gs[0] = lam[0] * Ls.gna;
    gs[1] = lam[0] * Ls.gk;
    gs[2] = lam[0] * Ls.gl;
  }
#pragma unroll
  for (int k = 0; k < 4; k++) nu[k] = __builtin_fma(dt, mu[k], lam[k]);
  Ly.jt(nu, jy);
#pragma unroll
  for (int k = 0; k < 4; k++) lam[k] = __builtin_fma(hdt, mu[k] + jy[k], lam[k]);
  gacc[0] = __builtin_fma(hdt, __builtin_fma(nu[0], Ly.gna, gs[0]), gacc[0]);
  gacc[1] = __builtin_fma(hdt, __builtin_fma(nu[0], Ly.gk, gs[1]), gacc[1]);
  gacc[2] = __builtin_fma(hdt, __builtin_fma(nu[0], Ly.gl, gs[2]), gacc[2]);
}

// current pulses as the reverse sweep sees them
struct AdjStim {
  int on;       // pulses are set
  int param;    // the stimulus parameter
  const double *onset, *duration, *amplitude;   // [F]
  const int *vc_centre;   // point-buffer order: [F], negative on fibres that are never stimulated; else null
};

// reverse of one reaction half of a node from its state y0 at t0: l in: adjoint of
// the half's output, out: adjoint of y0; g += dL/d(gNa, gK, gL). Heun step j is
// reversed from its recomputed input with the stimulus parameter of that step
// (params(t, p)).
template <class E, class Params>
__device__ __forceinline__ void reverse_half(Params &&params, const double *y0, double t0, double dt, int n0D,
                                             double *l, double *g) {
#pragma unroll 1
  for (int j = n0D - 1; j >= 0; j--) {
    double y[4] = {y0[0], y0[1], y0[2], y0[3]}, pj[4];
#pragma unroll 1
    for (int jj = 0; jj < j; jj++) {
      params(t0 + jj * dt, pj);
      heun_node<ModelHH, double, E, false>(y[0], y + 1, pj, t0 + jj * dt, dt, false, 0.0);
    }
    params(t0 + j * dt, pj);
    hh_heun_step_reverse<E>(y, pj, dt, l, g);
  }
}

// What one launch of the reverse sweep needs: kc split steps of one segment, steps
// s = kc-1 .. 0 (rows of `steps`). Tape: [kc][9][N] = y0 (4), y after half 1 (V^a and
// the gates, 4), V^b. lam: [4][N]; acc: [4][F * T], each thread's sums of dL/d(gNa, gK,
// gL) and of the prefactor's element terms.
struct AdjArgs {
  DevFibers fb;
  AdjStim st;
  const double *tape, *steps;
  int kc, n0D, ie;
  const int *sensor_slot;
  const double *dtrace;
  int n_sensors;
  double *lam, *acc;
  int raise_priority;
};

// Per step: the sensors' dL/dV, reverse of half 2 from y^b = (V^b, gates after half
// 1), reverse diffusion, reverse of half 1 from y0. A w = lambda_V is solved with the
// factored chunks of the forward (fms_chunk.h: A' x = lambda_V, w = -x), and B = A - K
// gives B w = lambda_V + K x, a difference of element fluxes; the same fluxes give
// the prefactor gradient w^T (dB/dpf V^a - dA/dpf V^b) = -theta sum_e (x_{e+1} - x_e)
// (v_{e+1} - v_e) / h_e with v = V^b, theta = 1 (IE) or v = V^a + V^b, theta = 1/2 (CN).
// lambda, and the sums of each thread, stay in registers for the whole segment; sums
// over threads are taken once after the last segment (k_adj_reduce), so the gradient
// does not depend on the segmentation.
template <class E, int T, int C>
__device__ __forceinline__ void adj_steps(const AdjArgs &a, int f, int off, int n, double *sh) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long long N = a.fb.n_total, FT = (long long)a.fb.n_fibers * T;
  const double pf = a.fb.prefactor[f];
  const ChunkLds<T, C> lds{sh, tid};
  const int lo = tid * C;
  const bool busy = wave * 64 * C < n;
  const bool ie = a.ie != 0;
  double p[4];
#pragma unroll
  for (int k = 0; k < 4; k++) p[k] = a.fb.params[(long long)f * 4 + k];
  const double onset = a.st.on ? a.st.onset[f] - 1e-13 : 0.0;
  const double end = a.st.on ? a.st.onset[f] + a.st.duration[f] - 1e-13 : 0.0;
  const double amp = a.st.on ? a.st.amplitude[f] : 0.0;
  double l[C][4], acc[4];
  int slot[C];
  unsigned inset = 0;
  {
    const bool checked = !a.st.vc_centre || a.st.vc_centre[f] >= 0;
    const int sb = a.fb.stim_begin[f], se = checked ? a.fb.stim_end[f] : sb;
#pragma unroll
    for (int q = 0; q < C; q++) {
      // threads past the fibre's end shadow its last node with a zero adjoint
      const bool valid = lo + q < n;
      const int i = off + (valid ? lo + q : n - 1);
#pragma unroll
      for (int k = 0; k < 4; k++) l[q][k] = valid ? a.lam[k * N + i] : 0.0;
      slot[q] = valid ? a.sensor_slot[i] : -1;
      inset |= (lo + q >= sb && lo + q < se ? 1u : 0u) << q;
    }
#pragma unroll
    for (int k = 0; k < 4; k++) acc[k] = a.acc[k * FT + (long long)f * T + tid];
  }
  // the element between the previous wave's last node and this wave's first
  const double ihl = lane == 0 && wave > 0 && lo < n ? recip_nr(a.fb.elem_len[off - f + lo - 1]) : 0.0;
  // half step hs: the second half of step hs / 2 and its diffusion (odd), or its
  // first half. One node at a time (its two linearisations hold about 100
  // registers; two waves per SIMD hide their chains), the next node's tape entries
  // in flight meanwhile, over the end of a half and the solve too.
  struct NodeTape {
    double y[4], va, dl;   // the state the half starts from; V^a; the sensor's dL/dV
  };
  double v[C];   // the diffusion's Vm
  auto load = [&](int hs, int q) {
    NodeTape in;
    const int s = hs >> 1;
    const double *tp = a.tape + (long long)s * 9 * N + off + (lo + q < n ? lo + q : n - 1);
    in.va = 0.0;
    in.dl = 0.0;
    if (hs & 1) {
      in.y[0] = tp[8 * N];
#pragma unroll
      for (int k = 1; k < 4; k++) in.y[k] = tp[(4 + k) * N];
      if (!ie) in.va = tp[4 * N];
      if (slot[q] >= 0) in.dl = a.dtrace[((long long)s * a.fb.n_fibers + f) * a.n_sensors + slot[q]];
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) in.y[k] = tp[k * N];
    }
    return in;
  };
#pragma unroll
  for (int q = 0; q < C; q++) v[q] = 0.0;
  int hs = 2 * a.kc - 1;
  NodeTape next{};
  if (busy) next = load(hs, 0);
  while (hs >= 0) {
    const double dt1 = a.steps[4 * (long long)(hs >> 1) + 3];
    ChunkFactor<C> fac;
    chunk_refactor<T, C, true>(fac, n, a.fb.elem_len + (off - f), pf, dt1, ie, lds);
#pragma unroll 1
    do {
      const int s = hs >> 1;
      const bool half = hs & 1;
      const double *row = a.steps + 4 * (long long)s;
      if (busy) {
        const double t0 = half_start(row, half), dt = row[2];
        constexpr_for<0, C, 1>([&](auto q_) {
          constexpr int q = decltype(q_)::value;
          const NodeTape in = next;
          if constexpr (q + 1 < C)
            next = load(hs, q + 1);
          else if (hs > 0)
            next = load(hs - 1, 0);
          if (half) {
            l[q][0] += in.dl;
            v[q] = in.va + in.y[0];   // V^b, or V^a + V^b
          }
          auto params = [&](double t, double *pj) {
            // the pulse's window as the forward has it (current_on)
            const bool on = a.st.on && t >= onset && t < end && ((inset >> q) & 1);
#pragma unroll
            for (int k = 0; k < 4; k++) pj[k] = on && k == a.st.param ? amp : p[k];
          };
          reverse_half<E>(params, in.y, t0, dt, a.n0D, l[q], acc);
        });
      }
      hs--;
      if (!half) continue;
      // A' x = lambda_V; rows past the fibre's end have no coefficients
      double z[C];
#pragma unroll
      for (int q = 0; q < C; q++) z[q] = lo + q < n ? l[q][0] : 0.0;
      double D = z[0], zlast = 0.0;
      chunk_interior<C>(fac, z);
      if constexpr (C > 1) {
        zlast = z[C - 1];
        D = __builtin_fma(-fac.o0, z[1], D);
      }
      D -= lane_prev(fac.ob * zlast);
      double X, Xn, Sn, Lp;
      chunk_separators<T, C>(fac, D, zlast, v[0], 0.0, s & 1, lds, X, Xn, Sn, Lp);
      constexpr_for<1, C, 1>([&](auto k_) {
        constexpr int k = decltype(k_)::value;
        z[k] = __builtin_fma(lds.zr(k), Xn, __builtin_fma(lds.zl(k), X, z[k]));
      });
      z[0] = X;
      // fluxes of x over the thread's elements: lambda_V += K x, prefactor terms
      double xn = lane_next(X), vn = lane_next(v[0]);
      if (lane == 63) {
        xn = Sn;
        vn = wave + 1 < T / 64 ? lds.iface(s & 1)[4 * (wave + 1)] : 0.0;
      }
      double fx[C], pfs = 0.0;
#pragma unroll
      for (int q = 0; q < C; q++) {
        const double ih = q == C - 1 ? fac.kapb : fac.kap[q];
        fx[q] = ih * ((q == C - 1 ? xn : z[q + 1 < C ? q + 1 : q]) - z[q]);
        pfs = __builtin_fma(fx[q], (q == C - 1 ? vn : v[q + 1 < C ? q + 1 : q]) - v[q], pfs);
      }
      acc[3] -= pfs;
      // the flux of the element left of the first row: the previous thread's last; at
      // the start of a wave from the previous wave's last row
      double fp = lane_prev(fx[C - 1]);
      if (lane == 0) fp = ihl * (X - Lp);
#pragma unroll
      for (int q = 0; q < C; q++) {
        l[q][0] = __builtin_fma(pf, fx[q] - fp, l[q][0]);
        fp = fx[q];
      }
    } while (hs >= 0 && (!(hs & 1) || a.steps[4 * (long long)(hs >> 1) + 3] == dt1));
  }
#pragma unroll
  for (int q = 0; q < C; q++)
    if (lo + q < n) {
#pragma unroll
      for (int k = 0; k < 4; k++) a.lam[k * N + off + lo + q] = l[q][k];
    }
#pragma unroll
  for (int k = 0; k < 4; k++) a.acc[k * FT + (long long)f * T + tid] = acc[k];
}

template <class E, int T, int CMAX>
__global__ __launch_bounds__(T, 2) void k_adj_steps(AdjArgs a) {
  extern __shared__ double sh[];
  // with raise_priority the reverse sweep's waves win issue over the next
  // segment's recompute that runs beside it on the same CUs
  if (a.raise_priority) __builtin_amdgcn_s_setprio(2);
  const int f = blockIdx.x;
  const int off = a.fb.fiber_off[f];
  const int n = a.fb.fiber_off[f + 1] - off;
  with_chunk_rows<CMAX>((n + T - 1) / T,
                        [&](auto c_) { adj_steps<E, T, decltype(c_)::value>(a, f, off, n, sh); });
}

// per-fibre sums of the threads' accumulators [4][F * T], in a fixed order: the
// conductances' gradients to grad [F][3], the prefactor's (scaled by theta) to
// pf_bar [F]
static __global__ __launch_bounds__(256) void k_adj_reduce(int n_fibers, int T, const double *acc, double theta,
                                                           double *grad, double *pf_bar) {
  const int f = blockIdx.x;
  const long long FT = (long long)n_fibers * T;
  __shared__ double part[4][256];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    double s = 0;
    for (int i = threadIdx.x; i < T; i += 256) s += acc[k * FT + (long long)f * T + i];
    part[k][threadIdx.x] = s;
  }
  __syncthreads();
  if (threadIdx.x < 4) {
    double s = 0;
    for (int q = 0; q < 256; q++) s += part[threadIdx.x][q];
    if (threadIdx.x < 3)
      grad[f * 3 + threadIdx.x] = s;
    else
      pf_bar[f] = theta * s;
  }
}

}  // namespace fms
