// Hodgkin-Huxley reaction with fused multiply-adds, for the runs that are held to
// a tolerance against the oracle and not to its bits (partitioned solve). The
// model is model_hh.h's; what differs is how its expressions are evaluated:
//
//  * The argument of an exponential is linear in V, so the base 1 + x/1024 of the
//    approximate exponential is one fused multiply-add (constants exact, or their
//    error below 1e-18 of the base) instead of an add, a division by a constant,
//    a multiply and an add: 7 instructions for the six instead of 36. Its rounding,
//    which the ten squarings multiply by 1024, stays the only one.
//  * alpha_m = x/(E(x) - 1) takes x = 1024 (base - 1), one exact instruction, and
//    alpha_n likewise.
//  * The three quotients share one reciprocal; under the device's exp, whose error is
//    as small as a product's, each is corrected by its remainder.
//  * d gate/dt = alpha - (alpha + beta) gate (under the device's exp
//    alpha (1 - gate) - beta gate), currents and Heun updates as fused multiply-adds.
//
// About 110 FP64 instructions per right-hand side instead of 175; FP64 issue is what
// bounds the kernels. In kernels that are otherwise the same, 4096 fibres of 400-2000
// nodes, 1000 steps and the states read back: 183 -> 156 ms (mixed 113 -> 95 ms).
// Mean errors of the rates against 80-bit arithmetic, Vm from -90 to 40 mV, as a share
// of the model form's, on the device: dV/dt 0.89, dm/dt, dh/dt and dn/dt 0.84, 1.00 and
// 0.80 (approximate exponential), 0.95, 1.00 and 0.96 (device's exp; no larger in any of
// the bands -90..-70, -70..-60, -55..-45 and -40..40 mV). With the approximate
// exponential alpha_m's x has the base's error of 1e-13: what it cancels around -50 mV
// is most of the former error; at -40..40 mV dm/dt has 4 times its small former one.
// Under the device's exp, en and ebh as multiples of em were 24 % faster (512 x 1001
// nodes, 300 steps: 4.3 against 5.4 ms; model form and its kernels 8.0) but gave dn/dt
// 1.75 times the model form's mean error and 9.5 times its rms one, around -65 mV.
#pragma once

#include "fms_math.h"
#include "model_hh.h"

namespace fms {

// the exponentials of one right-hand side, and the arguments of the two that
// have a removable singularity
struct HHExps {
  double em, en, ebh, ebm, eah, ebn;   // E(xm), E(xn), beta_h's, beta_m's, alpha_h's, beta_n's
  double xm, xn01;                     // xm and 0.1 xn
};

FMS_HD double pow1024(double b) {
#pragma unroll
  for (int i = 0; i < 10; i++) b *= b;
  return b;
}

// the bases 1 + x/1024 of the approximate exponentials, in HHExps's order
struct HHBases {
  double m, n, bh, bm, ah, bn;
};

// v (c + c_lo)
FMS_HD double hh_two_term(double v, double c, double c_lo) { return __builtin_fma(v, c, v * c_lo); }

template <class E> FMS_HD HHExps hh_exps(double V, HHBases *bases = nullptr) {
  HHExps e;
  const double v75 = V + 75.0;
  if constexpr (std::is_base_of<ExpApprox, E>::value) {
    const double bm = __builtin_fma(V, -1.0 / 10240, 1.0 - 5.0 / 1024);
    const double bn = __builtin_fma(V, -1.0 / 10240, 1.0 - 6.5 / 1024);
    const double bh = __builtin_fma(V, -1.0 / 10240, 1.0 - 4.5 / 1024);
    e.em = pow1024(bm);
    e.en = pow1024(bn);
    e.ebh = pow1024(bh);
    const double bbm = __builtin_fma(v75, -1.0 / 18432, 1.0);
    const double bah = __builtin_fma(V, -1.0 / 20480, 1.0 - 3.75 / 1024);
    const double bbn = __builtin_fma(V, 1.0 / 81920, 1.0 + 0.9375 / 1024);
    e.ebm = pow1024(bbm);
    e.eah = pow1024(bah);
    e.ebn = pow1024(bbn);
    if (bases) *bases = HHBases{bm, bn, bh, bbm, bah, bbn};
    e.xm = __builtin_fma(bm, 1024.0, -1024.0);
    e.xn01 = __builtin_fma(bn, 102.4, -102.4);
  } else {
    // six exponentials, each of its own argument: the quotient by the slope as the
    // product with its reciprocal in two terms, which is correctly rounded but for ties
    const double v50 = V + 50.0, v65 = V + 65.0, v45 = V + 45.0;
    e.em = E::exp(hh_two_term(v50, -0.1, 5.551115123125783e-18));
    e.en = E::exp(hh_two_term(v65, -0.1, 5.551115123125783e-18));
    e.ebh = E::exp(hh_two_term(v45, -0.1, 5.551115123125783e-18));
    e.ebm = E::exp(hh_two_term(v75, -1.0 / 18, -3.0839528461809902e-18));
    e.eah = E::exp(hh_two_term(v75, -0.05, 2.7755575615628915e-18));
    e.ebn = E::exp(v75 * 0.0125);
    e.xm = v50 * -0.1;
    e.xn01 = v65 * -0.01;
  }
  return e;
}

// 1/base of all six from one reciprocal
FMS_HD HHBases hh_inverse_bases(const HHBases &b) {
  const double p2 = b.m * b.n, p3 = p2 * b.bh, p4 = p3 * b.bm, p5 = p4 * b.ah;
  HHBases r;
  double q = recip_nr(p5 * b.bn);
  r.bn = q * p5;
  q *= b.bn;
  r.ah = q * p4;
  q *= b.ah;
  r.bm = q * p3;
  q *= b.bm;
  r.bh = q * p2;
  q *= b.bh;
  r.n = q * b.m;
  r.m = q * b.n;
  return r;
}

// 1/(em - 1), 1/(en - 1) and 1/(ebh + 1) from one reciprocal, for every Vm at which the
// three are finite: where their product overflows (below -2400 mV; above 23000 mV with
// the approximate exponential) each of the three is above 1e102 in size, the
// reciprocal is 0, not the Newton steps' NaN, and so are the quotients, multiplied by
// one factor at a time. (The two instructions cost 0 to 3 %: 4096 x 1000 nodes 66 -> 67
// us per step, 256 x 1000 6.9 -> 7.0, 1 x 100 2.75 -> 2.70. A branch to three
// reciprocals spilled 611 registers instead of 43, one per Heun step cost 5 %.)
FMS_HD void hh_inverses(const HHExps &e, double &im, double &in, double &ih) {
  const double dm = e.em - 1.0, dn = e.en - 1.0, dh = e.ebh + 1.0;
  const double p = (dm * dn) * dh;
  double r = recip_nr(p);
#if defined(__HIP_DEVICE_COMPILE__)
  r = __builtin_amdgcn_div_fixup(r, p, 1.0);
#endif
  ih = (r * dm) * dn;
  const double rh = r * dh;
  im = rh * dn;
  in = rh * dm;
}

// the device's exponential leaves the quotients and the sums of a rate as the largest
// errors of the rates; the approximate one's 1024-fold base error is above them
template <class E> constexpr bool hh_exact() { return !std::is_base_of<ExpApprox, E>::value; }

// alpha_m, alpha_n and beta_h from the shared reciprocal's im, in, ih
struct HHQuotients {
  double am, an, bh;
};
template <class E> FMS_HD HHQuotients hh_quotients(const HHExps &e, double im, double in, double ih) {
  HHQuotients q{e.xm * im, e.xn01 * in, ih};
  if constexpr (hh_exact<E>()) {
    // one step on the remainder each: the errors of the shared reciprocal's products go
    q.am = __builtin_fma(__builtin_fma(-(e.em - 1.0), q.am, e.xm), im, q.am);
    q.an = __builtin_fma(__builtin_fma(-(e.en - 1.0), q.an, e.xn01), in, q.an);
    q.bh = __builtin_fma(__builtin_fma(-(e.ebh + 1.0), ih, 1.0), ih, ih);
  }
  return q;
}

// alpha (1 - x) - beta x with beta = cb eb (cb a power of two), s = alpha + beta
template <class E> FMS_HD double hh_gate_rate(double alpha, double cb, double eb, double s, double x) {
  if constexpr (hh_exact<E>()) return __builtin_fma(alpha, 1.0 - x, -((cb * eb) * x));
  return __builtin_fma(-s, x, alpha);
}

// rates r[4] at (V, m, h, n), dV/dt without the stimulus; ALG: the algebraics of the model file in a[9]
template <class E, bool ALG>
FMS_HD void hh_rates_fused(double V, double m, double h, double n, const double *p, double *r, double *a) {
  const HHExps e = hh_exps<E>(V);
  double im, in, ih;
  hh_inverses(e, im, in, ih);
  const HHQuotients q = hh_quotients<E>(e, im, in, ih);
  const double am = q.am, an = q.an, ah = 0.07 * e.eah;
  r[1] = hh_gate_rate<E>(am, 4.0, e.ebm, __builtin_fma(4.0, e.ebm, am), m);
  r[2] = hh_gate_rate<E>(ah, 1.0, q.bh, ah + q.bh, h);
  r[3] = hh_gate_rate<E>(an, 0.125, e.ebn, __builtin_fma(0.125, e.ebn, an), n);
  const double gm3h = p[1] * (m * m * m * h), n2 = n * n, gn4 = p[2] * (n2 * n2);
  const double vna = V - 40.0, vk = V + 87.0, vl = V + (75.0 - 10.6130);
  r[0] = __builtin_fma(-gm3h, vna, __builtin_fma(-gn4, vk, -(p[3] * vl)));
  if constexpr (ALG) {
    a[0] = gm3h * vna;
    a[1] = am;
    a[2] = ah;
    a[3] = an;
    a[4] = gn4 * vk;
    a[5] = 4.0 * e.ebm;
    a[6] = q.bh;
    a[7] = 0.125 * e.ebn;
    a[8] = p[3] * vl;
  }
}

// Heun step of one node, as heun_node (fms_kernels.h), but for the second clamp, which
// is the caller's. i_stim: the node's i_Stim; clamp(v) holds Vm at the stimulus's value
// if the step's stimulus does so.
template <class G, class E, bool ALG, class Clamp>
FMS_HD void hh_step(double &V, G *g, const double *p, double i_stim, double dt, Clamp &&clamp, double *alg_out) {
  double r[4], ys[4], rs[4];
  hh_rates_fused<E, false>(V, (double)g[0], (double)g[1], (double)g[2], p, r, nullptr);
  r[0] += i_stim;
  ys[0] = __builtin_fma(dt, r[0], V);
#pragma unroll
  for (int k = 1; k < 4; k++) ys[k] = __builtin_fma(dt, r[k], (double)g[k - 1]);
  clamp(ys[0]);
  hh_rates_fused<E, ALG>(ys[0], ys[1], ys[2], ys[3], p, rs, alg_out);
  const double hdt = 0.5 * dt;
  rs[0] += i_stim;
  V = __builtin_fma(hdt, r[0] + rs[0], V);
#pragma unroll
  for (int k = 1; k < 4; k++) g[k - 1] = (G)__builtin_fma(hdt, r[k] + rs[k], (double)g[k - 1]);
}

// Heun step of one node, as heun_node
template <class G, class E, bool ALG>
FMS_HD void hh_step_fused(double &V, G *g, const double *p, double dt, bool clamp, double vstim, double *alg_out) {
  hh_step<G, E, ALG>(V, g, p, p[0], dt, [&](double &v) { if (clamp) v = vstim; }, alg_out);
  V = clamp ? vstim : V;
}

}  // namespace fms
