// Diffusion of one fibre by one workgroup whose threads own chunks of
// consecutive nodes, with the matrix factored ahead of the steps (models of at
// most 8 states, partitioned solve).
//
// The step solves A x = B u (assemble_row). B = A - K for both schemes, K the
// stiffness matrix with the fibre's prefactor, so x = u + w with A' w = K u,
// A' = -A. (K u)_i is a difference of element fluxes kap_e (u_{e+1} - u_e), so
// the right-hand side needs one coefficient per element, and the solve's
// rounding errors are relative to the step's change w instead of to u.
//
// A' depends on the element lengths, the prefactor and dt only. chunk_factor
// computes what every solve with it needs into registers (and a few boundary
// constants into LDS); chunk_diffuse applies it:
//
//  1. Thread t owns rows t*C .. t*C + C-1 (C = ceil(n / T)). Its first row
//     is a separator; its other rows are eliminated against the separators on
//     either side (LDL^T within the chunk).
//  2. The separators of a wave form a tridiagonal system of 64 rows, one per
//     lane: cyclic reduction with cross-lane shuffles. A level costs two fused
//     multiply-adds and two shuffles; the levels stop where the remaining
//     couplings of every row are below 2^-72 of its diagonal (after 2 to 4
//     levels at dt = 1e-3 ms and 0.01 cm elements, where a separator's influence
//     decays by 1e-4 or more per chunk), which leaves the bits of u + w alone.
//  3. Waves meet at boundary elements. Each wave publishes its separator and
//     last row at the boundary, solved without the neighbouring wave; one barrier
//     later every thread solves the 2x2 system of its wave's two boundaries. If
//     a wave is too short or the matrix too strongly coupled for its two ends to
//     be independent (below the same 2^-72), every thread solves the whole
//     chain of boundaries instead.
//
// Per step and row that is about 12 fused multiply-adds instead of the about 100
// instructions of the elimination that refactors in each step (lds_thomas_part),
// and one barrier instead of three.
#pragma once

#include "fms_kernels.h"

namespace fms {

// f(integral_constant k) for k = B, B + S, ... below N (S < 0: above N): loops
// over register arrays whose indices are constants whatever the optimiser does (a
// loop that it left rolled, or turned into an indexed store, put the array into
// scratch memory)
template <int B, int N, int S, class F> __device__ __forceinline__ void constexpr_for(F &&f) {
  if constexpr (S > 0 ? B < N : B > N) {
    f(std::integral_constant<int, B>{});
    constexpr_for<B + S, N, S>(f);
  }
}

// value of the next / previous lane; lane 63 / lane 0 receive 0
__device__ __forceinline__ double lane_next(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, 0x130, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, lo, 0x130, 0xf, 0xf, true));
}
__device__ __forceinline__ double lane_prev(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  return __hiloint2double(__builtin_amdgcn_update_dpp(0, hi, 0x138, 0xf, 0xf, true),
                          __builtin_amdgcn_update_dpp(0, lo, 0x138, 0xf, 0xf, true));
}

// couplings below this (relative to the diagonal) are dropped
constexpr double CHUNK_NEGLIGIBLE = 2.117582368135751e-22;   // 2^-72

// LDS doubles of the solve: per thread the cyclic reduction's multipliers (6 levels
// x 2) and the interior's responses to the separators (2 (C - 1)), which would
// otherwise take 50 of 256 registers at C = 8; for W waves their published boundary
// values, double-buffered over consecutive solves (2 x 4 W), the boundaries'
// constants (8 W) and the chain's scratch (4 W)
template <int T> constexpr int chunk_lds_doubles(int C) { return 20 * (T / 64) + T * (12 + 2 * (C - 1)); }

// the solve's LDS
template <int T, int C> struct ChunkLds {
  double *base;
  int tid;
  __device__ __forceinline__ double *iface(int parity) const { return base + parity * 4 * (T / 64); }
  __device__ __forceinline__ double *bnd() const { return base + 8 * (T / 64); }
  __device__ __forceinline__ double &at(int k) const { return base[20 * (T / 64) + k * T + tid]; }
  // cyclic reduction multipliers of level l
  __device__ __forceinline__ double &al(int l) const { return at(l); }
  __device__ __forceinline__ double &ga(int l) const { return at(6 + l); }
  // interior response of row k >= 1 to the own separator, and to the next thread's
  // (lane 63: to a unit right-hand side in the last row)
  __device__ __forceinline__ double &zl(int k) const { return at(11 + k); }
  __device__ __forceinline__ double &zr(int k) const { return at(10 + C + k); }
};

// the same with the per-thread values in registers, for a kernel of one solve (its
// LDS then allows more workgroups per CU)
template <int T, int C> struct ChunkRegs {
  double *base;
  int tid;
  double al_[6], ga_[6], zl_[C], zr_[C];
  __device__ __forceinline__ double *iface(int parity) const { return base + parity * 4 * (T / 64); }
  __device__ __forceinline__ double *bnd() const { return base + 8 * (T / 64); }
  __device__ __forceinline__ double &al(int l) { return al_[l]; }
  __device__ __forceinline__ double &ga(int l) { return ga_[l]; }
  __device__ __forceinline__ double &zl(int k) { return zl_[k]; }
  __device__ __forceinline__ double &zr(int k) { return zr_[k]; }
};

template <int C> struct ChunkFactor {
  double kap[C];   // flux coefficient of the element right of row k (0: none, or a boundary between waves)
  double s[C];     // s_k = -o_{k-1} / p_{k-1} of the interior rows k = 2..C-1
  double ip[C];    // 1 / p_k, k = 1..C-1
  double o0;       // off-diagonal between the separator and row 1
  double ob;       // off-diagonal to the next thread's separator (0 at a boundary between waves)
  double zll;      // zl of row C-1 (C = 1: 1, the separator is the last row)
  double ib;       // 1 / diagonal of the reduced separator row
  double vc, uc;   // separator responses to the couplings across the wave's left and right boundary
  double kapb;     // flux coefficient of the chunk's last element, also at a boundary between waves
  int nlev;        // cyclic reduction levels used
  int chain;       // the boundaries are coupled with each other
};

// boundary constants of wave w at bnd + 8 w: responses V0, U0 of its first separator
// and beta, VW of its last row; kap_b, o_b of the boundary between wave w and w + 1;
// the factors 1/(1 - V0 o_b^2 beta) of its right and left boundary
enum { BND_V0 = 0, BND_U0, BND_BETA, BND_VW, BND_KAP, BND_O, BND_KR, BND_KL };

// RHS_GIVEN: for solves with a right-hand side of their own instead of K u; kap is
// then 1/h and the boundaries carry no flux. AGAIN: the LDS holds an earlier factor.
// What the workgroup wrote to LDS before is visible afterwards.
template <int T, int C, bool RHS_GIVEN, bool AGAIN, class Store>
__device__ __forceinline__ void chunk_factor(ChunkFactor<C> &q, int n, const double *__restrict__ h, double pf,
                                             double dt, bool ie, Store &lds) {
  constexpr int W = T / 64;
  const int tid = lds.tid;
  double *bnd = lds.bnd();
  const int lane = tid & 63, wave = tid >> 6;
  const int lo = tid * C;
  const double theta = ie ? 1.0 : 0.5;
  const double idt6 = 1.0 / (6.0 * dt);
  double o[C], dg[C];   // off-diagonal of the element right of row k, diagonal
  double eprev = 0.0;   // diagonal contribution of the element left of row 0
  if (tid > 0 && lo < n) {
    const double hl = h[lo - 1];
    eprev = theta * (pf * recip_nr(hl)) + 2.0 * (hl * idt6);
  }
  constexpr_for<0, C, 1>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    double ih = 0.0, m = 0.0;
    if (lo + k + 1 < n) {
      const double hk = h[lo + k];
      ih = recip_nr(hk);
      m = hk * idt6;
    }
    const double kap = pf * ih;
    q.kap[k] = RHS_GIVEN ? ih : kap;
    o[k] = m - theta * kap;
    const double e = theta * kap + 2.0 * m;
    dg[k] = eprev + e;
    eprev = e;
    q.s[k] = 0.0;
    q.ip[k] = 0.0;
  });
  q.kapb = q.kap[C - 1];
  const double oB = o[C - 1];
  // interior rows 1..C-1; rows past the fibre's end keep 1/p = 0
  constexpr_for<1, C, 1>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    double p = dg[k];
    if constexpr (k > 1) {
      q.s[k] = -o[k - 1] * q.ip[k - 1];
      p += q.s[k] * o[k - 1];
    }
    q.ip[k] = lo + k < n ? recip_nr(p) : 0.0;
  });
  // responses of the interior to its separators
  double zl1 = 0.0, zr1 = 0.0, zll = 1.0, zrl = 0.0;
  if constexpr (C > 1) {
    double y[C], z = 0.0;
    y[1] = -o[0];
    constexpr_for<2, C, 1>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      y[k] = q.s[k] * y[k - 1];
    });
    constexpr_for<C - 1, 0, -1>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      z = k < C - 1 ? q.ip[k] * y[k] + q.s[k < C - 1 ? k + 1 : k] * z : q.ip[k] * y[k];
      lds.zl(k) = z;
      if (k == C - 1) zll = z;
    });
    zl1 = z;
    constexpr_for<C - 1, 0, -1>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      z = k < C - 1 ? q.s[k < C - 1 ? k + 1 : k] * z : q.ip[k] * (lane == 63 ? 1.0 : -oB);
      lds.zr(k) = z;
      if (k == C - 1) zrl = z;
    });
    zr1 = z;
  }
  q.zll = zll;
  q.o0 = C > 1 ? o[0] : 0.0;
  // reduced separator rows of the wave: a x_{l-1} + b x_l + cc x_{l+1}
  const double mA = C > 1 ? oB * zll : oB, mB = C > 1 ? oB * zrl : 0.0;
  double a = lane_prev(mA);
  double b = (lo < n ? dg[0] : 1.0) + q.o0 * zl1 + lane_prev(mB);
  double cc = lane == 63 ? 0.0 : (C > 1 ? o[0] * zr1 : oB);
  double V = lane == 0 ? 1.0 : 0.0;
  double U = lane == 63 ? (C > 1 ? -o[0] * zr1 : 1.0) : 0.0;
  q.nlev = 0;
  constexpr_for<0, 6, 1>([&](auto l_) {
    constexpr int l = decltype(l_)::value;
    const int sft = 1 << l;
    const double ab = b < 0.0 ? -b : b;
    const bool far = (a < 0.0 ? -a : a) > CHUNK_NEGLIGIBLE * ab || (cc < 0.0 ? -cc : cc) > CHUNK_NEGLIGIBLE * ab;
    if (q.nlev == l && __builtin_amdgcn_ballot_w64(far) != 0) {
      const int im = (lane - sft) & 63, ip = (lane + sft) & 63;
      const double r = recip_nr(b);
      // every lane shuffles; lanes without a neighbour drop what wrapped around
      const double rm = __shfl(r, im), rp = __shfl(r, ip);
      const double al = lane >= sft ? -a * rm : 0.0, ga = lane + sft < 64 ? -cc * rp : 0.0;
      const double am = __shfl(a, im), cm = __shfl(cc, im), ap = __shfl(a, ip), cp = __shfl(cc, ip);
      const double vm = __shfl(V, im), vp = __shfl(V, ip), um = __shfl(U, im), up = __shfl(U, ip);
      b += al * cm + ga * ap;
      a = al * am;
      cc = ga * cp;
      V += al * vm + ga * vp;
      U += al * um + ga * up;
      lds.al(l) = al;
      lds.ga(l) = ga;
      q.nlev = l + 1;
    }
  });
  q.ib = recip_nr(b);
  q.vc = V * q.ib;
  q.uc = U * q.ib;
  q.ob = lane == 63 ? 0.0 : (C > 1 ? oB : 0.0);
  // boundary constants
  if (AGAIN) __syncthreads();   // readers of the earlier factor's constants are done
  if (lane == 0) {
    bnd[8 * wave + BND_V0] = q.vc;
    bnd[8 * wave + BND_U0] = q.uc;
  }
  if (lane == 63) {
    bnd[8 * wave + BND_BETA] = zrl + zll * q.uc;
    bnd[8 * wave + BND_VW] = zll * q.vc;
    bnd[8 * wave + BND_KAP] = RHS_GIVEN ? 0.0 : q.kapb;
    bnd[8 * wave + BND_O] = oB;
    q.kap[C - 1] = 0.0;   // the boundary's flux is applied with its solution
  }
  __syncthreads();
  // lane w: wave w's two ends, and the boundary between waves w and w + 1
  const int w = lane < W ? lane : W - 1;
  const double *k = bnd + 8 * w, *kp = bnd + 8 * (w > 0 ? w - 1 : 0), *kn = bnd + 8 * (w + 1 < W ? w + 1 : w);
  const bool far = (w > 0 && fabs(k[BND_VW]) * (fabs(kp[BND_O]) + fabs(kp[BND_KAP])) > CHUNK_NEGLIGIBLE) ||
                   (w + 1 < W && fabs(k[BND_U0]) * (fabs(k[BND_O]) + fabs(k[BND_KAP])) > CHUNK_NEGLIGIBLE);
  q.chain = __builtin_amdgcn_ballot_w64(far) != 0;
  const double kb = recip_nr(1.0 - kn[BND_V0] * (k[BND_O] * k[BND_O]) * k[BND_BETA]);
  // each wave keeps its own copy of its two boundaries' factors
  if (lane == wave) bnd[8 * wave + BND_KR] = kb;
  if (lane == wave - 1) bnd[8 * wave + BND_KL] = kb;
}

// The same as a function of its own, with its result in the caller's stack frame, for
// the kernels of many steps: inlined, its temporaries and code (once per change of dt)
// took the registers of the steps.
template <int T, int C, bool RHS_GIVEN>
__device__ __noinline__ void chunk_factor_call(ChunkFactor<C> *out, int n, const double *__restrict__ h, double pf,
                                               double dt, bool ie, ChunkLds<T, C> lds) {
  ChunkFactor<C> q;
  chunk_factor<T, C, RHS_GIVEN, true>(q, n, h, pf, dt, ie, lds);
  *out = q;
}
template <int T, int C, bool RHS_GIVEN = false>
__device__ __forceinline__ void chunk_refactor(ChunkFactor<C> &q, int n, const double *__restrict__ h, double pf,
                                               double dt, bool ie, const ChunkLds<T, C> &lds) {
  ChunkFactor<C> r;
  chunk_factor_call<T, C, RHS_GIVEN>(&r, n, h, pf, dt, ie, lds);
  q = r;
  q.nlev = __builtin_amdgcn_readfirstlane(q.nlev);
  q.chain = __builtin_amdgcn_readfirstlane(q.chain);
}

// Boundary between wave w and w + 1 from the published values {u of the
// separator, separator, u of the last row, last row} of both waves: the
// separator of wave w + 1 and the last row of wave w couple through o_b and share
// the flux f_b. rho enters wave w's last row, -gamma wave w + 1's separator; S that
// separator's solution, L that last row's.
struct ChunkBoundary {
  double rho, gamma, S, L;
};
__device__ __forceinline__ ChunkBoundary chunk_boundary(const double *iface, const double *bnd, int w, double kb) {
  const double *k = bnd + 8 * w;
  const double f = k[BND_KAP] * (iface[4 * (w + 1)] - iface[4 * w + 2]);
  const double o = k[BND_O], beta = k[BND_BETA], V0 = k[8 + BND_V0];
  const double lhat = iface[4 * w + 3];
  const double t = __builtin_fma(o, __builtin_fma(beta, f, lhat), f);
  ChunkBoundary r;
  r.S = kb * __builtin_fma(-V0, t, iface[4 * (w + 1) + 1]);
  r.rho = __builtin_fma(-o, r.S, f);
  r.L = __builtin_fma(beta, r.rho, lhat);
  r.gamma = __builtin_fma(o, r.L, f);
  return r;
}

// the boundaries' chain when they are coupled with each other: F_w the separator
// at wave w's start, L_w its last row,
//   F_w = df - vf L_{w-1} - uf F_{w+1},  L_w = dl - vl L_{w-1} - ul F_{w+1}
// Every wave solves it with the same values (rolled, the elimination's results in
// LDS: this branch must not cost the common one its registers).
template <int W>
__device__ __forceinline__ void chunk_chain(const double *iface, const double *bnd, double *tmp, int wave,
                                            ChunkBoundary &left, ChunkBoundary &right) {
  double al_prev = 0.0, be_prev = 0.0, f_prev = 0.0, o_prev = 0.0;
#pragma unroll 1
  for (int w = 0; w < W; w++) {
    const double *k = bnd + 8 * w;
    double f = 0.0, o = 0.0;
    if (w < W - 1) {
      o = k[BND_O];
      f = k[BND_KAP] * (iface[4 * (w + 1)] - iface[4 * w + 2]);
    }
    const double df = iface[4 * w + 1] - k[BND_V0] * f_prev + k[BND_U0] * f, vf = k[BND_V0] * o_prev, uf = k[BND_U0] * o;
    const double dl = iface[4 * w + 3] - k[BND_VW] * f_prev + k[BND_BETA] * f, vl = k[BND_VW] * o_prev,
                 ul = k[BND_BETA] * o;
    const double r = recip_nr(1.0 + vf * be_prev);
    const double gam = r * (df - vf * al_prev), del = -r * uf;
    al_prev = dl - vl * (al_prev + be_prev * gam);
    be_prev = -vl * be_prev * del - ul;
    tmp[4 * w] = gam;
    tmp[4 * w + 1] = del;
    tmp[4 * w + 2] = al_prev;
    tmp[4 * w + 3] = be_prev;
    f_prev = f;
    o_prev = o;
  }
  double Fn = 0.0;
#pragma unroll 1
  for (int w = W - 1; w >= wave - 1 && w >= 0; w--) {
    const double L = tmp[4 * w + 2] + tmp[4 * w + 3] * Fn;
    if (w < W - 1 && (w == wave || w == wave - 1)) {
      const double o = bnd[8 * w + BND_O], f = bnd[8 * w + BND_KAP] * (iface[4 * (w + 1)] - iface[4 * w + 2]);
      // (selects: a reference to one of the two would put both into the stack frame)
      const bool r = w == wave;
      const double rho = f - o * Fn, gamma = f + o * L;
      right.rho = r ? rho : right.rho;
      right.S = r ? Fn : right.S;
      left.gamma = r ? left.gamma : gamma;
      left.L = r ? left.L : L;
    }
    Fn = tmp[4 * w] + tmp[4 * w + 1] * Fn;
  }
}

// the wave's separators without its neighbours, the boundary, and the separators
// of the whole fibre: D in: right-hand side of the lane's separator, X out: its
// solution, Xn out: the next thread's (lane 63: what multiplies zr). zlast: the
// chunk's last interior row without separators. Sn, Lp: the next wave's first
// separator and the previous wave's last row. One barrier.
template <int T, int C, class Store>
__device__ __forceinline__ void chunk_separators(const ChunkFactor<C> &q, double D, double zlast, double ufirst,
                                                 double ulast, int parity, Store &lds, double &X,
                                                 double &Xn, double &Sn, double &Lp) {
  constexpr int W = T / 64;
  const int lane = lds.tid & 63, wave = __builtin_amdgcn_readfirstlane(lds.tid >> 6);
  double *iface = lds.iface(parity), *bnd = lds.bnd();
  constexpr_for<0, 6, 1>([&](auto l_) {
    constexpr int l = decltype(l_)::value;
    if (l < q.nlev) {
      const int sft = 1 << l;
      const double Dm = l == 0 ? lane_prev(D) : __shfl(D, (lane - sft) & 63);
      const double Dp = l == 0 ? lane_next(D) : __shfl(D, (lane + sft) & 63);
      D = __builtin_fma(lds.ga(l), Dp, __builtin_fma(lds.al(l), Dm, D));
    }
  });
  X = q.ib * D;
  ChunkBoundary left{0, 0, 0, 0}, right{0, 0, 0, 0};
  if (lane == 0) {
    iface[4 * wave] = ufirst;
    iface[4 * wave + 1] = X;
  }
  if (lane == 63) {
    iface[4 * wave + 2] = ulast;
    iface[4 * wave + 3] = __builtin_fma(q.zll, X, zlast);
  }
  __syncthreads();
  if (q.chain) {
    chunk_chain<W>(iface, bnd, bnd + 8 * W, wave, left, right);
  } else {
    if (wave > 0) left = chunk_boundary(iface, bnd, wave - 1, bnd[8 * wave + BND_KL]);
    if (wave < W - 1) right = chunk_boundary(iface, bnd, wave, bnd[8 * wave + BND_KR]);
  }
  X = __builtin_fma(q.uc, right.rho, __builtin_fma(-q.vc, left.gamma, X));
  Xn = lane_next(X);
  Xn = lane == 63 ? right.rho : Xn;
  Sn = right.S;
  Lp = left.L;
}

// interior rows forward and backward: z[k] in: right-hand sides of rows 1..C-1,
// out: their solution without the separators
template <int C> __device__ __forceinline__ void chunk_interior(const ChunkFactor<C> &q, double *z) {
  constexpr_for<2, C, 1>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    z[k] = __builtin_fma(q.s[k], z[k - 1], z[k]);
  });
  if constexpr (C > 1) z[C - 1] = q.ip[C - 1] * z[C - 1];
  constexpr_for<C - 2, 0, -1>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    z[k] = __builtin_fma(q.s[k + 1], z[k + 1], q.ip[k] * z[k]);
  });
}

// one diffusion step of the thread's nodes V[0..C-1] in place; parity: consecutive
// solves alternate between 0 and 1
template <int T, int C, class Store>
__device__ __forceinline__ void chunk_diffuse(const ChunkFactor<C> &q, double *V, int parity, Store &lds) {
  const double un = lane_next(V[0]);
  double z[C], fp = 0.0, D = 0.0;
  constexpr_for<0, C, 1>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    const double ur = k + 1 < C ? V[k + 1 < C ? k + 1 : k] : un;
    const double f = q.kap[k] * (ur - V[k]);
    if constexpr (k == 0)
      D = f;
    else
      z[k] = f - fp;
    fp = f;
  });
  chunk_interior<C>(q, z);
  double zlast = 0.0;
  if constexpr (C > 1) {
    zlast = z[C - 1];
    D = __builtin_fma(-q.o0, z[1], D);
  }
  D -= lane_prev(__builtin_fma(q.ob, zlast, fp));
  double X, Xn, Sn, Lp;
  chunk_separators<T, C>(q, D, zlast, V[0], V[C - 1], parity, lds, X, Xn, Sn, Lp);
  V[0] += X;
  constexpr_for<1, C, 1>([&](auto k_) {
    constexpr int k = decltype(k_)::value;
    V[k] += __builtin_fma(lds.zr(k), Xn, __builtin_fma(lds.zl(k), X, z[k]));
  });
}

// calls f(integral_constant c) for the fibre's rows per thread c = 1..CMAX
template <int CMAX, class F> __device__ __forceinline__ void with_chunk_rows(int c, F &&f) {
  constexpr_for<1, CMAX + 1, 1>([&](auto k_) {
    if (c == decltype(k_)::value) f(k_);
  });
}

// split kernels: one workgroup per fibre, one diffusion step
template <int T, int CMAX>
__global__ __launch_bounds__(T) void k_diffuse_chunk(DevFibers fb, double *__restrict__ vm, StepRef sr, int ie) {
  extern __shared__ double sh[];
  const int f = blockIdx.x, tid = threadIdx.x;
  const double dt = sr.row()[3];
  const int off = fb.fiber_off[f];
  const int n = fb.fiber_off[f + 1] - off;
  const int c = (n + T - 1) / T;
  double *lv = sh + 20 * (T / 64);
  for (int i = tid; i < n; i += T) lv[i] = vm[off + i];
  with_chunk_rows<CMAX>(c, [&](auto c_) {
    constexpr int C = decltype(c_)::value;
    ChunkRegs<T, C> lds{sh, tid, {}, {}, {}, {}};
    ChunkFactor<C> q;
    chunk_factor<T, C, false, false>(q, n, fb.elem_len + (off - f), fb.prefactor[f], dt, ie != 0, lds);
    double V[C];
    constexpr_for<0, C, 1>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      V[k] = lv[tid * C + k < n ? tid * C + k : n - 1];
    });
    chunk_diffuse<T, C>(q, V, 0, lds);   // every thread has read lv before its barrier
    constexpr_for<0, C, 1>([&](auto k_) {
      constexpr int k = decltype(k_)::value;
      if (tid * C + k < n) lv[tid * C + k] = V[k];
    });
  });
  __syncthreads();
  for (int i = tid; i < n; i += T) vm[off + i] = lv[i];
}

}  // namespace fms
