// LJ + LK pair potentials as device functions, written for wave64 VALU code.
//
// Same functions as the reference (tmol/score/ljlk/potentials/lj.hh:21-177,
// lk_isotropic.hh:22-360, common.hh:13-44, tmol/score/common/
// cubic_hermite_polynomial.hh), arranged so that the regions of a piecewise
// potential share one evaluation of the underlying closed form at a clamped
// abscissa x, and the pieces that extend it (linear, Hermite to zero) are one
// expression in d - x:
//
//   LJ:  x = clamp(d, d_lin, cpoly_dmin); one 12-6 evaluation V(x), V'(x);
//        no branches.
//   LK:  one f_desolv evaluation at clamp(d, close_dmax, far_dmin) per
//        direction, a second one at d_min only where d < close_dmax; both
//        directions have the same knots, so their values are summed before
//        the (linear) interpolation.
//
// Float builds use the hardware rcp / sqrt / exp (1-2 ulp); the double
// instantiation (the oracle run) uses correctly rounded division, sqrt and
// exp.  Results agree with the reference's formulas to rounding.
#pragma once

#include <hip/hip_runtime.h>

namespace tmol_ljlk {

template <typename Real>
struct GlobalParams {
  Real max_dis;               // cpoly_dmax (lj.hh:125), cpoly_far_dmax (lk)
  Real dlin_factor;           // lj_dlin_sigma_factor
  Real lin6;                  // dlin_factor^-6
  Real hbond_dis;             // lj_hbond_dis
  Real hbond_oh_dis;          // lj_hbond_OH_donor_dis
  Real hbond_hdis;            // lj_hbond_hdis
  Real spline_start;          // max_dis - 1.5
  Real cpoly_cap;             // max_dis - 0.1
  Real max_dis2;              // max_dis^2 (pair culling)
};

// per-atom flag bits
enum : int {
  F_DONOR = 1,
  F_OH_DONOR = 2,  // donor and hydroxyl
  F_POLARH = 4,
  F_ACCEPTOR = 8,
  F_CARBON_LK = 16,
};

template <typename Real>
__device__ __forceinline__ Real fast_rcp(Real x);
template <>
__device__ __forceinline__ float fast_rcp<float>(float x) {
  return __builtin_amdgcn_rcpf(x);
}
template <>
__device__ __forceinline__ double fast_rcp<double>(double x) {
  return 1.0 / x;
}

template <typename Real>
__device__ __forceinline__ Real fast_sqrt(Real x);
template <>
__device__ __forceinline__ float fast_sqrt<float>(float x) {
  return __builtin_amdgcn_sqrtf(x);
}
template <>
__device__ __forceinline__ double fast_sqrt<double>(double x) {
  return __builtin_sqrt(x);
}

// 1 / sqrt(x): hardware v_rsq_f32 for float, correctly rounded ops for double
template <typename Real>
__device__ __forceinline__ Real fast_rsqrt(Real x);
template <>
__device__ __forceinline__ float fast_rsqrt<float>(float x) {
  return __builtin_amdgcn_rsqf(x);
}
template <>
__device__ __forceinline__ double fast_rsqrt<double>(double x) {
  return 1.0 / __builtin_sqrt(x);
}

template <typename Real>
__device__ __forceinline__ Real fast_exp(Real x);
template <>
__device__ __forceinline__ float fast_exp<float>(float x) {
  return __expf(x);
}
template <>
__device__ __forceinline__ double fast_exp<double>(double x) {
  return exp(x);
}

// v limited to [lo, hi], lo <= hi: one instruction for float
__device__ __forceinline__ float clamp(float v, float lo, float hi) {
  return __builtin_amdgcn_fmed3f(v, lo, hi);
}
__device__ __forceinline__ double clamp(double v, double lo, double hi) {
  return v > hi ? hi : (v > lo ? v : lo);
}

// connectivity weight: >4 bonds -> 1, ==4 -> 0.2, else 0 (common.hh:13-22)
template <typename Real>
__device__ __forceinline__ Real cp_weight(int sep) {
  return sep > 4 ? Real(1) : (sep == 4 ? Real(0.2) : Real(0));
}

// hbond-aware sigma (common.hh:24-44): donor-acceptor pairs use the hbond
// distance (the hydroxyl-donor one if either atom is a hydroxyl donor),
// polar-hydrogen-acceptor pairs the hbond-H distance, others r_i + r_j.
// With the flag bits D = 1, OH = 2, PH = 4, A = 8: bit 0 of
// (Ai & (Dj | PHj)) | (Aj & (Di | PHi)) is the donor-acceptor test and bit 2
// the polar-H-acceptor test, each the OR of both orientations.
template <typename Real>
__device__ __forceinline__ Real lj_sigma(int fi, int fj, Real ri, Real rj,
                                         const GlobalParams<Real>& g) {
  // bit 3 of each sign-extended to a mask
  const int both = (__builtin_amdgcn_sbfe(fi, 3, 1) & fj) | (__builtin_amdgcn_sbfe(fj, 3, 1) & fi);
  const bool da = both & F_DONOR;
  const bool ha = both & F_POLARH;
  const bool oh = (fi | fj) & F_OH_DONOR;
  Real s = ri + rj;
  s = ha ? g.hbond_hdis : s;
  s = da ? (oh ? g.hbond_oh_dis : g.hbond_dis) : s;
  return s;
}

// LJ for one pair: returns weighted (atr, rep) and d(atr+rep)/dd.
// Only one of atr/rep carries the derivative: rep inside sigma, atr outside.
// With u = d - x: u < 0 on the linear piece (V + V' u), 0 on the 12-6 piece,
// and on the Hermite piece to (0, 0) at max_dis, t = u / w, the value is
// (1 - t)^2 (V + V' u + 2 t V); t = 0 elsewhere, so one expression covers all
// three.
// Rounding: on the linear piece (sigma / x)^6 is dlin_factor^-6 for any sigma,
// a constant rounded once; sigma * rcp(x) is off by 2-3 ulp, and its sixth
// power by as much six times, in the pairs that carry most of the repulsion.
// V and V' come from s = (sigma/x)^6 - (sigma/x)^12, one rounding as an fma.
// Against float64, 512 poses: energies 9.4e-8 -> 4.6e-8, gradients 5.1e-7 ->
// 2.4e-7, at the same time (2.23 ms).
template <typename Real, bool DERIV>
__device__ __forceinline__ void lj_pair(Real dist, Real sigma, Real eps,
                                        Real weight,
                                        const GlobalParams<Real>& g,
                                        Real& atr, Real& rep, Real& dlj) {
  const Real d_lin = sigma * g.dlin_factor;
  const Real cpoly_dmin = clamp(sigma, g.spline_start, g.cpoly_cap);
  // evaluation point of the 12-6 form
  const bool linear = dist < d_lin;
  const Real x = linear ? d_lin : fmin(dist, cpoly_dmin);
  const Real inv_x = fast_rcp(x);
  const Real sd = sigma * inv_x;
  const Real sd2 = sd * sd;
  const Real sd6 = linear ? g.lin6 : sd2 * sd2 * sd2;
  const Real s = sd6 - sd6 * sd6;
  const Real V = -eps * (s + sd6);
  const Real dV = eps * Real(12) * s * inv_x;
  const Real u = dist - x;
  const Real iw = u > Real(0) ? fast_rcp(g.max_dis - cpoly_dmin) : Real(0);
  const Real t = u * iw;
  const Real q = fmax(Real(1) - t, Real(0));  // zero at and beyond max_dis
  const Real b = V + dV * u + Real(2) * t * V;
  const Real lj = q * q * b;
  const bool inside = dist < sigma;
  atr = weight * (inside ? -eps : lj);
  rep = weight * (inside ? lj + eps : Real(0));
  dlj = DERIV ? weight * (q * (q * (dV + Real(2) * iw * V) - Real(2) * iw * b)) : Real(0);
}

// LK knots on the 1/20 A^2 etable grid (lk_isotropic.hh:116-125)
template <typename Real>
__device__ __forceinline__ void lk_knots(Real sigma, bool is_cc, Real& d_min,
                                         Real& close_dmin, Real& close_dmax) {
  Real dm = Real(double(sigma) * 0.89);
  if (is_cc) dm = dm > Real(4.2) ? dm : Real(4.2);
  Real n = floor(Real(20) * dm * dm);
  Real lo = n - Real(29);
  lo = lo > Real(0) ? lo : Real(0);
  Real hi = n + Real(21);
  hi = hi < Real(405) ? hi : Real(405);
  d_min = dm;
  close_dmin = fast_sqrt(lo * Real(0.05));
  close_dmax = fast_sqrt(hi * Real(0.05));
}

// one direction of LK: c = -vol_j * K_i with K_i = dg_i / (2 pi^1.5 lambda_i),
// r_i and 1 / lambda_i^2
template <typename Real>
struct LkSide {
  Real c, r, inv_lam2;
};

// sum over the directions of f_desolv and its derivative at x
template <typename Real, int SIDES>
__device__ __forceinline__ void fdesolv(Real x, const LkSide<Real> (&side)[SIDES], Real& f,
                                        Real& df) {
  const Real inv_x = fast_rcp(x);
  const Real inv_x2 = inv_x * inv_x;
  f = df = Real(0);
#pragma unroll
  for (int k = 0; k < SIDES; ++k) {
    const Real dr = x - side[k].r;
    const Real sl = dr * side[k].inv_lam2;
    const Real e = side[k].c * inv_x2 * fast_exp(-dr * sl);
    f += e;
    df += e * (Real(-2) * (inv_x + sl));
  }
}

// isotropic LK (lk_isotropic.hh:167-235), unweighted, summed over the given
// directions (their knots are the same): f at clamp(d, cdmax, far_dmin), the
// Hermite piece to zero as in lj_pair, and below cdmax the Hermite piece from
// (cdmin, f(d_min), slope 0), constant below cdmin.
template <typename Real, bool DERIV, int SIDES>
__device__ __forceinline__ void lk_sides(Real dist, Real d_min, Real cdmin, Real cdmax,
                                         const LkSide<Real> (&side)[SIDES],
                                         const GlobalParams<Real>& g, Real& V, Real& dV) {
  const bool close = dist < cdmax;
  const Real x = close ? cdmax : (dist < g.spline_start ? dist : g.spline_start);
  Real f, df;
  fdesolv<Real, SIDES>(x, side, f, df);
  const Real u = dist - x;
  const Real iw = u > Real(0) ? fast_rcp(g.max_dis - g.spline_start) : Real(0);
  const Real t = u * iw;
  Real q = Real(1) - t;
  q = q > Real(0) ? q : Real(0);
  const Real b = f + df * u + Real(2) * t * f;
  V = q * q * b;
  dV = DERIV ? q * (q * (df + Real(2) * iw * f) - Real(2) * iw * b) : Real(0);
  if (close) {
    Real f0, df0;
    fdesolv<Real, SIDES>(d_min, side, f0, df0);
    const Real w = cdmax - cdmin;
    // below cdmin tc and the slope are 0 whatever w is: the knots' cap is on
    // cdmax alone, so from a sigma of 5.234 on cdmin is not below it
    const Real inv_w = dist < cdmin ? Real(0) : fast_rcp(w);
    const Real tc = (dist - cdmin) * inv_w;
    const Real dp1 = df * w;
    const Real c2 = Real(3) * (f - f0) - dp1;
    const Real c3 = dp1 - Real(2) * (f - f0);
    V = f0 + tc * tc * (c2 + tc * c3);
    dV = DERIV ? tc * (Real(2) * c2 + Real(3) * tc * c3) * inv_w : Real(0);
  }
}

// ---- elec (tmol/score/elec/potentials/potentials.hh)

// Per-launch constants of the potential (computed on the host in the
// reference's precision: eps() at max_dis and min_dis in float, the rest in
// Real).  Hermite pieces take the charge product out as a common factor.
template <typename Real>
struct ElecConst {
  Real D, S, hdd;       // hdd = 0.5 (D - D0)
  Real C1, C2;          // 322.0637, C1 / (max_dis eps(max_dis))
  Real lps, lpe;        // min_dis -+ 0.25
  Real hps, hpe;        // max_dis - 1, max_dis
  Real mds;             // C1 / (min_dis eps(min_dis)) - C2 (flat part)
  Real e_lo, de_lo;     // Coulomb value and slope at lpe (per unit q1 q2)
  Real e_hi, de_hi;     // ... at hps
  Real lw, hw;          // lpe - lps, hpe - hps
  Real inv_lw, inv_hw;
  Real cull2;           // (max_dis + 1e-3)^2: phase A keeps pairs below it
};

// V and dV/dd per unit charge product (potentials.hh:55-138).  Branch-free
// over the wave: the Coulomb form is evaluated at clamp(d, lpe, hps), and one
// Hermite piece, its ends chosen by region, covers both fades (below lps it
// sits at t = 0: the flat part, slope 0).
template <typename Real, bool DERIV>
__device__ __forceinline__ void elec_unit(Real dist, const ElecConst<Real>& k, Real& V,
                                          Real& dV) {
  const Real x = dist < k.lpe ? k.lpe : (dist < k.hps ? dist : k.hps);
  const Real ex = fast_exp(-x * k.S);
  const Real xs = x * k.S;
  const Real eps = k.D - k.hdd * (Real(2) + Real(2) * xs + xs * xs) * ex;
  const Real r = fast_rcp(eps);
  const Real ix = fast_rcp(x);
  const Real vc = k.C1 * ix * r - k.C2;
  Real dc = Real(0);
  if (DERIV) {
    const Real deps = k.hdd * xs * xs * k.S * ex;  // 0.5 (D - D0) x^2 S^3 e^{-xS}
    dc = -k.C1 * (eps + x * deps) * ix * ix * r * r;
  }
  const bool lo = dist < k.lpe;
  const bool hi = dist >= k.hps;
  const Real x0 = lo ? k.lps : k.hps;
  const Real w = lo ? k.lw : k.hw;
  const Real iw = lo ? k.inv_lw : k.inv_hw;
  const Real p0 = lo ? k.mds : k.e_hi;
  const Real p1 = lo ? k.e_lo : Real(0);
  const Real dp0 = lo ? Real(0) : k.de_hi * w;
  const Real dp1 = lo ? k.de_lo * w : Real(0);
  Real t = (dist - x0) * iw;
  t = t > Real(0) ? t : Real(0);
  const Real c2 = Real(-2) * dp0 - dp1 - Real(3) * p0 + Real(3) * p1;
  const Real c3 = dp0 + dp1 + Real(2) * p0 - Real(2) * p1;
  const Real vh = p0 + t * (dp0 + t * (c2 + t * c3));
  const Real dh = (dp0 + t * (Real(2) * c2 + Real(3) * t * c3)) * iw;
  const bool fade = lo || hi;
  V = fade ? vh : vc;
  dV = DERIV ? (fade ? dh : dc) : Real(0);
  const bool out = dist >= k.hpe;
  V = out ? Real(0) : V;
  dV = out ? Real(0) : dV;
}

}  // namespace tmol_ljlk
