// imexsw_profiles.h -- vertical-profile closures (VERTICAL_PROFILES_FLAG) as
// device functions: a log velocity profile u ~ log(30 z / k_s + 1) below a
// boundary-layer top h0 and uniform above it, exponential solid
// concentrations exp(a z) with a = -w_s / epsilon_s (Rouse), their depth
// averages by an n_quad-point Gauss-Legendre rule on [0, h0] plus the
// uniform part on [h0, h].
//   r_phys_var's mean speed (Aitken iteration on avg_profiles_mix),
//     src/constitutive_2d.f90:797-942, 970-1123
//   qp_to_qc's profile momentum, src/constitutive_2d.f90:1976-2107
//   eval_flux_coeffs, src/constitutive_2d.f90:2532-2823
//   eval_dep_coeffs, src/constitutive_2d.f90:2844-2986
//   Lambert W on both real branches, src/geometry_2d.f90:1776-2038
//   integrate_friction_term (rheology model 8), src/constitutive_2d.f90:
//     3252-3306
//
// The quadrature points stay out of arrays: every sum runs over the points
// in order, forming z_m, w_m and log(b z_m + 1) per point (one log) unless the
// logarithm is kept (the mean speed's iteration), and advances every solid
// class's sums together, so a cell holds a few accumulators per class instead
// of n_quad-long arrays.  Each sum is taken in the same order as the oracle's,
// so the results agree bit for bit.
#pragma once

#include "imexsw_math.h"

namespace imexsw {

// ---------------------------------------------------------------------------
// Lambert W for x in [-1/e, 0) (and x >= 0 on the principal branch)
// ---------------------------------------------------------------------------
// W = sum mu_k p^k about the branch point, p = +-sqrt(2 (e x + 1)) (Corless,
// Gonnet, Hare, Jeffrey & Knuth 1996, eqs. 4.22-4.24); used for |p| < 0.1
__device__ __forceinline__ double lw_series(double p) {
  constexpr double mu[13] = {
      -1.0, 1.0, -1.0 / 3.0, 11.0 / 72.0, -43.0 / 540.0, 769.0 / 17280.0,
      -221.0 / 8505.0, 680863.0 / 43545600.0, -1963.0 / 204120.0,
      226287557.0 / 37623398400.0, -5776369.0 / 1515591000.0,
      169709463197.0 / 69528040243200.0, -1118511313.0 / 709296588000.0};
  double s = mu[12];
#pragma unroll
  for (int k = 11; k >= 0; k--) s = s * p + mu[k];
  return s;
}

// Halley's iteration on w e^w = x until the step is below 1e-15 |w|
__device__ __forceinline__ double lw_halley(double x, double w) {
  for (int it = 0; it < 20; it++) {
    const double ew = det_exp(w);
    const double f = w * ew - x;
    const double wp1 = w + 1.0;
    const double dw = f / (ew * wp1 - (w + 2.0) * f / (2.0 * wp1));
    w = w - dw;
    if (!(fabs(dw) > 1.0e-15 * fabs(w))) break;
  }
  return w;
}

constexpr double kE = 2.718281828459045;

// W_0; -1 outside the domain (as lambertw0 returns)
__device__ __forceinline__ double lambertw0(double x) {
  const double p2 = 2.0 * (kE * x + 1.0);
  if (!(p2 > 0.0)) return -1.0;
  if (p2 < 0.01) return lw_series(sqrt(p2));
  double w;
  if (x < -0.25) {
    const double p = sqrt(p2);
    w = -1.0 + p * (1.0 + p * (-1.0 / 3.0 + p * (11.0 / 72.0)));
  } else {
    // Winitzki (2003): W ~ L (1 - log(1 + L) / (2 + L)), L = log(1 + x)
    const double L = det_log(1.0 + x);
    w = (x == 0.0) ? 0.0 : L * (1.0 - det_log(1.0 + L) / (2.0 + L));
  }
  return lw_halley(x, w);
}

// W_{-1}; -1 outside the domain and above -64 e^-64 (as lambertwm1 returns)
__device__ __forceinline__ double lambertwm1(double x) {
  const double p2 = 2.0 * (kE * x + 1.0);
  if (!(p2 > 0.0) || !(x < 0.0) || x > -1.0288423856755186e-26) return -1.0;
  if (p2 < 0.01) return lw_series(-sqrt(p2));
  double w;
  if (x < -0.25) {
    const double p = -sqrt(p2);
    w = -1.0 + p * (1.0 + p * (-1.0 / 3.0 + p * (11.0 / 72.0)));
  } else {
    const double L1 = det_log(-x), L2 = det_log(-L1);
    w = L1 - L2 + L2 / L1;
  }
  return lw_halley(x, w);
}

// ---------------------------------------------------------------------------
// profile geometry
// ---------------------------------------------------------------------------
// boundary-layer top: the smaller root z of b log(c z + 1) - z = a in units
// of k_s when h/k_s > H_crit_rel, else h (src/constitutive_2d.f90:821-854).
// The roots are -b W_0(arg) - 1/c and -b W_{-1}(arg) - 1/c with b > 0; as
// W_0 >= -1 >= W_{-1} the first is the smaller one, so W_{-1} is not formed.
__device__ __forceinline__ double vp_h0(const DevParams& P, double r_h) {
  const double h_rel = r_h / P.k_s;
  double h0_rel;
  if (h_rel > P.h_crit_rel) {
    const double a = h_rel * P.vonK / P.sqrt_ff;
    const double b = 1.0 / 30.0 + h_rel, c = 30.0;
    const double d = a / b - 1.0 / (b * c);
    const double arg = -det_exp(d) / (b * c);
    h0_rel = -(b * lambertw0(arg)) - 1.0 / c;
  } else {
    h0_rel = h_rel;
  }
  return h0_rel * P.k_s;
}

// The mean speed's iteration reads each point's logarithm four to twenty
// times: the first kVpCache points' stay in LDS, one column per lane of the
// workgroup (at most kVpLanes), the rest are formed again.  40 KB a workgroup:
// four fit a CU, the registers allow two or three.  500 x 386, model 8, two
// conversions a cell: stage kernel 630 us with every logarithm formed each time,
// 487 from LDS, 458 with the points unrolled and without range selects, 380 with
// full wavefronts (item_cell).
constexpr int kVpCache = 20, kVpLanes = 256;

// point m of the rule on [0, h0]: z, weight and log(b z + 1)
__device__ __forceinline__ void vp_point(const DevParams& P, int m, double h0, double b,
                                         double& z, double& w, double& lz) {
  z = 0.5 * h0 * (P.zq[m] + 1.0);
  w = 0.5 * h0 * P.wq[m];
  lz = det_log(b * z + 1.0);
}

// What the closures of one state share whatever its velocity: the
// boundary-layer top (from h) and the settling speeds (from the carrier
// density), so that a face side's momentum and flux coefficients form
// them once
template <int NS>
struct VpPre {
  double h0;
  double sv[NS > 0 ? NS : 1];
};
template <int NS>
__device__ __forceinline__ void vp_pre(const DevParams& P, double r_h, double rho_c,
                                       VpPre<NS>& r) {
  r.h0 = vp_h0(P, r_h);
  const double ikv = 1.0 / P.kin_visc_c;
#pragma unroll
  for (int i = 0; i < NS; i++) r.sv[i] = settling_velocity(P, P.diam_s[i], P.rho_s[i], rho_c, ikv);
}

// Rouse numbers w_s / (vonK u*) (zero without shear)
template <int NS>
__device__ __forceinline__ void vp_rouse(const DevParams& P, double shear_vel, const double* sv,
                                         double* rouse) {
#pragma unroll
  for (int i = 0; i < NS; i++) rouse[i] = (shear_vel > 0.0) ? sv[i] / (P.vonK * shear_vel) : 0.0;
}

// Exponents a_i = -w_s / epsilon_s of the solid profiles exp(a_i z)
template <int NS>
__device__ __forceinline__ void vp_exponents(const DevParams& P, double shear_vel, double h0,
                                             const double* sv, double* a) {
  const double eps_s = P.Sc * shear_vel * P.vonK * ((h0 / 6.0) + (P.k_s / 60.0));
  const double a_coeff = -(P.vonK * shear_vel / eps_s);
  double rouse[NS > 0 ? NS : 1];
  vp_rouse<NS>(P, shear_vel, sv, rouse);
#pragma unroll
  for (int i = 0; i < NS; i++) a[i] = a_coeff * rouse[i];
}

// The sums the closures start from, for the solid exponents a_i:
//   se_i = sum w e_i, sq_i = sum w (e_i lz), sl_i = sum e_i (w lz^2) (FULL),
// with e_i = exp(a_i z), over the points in order, and e_i at h0.
template <int NS>
struct VpSums {
  double se[NS > 0 ? NS : 1], sq[NS > 0 ? NS : 1], sl[NS > 0 ? NS : 1], eh0[NS > 0 ? NS : 1];
};
template <int NS>
__device__ __forceinline__ void vp_sums_zero(VpSums<NS>& S) {
#pragma unroll
  for (int i = 0; i < NS; i++) S.se[i] = S.sq[i] = S.sl[i] = 0.0;
}
// PLAIN: no exponent of the rule leaves the exponential's ordinary range
template <int NS, bool FULL, bool PLAIN>
__device__ __forceinline__ void vp_sums_add(const double* a, double z, double w, double lz,
                                            double wll, VpSums<NS>& S) {
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const double e = PLAIN ? det_exp_core(a[i] * z) : det_exp(a[i] * z);
    S.se[i] += w * e;
    S.sq[i] += w * (e * lz);
    if (FULL) S.sl[i] += e * wll;
  }
}
// the points lie in (0, h0): |a h0| <= 700 bounds every exponent (a NaN fails)
template <int NS>
__device__ __forceinline__ bool vp_plain(const double* a, double h0) {
  bool p = true;
#pragma unroll
  for (int i = 0; i < NS; i++) p = p && fabs(a[i] * h0) <= 700.0;
  return p;
}
template <int NS>
__device__ __forceinline__ void vp_sums_top(const double* a, double h0, VpSums<NS>& S) {
#pragma unroll
  for (int i = 0; i < NS; i++) S.eh0[i] = det_exp(a[i] * h0);
}

// What a state's momentum and flux coefficients share whatever its velocity
// (and each other's sums): slog = sum w lz, sll = sum w lz^2, lh0 the
// logarithm at h0.  mom and flx are the sums at the momentum's and at the
// fluxes' speed, which differ by the slope's vertical velocity alone: the
// logarithms are formed once for both, and without slope correction the
// exponentials too.
template <int NS>
struct VpState : VpPre<NS> {
  double slog, sll, lh0;
  VpSums<NS> mom, flx;
};
// FLX: the fluxes' sums too; two: at another speed than the momentum's
template <int NS, bool FLX, bool PLAIN>
__device__ __forceinline__ void vp_state_points(const DevParams& P, const double* a,
                                                const double* af, bool two, VpState<NS>& S) {
  const double b = 30.0 / P.k_s;
#pragma nounroll
  for (int m = 0; m < P.nq; m++) {
    double z, w, lz;
    vp_point(P, m, S.h0, b, z, w, lz);
    S.slog += w * lz;
    const double wll = w * (lz * lz);
    if (FLX) S.sll += wll;
    if (FLX && !two) {
      vp_sums_add<NS, true, PLAIN>(a, z, w, lz, wll, S.flx);
    } else {
      vp_sums_add<NS, false, PLAIN>(a, z, w, lz, wll, S.mom);
      if (FLX) vp_sums_add<NS, true, PLAIN>(af, z, w, lz, wll, S.flx);
    }
  }
}
template <int NS, bool FLX>
__device__ __forceinline__ void vp_state(const DevParams& P, double u2, double w2,
                                         VpState<NS>& S) {
  const double b = 30.0 / P.k_s;
  double a[NS > 0 ? NS : 1], af[NS > 0 ? NS : 1];
  vp_exponents<NS>(P, P.sqrt_ff * sqrt(u2 + 0.0 * 0.0), S.h0, S.sv, a);
  const bool two = FLX && P.slope;
  if (two) vp_exponents<NS>(P, P.sqrt_ff * sqrt(u2 + w2), S.h0, S.sv, af);
  S.slog = 0.0;
  S.sll = 0.0;
  vp_sums_zero<NS>(S.mom);
  if (FLX) vp_sums_zero<NS>(S.flx);
  if (__all(vp_plain<NS>(a, S.h0) && (!two || vp_plain<NS>(af, S.h0))))
    vp_state_points<NS, FLX, true>(P, a, af, two, S);
  else
    vp_state_points<NS, FLX, false>(P, a, af, two, S);
  S.lh0 = det_log(b * S.h0 + 1.0);
  if (two) {
    vp_sums_top<NS>(a, S.h0, S.mom);
    vp_sums_top<NS>(af, S.h0, S.flx);
  } else if (FLX) {
    vp_sums_top<NS>(a, S.h0, S.flx);
    S.mom = S.flx;
  } else {
    vp_sums_top<NS>(a, S.h0, S.mom);
  }
}

// avg_profiles_mix (src/constitutive_2d.f90:970-1123): the profile-averaged
// mixture momentum per unit depth at mean speed u_guess (its dynamic
// pressure output is overwritten by the caller and not formed)
// lc: the lane's log(b z + 1) of the first kVpCache points, kVpLanes apart;
// ncu, lh0: formed by the caller, they do not depend on the speed
template <int NS>
__device__ __forceinline__ double vp_avg_mix(const DevParams& P, double h, const double* sv,
                                             const double* ra, double u_guess, double h0,
                                             double b, double ncu, double u_rel0, double rho_c,
                                             const double* lc) {
  double a[NS > 0 ? NS : 1];
  vp_exponents<NS>(P, u_guess * P.sqrt_ff, h0, sv, a);
  VpSums<NS> S;
  vp_sums_zero<NS>(S);
  const int n0 = min(P.nq, kVpCache);
  int m = 0;
  if (__all(vp_plain<NS>(a, h0))) {
#pragma unroll 4
    for (; m < n0; m++)
      vp_sums_add<NS, false, true>(a, 0.5 * h0 * (P.zq[m] + 1.0), 0.5 * h0 * P.wq[m],
                                   lc[m * kVpLanes], 0.0, S);
  }
#pragma nounroll
  for (; m < P.nq; m++) {
    double z, w, lz;
    vp_point(P, m, h0, b, z, w, lz);
    vp_sums_add<NS, false, false>(a, z, w, lz, 0.0, S);
  }
  vp_sums_top<NS>(a, h0, S);
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const double nca = 1.0 / ((S.se[i] + S.eh0[i] * (h - h0)) / h);
    const double d1 = ncu * nca * S.sq[i];
    const double d2 = (h - h0) * u_rel0 * (nca * S.eh0[i]);
    const double rua = ra[i] * u_guess * (d1 + d2) / h;
    s += (P.rho_s[i] - rho_c) / P.rho_s[i] * rua;
  }
  return u_guess * rho_c + s;
}

// r_phys_var's mean speed (src/constitutive_2d.f90:797-942): the fixed point
// of u <- u |q| / (h M(u)) with Aitken's acceleration, at most ten rounds,
// tolerances 1e-8 as the reference's single-precision literals round
template <int NS>
__device__ __forceinline__ double vp_velocity(const DevParams& P, double r_h, double q2,
                                              double q3, double r_rho_m, double r_rho_c,
                                              const double* r_alphas) {
  const double ikv = 1.0 / P.kin_visc_c;
  double sv[NS > 0 ? NS : 1], ra[NS > 0 ? NS : 1];
#pragma unroll
  for (int i = 0; i < NS; i++) {
    ra[i] = r_alphas[i] * P.rho_s[i];
    sv[i] = settling_velocity(P, P.diam_s[i], P.rho_s[i], r_rho_c, ikv);
  }
  const double h0 = vp_h0(P, r_h);
  const double b = 30.0 / P.k_s;
  __shared__ double cache[kVpCache * kVpLanes];
  double* lc = cache + threadIdx.x;
  double slog = 0.0;
  for (int m = 0; m < P.nq; m++) {
    double z, w, lz;
    vp_point(P, m, h0, b, z, w, lz);
    slog += w * lz;
    if (m < kVpCache) lc[m * kVpLanes] = lz;
  }
  const double lh0 = det_log(b * h0 + 1.0);
  const double ncu = 1.0 / ((slog + lh0 * (r_h - h0)) / r_h);
  const double u_rel0 = ncu * lh0;
  const double uRho_avg = sqrt(q2 * q2 + q3 * q3) / r_h;
  double u_guess = uRho_avg / r_rho_m, u_new = u_guess;
  const double rel_tol = (double)1.e-8f, abs_tol = (double)1.e-8f;
  for (int it = 0; it < 10; it++) {
    // two steps of the fixed point from x0, one piece of code
    const double x0 = u_guess;
    double x1 = u_guess, x2 = u_guess;
#pragma nounroll
    for (int half = 0; half < 2; half++) {
      x1 = x2;
      x2 = x1 * uRho_avg /
           vp_avg_mix<NS>(P, r_h, sv, ra, x1, h0, b, ncu, u_rel0, r_rho_c, lc);
    }
    u_new = x2;
    const double den = (x2 - x1) - (x1 - x0);
    if (fabs(den) < (double)0.1f * abs_tol) break;
    u_new = x2 - ((x2 - x1) * (x2 - x1)) / den;
    if ((fabs(u_guess - u_new) / u_guess < rel_tol) || (fabs(u_guess - u_new) < abs_tol)) break;
    u_guess = u_new;
  }
  return u_new;
}

// qp_to_qc's profile momentum (src/constitutive_2d.f90:1976-2107) from the
// state's sums
template <int NS>
__device__ __forceinline__ void vp_momentum(const DevParams& P, double r_h, double r_u,
                                            double r_v, const VpState<NS>& S, double r_rho_c,
                                            const double* r_alphas, double& qc2, double& qc3) {
  const double mod_vel = sqrt(r_u * r_u + r_v * r_v + 0.0 * 0.0);
  const double h0 = S.h0;
  const double ncu = 1.0 / ((S.slog + S.lh0 * (r_h - h0)) / r_h);
  const double u_rel0 = ncu * S.lh0;
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const double eh0 = S.mom.eh0[i];
    const double nca = 1.0 / ((S.mom.se[i] + eh0 * (r_h - h0)) / r_h);
    const double d1 = (mod_vel * ncu) * (r_alphas[i] * nca) * S.mom.sq[i];
    const double d2 = (r_h - h0) * (mod_vel * u_rel0) * ((nca * eh0) * r_alphas[i]);
    const double rua = P.rho_s[i] * (d1 + d2) / r_h;
    s += (P.rho_s[i] - r_rho_c) / P.rho_s[i] * rua;
  }
  const double uRho_avg = mod_vel * r_rho_c + s;
  qc2 = r_h * uRho_avg * r_u / mod_vel;
  qc3 = r_h * uRho_avg * r_v / mod_vel;
}

// eval_flux_coeffs (src/constitutive_2d.f90:2532-2823); sc[0..NV-1], from
// the state's sums
template <int NS>
__device__ __forceinline__ void vp_flux_coeffs(const DevParams& P, const double* qp, double Bx,
                                               double By, const VpState<NS>& S, double r_rho_c,
                                               double r_rho_m, double* sc) {
  constexpr int NV = 4 + NS;
  const double r_h = qp[0], r_hu = qp[1], r_hv = qp[2], r_u = qp[NV], r_v = qp[NV + 1];
  double al[NS > 0 ? NS : 1];
#pragma unroll
  for (int i = 0; i < NS; i++) al[i] = P.alpha ? qp[4 + i] : qp[4 + i] / qp[0];
  const double r_hw = P.slope ? r_hu * Bx + r_hv * By : 0.0;
  const double r_w = P.slope ? r_u * Bx + r_v * By : 0.0;
  const double mod_hvel = sqrt(r_hu * r_hu + r_hv * r_hv + r_hw * r_hw);
  const double mod_vel = sqrt(r_u * r_u + r_v * r_v + r_w * r_w);
  const double h0 = S.h0;
  const double lt_h0 = S.lh0 * S.lh0;
  const double ncu = 1.0 / ((S.slog + S.lh0 * (r_h - h0)) / r_h);
  const double u_rel0 = ncu * S.lh0;
  double irhv = 0.0, rua[NS > 0 ? NS : 1];
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const double eh0 = S.flx.eh0[i];
    const double nca = 1.0 / ((S.flx.se[i] + eh0 * (r_h - h0)) / r_h);
    const double d1 = (mod_vel * ncu) * (al[i] * nca) * S.flx.sq[i];
    const double d2 = (r_h - h0) * (mod_vel * u_rel0) * (al[i] * (nca * eh0));
    rua[i] = P.rho_s[i] * (d1 + d2) / r_h;
    const double d3 = (r_h - h0) * eh0 * lt_h0;
    irhv = irhv + (P.rho_s[i] - r_rho_c) * (nca * al[i]) * (mod_hvel * mod_vel * (ncu * ncu)) *
                      (S.flx.sl[i] + d3);
  }
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < NS; i++) s += (P.rho_s[i] - r_rho_c) / P.rho_s[i] * rua[i];
  const double uRho_avg = mod_vel * r_rho_c + s;
  const double ihv = mod_hvel * mod_vel * (ncu * ncu) * (S.sll + (r_h - h0) * lt_h0);
  const double rvv = (irhv + r_rho_c * ihv) / (r_h * r_h);
  sc[0] = uRho_avg / (mod_vel * r_rho_m);
  sc[1] = rvv / (uRho_avg * mod_vel);
  sc[2] = sc[1];
  sc[3] = sc[0];
#pragma unroll
  for (int i = 0; i < NS; i++) sc[4 + i] = rua[i] / (P.rho_s[i] * al[i] * mod_vel);
}

// eval_dep_coeffs (src/constitutive_2d.f90:2844-2986): bottom over mean
// concentration of each class; sv: their settling speeds
template <int NS>
__device__ __forceinline__ void vp_dep_coeffs(const DevParams& P, double r_h, double mod_vel,
                                              double r_rho_c, double* dep, double* sv) {
  const double shear_vel = P.sqrt_ff * mod_vel;
  VpPre<NS> pre;
  vp_pre<NS>(P, r_h, r_rho_c, pre);
  const double h0 = pre.h0;
  double a[NS > 0 ? NS : 1], se[NS > 0 ? NS : 1];
  vp_exponents<NS>(P, shear_vel, h0, pre.sv, a);
#pragma unroll
  for (int i = 0; i < NS; i++) {
    se[i] = 0.0;
    sv[i] = pre.sv[i];
  }
  for (int m = 0; m < P.nq; m++) {
    const double z = 0.5 * h0 * (P.zq[m] + 1.0);
    const double w = 0.5 * h0 * P.wq[m];
#pragma unroll
    for (int i = 0; i < NS; i++) se[i] += w * det_exp(a[i] * z);
  }
#pragma unroll
  for (int i = 0; i < NS; i++) dep[i] = 1.0 / ((se[i] + det_exp(a[i] * h0) * (r_h - h0)) / r_h);
}

}  // namespace imexsw
