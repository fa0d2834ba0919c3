// imexsw_newton.h -- the per-cell implicit Runge-Kutta stage (one lane per
// cell, everything in registers): semi-implicit Coulomb predictor, Newton
// with complex-step Jacobian and backtracking line search for the Voellmy
// drag, velocity realignment, and the assembly checks of imex_RK_solver.
#pragma once

#include "imexsw_physics.h"

namespace imexsw {

// eval_f (src/solver_2d.f90:2243-2282) from the implicit terms' real parts
// nh1, nh2 at qj
template <int NS>
__device__ __forceinline__ void finish_f(const double* qj, const double* qold,
                                         const double* Rj, double a_diag, double dt,
                                         double nh1, double nh2, double* f, double& scal) {
  constexpr int NV = 4 + NS;
  double s = 0.0;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const double R = (i == 1) ? Rj[1] - a_diag * nh1 : (i == 2) ? Rj[2] - a_diag * nh2 : Rj[i];
    f[i] = qj[i] - qold[i] + dt * R;
  }
#pragma unroll
  for (int i = 0; i < NV; i++) s += f[i] * f[i];
  scal = 0.5 * s;
}
template <int NS, int RM = 1>
__device__ __forceinline__ void eval_f(const DevParams& P, const double* qj,
                                       const double* qold, const double* Rj,
                                       double a_diag, double dt, double Bx,
                                       double By, double* f, double& scal) {
  ImplPt b;
  implicit_real<NS, RM>(P, qj, Bx, By, b);
  finish_f<NS>(qj, qold, Rj, a_diag, dt, b.n1, b.n2, f, scal);
}

// gfortran NORM2 (scaled sum of squares)
template <int NV>
__device__ __forceinline__ double norm2_(const double* x) {
  double scale = 0.0, res = 1.0;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    if (x[i] != 0.0) {
      double ax = fabs(x[i]);
      if (scale < ax) {
        double r = scale / ax;
        res = 1.0 + res * (r * r);
        scale = ax;
      } else {
        double r = ax / scale;
        res = res + r * r;
      }
    }
  }
  return scale * sqrt(res);
}

struct NewtonOut {
  int iters;
  int conv;
  int ls_evals;  // residual evaluations inside the line search
};

// The Newton step from the residual rt and the implicit terms' derivatives
// J1[], J2[] (d nh_{1,2} / d rel_1, rel_2): the partitioned solve of
// src/solver_2d.f90:1846-1925 on the 2x2 momentum block (the other unknowns'
// columns are the diagonal org, their right-hand side terms are zero).
// L receives the block (11, 21, 12, 22).  first: the first iteration, in which
// another unknown's residual that is not finite makes the momenta NaN through
// those zero terms (later ones have small residuals or NaN momenta already).
template <int NS>
__device__ __forceinline__ void newton_step(const double* org, const double* rt, double dta,
                                            const double* J1, const double* J2, double* L,
                                            double* desc, bool first) {
  constexpr int NV = 4 + NS;
  L[0] = org[1] - dta * J1[0];
  L[1] = 0.0 - dta * J1[1];
  L[2] = 0.0 - dta * J2[0];
  L[3] = org[2] - dta * J2[1];
  const double inv_det = fdiv(1.0, L[0] * L[3] - L[1] * L[2]);
#pragma unroll
  for (int i = 0; i < NV; i++) {
    if (i == 1) desc[i] = -((rt[1] * L[3] - rt[2] * L[2]) * inv_det) + 0.0;
    else if (i == 2) desc[i] = -((L[0] * rt[2] - L[1] * rt[1]) * inv_det) + 0.0;
    else desc[i] = 0.0 + -fdiv(rt[i], org[i]);
  }
  if (first) {
    double z = 0.0;
#pragma unroll
    for (int i = 0; i < NV; i++)
      if (i != 1 && i != 2) z += desc[i] * 0.0;
    desc[1] += z;
    desc[2] += z;
  }
}

// What lnsrch (src/solver_2d.f90:2019-2224) forms ahead of its first trial.
// The step's norm is only compared with stpmax >= 100 NV, and the smallest
// step alamin only matters after a rejected trial, so neither is formed
// while the largest component of the step is at most 100: the norm is then
// below stpmax / 2.  slope: desc . (rt . L) with L's zero entries left out.
struct LineSearch {
  double slope, dmax, mx;
  bool have_mx;  // mx is known (else formed by below_alamin when needed)
  bool none;     // alamin == 0: no trial, the step is dropped
};
constexpr double kTolX = kEps;

template <int NV>
__device__ __forceinline__ double ls_mx(const double* desc, const double* old) {
  double mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const double v = fdiv(fabs(desc[i]), fmax(fabs(old[i]), 1.0));
    if (v > mx) mx = v;
  }
  return mx;
}
template <int NS>
__device__ __forceinline__ LineSearch ls_begin(const double* org, const double* old,
                                               const double* rt, const double* L,
                                               double* desc) {
  constexpr int NV = 4 + NS;
  LineSearch s{0.0, -1.0, 0.0, false, false};
#pragma unroll
  for (int i = 0; i < NV; i++) s.dmax = fmax(s.dmax, fabs(desc[i]));
  if (!(s.dmax >= 0.0 && s.dmax <= 100.0)) {
    double dd = 0.0;
#pragma unroll
    for (int i = 0; i < NV; i++) dd += old[i] * old[i];
    const double stpmax = 100.0 * fmax(sqrt(dd), (double)NV);
    const double dabs = norm2_<NV>(desc);
    if (dabs > stpmax) {
#pragma unroll
      for (int i = 0; i < NV; i++) desc[i] = desc[i] * stpmax / dabs;
    }
    s.mx = ls_mx<NV>(desc, old);
    s.have_mx = true;
    s.none = (kTolX / s.mx) == 0.0;
  }
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const double g = (i == 1) ? rt[1] * L[0] + rt[2] * L[1]
                     : (i == 2) ? rt[1] * L[2] + rt[2] * L[3] : rt[i] * org[i];
    s.slope += g * desc[i];
  }
  return s;
}
// alam < alamin = TOLX / mx, mx the largest |desc| / max(|old|, 1): decided
// without the divisions unless alam is within 1e-6 of alamin's bounds
template <int NV>
__device__ __forceinline__ bool below_alamin(LineSearch& s, double alam, const double* desc,
                                             const double* old) {
  if (!s.have_mx) {
    double om = 1.0;
#pragma unroll
    for (int i = 0; i < NV; i++) om = fmax(om, fabs(old[i]));
    const double hi = alam * s.dmax;
    if (hi < 0.999999 * kTolX) return true;
    if (hi > 1.000001 * kTolX * om) return false;
    s.mx = ls_mx<NV>(desc, old);
    s.have_mx = true;
  }
  return alam < kTolX / s.mx;
}

// org = max(|q|, 1e-3), rel = q / org (+-1 where |q| is the larger).  Returns
// whether rel * org is q again (it may be a rounding off below 1e-3).
template <int NV>
__device__ __forceinline__ bool newton_scale(const double* q, double* org, double* rel) {
  const Rcp rm = rcp_of(1.0e-3);
  bool same = true;
#pragma unroll
  for (int i = 0; i < NV; i++) {
    const double a = fabs(q[i]);
    org[i] = fmax(a, 1.0e-3);
    rel[i] = (a >= 1.0e-3 && a < INFINITY) ? copysign(1.0, q[i]) : div_by(q[i], rm);
    if (a == INFINITY) rel[i] = __builtin_nan("");
    same = same && rel[i] * org[i] == q[i];
  }
  return same;
}

template <int NV>
__device__ __forceinline__ double max_abs(const double* x) {
  double m = 0.0;
#pragma unroll
  for (int i = 0; i < NV; i++) m = fmax(m, fabs(x[i]));
  return m;
}
// max |rel - old| / max(|rel|, 1) < TOLX (a power of two: the product is exact)
template <int NV>
__device__ __forceinline__ bool step_below_tolx(const double* rel, const double* old) {
  bool below = true;
#pragma unroll
  for (int i = 0; i < NV; i++)
    below = below && !(fabs(rel[i] - old[i]) >= kTolX * fmax(fabs(rel[i]), 1.0));
  return below;
}

// solve_rk_step with eval_jacobian and lnsrch (src/solver_2d.f90:1660-2365);
// RM = 6: the implicit terms of rheology model 6.
// The implicit unknowns are the momenta (implicit_flag = F,T,T,F,...,
// src/constitutive_2d.f90:478-480): the Jacobian has the 2x2 momentum block
// plus the diagonal scaling of the other unknowns, which is what the
// reference's packed partitioned solve reduces to.
template <int NS, int RM = 1>
__device__ __forceinline__ NewtonOut solve_rk_step(const DevParams& P, double* qj,
                                                  const double* qold,
                                                  const double* Rj, double a_diag,
                                                  double dt, double Bx, double By) {
  constexpr int NV = 4 + NS;
  const double TOLF = 1.0e-10;
  double org[NV], rel[NV], rt[NV], old[NV], desc[NV];
  double scal = 0.0;
  const bool same = newton_scale<NV>(qj, org, rel);
  NewtonOut out{0, 0, 0};
  int it;
  // b, rt and scal already belong to qj when the previous iteration ended
  // on an evaluated point (an accepted line-search point or the full first
  // step); the reference evaluates it again at the top of the iteration,
  // with the same operands, so that evaluation is skipped
  ImplPt b;
  bool fresh = false;
  for (it = 1; it <= 100; it++) {
    if (!fresh) {
      // the residual at qj; the Jacobian's point is rel * org, which in the
      // first iteration may be a rounding off qj
#pragma unroll 1
      for (int e = 0; e < 2; e++) {
        double q[NV];
#pragma unroll
        for (int m = 0; m < NV; m++) q[m] = e ? rel[m] * org[m] : qj[m];
        implicit_real<NS, RM>(P, q, Bx, By, b);
        if (e == 0) finish_f<NS>(qj, qold, Rj, a_diag, dt, b.n1, b.n2, rt, scal);
        if (it > 1 || same) break;
      }
    }
    bool restored = false;
    if (max_abs<NV>(rt) < TOLF) {
      out.conv = 1;
      break;
    }
    // --- Jacobian: complex step on the two momentum columns
    double J1[2], J2[2], L[4];
    {
      const double q1 = rel[1] * org[1], q2 = rel[2] * org[2];
      const double d1 = P.h_cs * org[1], d2 = P.h_cs * org[2];
      bool ok = implicit_col<RM>(P, b, q1, q2, d1, 0.0, Bx, By, J1[0], J1[1]);
      ok = implicit_col<RM>(P, b, q1, q2, 0.0, d2, Bx, By, J2[0], J2[1]) && ok;
      if (!ok) {
        double q[NV];
#pragma unroll
        for (int m = 0; m < NV; m++) q[m] = rel[m] * org[m];
#pragma unroll 1
        for (int p = 0; p < 2; p++) {
          double a, c;
          implicit_col_c<NS, RM>(P, q, p ? 0.0 : d1, p ? d2 : 0.0, Bx, By, a, c);
          J1[0] = p ? J1[0] : a;
          J1[1] = p ? J1[1] : c;
          J2[0] = a;
          J2[1] = c;
        }
      }
      J1[0] = J1[0] * P.one_by_h;
      J1[1] = J1[1] * P.one_by_h;
      J2[0] = J2[0] * P.one_by_h;
      J2[1] = J2[1] * P.one_by_h;
    }
    newton_step<NS>(org, rt, dt * a_diag, J1, J2, L, desc, it == 1);
#pragma unroll
    for (int i = 0; i < NV; i++) old[i] = rel[i];
    double alam = 1.0;
    LineSearch ls{};
    if (it > 1) ls = ls_begin<NS>(org, old, rt, L, desc);
    const double scal_old = scal;
    // The trials of lnsrch: the full step (accepted as it is in the first
    // iteration), then max(quadratic model, 0.5), then halvings (the cubic
    // model is capped at half the last step, so max(model, 0.5 * alam) is
    // always 0.5 * alam).  alam at least halves every pass after the first,
    // so it falls below alamin (>= ~1e-16 relative) within a few dozen
    // passes; the bound only guards against NaN states.
    for (int tr = 0; tr < 256 && !ls.none; tr++) {
#pragma unroll
      for (int i = 0; i < NV; i++) rel[i] = old[i] + alam * desc[i];
#pragma unroll
      for (int i = 0; i < NV; i++) qj[i] = rel[i] * org[i];
      implicit_real<NS, RM>(P, qj, Bx, By, b);
      finish_f<NS>(qj, qold, Rj, a_diag, dt, b.n1, b.n2, rt, scal);
      if (it == 1) break;
      out.ls_evals++;
      if (scal <= 0.9 * scal_old) break;
      if (below_alamin<NV>(ls, alam, desc, old)) {
#pragma unroll
        for (int i = 0; i < NV; i++) rel[i] = old[i];
        scal = scal_old;
        restored = true;  // rt belongs to the rejected trial point
        break;
      }
      const double half = 0.5 * alam;
      alam = (tr == 0)
                 ? fmax(-fdiv(ls.slope, 2.0 * (scal - scal_old - ls.slope)), half)
                 : half;
    }
#pragma unroll
    for (int i = 0; i < NV; i++) qj[i] = rel[i] * org[i];
    fresh = !restored;
    if (max_abs<NV>(rt) < TOLF || step_below_tolx<NV>(rel, old)) {
      out.conv = 1;
      break;
    }
  }
  out.iters = it > 100 ? 100 : it;
  return out;
}

// solve_rk_step on four lanes (4i .. 4i+3, the same cell and operands on
// each).  Each evaluation runs the real chain on every lane and the two
// complex-step Jacobian columns on lanes 0 and 1 of the quad, so residual and
// Jacobian of a point come from one round: at the start, at the full first
// step and at the line search's first trial (alam = 1), where lane 3
// evaluates the trial 0.5 that usually follows a rejection.  The operands are
// the plain solver's, so the same bits.  Every value the control flow depends
// on is taken from one lane of the quad, so the four lanes stay together.
template <int NS>
__device__ __forceinline__ double quad_from(double v, int role) {
  const int src = (threadIdx.x & 60) | role;
  int lo = __double2loint(v), hi = __double2hiint(v);
  lo = __shfl(lo, src, 64);
  hi = __shfl(hi, src, 64);
  return __hiloint2double(hi, lo);
}

// One quad round: this lane's implicit terms nh1, nh2 at its own point q,
// and J1/J2 (columns 1, 2) at the point of lanes 0 and 1
template <int NS>
__device__ __forceinline__ void quad_round(const DevParams& P, const double* q, const double* org,
                                           double Bx, double By, double* J1, double* J2,
                                           double& nh1, double& nh2) {
  const int role = threadIdx.x & 3;
  ImplPt b;
  implicit_real<NS>(P, q, Bx, By, b);
  nh1 = b.n1;
  nh2 = b.n2;
  const double d1 = (role == 0) ? P.h_cs * org[1] : 0.0;
  const double d2 = (role == 1) ? P.h_cs * org[2] : 0.0;
  double a, c;
  const bool ok = implicit_col<1>(P, b, q[1], q[2], d1, d2, Bx, By, a, c);
  if (!ok && role < 2) implicit_col_c<NS>(P, q, d1, d2, Bx, By, a, c);
  a = a * P.one_by_h;
  c = c * P.one_by_h;
  J1[0] = quad_from<NS>(a, 0);
  J1[1] = quad_from<NS>(c, 0);
  J2[0] = quad_from<NS>(a, 1);
  J2[1] = quad_from<NS>(c, 1);
}

template <int NS>
__device__ __forceinline__ NewtonOut solve_rk_step_quad(const DevParams& P, double* qj,
                                                       const double* qold, const double* Rj,
                                                       double a_diag, double dt, double Bx,
                                                       double By) {
  constexpr int NV = 4 + NS;
  const double TOLF = 1.0e-10;
  const int role = threadIdx.x & 3;
  double org[NV], rel[NV], rt[NV], old[NV], desc[NV];
  double scal = 0.0;
  (void)newton_scale<NV>(qj, org, rel);
  NewtonOut out{0, 0, 0};
  int it;
  bool fresh = false;  // rt and scal belong to qj, J1/J2 too
  double J1[2] = {0.0, 0.0}, J2[2] = {0.0, 0.0};
  for (it = 1; it <= 100; it++) {
    if (!fresh) {
      // the residual at qj (lane 2), the Jacobian at rel * org, which in the
      // first iteration may be a rounding off qj (lanes 0, 1)
      double q[NV], h1, h2;
#pragma unroll
      for (int m = 0; m < NV; m++) q[m] = (role < 2) ? rel[m] * org[m] : qj[m];
      quad_round<NS>(P, q, org, Bx, By, J1, J2, h1, h2);
      finish_f<NS>(qj, qold, Rj, a_diag, dt, quad_from<NS>(h1, 2), quad_from<NS>(h2, 2), rt, scal);
    }
    bool restored = false;
    if (max_abs<NV>(rt) < TOLF) {
      out.conv = 1;
      break;
    }
    double L[4];
    newton_step<NS>(org, rt, dt * a_diag, J1, J2, L, desc, it == 1);
#pragma unroll
    for (int i = 0; i < NV; i++) old[i] = rel[i];
    LineSearch ls{};
    if (it > 1) ls = ls_begin<NS>(org, old, rt, L, desc);
    const double scal_old = scal;
    if (!ls.none) {
      double n1a, n2a;  // this lane's implicit terms
      // trial `alam` from the implicit terms of lane `src`; returns true
      // when the search ends with it (accepted, or below alamin)
      bool acc = false;
      auto take = [&](double alam, int src) -> bool {
        const double h1 = quad_from<NS>(n1a, src), h2 = quad_from<NS>(n2a, src);
#pragma unroll
        for (int i = 0; i < NV; i++) rel[i] = old[i] + alam * desc[i];
#pragma unroll
        for (int i = 0; i < NV; i++) qj[i] = rel[i] * org[i];
        finish_f<NS>(qj, qold, Rj, a_diag, dt, h1, h2, rt, scal);
        if (it == 1) {
          acc = true;
          return true;
        }
        out.ls_evals++;
        acc = scal <= 0.9 * scal_old;
        if (acc) return true;
        if (below_alamin<NV>(ls, alam, desc, old)) {
#pragma unroll
          for (int i = 0; i < NV; i++) rel[i] = old[i];
          scal = scal_old;
          restored = true;
          return true;
        }
        return false;
      };
      {
        double q[NV];
        const double al = (role == 3 && it > 1) ? 0.5 : 1.0;
#pragma unroll
        for (int m = 0; m < NV; m++) q[m] = (old[m] + al * desc[m]) * org[m];
        quad_round<NS>(P, q, org, Bx, By, J1, J2, n1a, n2a);
      }
      bool end = take(1.0, 2);
      fresh = end && acc;
      if (!end) {
        // max(quadratic model, 0.5), then halvings (see solve_rk_step), four
        // at a time: lane r evaluates alam * 0.5^r, and the trials are taken
        // in order with the serial rules
        double alam = fmax(-fdiv(ls.slope, 2.0 * (scal - scal_old - ls.slope)), 0.5);
        int trials = 1;
        if (alam == 0.5) {
          end = take(0.5, 3);
          alam = 0.25;
          trials++;
        }
        while (!end && trials < 256) {
          double al = alam;
#pragma unroll
          for (int r = 0; r < 3; r++)
            if (role > r) al = al * 0.5;
          double q[NV];
#pragma unroll
          for (int m = 0; m < NV; m++) q[m] = (old[m] + al * desc[m]) * org[m];
          ImplPt b;
          implicit_real<NS>(P, q, Bx, By, b);
          n1a = b.n1;
          n2a = b.n2;
          for (int r = 0; r < 4 && !end && trials < 256; r++) {
            end = take(alam, r);
            alam = alam * 0.5;
            trials++;
          }
        }
      }
    } else {
      fresh = false;
    }
#pragma unroll
    for (int i = 0; i < NV; i++) qj[i] = rel[i] * org[i];
    // an accepted shorter trial has its residual but not its Jacobian: the
    // round at the top of the next iteration gives both (the same residual)
    if (restored) fresh = false;
    if (max_abs<NV>(rt) < TOLF || step_below_tolx<NV>(rel, old)) {
      out.conv = 1;
      break;
    }
  }
  out.iters = it > 100 ? 100 : it;
  return out;
}

// Raw warm-start features of one cell entering Newton: log h, the
// predictor's velocity (u, v), T, three solid volume fractions, log dt and
// the bed slope magnitude.
template <int NS>
__device__ __forceinline__ void mlp_features_raw(const DevParams& P, const double* q_fv,
                                                 const double* qp, const double* q_si,
                                                 double dt, double Bx, double By, float* f) {
  const double h = qp[0];
  f[0] = (float)log(h);
  f[1] = (float)(q_si[1] / q_fv[0]);
  f[2] = (float)(q_si[2] / q_fv[0]);
  f[3] = (float)qp[3];
#pragma unroll
  for (int s = 0; s < 3; s++)
    f[4 + s] = (s < NS) ? (float)(P.alpha ? qp[4 + s] : qp[4 + s] / h) : 0.f;
  f[7] = (float)log(dt);
  f[8] = (float)sqrt(Bx * Bx + By * By);
}

// Mixture density and reduced gravity of a state whose momenta are (mx, my),
// the real part of the chain in implicit_c (c_phys_var and mixt_var,
// src/constitutive_2d.f90:1145-1313, 1333-1483) for q1 > eps_sing.
template <int NS>
__device__ __forceinline__ void rho_rg_of(const DevParams& P, const double* q, double mx,
                                          double my, double& rho_m, double& rg) {
  const double inv_q1 = 1.0 / q[0];
  double xs_tot = 0.0, dsh = 0.0, dinv = 0.0;
#pragma unroll
  for (int i = 0; i < NS; i++) {
    const double xs = q[4 + i] * inv_q1;
    xs_tot += xs;
    dsh += xs * P.sp_heat_s[i];
    dinv += xs * P.inv_rho_s[i];
  }
  const double xc = 1.0 - xs_tot;
  const double shm = dsh + xc * P.sp_heat_a;
  double T = P.energy ? (q[3] - 0.5 * (mx * mx + my * my) * inv_q1) / (q[0] * shm)
                      : q[3] / (q[0] * shm);
  if (T <= 0.0) T = P.T_ambient;
  rho_m = 1.0 / (dinv + xc * (P.sp_gas_const_a * T * P.inv_pres));
  rg = (rho_m - P.rho_a_amb) / rho_m * P.grav;
}

// A starting point for the implicit Voellmy solve (no reference
// counterpart: the reference starts Newton at q_si, src/solver_2d.f90:1196).
// The momenta solve m = m_si + dt a NH(m) with NH = -(rho_m g'/xi) |U| u,
// u = m/q1 and |U| = |u| sqrt(1 + (u.grad B)^2/|u|^2) with slope correction.
// m is parallel to m_si, so with the mixture density frozen the speed s =
// |m| solves s + C c s^2 = |m_si| with C = dt a rho_m g'/(xi q1^2), c the
// slope factor: s = 2|m_si| / (1 + sqrt(1 + 4 C c |m_si|)).  The density
// depends on s only through the kinetic energy in the temperature, weakly,
// so three refreshes of rho_m, g' at the current s make the root exact to
// rounding.  Returns false where it does not apply (no Voellmy term, thin
// or lighter-than-air cells, no momentum); Newton then starts at q_si.
template <int NS>
__device__ __forceinline__ bool voellmy_closed_form(const DevParams& P, const double* q_si,
                                                    double a_diag, double dt, double Bx,
                                                    double By, double* m) {
  if (!P.rheo || P.rheo_model != 1 || !(q_si[0] > P.eps_sing)) return false;
  const double mx = q_si[1], my = q_si[2];
  const double ms = sqrt(mx * mx + my * my);
  if (!(ms > 0.0)) return false;
  const double ex = mx / ms, ey = my / ms;
  const double wn = P.slope ? ex * Bx + ey * By : 0.0;
  const double c = sqrt(1.0 + wn * wn);
  const double k0 = dt * a_diag / (P.xi * q_si[0] * q_si[0]) * c;
  double s = ms;
#pragma unroll
  for (int it = 0; it < 4; it++) {
    double rho_m, rg;
    rho_rg_of<NS>(P, q_si, s * ex, s * ey, rho_m, rg);
    const double C = k0 * rho_m * rg;
    if (!(C > 0.0)) return false;
    s = 2.0 * ms / (1.0 + sqrt(1.0 + 4.0 * C * ms));
  }
  m[0] = s * ex;
  m[1] = s * ey;
  return isfinite(m[0]) && isfinite(m[1]);
}

// The stage-2 predictor (src/solver_2d.f90:1132-1196): q_fv = q0 - dt*D, its
// physical variables, and the semi-implicit Coulomb step q_si realigned with
// q_fv.  Returns false when q_fv has no mass (no Newton solve).
template <int NS>
__device__ __forceinline__ bool predictor(const DevParams& P, const double* q0,
                                          const double* D, double dt, double Bx,
                                          double By, double Bxx, double Bxy, double Byy,
                                          double gc, double* q_fv, double* qp,
                                          double* q_si) {
  constexpr int NV = 4 + NS;
#pragma unroll
  for (int i = 0; i < NV; i++) q_fv[i] = q0[i] - dt * (D[i] - 0.0);
  phys<NS>(P, q_fv, qp);
  if (!(q_fv[0] > 0.0)) return false;
  double s1, s2;
  semi_impl<NS>(P, Bx, By, Bxx, Bxy, Byy, gc, qp, s1, s2);
#pragma unroll
  for (int i = 0; i < NV; i++) {
    double si = (i == 1) ? s1 : (i == 2) ? s2 : 0.0;
    q_si[i] = q_fv[i] + dt * 1.0 * si;
  }
  const double f2 = q_fv[1], f3 = q_fv[2];
  if ((f2 * f2 + f3 * f3) == 0.0) {
    q_si[1] = 0.0;
    q_si[2] = 0.0;
  } else if ((q_si[1] * f2 < 0.0) || (q_si[2] * f3 < 0.0)) {
    q_si[1] = 0.0;
    q_si[2] = 0.0;
  } else {
    double m = fsqrt(q_si[1] * q_si[1] + q_si[2] * q_si[2]);
    const Rcp den = rcp_of(fsqrt(f2 * f2 + f3 * f3));
    q_si[1] = div_by(m * f2, den);
    q_si[2] = div_by(m * f3, den);
  }
  return true;
}

// Stage 2 of the N_RK = 2 IMEX scheme for one cell (src/solver_2d.f90:
// 1105-1280), from q0 = q^n and D = divFlux - expl_terms of stage 1.  The
// implicit term refresh of :1234-1236 is not evaluated: for the stiffly
// accurate N_RK = 2 tableau it is overwritten at :1271-1277 and never enters
// q.  Returns the Newton iteration count (0: no Newton).
// LANES: lanes per cell, 1 or 4 (the quad solver)
template <int NS, int LANES = 1>
__device__ __forceinline__ int stage2(const DevParams& P, const double* q0,
                                      const double* D, double dt, double Bx,
                                      double By, double Bxx, double Bxy,
                                      double Byy, double gc, double* q,
                                      int& nonconv, int& ls_evals,
                                      const double* warm = nullptr, int* warm_used = nullptr,
                                      float* harvest = nullptr, bool* harvested = nullptr,
                                      bool closed = false) {
  constexpr int NV = 4 + NS;
  double q_fv[NV], qp[NV + 2], q_si[NV];
  nonconv = 0;
  ls_evals = 0;
  if (!predictor<NS>(P, q0, D, dt, Bx, By, Bxx, Bxy, Byy, gc, q_fv, qp, q_si)) {
#pragma unroll
    for (int i = 0; i < NV; i++) q[i] = q_fv[i];
    return 0;
  }
  double Rj[NV];
  const Rcp rdt = rcp_of(dt * 1.0);
#pragma unroll
  for (int i = 0; i < NV; i++) {
    // (only the momenta differ from q_fv)
    const double si = (i == 1 || i == 2) ? div_by(q_si[i] - q_fv[i], rdt) : 0.0;
    Rj[i] = (D[i] - 0.0) - 1.0 * si;
    q[i] = q_si[i];
  }
  NewtonOut no;
  double mg[2];
  bool have = false;
  if (closed) {
    have = voellmy_closed_form<NS>(P, q_si, 1.0, dt, Bx, By, mg);
  } else if (warm && warm[0] == warm[0] && warm[1] == warm[1]) {
    mg[0] = warm[0];
    mg[1] = warm[1];
    have = true;
  }
  if (have) {
    // a starting point for the momenta (learned, or the closed form): Newton
    // starts from it when it already meets the tolerance or has the smaller
    // residual of it and the plain predictor (the plain one stays the
    // fallback), and the equation solved is the same
    double qw[NV], rtw[NV], sw;
#pragma unroll
    for (int i = 0; i < NV; i++) qw[i] = q_si[i];
    qw[1] = mg[0];
    qw[2] = mg[1];
    eval_f<NS>(P, qw, q0, Rj, 1.0, dt, Bx, By, rtw, sw);
    bool use = max_abs<NV>(rtw) < 1.0e-10;
    if (!use) {
      double rtp[NV], sp;
      eval_f<NS>(P, q, q0, Rj, 1.0, dt, Bx, By, rtp, sp);
      use = sw < sp;
    }
    *warm_used = use ? 1 : 0;
    q[1] = use ? qw[1] : q[1];
    q[2] = use ? qw[2] : q[2];
  } else if (warm_used) {
    *warm_used = (closed || warm) ? 0 : -1;
  }
  no = (LANES == 4) ? solve_rk_step_quad<NS>(P, q, q0, Rj, 1.0, dt, Bx, By)
                    : solve_rk_step<NS>(P, q, q0, Rj, 1.0, dt, Bx, By);
  nonconv = !no.conv;
  ls_evals = no.ls_evals;
  if (harvest && no.conv) {
    // (state entering Newton, converged momenta) pair for the warm start;
    // a momentum component below 1e-6 of the predictor's magnitude gets a
    // zero target, and pairs with non-finite values are not recorded
    float f[9];
    mlp_features_raw<NS>(P, q_fv, qp, q_si, dt, Bx, By, f);
    const double mag = sqrt(q_si[1] * q_si[1] + q_si[2] * q_si[2]);
    bool ok = mag > 0.0;
#pragma unroll
    for (int i = 0; i < 9; i++) {
      harvest[i] = f[i];
      ok = ok && isfinite(f[i]);
    }
    harvest[9] = (fabs(q_si[1]) > 1e-6 * mag) ? (float)(q[1] / q_si[1] - 1.0) : 0.f;
    harvest[10] = (fabs(q_si[2]) > 1e-6 * mag) ? (float)(q[2] / q_si[2] - 1.0) : 0.f;
    ok = ok && isfinite(harvest[9]) && isfinite(harvest[10]);
    *harvested = ok;
  }
  if (P.ny == 1) q[2] = 0.0;
  if (P.nx == 1) q[1] = 0.0;
  if (q_si[1] * q_si[1] + q_si[2] * q_si[2] == 0.0) {
    q[1] = 0.0;
    q[2] = 0.0;
  } else if ((q[1] * q_si[1] <= 0.0) && (q[2] * q_si[2] <= 0.0)) {
    q[1] = 0.0;
    q[2] = 0.0;
  } else {
    double m = fsqrt(q[1] * q[1] + q[2] * q[2]);
    const Rcp den = rcp_of(fsqrt(q_si[1] * q_si[1] + q_si[2] * q_si[2]));
    q[1] = div_by(m * q_si[1], den);
    q[2] = div_by(m * q_si[2], den);
  }
  return no.iters;
}

// eval_mass_exchange_terms, supported branches (src/constitutive_2d.f90:
// 4424-5003).  Returns false when every term is zero.
// LANES > 1: the cell runs on LANES lanes (the same operands on each); the
// solid classes' settling velocities are split between them (class
// LANES*s + r on lane r, the same instructions on every lane) and
// exchanged, so the cell waits for about 1/LANES of them.
template <int NS, int LANES = 1, bool VP = false>
__device__ __forceinline__ void mass_exchange(const DevParams& P, const double* qp,
                                              double Bx, double By,
                                              const double* erodible, double dt,
                                              double* er, double* dep, double* eq,
                                              double& topo) {
  constexpr int NV = 4 + NS;
#pragma unroll
  for (int i = 0; i < NS; i++) {
    er[i] = 0.0;
    dep[i] = 0.0;
  }
#pragma unroll
  for (int i = 0; i < NV; i++) eq[i] = 0.0;
  topo = 0.0;
  if (qp[0] <= kEps) return;
  const double alpha_max = 0.6, hind_exp = 4.65;
  double r_h = qp[0], r_u = qp[NV], r_v = qp[NV + 1];
  double al[NS > 0 ? NS : 1], at = 0.0;
  const Rcp rh = rcp_of(qp[0]), rdt = rcp_of(dt);
#pragma unroll
  for (int i = 0; i < NS; i++) al[i] = P.alpha ? qp[4 + i] : div_by(qp[4 + i], rh);
#pragma unroll
  for (int i = 0; i < NS; i++) at += al[i];
  double r_w = P.slope ? r_u * Bx + r_v * By : 0.0;
  double mv2 = r_u * r_u + r_v * r_v + r_w * r_w;
  double mv = fsqrt(mv2);
  if (P.erosion_coeff > 0.0) {
    double te = P.erosion_coeff * mv * r_h * (1.0 - at);
    double tse = te * (1.0 - P.erodible_porosity);
#pragma unroll
    for (int i = 0; i < NS; i++) er[i] = P.erodible_fract[i] * tse;
  }
#pragma unroll
  for (int i = 0; i < NS; i++) er[i] = fmax(0.0, fmin(er[i], div_by(erodible[i], rdt)));
  double tse = 0.0;
#pragma unroll
  for (int i = 0; i < NS; i++) tse += er[i];
  double te = fdiv(tse, 1.0 - P.erodible_porosity);
  double cont_erosion = te * P.erodible_porosity;
  if (at <= P.alphastot_min) return;
  double r_T = qp[3];
  Mixt m = mixt<NS, true>(P, qp);
  double inv_kin_visc = fdiv(1.0, P.kin_visc_c);
  // bottom over mean concentration with the profiles (:4676-4683)
  double dcf[NS > 0 ? NS : 1];
#pragma unroll
  for (int i = 0; i < NS; i++) dcf[i] = 1.0;
  double svp[NS > 0 ? NS : 1];
  if (VP && P.bottom_conc) vp_dep_coeffs<NS>(P, r_h, mv, m.rho_c, dcf, svp);
  if (P.settling) {
    // hindered settling factor, the same for every class
    const double hind = det_pow(1.0 - fmin(1.0, fdiv(at, alpha_max)), hind_exp);
    double svs[NS > 0 ? NS : 1];
    if (LANES > 1) {
      constexpr int NSL = (NS + LANES - 1) / LANES;
      const int p = threadIdx.x & (LANES - 1);
      double mine[NSL > 0 ? NSL : 1];
#pragma unroll
      for (int sl = 0; sl < NSL; sl++) {
        double a = 0.0, diam = 0.0, rhos = 0.0;
        bool has = false;
#pragma unroll
        for (int r = 0; r < LANES; r++) {
          const int c = sl * LANES + r;
          if (c < NS && p == r) {
            a = al[c];
            diam = P.diam_s[c];
            rhos = P.rho_s[c];
            has = true;
          }
        }
        mine[sl] = (has && a > 0.0) ? settling_velocity(P, diam, rhos, m.rho_c, inv_kin_visc)
                                    : 0.0;
      }
#pragma unroll
      for (int i = 0; i < NS; i++) {
        const int src = (threadIdx.x & (64 - LANES)) | (i % LANES);
        int lo = __double2loint(mine[i / LANES]), hi = __double2hiint(mine[i / LANES]);
        lo = __shfl(lo, src, 64);
        hi = __shfl(hi, src, 64);
        svs[i] = __hiloint2double(hi, lo);
      }
    }
#pragma unroll
    for (int i = 0; i < NS; i++) {
      if (al[i] > 0.0) {
        const double sv = (LANES > 1) ? svs[i]
                          : (VP && P.bottom_conc)
                              ? svp[i]
                              : settling_velocity(P, P.diam_s[i], P.rho_s[i], m.rho_c,
                                                  inv_kin_visc);
        double d = al[i] * sv * dcf[i];
        d = d * hind;
        dep[i] = fmin(d, div_by(r_h * al[i], rdt));
      }
    }
  }
  double sdep = 0.0;
#pragma unroll
  for (int i = 0; i < NS; i++) sdep += dep[i];
  double cl = 0.0 + P.coeff_porosity * sdep;
  double sal = 0.0;
#pragma unroll
  for (int i = 0; i < NS; i++) sal += al[i];
  cl = fmin(cl, div_by(r_h * fmax(0.0, P.max_packing - sal), rdt));
  cl = fmin(cl, div_by(r_h * (1.0 - sal) - P.coeff_porosity * (r_h * sal - dt * sdep), rdt));
  double T_erodible = P.erod_dep ? r_T : P.T_erodible;
  double air = 0.0;
  if (P.entrain && (r_h > 0.0) && (m.ri > 0.0)) {
    double ec = fdiv(0.075, fsqrt(1.0 + 718.0 * det_pow(m.ri, 2.4)));
    air = ec * fsqrt(mv2);
  }
  double dep_tot = 0.0, ers_tot = 0.0, rdep = 0.0, rers = 0.0, sdc = 0.0, sec = 0.0;
#pragma unroll
  for (int i = 0; i < NS; i++) dep_tot += dep[i];
#pragma unroll
  for (int i = 0; i < NS; i++) ers_tot += er[i];
#pragma unroll
  for (int i = 0; i < NS; i++) rdep += P.rho_s[i] * dep[i];
#pragma unroll
  for (int i = 0; i < NS; i++) rers += P.rho_s[i] * er[i];
  eq[0] = P.rho_a_amb * air + rers - rdep + P.rho_c_sub * cont_erosion - m.rho_c * cl;
  eq[1] = -(r_u * (rdep + m.rho_c * cl));
  eq[2] = -(r_v * (rdep + m.rho_c * cl));
#pragma unroll
  for (int i = 0; i < NS; i++) sdc += P.rho_s[i] * P.sp_heat_s[i] * dep[i];
#pragma unroll
  for (int i = 0; i < NS; i++) sec += P.rho_s[i] * P.sp_heat_s[i] * er[i];
  if (P.energy)
    eq[3] = -(r_T * (sdc + m.rho_c * m.shc * cl)) - 0.5 * mv2 * (rdep + m.rho_c * cl) +
            T_erodible * (sec + P.rho_c_sub * m.shc * cont_erosion) +
            P.T_ambient * P.sp_heat_a * P.rho_a_amb * air;
  else
    eq[3] = -(r_T * (sdc + m.rho_c * m.shc * cl)) +
            T_erodible * (sec + P.rho_c_sub * m.shc * cont_erosion) +
            P.T_ambient * P.sp_heat_a * P.rho_a_amb * air;
#pragma unroll
  for (int i = 0; i < NS; i++) eq[4 + i] = P.rho_s[i] * (er[i] - dep[i]);
  topo = fdiv(dep_tot - ers_tot, 1.0 - P.erodible_porosity);
}

}  // namespace imexsw
