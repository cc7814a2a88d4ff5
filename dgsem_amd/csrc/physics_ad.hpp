// Tangent (JVP) and adjoint (VJP) of the pointwise physics in physics.hpp
// and parabolic_impl.hpp, derived by hand from the implemented formulas.
//
// Every nonlinear map y = F(x) here has a pair of functions:
//   *_jvp: dy = F'(x) dx
//   *_vjp: xbar += F'(x)^T ybar   (accumulates)
// built from the same partial derivatives, so <ybar, F' dx> = <F'^T ybar, dx>
// holds to rounding.  Branches (the series / logarithm forms of the
// logarithmic mean, the max in the LLF wave speed) follow the forward
// evaluation's choice at x: these are the derivatives of the function the
// forward kernels compute, i.e. a discrete tangent and adjoint.  Where the
// LLF wave speed's max() ties exactly, the flux has no derivative and the
// two sides share it (the mean of the one-sided derivatives).
//
// The blending factor of shock capturing is not differentiated (it is frozen
// at its forward value by the callers).
#pragma once

#include "physics.hpp"

namespace dgsem {

// Node primitives used by the two-point flux: q = (rho, v[DIM], beta, kin),
// beta = rho / (2 p), kin = |v|^2 / 2, p = (gamma - 1)(E - rho kin).
template <int DIM>
struct PrimTangent {
  double rho, v[DIM], beta, kin;
};

template <int DIM>
DG_HD void prims_jvp(double gamma, const double* u, const NodePrims<DIM>& q, const double* du,
                     PrimTangent<DIM>& dq) {
  const double ir = recip(q.rho);
  dq.rho = du[0];
  double dkin = 0.0;
  for (int k = 0; k < DIM; ++k) {
    dq.v[k] = (du[k + 1] - q.v[k] * du[0]) * ir;
    dkin += q.v[k] * dq.v[k];
  }
  dq.kin = dkin;
  const double dp = (gamma - 1.0) * (du[DIM + 1] - q.kin * du[0] - q.rho * dkin);
  dq.beta = q.beta * (du[0] * ir - dp * recip(q.p));
  (void)u;
}

// ubar += (dq/du)^T qbar; pbar is an extra cotangent of the pressure.
template <int DIM>
DG_HD void prims_vjp(double gamma, const NodePrims<DIM>& q, const PrimTangent<DIM>& qbar,
                     double pbar, double* ubar) {
  const double ir = recip(q.rho);
  double rb = qbar.rho + qbar.beta * q.beta * ir;
  double pb = pbar - qbar.beta * q.beta * recip(q.p);
  double vb[DIM];
  for (int k = 0; k < DIM; ++k) vb[k] = qbar.v[k] + qbar.kin * q.v[k];
  // p = (gamma - 1) (E - rho kin(v)), with v held as an independent variable
  ubar[DIM + 1] += (gamma - 1.0) * pb;
  rb -= (gamma - 1.0) * q.kin * pb;
  for (int k = 0; k < DIM; ++k) vb[k] -= (gamma - 1.0) * q.rho * q.v[k] * pb;
  // v = m / rho
  for (int k = 0; k < DIM; ++k) {
    ubar[k + 1] += vb[k] * ir;
    rb -= vb[k] * q.v[k] * ir;
  }
  ubar[0] += rb;
}

// Q = artanh(xi) / xi of a pair (physics.hpp) and dQ/df2, f2 = xi^2: the series
// and its derivative term by term, or the identity dQ/df2 = (1 / (1 - f2) - Q) /
// (2 f2) with 1 - f2 = 4 x y / (x + y)^2.
DG_HD void artanh_ratio_jet(double x, double y, double f2, double& Q, double& dQ) {
  Q = artanh_ratio(x, y, f2);
  if (f2 < kSeriesMax) {
    double d = 10.0 / 21.0;
    d = 9.0 / 19.0 + f2 * d;
    d = 8.0 / 17.0 + f2 * d;
    d = 7.0 / 15.0 + f2 * d;
    d = 6.0 / 13.0 + f2 * d;
    d = 5.0 / 11.0 + f2 * d;
    d = 4.0 / 9.0 + f2 * d;
    d = 3.0 / 7.0 + f2 * d;
    d = 2.0 / 5.0 + f2 * d;
    dQ = 1.0 / 3.0 + f2 * d;
  } else {
    const double s = x + y;
    dQ = (s * s * recip(4.0 * x * y) - Q) * recip(2.0 * f2);
  }
}

// Means of the Chandrashekar flux and their partial derivatives with
// respect to (rho_a, rho_b) and (beta_a, beta_b): rho_mean, its inverse
// beta mean B, one over the logarithmic mean of beta, and p_mean = (rho_a + rho_b) /
// (2 (beta_a + beta_b)), as flux_chandrashekar forms them, with its branches.
// rho_mean = s / 2 P and B = 2 Q / s; xi_x = 2 y / s^2, xi_y = -2 x / s^2.  With
// both branches and IEEE quotients evaluated for every pair (selected without a
// branch) the derivative kernels spent four times the FP64 instructions; their
// callers pin the sums after each pair, so the branch costs no registers.
struct ChandrashekarMeans {
  double rho, rho_a, rho_b;  // rho_mean and partials
  double B, B_a, B_b;        // inverse beta mean and partials
  double p, p_rho, p_beta;   // p_mean, d/d(rho_a or rho_b), d/d(beta_a or beta_b)
};

template <int DIM>
DG_HD ChandrashekarMeans chandrashekar_means(const NodePrims<DIM>& a, const NodePrims<DIM>& b) {
  const double sr = a.rho + b.rho, sb = a.beta + b.beta;
  const double r = recip(sr * sb);
  const double isr = r * sb, isb = r * sr;
  const double xr = (a.rho - b.rho) * isr, xb = (a.beta - b.beta) * isb;
  const double fr = xr * xr, fb = xb * xb;
  double P, dP, Q, dQ;  // functions of f2 and their derivatives
  if (fr < 1.0e-4 && fb < 1.0e-4) {
    P = 1.0 - fr * (1.0 / 3.0 + fr * (4.0 / 45.0 + fr * (44.0 / 945.0)));
    dP = -(1.0 / 3.0 + fr * (8.0 / 45.0 + fr * (44.0 / 315.0 + fr * (1712.0 / 14175.0))));
    Q = 1.0 + fb * (1.0 / 3.0 + fb * (1.0 / 5.0 + fb * (1.0 / 7.0)));
    dQ = 1.0 / 3.0 + fb * (2.0 / 5.0 + fb * (3.0 / 7.0 + fb * (4.0 / 9.0)));
  } else {
    artanh_ratio_jet(a.rho, b.rho, fr, P, dP);
    P = recip(P);
    dP = -dP * P * P;
    artanh_ratio_jet(a.beta, b.beta, fb, Q, dQ);
  }
  ChandrashekarMeans m;
  m.rho = 0.5 * sr * P;
  const double t = 2.0 * xr * isr * dP;
  m.rho_a = 0.5 * P + t * b.rho;
  m.rho_b = 0.5 * P - t * a.rho;
  m.B = 2.0 * isb * Q;
  const double c = 2.0 * isb * isb, w = 4.0 * xb * isb * dQ;
  m.B_a = c * (w * b.beta - Q);
  m.B_b = -c * (w * a.beta + Q);
  m.p = 0.5 * sr * isb;
  m.p_rho = 0.5 * isb;
  m.p_beta = -m.p * isb;
  return m;
}

// Tangent of the Chandrashekar flux with respect to both nodes' primitives
// (the normal n is geometry, not differentiated), in flux_chandrashekar's form:
// f = (2 h, h vs + p n, h (B / (gamma - 1) + v_a . v_b) + p vn / 2) with vs =
// v_a + v_b, vn = vs . n and h = rho_mean vn / 4.
template <int DIM>
DG_HD void chandrashekar_jvp(double inv_gm1, const NodePrims<DIM>& a, const NodePrims<DIM>& b,
                             const PrimTangent<DIM>& da, const PrimTangent<DIM>& db,
                             const double* n, double* df) {
  const ChandrashekarMeans m = chandrashekar_means<DIM>(a, b);
  double vs[DIM], dvs[DIM], vn = 0.0, dvn = 0.0, dot = 0.0, ddot = 0.0;
  for (int k = 0; k < DIM; ++k) {
    vs[k] = a.v[k] + b.v[k];
    dvs[k] = da.v[k] + db.v[k];
    vn += vs[k] * n[k];
    dvn += dvs[k] * n[k];
    dot += a.v[k] * b.v[k];
    ddot += da.v[k] * b.v[k] + a.v[k] * db.v[k];
  }
  const double drm = m.rho_a * da.rho + m.rho_b * db.rho;
  const double dB = m.B_a * da.beta + m.B_b * db.beta;
  const double dp = m.p_rho * (da.rho + db.rho) + m.p_beta * (da.beta + db.beta);
  const double h = 0.25 * m.rho * vn;
  const double dh = 0.25 * (drm * vn + m.rho * dvn);
  df[0] = 2.0 * dh;
  for (int k = 0; k < DIM; ++k) df[k + 1] = dh * vs[k] + h * dvs[k] + dp * n[k];
  df[DIM + 1] = dh * (inv_gm1 * m.B + dot) + h * (inv_gm1 * dB + ddot) + 0.5 * (dp * vn + m.p * dvn);
}

// abar += (df/dq_a)^T g, bbar += (df/dq_b)^T g (kin, which the flux does not
// take, untouched).
template <int DIM>
DG_HD void chandrashekar_vjp(double inv_gm1, const NodePrims<DIM>& a, const NodePrims<DIM>& b,
                             const double* n, const double* g, PrimTangent<DIM>& abar,
                             PrimTangent<DIM>& bbar) {
  const ChandrashekarMeans m = chandrashekar_means<DIM>(a, b);
  const double gE = g[DIM + 1];
  double vs[DIM], vn = 0.0, dot = 0.0, hb = 2.0 * g[0], pb = 0.0;
  for (int k = 0; k < DIM; ++k) {
    vs[k] = a.v[k] + b.v[k];
    vn += vs[k] * n[k];
    dot += a.v[k] * b.v[k];
    hb += g[k + 1] * vs[k];
    pb += g[k + 1] * n[k];
  }
  const double h = 0.25 * m.rho * vn;
  hb += gE * (inv_gm1 * m.B + dot);
  pb += 0.5 * gE * vn;
  const double vnb = 0.25 * m.rho * hb + 0.5 * gE * m.p, dotb = gE * h;
  for (int k = 0; k < DIM; ++k) {
    const double vsb = h * g[k + 1] + vnb * n[k];
    abar.v[k] += vsb + dotb * b.v[k];
    bbar.v[k] += vsb + dotb * a.v[k];
  }
  const double rmb = 0.25 * vn * hb, Bb = dotb * inv_gm1;
  abar.rho += m.rho_a * rmb + m.p_rho * pb;
  bbar.rho += m.rho_b * rmb + m.p_rho * pb;
  abar.beta += m.B_a * Bb + m.p_beta * pb;
  bbar.beta += m.B_b * Bb + m.p_beta * pb;
}

// ---------------------------------------------------------------------
// Physical flux F(u).n and the LLF flux, in terms of u with the node
// primitives q (rho, v, p, c) of u.
// ---------------------------------------------------------------------

// Tangent of (v, p) of a state: dv_k = (dm_k - v_k drho) / rho,
// dp = (gamma - 1)(dE - v.dm + kin drho).
template <int DIM>
DG_HD void vp_jvp(double gamma, const NodePrims<DIM>& q, const double* du, double* dv, double& dp) {
  const double ir = recip(q.rho);
  double vdm = 0.0;
  for (int k = 0; k < DIM; ++k) {
    dv[k] = (du[k + 1] - q.v[k] * du[0]) * ir;
    vdm += q.v[k] * du[k + 1];
  }
  dp = (gamma - 1.0) * (du[DIM + 1] - vdm + q.kin * du[0]);
}

// ubar += (d(v, p)/du)^T (vbar, pbar).
template <int DIM>
DG_HD void vp_vjp(double gamma, const NodePrims<DIM>& q, const double* vbar, double pbar,
                  double* ubar) {
  const double ir = recip(q.rho);
  double rb = (gamma - 1.0) * q.kin * pbar;
  for (int k = 0; k < DIM; ++k) {
    ubar[k + 1] += vbar[k] * ir - (gamma - 1.0) * q.v[k] * pbar;
    rb -= vbar[k] * q.v[k] * ir;
  }
  ubar[0] += rb;
  ubar[DIM + 1] += (gamma - 1.0) * pbar;
}

// d(F(u).n) for F0 = rho vn, F_k = m_k vn + p n_k, F_E = (E + p) vn.
template <int DIM>
DG_HD void flux_n_jvp(double gamma, const double* u, const NodePrims<DIM>& q, const double* du,
                      const double* n, double* dF) {
  double dv[DIM], dp, vn = 0.0, dvn = 0.0;
  vp_jvp<DIM>(gamma, q, du, dv, dp);
  for (int k = 0; k < DIM; ++k) {
    vn += q.v[k] * n[k];
    dvn += dv[k] * n[k];
  }
  dF[0] = du[0] * vn + u[0] * dvn;
  for (int k = 0; k < DIM; ++k) dF[k + 1] = du[k + 1] * vn + u[k + 1] * dvn + dp * n[k];
  dF[DIM + 1] = (du[DIM + 1] + dp) * vn + (u[DIM + 1] + q.p) * dvn;
}

// ubar += (d(F(u).n)/du)^T g
template <int DIM>
DG_HD void flux_n_vjp(double gamma, const double* u, const NodePrims<DIM>& q, const double* n,
                      const double* g, double* ubar) {
  double vn = 0.0;
  for (int k = 0; k < DIM; ++k) vn += q.v[k] * n[k];
  const double gE = g[DIM + 1];
  ubar[0] += g[0] * vn;
  double vnb = g[0] * u[0] + gE * (u[DIM + 1] + q.p);
  double pb = gE * vn;
  for (int k = 0; k < DIM; ++k) {
    ubar[k + 1] += g[k + 1] * vn;
    vnb += g[k + 1] * u[k + 1];
    pb += g[k + 1] * n[k];
  }
  ubar[DIM + 1] += gE * vn;
  double vb[DIM];
  for (int k = 0; k < DIM; ++k) vb[k] = vnb * n[k];
  vp_vjp<DIM>(gamma, q, vb, pb, ubar);
}

// Gradient of the LLF wave speed max(|vn_L|, |vn_R|) + max(c_L, c_R)|n| with
// respect to one side's state: `left` selects the side, and only the terms
// whose max that side attains (the forward's dmax choice) contribute.
template <int DIM>
DG_HD void llf_lambda_grad(double gamma, const NodePrims<DIM>& ql, const NodePrims<DIM>& qr,
                           const double* n, bool left, double* grad) {
  double vnl = 0.0, vnr = 0.0, nn = 0.0;
  for (int k = 0; k < DIM; ++k) {
    vnl += ql.v[k] * n[k];
    vnr += qr.v[k] * n[k];
    nn += n[k] * n[k];
  }
  const NodePrims<DIM>& q = left ? ql : qr;
  for (int i = 0; i < DIM + 2; ++i) grad[i] = 0.0;
  // The side a max() takes gets the whole gradient.  On an exact tie the max
  // has no derivative; each side then gets half of its own, the mean of the
  // two one-sided derivatives, which is what a central difference sees.
  // Symmetric states put ties on many faces (equal traces, or a velocity or
  // sound speed that does not vary along the face normal).
  const double avl = fabs(vnl), avr = fabs(vnr);
  const double wvn = avl == avr ? 0.5 : ((avl > avr) == left ? 1.0 : 0.0);
  const double wc = ql.c == qr.c ? 0.5 : ((ql.c > qr.c) == left ? 1.0 : 0.0);
  double vb[DIM] = {};
  double pb = 0.0;
  if (wvn != 0.0) {
    const double vn = left ? vnl : vnr;
    const double s = vn > 0.0 ? 1.0 : (vn < 0.0 ? -1.0 : 0.0);
    for (int k = 0; k < DIM; ++k) vb[k] += wvn * s * n[k];
  }
  if (wc != 0.0) {
    // c = sqrt(gamma p / rho): dc = c/2 (dp/p - drho/rho)
    const double w = wc * sqrt(nn) * 0.5 * q.c;
    pb += w * recip(q.p);
    grad[0] -= w * recip(q.rho);
  }
  vp_vjp<DIM>(gamma, q, vb, pb, grad);
}

// Tangent of the LLF flux 0.5 (F_L + F_R).n - 0.5 lambda (u_R - u_L).
template <int DIM>
DG_HD void llf_jvp(double gamma, const double* ul, const NodePrims<DIM>& ql, const double* ur,
                   const NodePrims<DIM>& qr, const double* dul, const double* dur, const double* n,
                   double* df) {
  constexpr int NV = DIM + 2;
  double dfl[NV], dfr[NV], gl[NV], gr[NV];
  flux_n_jvp<DIM>(gamma, ul, ql, dul, n, dfl);
  flux_n_jvp<DIM>(gamma, ur, qr, dur, n, dfr);
  llf_lambda_grad<DIM>(gamma, ql, qr, n, true, gl);
  llf_lambda_grad<DIM>(gamma, ql, qr, n, false, gr);
  double vnl = 0.0, vnr = 0.0, nn = 0.0;
  for (int k = 0; k < DIM; ++k) {
    vnl += ql.v[k] * n[k];
    vnr += qr.v[k] * n[k];
    nn += n[k] * n[k];
  }
  const double lam = dmax(fabs(vnl), fabs(vnr)) + dmax(ql.c, qr.c) * sqrt(nn);
  double dlam = 0.0;
  for (int i = 0; i < NV; ++i) dlam += gl[i] * dul[i] + gr[i] * dur[i];
  for (int i = 0; i < NV; ++i)
    df[i] = 0.5 * (dfl[i] + dfr[i]) - 0.5 * dlam * (ur[i] - ul[i]) - 0.5 * lam * (dur[i] - dul[i]);
}

// ubar_side += (df/du_side)^T g for one side of the LLF flux.
template <int DIM>
DG_HD void llf_vjp_side(double gamma, const double* ul, const NodePrims<DIM>& ql, const double* ur,
                        const NodePrims<DIM>& qr, const double* n, const double* g, bool left,
                        double* ubar) {
  constexpr int NV = DIM + 2;
  double vnl = 0.0, vnr = 0.0, nn = 0.0;
  for (int k = 0; k < DIM; ++k) {
    vnl += ql.v[k] * n[k];
    vnr += qr.v[k] * n[k];
    nn += n[k] * n[k];
  }
  const double lam = dmax(fabs(vnl), fabs(vnr)) + dmax(ql.c, qr.c) * sqrt(nn);
  double gh[NV], lg[NV], gdu = 0.0;
  for (int i = 0; i < NV; ++i) {
    gh[i] = 0.5 * g[i];
    gdu += g[i] * (ur[i] - ul[i]);
  }
  flux_n_vjp<DIM>(gamma, left ? ul : ur, left ? ql : qr, n, gh, ubar);
  llf_lambda_grad<DIM>(gamma, ql, qr, n, left, lg);
  const double sgn = left ? 0.5 : -0.5;
  for (int i = 0; i < NV; ++i) ubar[i] += sgn * lam * g[i] - 0.5 * gdu * lg[i];
}

// ---------------------------------------------------------------------
// HLLC: the tangent by forward-mode dual numbers through the flux as
// physics.hpp writes it (flux_hllc is templated on its scalar type), so it
// follows the branches (wave-speed bounds, star region, side) the forward
// evaluation takes; the adjoint by hand in reverse mode, through the same
// branches.
// ---------------------------------------------------------------------

// value and derivative; arithmetic by the usual rules, comparisons on values
struct Dual {
  double v, d;
  DG_HD Dual(double x = 0.0, double dx = 0.0) : v(x), d(dx) {}
  DG_HD Dual& operator+=(Dual b) {
    v += b.v;
    d += b.d;
    return *this;
  }
  DG_HD Dual& operator*=(Dual b) {
    d = d * b.v + v * b.d;
    v *= b.v;
    return *this;
  }
};
DG_HD Dual operator+(Dual a, Dual b) { return Dual(a.v + b.v, a.d + b.d); }
DG_HD Dual operator-(Dual a, Dual b) { return Dual(a.v - b.v, a.d - b.d); }
DG_HD Dual operator-(Dual a) { return Dual(-a.v, -a.d); }
DG_HD Dual operator*(Dual a, Dual b) { return Dual(a.v * b.v, a.d * b.v + a.v * b.d); }
DG_HD Dual operator/(Dual a, Dual b) {
  const double y = recip(b.v), q = div_by(a.v, b.v, y);
  return Dual(q, (a.d - q * b.d) * y);
}
DG_HD Dual recip(Dual a) {
  const double y = recip(a.v);
  return Dual(y, -a.d * y * y);
}
// a / b with y = recip(b)
DG_HD Dual div_by(Dual a, Dual b, Dual y) {
  const double q = div_by(a.v, b.v, y.v);
  return Dual(q, (a.d - q * b.d) * y.v);
}
DG_HD Dual sqrt(Dual a) {
  const double r = sqrt(a.v);
  return Dual(r, 0.5 * a.d / r);
}
DG_HD bool operator<(Dual a, Dual b) { return a.v < b.v; }
DG_HD bool operator<=(Dual a, Dual b) { return a.v <= b.v; }
DG_HD bool operator>=(Dual a, Dual b) { return a.v >= b.v; }

// df = (dF/du_l) du_l + (dF/du_r) du_r for the HLLC flux F(u_l, u_r; n)
template <int DIM>
DG_HD void hllc_jvp(double gamma, const double* ul, const double* ur, const double* dul,
                    const double* dur, const double* n, double* df) {
  constexpr int NV = DIM + 2;
  Dual a[NV], b[NV], f[NV];
  for (int i = 0; i < NV; ++i) {
    a[i] = Dual(ul[i], dul[i]);
    b[i] = Dual(ur[i], dur[i]);
  }
  flux_hllc<DIM, Dual>(gamma, a, b, n, f);
  for (int i = 0; i < NV; ++i) df[i] = f[i].d;
}

// ubar_side += (dF/du_side)^T g for the sides selected, by forward-mode
// dual numbers: one column of the Jacobian per input component.  The
// kernels use the reverse-mode hllc_vjp below; this form serves as its check.
template <int DIM>
DG_HD void hllc_vjp_columns(double gamma, const double* ul, const double* ur, const double* n,
                            const double* g, bool with_left, bool with_right, double* ubar_l,
                            double* ubar_r) {
  constexpr int NV = DIM + 2;
  for (int side = 0; side < 2; ++side) {
    if (side == 0 ? !with_left : !with_right) continue;
    double* ub = side == 0 ? ubar_l : ubar_r;
    for (int j = 0; j < NV; ++j) {
      Dual a[NV], b[NV], f[NV];
      for (int i = 0; i < NV; ++i) {
        a[i] = Dual(ul[i], side == 0 && i == j ? 1.0 : 0.0);
        b[i] = Dual(ur[i], side == 1 && i == j ? 1.0 : 0.0);
      }
      flux_hllc<DIM, Dual>(gamma, a, b, n, f);
      double s = 0.0;
      for (int i = 0; i < NV; ++i) s += g[i] * f[i].d;
      ub[j] += s;
    }
  }
}

// ubar_side += (dF/du_side)^T g for the sides selected, in reverse mode: the
// forward pass of flux_hllc (the same expressions, so the same wave-speed,
// star-region and side choices), then the cotangents back through it, about
// the cost of two flux evaluations where the dual-number columns cost ten.
template <int DIM>
DG_HD void hllc_vjp(double gamma, const double* ul, const double* ur, const double* n,
                    const double* g, bool with_left, bool with_right, double* ubar_l,
                    double* ubar_r) {
  constexpr int NV = DIM + 2;
  const double gm1 = gamma - 1.0;
  // forward
  double nrm = 0.0, nh[DIM], vl[DIM], vr[DIM];
  for (int d = 0; d < DIM; ++d) nrm += n[d] * n[d];
  nrm = sqrt(nrm);
  const double inrm = recip(nrm);
  for (int d = 0; d < DIM; ++d) nh[d] = div_by(n[d], nrm, inrm);
  const double rl = ul[0], rr = ur[0], El = ul[NV - 1], Er = ur[NV - 1];
  const double il = recip(rl), ir = recip(rr);
  double v2l = 0.0, v2r = 0.0, vnl = 0.0, vnr = 0.0;
  for (int d = 0; d < DIM; ++d) {
    vl[d] = div_by(ul[d + 1], rl, il);
    vr[d] = div_by(ur[d + 1], rr, ir);
    v2l += vl[d] * vl[d];
    v2r += vr[d] * vr[d];
    vnl += vl[d] * nh[d];
    vnr += vr[d] * nh[d];
  }
  const double el = div_by(El, rl, il), er = div_by(Er, rr, ir);
  const double pl = (gamma - 1.0) * (El - 0.5 * rl * v2l);
  const double pr = (gamma - 1.0) * (Er - 0.5 * rr * v2r);
  const double cl = sqrt(div_by(gamma * pl, rl, il)), cr = sqrt(div_by(gamma * pr, rr, ir));
  const double sl = sqrt(rl), sr = sqrt(rr), ss = sl + sr, is = recip(ss);
  double vd[DIM], vroe2 = 0.0;
  for (int d = 0; d < DIM; ++d) {
    vd[d] = div_by(sl * vl[d] + sr * vr[d], ss, is);
    vroe2 += vd[d] * vd[d];
  }
  const double vroe = div_by(sl * vnl + sr * vnr, ss, is);
  const double Hl = div_by(El + pl, rl, il), Hr = div_by(Er + pr, rr, ir);
  const double Hroe = div_by(sl * Hl + sr * Hr, ss, is);
  const double croe = sqrt((gamma - 1.0) * (Hroe - 0.5 * vroe2));
  // SL = dmin(vnl - cl, vroe - croe), SR = dmax(vnr + cr, vroe + croe)
  const double aL = vnl - cl, bL = vroe - croe, aR = vnr + cr, bR = vroe + croe;
  const bool SL_roe = bL < aL, SR_roe = aR < bR;
  const double SL = SL_roe ? bL : aL, SR = SR_roe ? bR : aR;
  const double mL = SL - vnl, mR = SR - vnr;
  const bool star = !(SL >= 0) && !(SR <= 0);
  double Ss = 0.0, iden = 1.0;
  if (star) {
    const double den = rl * mL - rr * mR;
    iden = recip(den);
    Ss = div_by(pr - pl + rl * vnl * mL - rr * vnr * mR, den, iden);
  }
  const bool left = star ? Ss >= 0 : SL >= 0;
  const double* uk = left ? ul : ur;

  // reverse: f = nrm * (fk(uk) [+ Sk (star terms)])
  double G[NV];
  for (int i = 0; i < NV; ++i) G[i] = g[i] * nrm;
  double ulb[NV], urb[NV], ukb[NV];
  for (int i = 0; i < NV; ++i) ulb[i] = urb[i] = ukb[i] = 0.0;
  flux_n_vjp<DIM>(gamma, uk, node_prims<DIM>(gamma, uk), nh, G, ukb);
  double rl_b = 0.0, rr_b = 0.0, El_b = 0.0, Er_b = 0.0, vnl_b = 0.0, vnr_b = 0.0;
  double pl_b = 0.0, pr_b = 0.0, el_b = 0.0, er_b = 0.0, vl_b[DIM], vr_b[DIM];
  for (int d = 0; d < DIM; ++d) vl_b[d] = vr_b[d] = 0.0;
  if (star) {
    const double* vk = left ? vl : vr;
    const double rk = left ? rl : rr, vnk = left ? vnl : vnr, ek = left ? el : er;
    const double pk = left ? pl : pr, Sk = left ? SL : SR, mk = left ? mL : mR;
    const double iD = recip(Sk - Ss), rs = rk * mk * iD;
    const double X = Ss - vnk, irkmk = recip(rk * mk), Z = pk * irkmk, Y = Ss + Z, es = ek + X * Y;
    // f0 = fk0 + Sk (rs - uk0), f_d = fk_d + Sk (rs (vk_d + X nh_d) - uk_d),
    // fE = fkE + Sk (rs es - ukE)
    double Sk_b = G[0] * (rs - uk[0]) + G[NV - 1] * (rs * es - uk[NV - 1]);
    double rs_b = Sk * (G[0] + G[NV - 1] * es), gn = 0.0, vk_b[DIM];
    for (int d = 0; d < DIM; ++d) {
      const double w = vk[d] + X * nh[d];
      Sk_b += G[d + 1] * (rs * w - uk[d + 1]);
      rs_b += Sk * G[d + 1] * w;
      vk_b[d] = Sk * rs * G[d + 1];
      gn += G[d + 1] * nh[d];
    }
    for (int i = 0; i < NV; ++i) ukb[i] -= Sk * G[i];
    const double es_b = Sk * rs * G[NV - 1];
    double X_b = Sk * rs * gn + es_b * Y, Ss_b = 0.0;
    const double Y_b = es_b * X, ek_b = es_b;
    // Y = Ss + pk / (rk mk)
    Ss_b += Y_b;
    const double pk_b = Y_b * irkmk, rkmk_b = -Y_b * Z * irkmk;
    // X = Ss - vnk
    Ss_b += X_b;
    double vnk_b = -X_b;
    // rs = rk mk / (Sk - Ss)
    const double rk_b = rs_b * mk * iD + rkmk_b * mk;
    double mk_b = rs_b * rk * iD + rkmk_b * rk;
    const double D_b = -rs_b * rs * iD;
    Sk_b += D_b;
    Ss_b -= D_b;
    double SL_b = 0.0, SR_b = 0.0, mL_b = 0.0, mR_b = 0.0;
    if (left) {
      rl_b += rk_b; vnl_b += vnk_b; el_b += ek_b; pl_b += pk_b; SL_b += Sk_b; mL_b += mk_b;
      for (int d = 0; d < DIM; ++d) vl_b[d] += vk_b[d];
    } else {
      rr_b += rk_b; vnr_b += vnk_b; er_b += ek_b; pr_b += pk_b; SR_b += Sk_b; mR_b += mk_b;
      for (int d = 0; d < DIM; ++d) vr_b[d] += vk_b[d];
    }
    // Ss = (pr - pl + rl vnl mL - rr vnr mR) / (rl mL - rr mR)
    const double Num_b = Ss_b * iden, Den_b = -Ss_b * Ss * iden;
    pr_b += Num_b;
    pl_b -= Num_b;
    rl_b += Num_b * vnl * mL + Den_b * mL;
    vnl_b += Num_b * rl * mL;
    mL_b += Num_b * rl * vnl + Den_b * rl;
    rr_b -= Num_b * vnr * mR + Den_b * mR;
    vnr_b -= Num_b * rr * mR;
    mR_b -= Num_b * rr * vnr + Den_b * rr;
    // mL = SL - vnl, mR = SR - vnr
    SL_b += mL_b;
    vnl_b -= mL_b;
    SR_b += mR_b;
    vnr_b -= mR_b;
    // the wave-speed bounds, through the branch the forward took
    double vroe_b = 0.0, croe_b = 0.0, cl_b = 0.0, cr_b = 0.0;
    if (SL_roe) {
      vroe_b += SL_b;
      croe_b -= SL_b;
    } else {
      vnl_b += SL_b;
      cl_b -= SL_b;
    }
    if (SR_roe) {
      vroe_b += SR_b;
      croe_b += SR_b;
    } else {
      vnr_b += SR_b;
      cr_b += SR_b;
    }
    // croe = sqrt((gamma - 1)(Hroe - vroe2 / 2))
    const double W_b = croe_b * recip(2.0 * croe);
    const double Hroe_b = gm1 * W_b, vroe2_b = -0.5 * gm1 * W_b;
    double sl_b = Hroe_b * (Hl - Hroe) * is + vroe_b * (vnl - vroe) * is;
    double sr_b = Hroe_b * (Hr - Hroe) * is + vroe_b * (vnr - vroe) * is;
    const double Hl_b = Hroe_b * sl * is, Hr_b = Hroe_b * sr * is;
    vnl_b += vroe_b * sl * is;
    vnr_b += vroe_b * sr * is;
    for (int d = 0; d < DIM; ++d) {
      const double vd_b = 2.0 * vd[d] * vroe2_b;
      vl_b[d] += vd_b * sl * is;
      vr_b[d] += vd_b * sr * is;
      sl_b += vd_b * (vl[d] - vd[d]) * is;
      sr_b += vd_b * (vr[d] - vd[d]) * is;
    }
    // H = (E + p) / rho, s = sqrt(rho), c = sqrt(gamma p / rho)
    El_b += Hl_b * il;
    pl_b += Hl_b * il;
    rl_b -= Hl_b * Hl * il;
    Er_b += Hr_b * ir;
    pr_b += Hr_b * ir;
    rr_b -= Hr_b * Hr * ir;
    rl_b += sl_b * recip(2.0 * sl);
    rr_b += sr_b * recip(2.0 * sr);
    if (cl_b != 0.0) {
      const double Q_b = cl_b * recip(2.0 * cl);
      pl_b += Q_b * gamma * il;
      rl_b -= Q_b * cl * cl * il;
    }
    if (cr_b != 0.0) {
      const double Q_b = cr_b * recip(2.0 * cr);
      pr_b += Q_b * gamma * ir;
      rr_b -= Q_b * cr * cr * ir;
    }
  }
  // e = E / rho, p = (gamma - 1)(E - rho |v|^2 / 2), v = m / rho
  El_b += el_b * il + gm1 * pl_b;
  rl_b -= el_b * el * il + 0.5 * gm1 * v2l * pl_b;
  Er_b += er_b * ir + gm1 * pr_b;
  rr_b -= er_b * er * ir + 0.5 * gm1 * v2r * pr_b;
  const double v2l_b = -0.5 * gm1 * rl * pl_b, v2r_b = -0.5 * gm1 * rr * pr_b;
  for (int d = 0; d < DIM; ++d) {
    vl_b[d] += 2.0 * vl[d] * v2l_b + vnl_b * nh[d];
    vr_b[d] += 2.0 * vr[d] * v2r_b + vnr_b * nh[d];
    ulb[d + 1] += vl_b[d] * il;
    rl_b -= vl_b[d] * vl[d] * il;
    urb[d + 1] += vr_b[d] * ir;
    rr_b -= vr_b[d] * vr[d] * ir;
  }
  ulb[0] += rl_b;
  ulb[NV - 1] += El_b;
  urb[0] += rr_b;
  urb[NV - 1] += Er_b;
  double* ukside = left ? ulb : urb;
  for (int i = 0; i < NV; ++i) ukside[i] += ukb[i];
  if (with_left)
    for (int i = 0; i < NV; ++i) ubar_l[i] += ulb[i];
  if (with_right)
    for (int i = 0; i < NV; ++i) ubar_r[i] += urb[i];
}

// ---------------------------------------------------------------------
// Navier-Stokes: gradient variables q = (rho, v, T = p / rho) and the
// Newtonian viscous flux (parabolic_impl.hpp grad_vars, viscous_flux_dir).
// ---------------------------------------------------------------------

template <int DIM>
DG_HD void grad_vars_jvp(double gamma, const double* u, const double* du, double* dq) {
  const double ir = recip(u[0]);
  double m2 = 0.0, mdm = 0.0;
  for (int k = 0; k < DIM; ++k) {
    m2 += u[k + 1] * u[k + 1];
    mdm += u[k + 1] * du[k + 1];
  }
  const double p = (gamma - 1.0) * (u[DIM + 1] - 0.5 * m2 * ir);
  const double dp = (gamma - 1.0) * (du[DIM + 1] - mdm * ir + 0.5 * m2 * ir * ir * du[0]);
  dq[0] = du[0];
  for (int k = 0; k < DIM; ++k) dq[k + 1] = (du[k + 1] - u[k + 1] * ir * du[0]) * ir;
  dq[DIM + 1] = (dp - p * ir * du[0]) * ir;
}

template <int DIM>
DG_HD void grad_vars_vjp(double gamma, const double* u, const double* qbar, double* ubar) {
  const double ir = recip(u[0]);
  double m2 = 0.0;
  for (int k = 0; k < DIM; ++k) m2 += u[k + 1] * u[k + 1];
  const double p = (gamma - 1.0) * (u[DIM + 1] - 0.5 * m2 * ir);
  const double Tb = qbar[DIM + 1];
  // T = p / rho
  const double pb = Tb * ir;
  double rb = qbar[0] - Tb * p * ir * ir;
  // p = (gamma - 1)(E - |m|^2 / (2 rho))
  ubar[DIM + 1] += (gamma - 1.0) * pb;
  rb += (gamma - 1.0) * 0.5 * m2 * ir * ir * pb;
  for (int k = 0; k < DIM; ++k) {
    ubar[k + 1] += -(gamma - 1.0) * u[k + 1] * ir * pb + qbar[k + 1] * ir;
    rb -= qbar[k + 1] * u[k + 1] * ir * ir;
  }
  ubar[0] += rb;
}

DG_HD double third(double x) { return div_by(x, 3.0, 1.0 / 3.0); }

// Symmetric viscous stress tau (without mu) from the velocity gradients
// g[c][1 + k] = d v_k / d x_c, as viscous_flux_dir forms it.
template <int DIM>
DG_HD void stress(const double g[DIM][DIM + 2], double tau[DIM][DIM]) {
  if constexpr (DIM == 2) {
    tau[0][0] = third(4.0 * g[0][1] - 2.0 * g[1][2]);
    tau[1][1] = third(4.0 * g[1][2] - 2.0 * g[0][1]);
    tau[0][1] = tau[1][0] = g[1][1] + g[0][2];
  } else {
    tau[0][0] = third(4.0 * g[0][1] - 2.0 * (g[1][2] + g[2][3]));
    tau[1][1] = third(4.0 * g[1][2] - 2.0 * (g[0][1] + g[2][3]));
    tau[2][2] = third(4.0 * g[2][3] - 2.0 * (g[0][1] + g[1][2]));
    tau[0][1] = tau[1][0] = g[1][1] + g[0][2];
    tau[0][2] = tau[2][0] = g[2][1] + g[0][3];
    tau[1][2] = tau[2][1] = g[2][2] + g[1][3];
  }
}

// gbar += (dtau/dg)^T taubar (taubar as a full, not necessarily symmetric,
// matrix of cotangents of the entries tau[c][k]).
template <int DIM>
DG_HD void stress_vjp(const double taubar[DIM][DIM], double gbar[DIM][DIM + 2]) {
  if constexpr (DIM == 2) {
    const double t00 = taubar[0][0], t11 = taubar[1][1], t01 = taubar[0][1] + taubar[1][0];
    gbar[0][1] += third(4.0 * t00 - 2.0 * t11);
    gbar[1][2] += third(4.0 * t11 - 2.0 * t00);
    gbar[1][1] += t01;
    gbar[0][2] += t01;
  } else {
    const double t00 = taubar[0][0], t11 = taubar[1][1], t22 = taubar[2][2];
    const double t01 = taubar[0][1] + taubar[1][0];
    const double t02 = taubar[0][2] + taubar[2][0];
    const double t12 = taubar[1][2] + taubar[2][1];
    gbar[0][1] += third(4.0 * t00 - 2.0 * (t11 + t22));
    gbar[1][2] += third(4.0 * t11 - 2.0 * (t00 + t22));
    gbar[2][3] += third(4.0 * t22 - 2.0 * (t00 + t11));
    gbar[1][1] += t01;
    gbar[0][2] += t01;
    gbar[2][1] += t02;
    gbar[0][3] += t02;
    gbar[2][2] += t12;
    gbar[1][3] += t12;
  }
}

// Tangent of the viscous flux in every direction c: f[c] = (0, mu tau[c][.],
// mu (v . tau[c][.] + kappa dT/dx_c)), tau the stress of the gradient.
template <int DIM>
DG_HD void viscous_flux_jvp_stress(double mu, double kappa, const double* q,
                                   const double tau[DIM][DIM], const double* dq,
                                   const double dg[DIM][DIM + 2], double df[DIM][DIM + 2]) {
  double dtau[DIM][DIM];
  stress<DIM>(dg, dtau);
  for (int c = 0; c < DIM; ++c) {
    df[c][0] = 0.0;
    double e = kappa * dg[c][DIM + 1];
    for (int k = 0; k < DIM; ++k) {
      df[c][k + 1] = mu * dtau[c][k];
      e += dq[k + 1] * tau[c][k] + q[k + 1] * dtau[c][k];
    }
    df[c][DIM + 1] = mu * e;
  }
}

template <int DIM>
DG_HD void viscous_flux_jvp(double mu, double kappa, const double* q, const double g[DIM][DIM + 2],
                            const double* dq, const double dg[DIM][DIM + 2],
                            double df[DIM][DIM + 2]) {
  double tau[DIM][DIM];
  stress<DIM>(g, tau);
  viscous_flux_jvp_stress<DIM>(mu, kappa, q, tau, dq, dg, df);
}

// qbar += (df/dq)^T fbar, gbar += (df/dg)^T fbar over all directions c.
template <int DIM>
DG_HD void viscous_flux_vjp_stress(double mu, double kappa, const double* q,
                                   const double tau[DIM][DIM], const double fbar[DIM][DIM + 2],
                                   double* qbar, double gbar[DIM][DIM + 2]) {
  double taubar[DIM][DIM];
  for (int c = 0; c < DIM; ++c) {
    const double fe = mu * fbar[c][DIM + 1];
    gbar[c][DIM + 1] += kappa * fe;
    for (int k = 0; k < DIM; ++k) {
      taubar[c][k] = mu * fbar[c][k + 1] + fe * q[k + 1];
      qbar[k + 1] += fe * tau[c][k];
    }
  }
  stress_vjp<DIM>(taubar, gbar);
}

template <int DIM>
DG_HD void viscous_flux_vjp(double mu, double kappa, const double* q, const double g[DIM][DIM + 2],
                            const double fbar[DIM][DIM + 2], double* qbar,
                            double gbar[DIM][DIM + 2]) {
  double tau[DIM][DIM];
  stress<DIM>(g, tau);
  viscous_flux_vjp_stress<DIM>(mu, kappa, q, tau, fbar, qbar, gbar);
}

}  // namespace dgsem
