// Pointwise physics for the compressible Euler / Navier-Stokes equations in
// 2D and 3D: physical flux, LLF and HLLC surface fluxes, the Chandrashekar
// entropy-conservative / kinetic-energy-preserving two-point flux and the
// logarithmic mean.  Expressions keep the reference's evaluation order so the
// results agree with it to rounding.
//
// Reference: src/base/math_utils.hpp:8-24 (the logarithmic mean),
// src/equations/compressible_euler{2D,3D}.hpp (flux, wave speed),
// src/base/numerical_flux.hpp:39-135,198-228 (LLF), :436-594 (Chandrashekar),
// src/base/numerical_flux_detail.hpp:9-21.
#pragma once

#include <cmath>

// The functions are used by the HIP kernels and, compiled by a host C++
// compiler, by the CPU unit tests of their derivatives.
#if defined(__HIPCC__)
#include <hip/hip_runtime.h>
#define DG_HD __host__ __device__ __forceinline__
#else
#define DG_HD inline
#endif

namespace dgsem {

using std::fabs;
using std::log;
using std::sqrt;

// Numerical flux kinds (include/dgsem_amd.h DGSEM_FLUX_*).  kFluxAny is a
// template value only: the kernel instantiation that reads the volume,
// surface and subcell flux kinds from its parameters at run time.
enum FluxKind : int { kFluxLLF = 0, kFluxHLLC = 1, kFluxCentral = 2, kFluxAny = 3 };
// volume flux kinds
enum VolumeFluxKind : int { kVolumeChandrashekar = 0, kVolumeCentral = 2 };

DG_HD double dmax(double a, double b) { return (a < b) ? b : a; }
DG_HD double dmin(double a, double b) { return (b < a) ? b : a; }
// the same for other scalar types (the derivative code's dual numbers)
template <class T>
DG_HD T dmax(T a, T b) {
  return (a < b) ? b : a;
}
template <class T>
DG_HD T dmin(T a, T b) {
  return (b < a) ? b : a;
}

// 1 / x: on the GPU the hardware reciprocal r (relative error e below 5e-8)
// refined by one third-order step r (1 + e + e^2), which leaves e^3 < 2e-22,
// so the result is within an ulp of the IEEE quotient for a third of the
// instructions of the division sequence (the parity tests bound the effect on
// the RHS).  Over 1e9 random operands on an MI355X: r within 4.7e-8, 13 results off
// by an ulp, none by more.
DG_HD double recip(double x) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double r = __builtin_amdgcn_rcp(x);
  const double e = fma(-x, r, 1.0);
  return fma(r, fma(e, e, e), r);
#else
  return 1.0 / x;
#endif
}

// a / b from y = recip(b): the quotient estimate corrected by its residual
// (Markstein's method).  The residual is exact to an ulp of the estimate's
// error, so the result is the IEEE quotient (of all 1e9 random operand pairs on an
// MI355X); several quotients by one b share its reciprocal.
DG_HD double div_by(double a, double b, double y) {
#if defined(__HIP_DEVICE_COMPILE__)
  const double q = a * y;
  return fma(fma(-b, q, a), y, q);
#else
  (void)y;
  return a / b;
#endif
}

// Pressure of a conservative state.
template <int DIM>
DG_HD double pressure(double gamma, const double* u) {
  double v2 = 0.0;
  for (int k = 0; k < DIM; ++k) {
    const double v = u[k + 1] / u[0];
    v2 += v * v;
  }
  return (gamma - 1.0) * (u[DIM + 1] - 0.5 * u[0] * v2);
}

// Physical flux F(u) . n: compressible_euler2D.hpp:25-57,
// compressible_euler3D.hpp:26-67 (sum of the per-direction fluxes).  T is
// double, or the dual numbers of the derivative code (physics_ad.hpp).
template <int DIM, class T = double>
DG_HD void physical_flux_n(double gamma, const T* u, const double* n, T* f) {
  constexpr int NV = DIM + 2;
  const T rho = u[0], rhoE = u[NV - 1];
  T v[DIM];
  T v2 = 0.0;
  const T ir = recip(rho);
  for (int k = 0; k < DIM; ++k) v[k] = div_by(u[k + 1], rho, ir);
  for (int k = 0; k < DIM; ++k) v2 += v[k] * v[k];
  const T p = (gamma - 1.0) * (rhoE - 0.5 * rho * v2);
  for (int i = 0; i < NV; ++i) f[i] = 0.0;
  for (int d = 0; d < DIM; ++d) {
    // flux in direction d: (m_d, m_d v + p e_d, v_d (E + p))
    T fd[NV];
    fd[0] = u[d + 1];
    for (int k = 0; k < DIM; ++k) fd[k + 1] = u[d + 1] * v[k] + (k == d ? p : 0.0);
    fd[NV - 1] = v[d] * (rhoE + p);
    for (int i = 0; i < NV; ++i) f[i] = f[i] + n[d] * fd[i];
  }
}

// max(|v_L.n|, |v_R.n|) + max(c_L, c_R) |n|, compressible_euler3D.hpp:121-166.
template <int DIM>
DG_HD double llf_wave_speed(double gamma, const double* ul, const double* ur, const double* n) {
  double vnl = 0.0, vnr = 0.0, nn = 0.0;
  for (int k = 0; k < DIM; ++k) {
    vnl += (ul[k + 1] / ul[0]) * n[k];
    vnr += (ur[k + 1] / ur[0]) * n[k];
    nn += n[k] * n[k];
  }
  const double al = sqrt(gamma * pressure<DIM>(gamma, ul) / ul[0]);
  const double ar = sqrt(gamma * pressure<DIM>(gamma, ur) / ur[0]);
  return dmax(fabs(vnl), fabs(vnr)) + dmax(al, ar) * sqrt(nn);
}

// Local Lax-Friedrichs: 0.5 (F_L + F_R).n - 0.5 lambda (u_R - u_L) with lambda =
// max(|v_L.n|, |v_R.n|) + max(c_L, c_R) |n| (numerical_flux.hpp:54-68,
// compressible_euler3D.hpp:121-166).  One reciprocal per state and one square
// root: max(c_L, c_R) |n| = sqrt(max(c_L^2, c_R^2) |n|^2).  Like the maximum of
// the two roots, that is NaN for a left state of negative pressure.
template <int DIM>
DG_HD void flux_llf(double gamma, const double* ul, const double* ur, const double* n, double* f) {
  constexpr int NV = DIM + 2;
  const double il = recip(ul[0]), ir = recip(ur[0]);
  double vnl = 0.0, vnr = 0.0, v2l = 0.0, v2r = 0.0, nn = 0.0;
  for (int k = 0; k < DIM; ++k) {
    const double vl = ul[k + 1] * il, vr = ur[k + 1] * ir;
    vnl += vl * n[k];
    vnr += vr * n[k];
    v2l += vl * vl;
    v2r += vr * vr;
    nn += n[k] * n[k];
  }
  const double pl = (gamma - 1.0) * (ul[NV - 1] - 0.5 * ul[0] * v2l);
  const double pr = (gamma - 1.0) * (ur[NV - 1] - 0.5 * ur[0] * v2r);
  const double cl = gamma * pl * il, cr = gamma * pr * ir;  // squared speeds of sound
  const double c2 = cl >= 0.0 && cl < cr ? cr : cl;
  const double lam = dmax(fabs(vnl), fabs(vnr)) + sqrt(c2 * nn);
  const double ps = pl + pr;
  f[0] = 0.5 * (ul[0] * vnl + ur[0] * vnr - lam * (ur[0] - ul[0]));
  for (int k = 0; k < DIM; ++k)
    f[k + 1] = 0.5 * (ul[k + 1] * vnl + ur[k + 1] * vnr + ps * n[k] - lam * (ur[k + 1] - ul[k + 1]));
  f[NV - 1] = 0.5 * ((ul[NV - 1] + pl) * vnl + (ur[NV - 1] + pr) * vnr - lam * (ur[NV - 1] - ul[NV - 1]));
}

// HLLC with a normal vector.  The reference has HLLC for 1D Euler only
// (numerical_flux.hpp:283-378); this applies the same construction
// (Roe-averaged wave-speed bounds, contact speed, star states) in the frame of
// the unit normal with the tangential velocity carried through, and scales
// the result by |n|.  Its quotients are correctly rounded, from one reciprocal
// per denominator: at low Mach number the pressure differences keep the last
// bits of the velocities (plain reciprocals put the N = 5 Taylor-Green vortex
// 1.6e-12 from a scalar evaluation, these 6e-13).
template <int DIM, class T = double>
DG_HD void flux_hllc(double gamma, const T* ul, const T* ur, const double* n, T* f) {
  constexpr int NV = DIM + 2;
  double nrm = 0.0, nh[DIM];
  T vl[DIM], vr[DIM];
  for (int d = 0; d < DIM; ++d) nrm += n[d] * n[d];
  nrm = sqrt(nrm);
  const double inrm = recip(nrm);
  for (int d = 0; d < DIM; ++d) nh[d] = div_by(n[d], nrm, inrm);
  const T rl = ul[0], rr = ur[0], El = ul[NV - 1], Er = ur[NV - 1];
  const T il = recip(rl), ir = recip(rr);
  T v2l = 0.0, v2r = 0.0, vnl = 0.0, vnr = 0.0;
  for (int d = 0; d < DIM; ++d) {
    vl[d] = div_by(ul[d + 1], rl, il);
    vr[d] = div_by(ur[d + 1], rr, ir);
    v2l += vl[d] * vl[d];
    v2r += vr[d] * vr[d];
    vnl += vl[d] * nh[d];
    vnr += vr[d] * nh[d];
  }
  const T el = div_by(El, rl, il), er = div_by(Er, rr, ir);
  const T pl = (gamma - 1.0) * (El - 0.5 * rl * v2l);
  const T pr = (gamma - 1.0) * (Er - 0.5 * rr * v2r);
  const T cl = sqrt(div_by(gamma * pl, rl, il)), cr = sqrt(div_by(gamma * pr, rr, ir));
  const T sl = sqrt(rl), sr = sqrt(rr), ss = sl + sr, is = recip(ss);
  T vroe2 = 0.0;
  for (int d = 0; d < DIM; ++d) {
    const T vd = div_by(sl * vl[d] + sr * vr[d], ss, is);
    vroe2 += vd * vd;
  }
  const T vroe = div_by(sl * vnl + sr * vnr, ss, is);
  const T Hl = div_by(El + pl, rl, il), Hr = div_by(Er + pr, rr, ir);
  const T Hroe = div_by(sl * Hl + sr * Hr, ss, is);
  const T croe = sqrt((gamma - 1.0) * (Hroe - 0.5 * vroe2));
  const T SL = dmin(vnl - cl, vroe - croe);
  const T SR = dmax(vnr + cr, vroe + croe);
  const T mL = SL - vnl, mR = SR - vnr;
  // the side whose state (or star state) gives the flux; only that side's
  // physical flux is formed
  const bool star = !(SL >= 0) && !(SR <= 0);
  const T den = rl * mL - rr * mR;
  const T Ss = star ? div_by(pr - pl + rl * vnl * mL - rr * vnr * mR, den, recip(den)) : T(0.0);
  const bool left = star ? Ss >= 0 : SL >= 0;
  const T* uk = left ? ul : ur;
  T fk[NV];
  physical_flux_n<DIM>(gamma, uk, nh, fk);
  if (!star) {
    for (int i = 0; i < NV; ++i) f[i] = fk[i];
  } else {
    const T* vk = left ? vl : vr;
    const T rk = left ? rl : rr, vnk = left ? vnl : vnr, ek = left ? el : er;
    const T pk = left ? pl : pr, Sk = left ? SL : SR, mk = left ? mL : mR;
    const T D = Sk - Ss, rkmk = rk * mk;
    const T rs = div_by(rkmk, D, recip(D));
    const T es = ek + (Ss - vnk) * (Ss + div_by(pk, rkmk, recip(rkmk)));
    f[0] = fk[0] + Sk * (rs - uk[0]);
    for (int d = 0; d < DIM; ++d) f[d + 1] = fk[d + 1] + Sk * (rs * (vk[d] + (Ss - vnk) * nh[d]) - uk[d + 1]);
    f[NV - 1] = fk[NV - 1] + Sk * (rs * es - uk[NV - 1]);
  }
  for (int i = 0; i < NV; ++i) f[i] *= nrm;
}

// CentralFlux with a normal, numerical_flux.hpp:247-257 (2D in the
// reference): 0.5 (F(u_L).n + F(u_R).n), numerical_flux_detail.hpp:23-32.
template <int DIM>
DG_HD void flux_central(double gamma, const double* ul, const double* ur, const double* n, double* f) {
  constexpr int NV = DIM + 2;
  double fl[NV], fr[NV];
  physical_flux_n<DIM>(gamma, ul, n, fl);
  physical_flux_n<DIM>(gamma, ur, n, fr);
  for (int i = 0; i < NV; ++i) f[i] = 0.5 * (fl[i] + fr[i]);
}

template <int DIM>
DG_HD void surface_flux(int kind, double gamma, const double* ul, const double* ur, const double* n,
                        double* f) {
  if (kind == kFluxHLLC)
    flux_hllc<DIM>(gamma, ul, ur, n, f);
  else if (kind == kFluxCentral)
    flux_central<DIM>(gamma, ul, ur, n, f);
  else
    flux_llf<DIM>(gamma, ul, ur, n, f);
}

// Per-node quantities hoisted out of the two-point and surface fluxes:
// rho, v[DIM], beta = rho / (2 p), the specific kinetic energy |v|^2 / 2,
// the pressure and the speed of sound.
template <int DIM>
struct NodePrims {
  double rho, v[DIM], beta, kin, p, c;
};

template <int DIM>
DG_HD NodePrims<DIM> node_prims(double gamma, const double* u) {
  NodePrims<DIM> q;
  q.rho = u[0];
  double v2 = 0.0;
  const double ir = recip(u[0]);
  for (int k = 0; k < DIM; ++k) q.v[k] = u[k + 1] * ir;
  for (int k = 0; k < DIM; ++k) v2 += q.v[k] * q.v[k];
  q.p = (gamma - 1.0) * (u[DIM + 1] - 0.5 * u[0] * v2);
  q.beta = 0.5 * u[0] * recip(q.p);
  q.kin = 0.5 * v2;
  q.c = sqrt(gamma * q.p * ir);
  return q;
}

// The logarithmic mean of x and y is (x + y) / 2 over Q = artanh(xi) / xi with
// xi = (x - y) / (x + y), since log(y / x) = 2 artanh((y - x) / (y + x)).  Q and
// its inverse are series in f2 = xi^2; the reference switches from its own
// series to the quotient (y - x) / log(y / x) at f2 = 1e-4 (math_utils.hpp:8-24).

// Q = sum_k f2^k / (2k + 1) for f2 < kSeriesMax, to rounding.
constexpr double kSeriesMax = 0.0295;  // x / y up to sqrt(2)
DG_HD double artanh_series(double f2) {
  double q = 1.0 / 21.0;
  q = 1.0 / 19.0 + f2 * q;
  q = 1.0 / 17.0 + f2 * q;
  q = 1.0 / 15.0 + f2 * q;
  q = 1.0 / 13.0 + f2 * q;
  q = 1.0 / 11.0 + f2 * q;
  q = 1.0 / 9.0 + f2 * q;
  q = 1.0 / 7.0 + f2 * q;
  q = 1.0 / 5.0 + f2 * q;
  q = 1.0 / 3.0 + f2 * q;
  return 1.0 + f2 * q;
}

// log(hi / lo): binary exponents apart, the ratio of the significands is
// brought into [1/sqrt(2), sqrt(2)] and its logarithm is 2 artanh of
// (a - b) / (a + b).  NaN unless both have one sign, as the logarithm's.
DG_HD double log_quotient(double hi, double lo) {
  int eh, el;
  const double a = std::frexp(hi, &eh);
  double b = std::frexp(lo, &el);
  int k = eh - el;
  const double root2 = 1.4142135623730951;
  if (fabs(a) > root2 * fabs(b)) {
    b *= 2.0;
    ++k;
  } else if (root2 * fabs(a) < fabs(b)) {
    b *= 0.5;
    --k;
  }
  const double xi = (a - b) * recip(a + b);
  const double r = 0.6931471805599453 * (double)k + 2.0 * xi * artanh_series(xi * xi);
  return lo > 0.0 || hi < 0.0 ? r : __builtin_nan("");
}

// Q of x and y, f2 their xi^2.  Symmetric in x and y.
DG_HD double artanh_ratio(double x, double y, double f2) {
  if (f2 < kSeriesMax) return artanh_series(f2);
  const double lo = dmin(x, y), hi = dmax(x, y);
  return log_quotient(hi, lo) * (0.5 * (hi + lo)) * recip(hi - lo);
}

// Chandrashekar two-point flux from hoisted node quantities (rho, v, beta),
// numerical_flux.hpp:436-500 (2D) and :520-594 (3D).  inv_gm1 = 1/(gamma-1).
//
// One reciprocal, of s_rho s_beta with s = x + y, gives 1/s_rho and 1/s_beta and
// with them xi of both means, p_mean = s_rho / (2 s_beta) and 1/beta_mean =
// 2 Q(f2_beta) / s_beta; rho_mean is s_rho / 2 times 1 / Q(f2_rho), whose own
// series (xi / artanh xi = 1 - f2/3 - 4 f2^2/45 - 44 f2^3/945 - ...) serves the
// usual case.  With both f2 < 1e-4 three terms are exact to rounding; beyond,
// the longer series and the logarithm take over (a divergent branch: about 30
// instructions up to a ratio of sqrt(2), 45 above, against 150 for a library
// logarithm and its two divisions).  Largest error of a component over all
// branches: 3 epsilon of the magnitudes it sums (25 in the quotient form).
// Together with the register and LDS changes of the line kernels, one MI355X:
// SSPRK3 step at 64^3 N = 3 2.12 -> 1.84 ms, 2D N = 5 Riemann problem (101 x 97,
// 12 launches) 475 -> 261 us, warped 27 x 19 x 22 N = 4 right-hand side 197 ->
// 104 us.
//
// The energy flux f1 (1 / ((gamma-1) beta_mean) - (|v_a|^2 + |v_b|^2) / 2) / 2 +
// f_m . v_avg, with f_m = f1 v_avg + p_mean n, equals f1 / 2 (1 / ((gamma-1)
// beta_mean) + v_a . v_b) + p_mean v_avg . n: the squares cancel.
//
// Every expression is symmetric in the two nodes, so f(a, b) and f(b, a)
// are the same bits: a kernel may evaluate a pair from either side.
template <int DIM>
DG_HD void flux_chandrashekar(double inv_gm1, const NodePrims<DIM>& a, const NodePrims<DIM>& b,
                              const double* n, double* f) {
  double vs[DIM], vn = 0.0, dot = 0.0;
  for (int k = 0; k < DIM; ++k) {
    vs[k] = a.v[k] + b.v[k];
    vn += vs[k] * n[k];
    dot += a.v[k] * b.v[k];
  }
  const double sr = a.rho + b.rho, sb = a.beta + b.beta;
  const double r = recip(sr * sb);
  const double ib = r * sr;  // 1 / s_beta
  const double xr = (a.rho - b.rho) * (r * sb), xb = (a.beta - b.beta) * ib;
  const double f2r = xr * xr, f2b = xb * xb;
  double P, Q;  // rho_mean = s_rho / 2 P, 1 / beta_mean = 2 Q / s_beta
  if (f2r < 1.0e-4 && f2b < 1.0e-4) {
    P = 1.0 - f2r * (1.0 / 3.0 + f2r * (4.0 / 45.0 + f2r * (44.0 / 945.0)));
    Q = 1.0 + f2b * (1.0 / 3.0 + f2b * (1.0 / 5.0 + f2b * (1.0 / 7.0)));
  } else {
    P = recip(artanh_ratio(a.rho, b.rho, f2r));
    Q = artanh_ratio(a.beta, b.beta, f2b);
  }
  const double hr = 0.5 * sr;
  const double p_mean = hr * ib;
  const double h = 0.25 * (hr * P) * vn;  // f1 / 2, vn = 2 v_avg . n
  f[0] = 2.0 * h;
  for (int k = 0; k < DIM; ++k) f[k + 1] = h * vs[k] + p_mean * n[k];
  f[DIM + 1] = h * (2.0 * inv_gm1 * (ib * Q) + dot) + 0.5 * p_mean * vn;
}

// Primitive quantities of a state read from memory: one reciprocal of rho
// and one square root.
template <int DIM>
DG_HD NodePrims<DIM> face_prims(double gamma, const double* u) {
  NodePrims<DIM> q;
  const double ir = recip(u[0]);
  double v2 = 0.0;
  q.rho = u[0];
  for (int k = 0; k < DIM; ++k) q.v[k] = u[k + 1] * ir;
  for (int k = 0; k < DIM; ++k) v2 += q.v[k] * q.v[k];
  q.p = (gamma - 1.0) * (u[DIM + 1] - 0.5 * u[0] * v2);
  q.c = sqrt(gamma * q.p * ir);
  q.beta = 0.0;
  q.kin = 0.5 * v2;
  return q;
}

// The LLF flux from conservative states and their primitives, as the derivatives in
// physics_ad.hpp are written out.  The kernels evaluate flux_llf; the CPU checks hold
// the derivatives to both.
// 0.5 (F_L + F_R).n - 0.5 lambda (u_R - u_L), lambda = max|v.n| + max(c)|n|
// (numerical_flux.hpp:54-68, compressible_euler3D.hpp:121-166).
template <int DIM>
DG_HD void flux_llf_prims(const double* ul, const NodePrims<DIM>& ql, const double* ur,
                          const NodePrims<DIM>& qr, const double* n, double* f) {
  constexpr int NV = DIM + 2;
  double vnl = 0.0, vnr = 0.0, nn = 0.0;
  for (int k = 0; k < DIM; ++k) {
    vnl += ql.v[k] * n[k];
    vnr += qr.v[k] * n[k];
    nn += n[k] * n[k];
  }
  const double lam = dmax(fabs(vnl), fabs(vnr)) + dmax(ql.c, qr.c) * sqrt(nn);
  double fl[NV], fr[NV];
  fl[0] = ul[0] * vnl;
  fr[0] = ur[0] * vnr;
  for (int k = 0; k < DIM; ++k) {
    fl[k + 1] = ul[k + 1] * vnl + ql.p * n[k];
    fr[k + 1] = ur[k + 1] * vnr + qr.p * n[k];
  }
  fl[NV - 1] = (ul[NV - 1] + ql.p) * vnl;
  fr[NV - 1] = (ur[NV - 1] + qr.p) * vnr;
  for (int i = 0; i < NV; ++i) f[i] = 0.5 * (fl[i] + fr[i]) - 0.5 * lam * (ur[i] - ul[i]);
}

// gradient_variables (rho, v, T = p/rho), compressible_navier_stokes3D.hpp:55-70
template <int DIM>
DG_HD void grad_vars(double gamma, const double* u, double* q) {
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
  const double inv_rho = div_by(1.0, u[0], recip(u[0]));
  double m2 = 0.0;
  for (int k = 0; k < DIM; ++k) m2 += u[k + 1] * u[k + 1];
  const double p = (gamma - 1.0) * (u[DIM + 1] - 0.5 * m2 * inv_rho);
  q[0] = u[0];
  for (int k = 0; k < DIM; ++k) q[k + 1] = u[k + 1] * inv_rho;
  q[DIM + 1] = p * inv_rho;
}

// Newtonian viscous flux in direction dim, compressible_navier_stokes{2D,3D}.hpp
// viscous_flux.  g[c][var] = d q_var / d x_c.
template <int DIM>
DG_HD void viscous_flux_dir(double mu, double kappa, const double* q,
                                                 const double g[DIM][DIM + 2], int dim, double* f) {
#if defined(__clang__)
#pragma clang fp contract(off)
#endif
  auto third = [](double x) { return div_by(x, 3.0, 1.0 / 3.0); };
  if constexpr (DIM == 2) {
    const double tau11 = third(4.0 * g[0][1] - 2.0 * g[1][2]);
    const double tau22 = third(4.0 * g[1][2] - 2.0 * g[0][1]);
    const double tau12 = g[1][1] + g[0][2];
    const double t1 = dim == 0 ? tau11 : tau12, t2 = dim == 0 ? tau12 : tau22;
    f[0] = 0.0;
    f[1] = mu * t1;
    f[2] = mu * t2;
    f[3] = mu * (q[1] * t1 + q[2] * t2 + kappa * g[dim][3]);
  } else {
    const double tau11 = third(4.0 * g[0][1] - 2.0 * (g[1][2] + g[2][3]));
    const double tau22 = third(4.0 * g[1][2] - 2.0 * (g[0][1] + g[2][3]));
    const double tau33 = third(4.0 * g[2][3] - 2.0 * (g[0][1] + g[1][2]));
    const double tau12 = g[1][1] + g[0][2];
    const double tau13 = g[2][1] + g[0][3];
    const double tau23 = g[2][2] + g[1][3];
    const double t1 = dim == 0 ? tau11 : (dim == 1 ? tau12 : tau13);
    const double t2 = dim == 0 ? tau12 : (dim == 1 ? tau22 : tau23);
    const double t3 = dim == 0 ? tau13 : (dim == 1 ? tau23 : tau33);
    f[0] = 0.0;
    f[1] = mu * t1;
    f[2] = mu * t2;
    f[3] = mu * t3;
    f[4] = mu * (q[1] * t1 + q[2] * t2 + q[3] * t3 + kappa * g[dim][4]);
  }
}

// p * rho with gamma fixed at 1.4, the indicator variable of
// subcell_limiting/indicator.hpp:140-215.  The velocities are true quotients,
// so that alpha keeps the reference's bits.
template <int DIM>
DG_HD double indicator_variable(const double* u) {
  const double g = 1.4;
  const double y = recip(u[0]);
  double v2 = 0.0;
  for (int k = 0; k < DIM; ++k) {
    const double v = div_by(u[k + 1], u[0], y);
    v2 += v * v;
  }
  const double p = (g - 1.0) * (u[DIM + 1] - 0.5 * u[0] * v2);
  return p * u[0];
}

}  // namespace dgsem
