// Node-parallel variant of the fused RHS / SSPRK3 stage kernel for
// split-form elements of high polynomial degree, 2D and 3D (periodic
// meshes, no shock capturing).
//
// The line-thread kernel (rhs_kernel) keeps all N+1 node sums of a line in
// registers; at N = 7 in 3D that is 40 accumulators plus the line's metric
// rows, which takes the kernel past 400 registers and down to one wave per
// SIMD.
// Here one workgroup owns one element and one thread owns one node: it
// walks the lines through its node (three in 3D, two in 2D) and sums
// D_split(x, m) f(u_x, u_m)
// over the partners m, evaluating every pair flux itself.  Each pair is thus
// evaluated twice, once from either end (the flux is symmetric in its two
// nodes to the bit, so both ends agree and conservation is exact), but a
// thread holds only its node's five sums and one partner, so the kernel
// fits four waves per SIMD with two elements per CU, and there is no
// cross-thread accumulation: the node's result goes straight from registers
// to memory.  It is bound by instruction issue (the pair fluxes), so what it
// saves is instructions: the shared reciprocals of the pair flux, the face
// fluxes on fully active waves and the staged viscous terms took the 32^3 step
// from 6.72 to 5.02 ms and the 24^3 Navier-Stokes step from 5.61 to 4.12 ms
// (one MI355X), with the same bits.
//
// At N = 7 the split-form sums cancel terms some thousand times larger than
// their result, so the RHS carries the last bits of every term and the
// order of the sums at the 1e-12 level.  This kernel therefore takes each
// node's terms in the reference's order and rounds every operation of the
// pair flux, the face flux and the sums as its scalar code does (true
// quotients, no fused multiply-adds).  Against a scalar restatement of the
// reference's algorithm this kernel stays within a few 1e-13 on the hardest
// small case (TGV, 3x2x4 elements), where the line kernel's faster
// arithmetic is at 2e-12.
//
// Reference kernels replaced: the same as rhs_kernel's split-form path
// (volume_flux.hpp:221-410, surface_flux.hpp:45-271,
// surface_integral.hpp:35-154, jacobian.hpp:22-105, SSPRK3.hpp:12-143).
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "physics.hpp"

namespace dgsem {
namespace detail {

template <int DIM, int N, bool SC, bool BCS>
constexpr bool use_node_kernel() {
  return node_kernel_for(N, SC, BCS);
}

// The functions below round every operation as the reference's scalar code
// does (numerical_flux.hpp:520-594, compressible_euler3D.hpp:26-166,
// math_utils.hpp:8-24): true quotients and no fused multiply-adds.  At high
// degree the split-form sums cancel terms some thousand times larger than
// their result, so the last bits of each pair flux and the order of the sums
// show in the RHS at the 1e-12 level; with the reference's roundings and its
// summation order the kernel reproduces its results.

// Quotients are div_by (physics.hpp): the estimate a y, y within 5e-14 of 1 / b,
// corrected by its residual, which leaves less than 2e-11 of an ulp before the
// final rounding.  A quotient then costs three instructions beside its share of
// a reciprocal, against eleven for the IEEE sequence, with the same bits.

// Sums below run left to right from their first term, as the reference's
// written-out expressions do ((a + b) + c), in 2D and 3D alike.

// rho, v, beta = rho / (2 p), |v|^2 / 2 and p of a conservative state.
template <int DIM>
__device__ __forceinline__ NodePrims<DIM> node_prims_exact(double g, const double* u) {
#pragma clang fp contract(off)
  NodePrims<DIM> q;
  const double y = recip(u[0]);
  q.rho = u[0];
#pragma unroll
  for (int k = 0; k < DIM; ++k) q.v[k] = div_by(u[k + 1], u[0], y);
  double v2 = q.v[0] * q.v[0];
#pragma unroll
  for (int k = 1; k < DIM; ++k) v2 = v2 + q.v[k] * q.v[k];
  q.kin = 0.5 * v2;
  q.p = (g - 1.0) * (u[DIM + 1] - 0.5 * u[0] * v2);
  q.beta = div_by(0.5 * u[0], q.p, recip(q.p));
  q.c = 0.0;  // not needed per node
  return q;
}

// A node of the pair flux: rho / 4, v, beta / 2 and |v|^2 / 2.  Scaling by a
// power of two is exact, so the halvings of the reference's expressions move
// into the stored values and drop out of the flux.
template <int DIM>
struct PairNode {
  double r, v[DIM], b, kin;
};

// Logarithmic mean of lo <= hi by the reference's quotient.
__device__ __forceinline__ double log_mean_exact(double x, double y) {
  const double lo = dmin(x, y), hi = dmax(x, y);
  return (hi - lo) / log(hi / lo);
}

// Chandrashekar flux, symmetric in (a, b) to the bit: the series test uses
// ((x - y) / (x + y))^2 (whose rounding cannot reach the polynomial, which
// is 2 to within 1e-4), and the log branch orders its arguments by value.
// One reciprocal, of s_rho s_beta, serves the two ratios and both quotients by
// s_beta; the reciprocal of a polynomial 1 + f2 / 3 + ... comes from its own
// series.  88 FP64 issue slots a pair, against 125 with a reciprocal estimate
// and refinement for each of the five quotients.  The last component is twice
// the energy flux: its weight takes the half.
template <int DIM>
__device__ __forceinline__ void flux_chandrashekar_exact(double inv_gm1, const PairNode<DIM>& a,
                                                         const PairNode<DIM>& b, const double* n,
                                                         double* f) {
#pragma clang fp contract(off)
  double vna = a.v[0] * n[0], vnb = b.v[0] * n[0];
#pragma unroll
  for (int k = 1; k < DIM; ++k) {
    vna = vna + a.v[k] * n[k];
    vnb = vnb + b.v[k] * n[k];
  }
  const double sr = a.r + b.r, sb = a.b + b.b;  // s_rho / 4, s_beta / 2
  const double rc = recip(sr * sb);
  const double ysb = rc * sr;  // 2 / s_beta
  const double xr = (a.r - b.r) * (rc * sb), xb = (a.b - b.b) * ysb;
  const double f2r = xr * xr, f2b = xb * xb;
  double q, gb;  // rho_mean / 2 and 1 / ((gamma - 1) beta_mean)
  if (f2r < 1.0e-4 && f2b < 1.0e-4) {
    // s_rho / (2 + 2/3 f2 + ...) over 4, 2 and 2
    const double pr = fma(f2r, fma(f2r, fma(f2r, 1.0 / 7.0, 1.0 / 5.0), 1.0 / 3.0), 1.0);
    const double pb = fma(f2b, fma(f2b, fma(f2b, 1.0 / 7.0, 1.0 / 5.0), 1.0 / 3.0), 1.0);
    const double yr = fma(f2r, fma(f2r, -4.0 / 45.0, -1.0 / 3.0), 1.0);  // 1 / pr to 5e-14
    const double yb = fma(f2b, fma(f2b, -4.0 / 45.0, -1.0 / 3.0), 1.0);
    q = div_by(sr, pr, yr);
    const double bm = div_by(sb, pb, yb);
    gb = div_by(inv_gm1, bm, pb * ysb);
  } else {
    const double pr = fma(f2r, fma(f2r, fma(f2r, 1.0 / 7.0, 1.0 / 5.0), 1.0 / 3.0), 1.0);
    const double pb = fma(f2b, fma(f2b, fma(f2b, 1.0 / 7.0, 1.0 / 5.0), 1.0 / 3.0), 1.0);
    q = f2r < 1.0e-4 ? sr / pr : 2.0 * log_mean_exact(a.r, b.r);
    const double bm = f2b < 1.0e-4 ? sb / pb : 2.0 * log_mean_exact(a.b, b.b);
    gb = inv_gm1 / bm;
  }
  const double p_mean = div_by(sr, sb, ysb);
  const double vsq = a.kin + b.kin;
  const double f1 = q * (vna + vnb);
  const double h = 0.5 * f1;
  double fe = f1 * (gb - vsq);
  f[0] = f1;
#pragma unroll
  for (int k = 0; k < DIM; ++k) {
    const double vs = a.v[k] + b.v[k];
    f[k + 1] = h * vs + p_mean * n[k];
    fe = fe + f[k + 1] * vs;
  }
  f[DIM + 1] = fe;
}

// n . (F_1, ..., F_DIM)(u) (compressible_euler2D.hpp:25-57,
// compressible_euler3D.hpp:26-67) and the state's pressure.
template <int DIM>
__device__ __forceinline__ double physical_flux_exact(double g, const double* u, const double* n,
                                                      double* f) {
#pragma clang fp contract(off)
  constexpr int NV = DIM + 2;
  double v[DIM];
  const double y = recip(u[0]);
#pragma unroll
  for (int k = 0; k < DIM; ++k) v[k] = div_by(u[k + 1], u[0], y);
  double v2 = v[0] * v[0];
#pragma unroll
  for (int k = 1; k < DIM; ++k) v2 = v2 + v[k] * v[k];
  const double p = (g - 1.0) * (u[NV - 1] - 0.5 * u[0] * v2);
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    double fd[NV];
    fd[0] = u[d + 1];
#pragma unroll
    for (int k = 0; k < DIM; ++k) fd[k + 1] = k == d ? u[d + 1] * v[k] + p : u[d + 1] * v[k];
    fd[NV - 1] = v[d] * (u[NV - 1] + p);
#pragma unroll
    for (int i = 0; i < NV; ++i) f[i] = d == 0 ? n[0] * fd[i] : f[i] + n[d] * fd[i];
  }
  return p;
}

// Local Lax-Friedrichs flux from conservative states (numerical_flux.hpp:54-68
// with compressible_euler{2D,3D}.hpp get_wave_speed).
template <int DIM>
__device__ __forceinline__ void flux_llf_exact(double g, const double* ul, const double* ur,
                                               const double* n, double* f) {
#pragma clang fp contract(off)
  constexpr int NV = DIM + 2;
  double fl[NV], fr[NV], vn[2], a[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const double* u = s == 0 ? ul : ur;
    const double p = physical_flux_exact<DIM>(g, u, n, s == 0 ? fl : fr);
    const double y = recip(u[0]);
    a[s] = sqrt(div_by(g * p, u[0], y));
    double vnn = div_by(u[1], u[0], y) * n[0];
#pragma unroll
    for (int k = 1; k < DIM; ++k) vnn = vnn + div_by(u[k + 1], u[0], y) * n[k];
    vn[s] = vnn;
  }
  double nn2 = n[0] * n[0];
#pragma unroll
  for (int k = 1; k < DIM; ++k) nn2 = nn2 + n[k] * n[k];
  const double lam = dmax(fabs(vn[0]), fabs(vn[1])) + dmax(a[0], a[1]) * sqrt(nn2);
#pragma unroll
  for (int v = 0; v < NV; ++v) f[v] = 0.5 * (fl[v] + fr[v]) - 0.5 * lam * (ur[v] - ul[v]);
}

// HLLC flux with a normal vector (a build extension: the reference has
// HLLC for 1D Euler only, numerical_flux.hpp:283-378, whose structure this
// follows in the frame of the unit normal, scaled by |n|).
template <int DIM>
__device__ __forceinline__ void flux_hllc_exact(double g, const double* ul, const double* ur,
                                                const double* n, double* f) {
#pragma clang fp contract(off)
  constexpr int NV = DIM + 2;
  double nh[DIM], vl[DIM], vr[DIM], fl[NV], fr[NV];
  double nn2 = n[0] * n[0];
#pragma unroll
  for (int k = 1; k < DIM; ++k) nn2 = nn2 + n[k] * n[k];
  const double nrm = sqrt(nn2);
#pragma unroll
  for (int d = 0; d < DIM; ++d) nh[d] = n[d] / nrm;
  const double rho_ll = ul[0], rho_rr = ur[0], rhoE_ll = ul[NV - 1], rhoE_rr = ur[NV - 1];
  const double yl = recip(rho_ll), yr = recip(rho_rr);
  double v2l = 0.0, v2r = 0.0, vn_l = 0.0, vn_r = 0.0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    vl[d] = div_by(ul[d + 1], rho_ll, yl);
    vr[d] = div_by(ur[d + 1], rho_rr, yr);
    v2l += vl[d] * vl[d];
    v2r += vr[d] * vr[d];
    vn_l += vl[d] * nh[d];
    vn_r += vr[d] * nh[d];
  }
  const double E_ll = rhoE_ll / rho_ll, E_rr = rhoE_rr / rho_rr;
  const double p_ll = (g - 1.0) * (rhoE_ll - 0.5 * rho_ll * v2l);
  const double p_rr = (g - 1.0) * (rhoE_rr - 0.5 * rho_rr * v2r);
  const double c_ll = sqrt(g * p_ll / rho_ll), c_rr = sqrt(g * p_rr / rho_rr);
  physical_flux_exact<DIM>(g, ul, nh, fl);
  physical_flux_exact<DIM>(g, ur, nh, fr);
  const double srl = sqrt(rho_ll), srr = sqrt(rho_rr), ssum = srl + srr;
  double vroe2 = 0.0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const double vroe_d = (srl * vl[d] + srr * vr[d]) / ssum;
    vroe2 += vroe_d * vroe_d;
  }
  const double vel_roe = (srl * vn_l + srr * vn_r) / ssum;
  const double ekin_roe = 0.5 * vroe2;
  const double H_ll = (rhoE_ll + p_ll) / rho_ll, H_rr = (rhoE_rr + p_rr) / rho_rr;
  const double H_roe = (srl * H_ll + srr * H_rr) / ssum;
  const double c_roe = sqrt((g - 1.0) * (H_roe - ekin_roe));
  const double Ssl = dmin(vn_l - c_ll, vel_roe - c_roe);
  const double Ssr = dmax(vn_r + c_rr, vel_roe + c_roe);
  const double sMu_L = Ssl - vn_l, sMu_R = Ssr - vn_r;
  if (Ssl >= 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) f[i] = fl[i];
  } else if (Ssr <= 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) f[i] = fr[i];
  } else {
    const double SStar = (p_rr - p_ll + rho_ll * vn_l * sMu_L - rho_rr * vn_r * sMu_R) /
                         (rho_ll * sMu_L - rho_rr * sMu_R);
    const bool left = SStar >= 0;
    const double* uk = left ? ul : ur;
    const double* fk = left ? fl : fr;
    const double* vk = left ? vl : vr;
    const double rk = left ? rho_ll : rho_rr, vnk = left ? vn_l : vn_r;
    const double Ek = left ? E_ll : E_rr, pk = left ? p_ll : p_rr;
    const double Sk = left ? Ssl : Ssr, sMu = left ? sMu_L : sMu_R;
    const double densStar = rk * sMu / (Sk - SStar);
    const double enerStar = Ek + (SStar - vnk) * (SStar + pk / (rk * sMu));
    f[0] = fk[0] + Sk * (densStar - uk[0]);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const double mstar = densStar * (vk[d] + (SStar - vnk) * nh[d]);
      f[d + 1] = fk[d + 1] + Sk * (mstar - uk[d + 1]);
    }
    f[NV - 1] = fk[NV - 1] + Sk * (densStar * enerStar - uk[NV - 1]);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) f[i] *= nrm;
}

// The face fluxes of an element, one per line end, and the rounds in which its NN
// threads form them: thread a takes line end a + k NN in round k.  From N = 5 in 3D
// and N = 3 in 2D on there is a thread for each; a kernel built for lower degrees
// (DGSEM_NODE_KERNEL_MIN_N) takes further rounds.
template <int DIM, int N>
struct NodeFaces {
  static constexpr int NN = Shape<DIM, N>::NN, COUNT = 2 * DIM * Shape<DIM, N>::FN;
  static constexpr int ROUNDS = (COUNT + NN - 1) / NN;
};

template <int DIM, int N, bool NODAL, int SF>
__global__ void __launch_bounds__((Shape<DIM, N>::NN)) __attribute__((amdgpu_waves_per_eu(4)))
    rhs_node_kernel(const KParams p) {
  constexpr int n = N + 1, NV = DIM + 2, NN = Shape<DIM, N>::NN;
  constexpr int PN = NN + NN / n;  // padded plane (lds_pos)
  constexpr int DS = n + 1;        // padded row of the D_split table
  constexpr int QB = DIM + 1;      // plane of beta; kin follows
  constexpr int FN = Shape<DIM, N>::FN;
  using Faces = NodeFaces<DIM, N>;
  // LDS planes: rho, v[DIM], beta, kin, then (NODAL) Ja^d_c / 2.  Once the term
  // loops are done with them they take the face fluxes (FPL planes) and the
  // viscous fluxes (VPL planes: the mass component is zero).
  constexpr int QPL = DIM + 3, FPL = (Faces::COUNT * NV + PN - 1) / PN, VPL = DIM * (NV - 1);
  constexpr int JPL = NODAL ? DIM * DIM : 0;
  constexpr int PLANES = QPL + JPL > FPL + VPL ? QPL + JPL : FPL + VPL;
  __shared__ double s_q[PLANES * PN];
  double* const s_ja = s_q + QPL * PN;
  double* const s_face = s_q;                 // [dir][side][var][line]
  double* const s_vf = s_q + FPL * PN;        // [dir][var - 1][node], padded
  __shared__ double s_D[n * DS];
  __shared__ double s_Dh[n * DS];  // D_hat (Navier-Stokes viscous terms)

  const int a = threadIdx.x;
  const int64_t e = xcd_block(blockIdx.x, gridDim.x);
  const int idx[3] = {a % n, (a / n) % n, DIM == 3 ? a / (n * n) : 0};
  constexpr int stride[3] = {1, n, n * n};
  const int pa = lds_pos<N>(a);
  int eid[3];
  element_indices<DIM>(p, (int)e, eid);

  // 1. the node's state, metric rows and 1/J (the face data follows the
  // term loops, phase 4)
  double u[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) u[v] = p.u[(e * NV + v) * NN + a];
  double jm[DIM][DIM];
#pragma unroll
  for (int d = 0; d < DIM; ++d)
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      jm[d][c] = NODAL ? p.Ja[((e * DIM + d) * DIM + c) * NN + a] : p.Ja[(e * DIM + d) * DIM + c];
  const double ij = NODAL ? p.invJ[e * NN + a] : p.invJ[e];

  // 2. the node's primitives and halved metric rows into LDS
  const NodePrims<DIM> q = node_prims_exact<DIM>(p.gamma, u);
  PairNode<DIM> qa;  // scaled as the flux takes it
  qa.r = 0.25 * q.rho;
#pragma unroll
  for (int c = 0; c < DIM; ++c) qa.v[c] = q.v[c];
  qa.b = 0.5 * q.beta;
  qa.kin = q.kin;
  s_q[pa] = qa.r;
#pragma unroll
  for (int c = 0; c < DIM; ++c) s_q[(1 + c) * PN + pa] = qa.v[c];
  s_q[QB * PN + pa] = qa.b;
  s_q[(QB + 1) * PN + pa] = qa.kin;
  if constexpr (NODAL) {
#pragma unroll
    for (int d = 0; d < DIM; ++d)
#pragma unroll
      for (int c = 0; c < DIM; ++c) s_ja[(d * DIM + c) * PN + pa] = 0.5 * jm[d][c];
  }
  if (a < n * n) {
    s_D[(a / n) * DS + a % n] = p.basis[a];
    s_Dh[(a / n) * DS + a % n] = p.basis[n * n + a];
  }
  __syncthreads();

  // 3. flux differencing.  The reference (volume_flux.hpp:296-410) visits
  // the nodes in memory order and adds each pair's two terms as it goes, so
  // a node's sum takes its terms in the order: partners below it on its
  // z-line, y-line and x-line, then partners above it on its x-, y- and
  // z-lines, each line in increasing position.  Every node has 3N terms, so
  // each lane walks its own sequence in one uniform loop, and the face terms
  // follow in direction order (surface_integral.hpp:82-154).
  const int ix = idx[0], iy = idx[1], iz = idx[2];
  double acc[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) acc[v] = 0.0;
  // One term D_split(x_d, m) f(u_a, u_b) of line direction d, partner m at LDS
  // position pb.  The node's own metric row is read again from LDS for each
  // term (affine: the element's, from the registers): selecting it from
  // registers by the lane's direction costs more than the three reads.
  auto term = [&](int d, int xd, int m, int pb) {
    PairNode<DIM> qb;
    qb.r = s_q[pb];
#pragma unroll
    for (int c = 0; c < DIM; ++c) qb.v[c] = s_q[(1 + c) * PN + pb];
    qb.b = s_q[QB * PN + pb];
    qb.kin = s_q[(QB + 1) * PN + pb];
    double nrm[DIM], f[NV];
    if constexpr (NODAL) {
      // (Ja_x + Ja_m) / 2 from the halved rows (halving is exact)
      const double* row = s_ja + d * (DIM * PN);
#pragma unroll
      for (int c = 0; c < DIM; ++c) nrm[c] = row[c * PN + pa] + row[c * PN + pb];
    } else {
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        nrm[c] = d == 0 ? jm[0][c] : jm[1][c];
        if constexpr (DIM == 3) nrm[c] = d == 2 ? jm[2][c] : nrm[c];
      }
    }
    const double w = s_D[xd * DS + m];
    flux_chandrashekar_exact<DIM>(p.inv_gm1, qa, qb, nrm, f);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
#pragma clang fp contract(off)
      acc[v] = acc[v] + (v == NV - 1 ? 0.5 * w : w) * f[v];
    }
  };
  // LDS positions of the node's lines' first nodes and their strides
  constexpr int PY = n + 1, PZ = n * (n + 1);
  const int xb = pa - ix, yb = pa - iy * PY, zb = DIM == 3 ? pa - iz * PZ : 0;
  // partners below on the z-line (3D)
  if constexpr (DIM == 3) {
#pragma unroll 1
    for (int m = 0; m < iz; ++m) term(2, iz, m, zb + m * PZ);
  }
  // The lane's y- and x-lines: below on the y-line, below and above on the x-line,
  // above on the y-line (2N terms for every node).  A term is set up with selects
  // only, and its weight read beside the partner: branches and a late read there
  // cost a 2D grid that leaves the SIMDs a wave each 7% (2D, 8 x 8, N = 7, us a
  // step: LLF 54.1 -> 50.7, HLLC 57.0 -> 53.4; 3D 32^3 5082 -> 5042).
#pragma unroll 1
  for (int t = 0; t < 2 * N; ++t) {
    const bool below = t < iy, dy = below || t >= iy + N;
    const int skip_y = below ? 0 : N - 1, skip_x = t < iy + ix ? iy : iy - 1;
    const int m = t - (dy ? skip_y : skip_x);
    const int first = dy ? yb : xb, step = dy ? PY : 1;
    term(dy ? 1 : 0, dy ? iy : ix, m, first + m * step);
  }
  // partners above on the z-line (3D)
  if constexpr (DIM == 3) {
#pragma unroll 1
    for (int m = iz + 1; m <= N; ++m) term(2, iz, m, zb + m * PZ);
  }

  // 4. numerical fluxes on the element's faces, one thread for each line end:
  // item (dir, side, line) to a thread (NodeFaces), so that a wave takes one side
  // of one direction (3D) and every lane works.  Formed by the face
  // nodes' own threads they ran once per direction in every wave, a quarter of
  // its lanes active.  The lower face takes the lower neighbour's node with
  // index N, the upper face the upper neighbour's node with index 0 and its
  // metric row and 1/J, whose sign and row make the interface normal.
  {
    double f[Faces::ROUNDS][NV];
#pragma unroll
    for (int k = 0; k < Faces::ROUNDS; ++k) {
      const int t = a + k * NN;
      if (t >= Faces::COUNT) break;
      const int fd = t / (2 * FN), rem = t - fd * (2 * FN), line = rem % FN;
      const bool lower = rem < FN;
      const LineNodes<DIM, N> ln(fd, line);
      const int first = ln.base, last = ln.base + N * ln.stride;
      int64_t lo, hi;
      face_neighbours<DIM, false>(p, eid, e, fd, lo, hi);
      const int64_t ne = lower ? lo : hi;
      const int on = lower ? first : last, nn = lower ? last : first;
      const double* uo = p.u + e * (NV * NN) + on;
      const double* un = p.u + ne * (NV * NN) + nn;
      // the face's upper element, whose first node makes the normal
      const int64_t ue = lower ? e : hi;
      const double uij = NODAL ? p.invJ[ue * NN + first] : p.invJ[ue];
      const double sg = uij >= 0.0 ? 1.0 : -1.0;
      double so[NV], sn[NV], ul[NV], ur[NV], nrm[DIM];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        so[v] = uo[v * NN];
        sn[v] = un[v * NN];
      }
#pragma unroll
      for (int c = 0; c < DIM; ++c)
        nrm[c] = sg * (NODAL ? p.Ja[((ue * DIM + fd) * DIM + c) * NN + first]
                             : p.Ja[(ue * DIM + fd) * DIM + c]);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        ul[v] = lower ? sn[v] : so[v];
        ur[v] = lower ? so[v] : sn[v];
      }
      if constexpr (SF == kFluxLLF) {
        flux_llf_exact<DIM>(p.gamma, ul, ur, nrm, f[k]);
      } else {
        flux_hllc_exact<DIM>(p.gamma, ul, ur, nrm, f[k]);
      }
    }
    __syncthreads();  // the term loops are done with the primitives
#pragma unroll
    for (int k = 0; k < Faces::ROUNDS; ++k) {
      const int t = a + k * NN;
      if (t >= Faces::COUNT) break;
      const int face = t / FN, line = t % FN;  // face = 2 dir + upper
#pragma unroll
      for (int v = 0; v < NV; ++v) s_face[(face * NV + v) * FN + line] = f[k][v];
    }
  }

  // 3b. Navier-Stokes: the viscous volume integral adds
  // D_hat(x_d, m) Ja^d . (-F_v)(m) over every partner m of each line through
  // the node (the node itself included) into the same sums, after the
  // split-form terms (parabolic_viscous.hpp:103-163 3D, :412-447 2D).  It
  // visits the source nodes in memory order, so a node takes: sources below
  // it on its z-line and y-line, its x-line up to itself, its own y and z
  // terms, then the rest of its x-, y- and z-lines.  At a face node the sums
  // hold the uncancelled half of the face balance, about a thousand times
  // the RHS, so this order fixes the RHS's last bits whatever the viscosity.
  // The element's fluxes are staged in the planes the term loops have left;
  // the mass component is zero and adds nothing.
  const double* vf = p.visc;  // [E][d][var][dof], or null (Euler)
  if (vf) {
    double own[DIM][NV - 1];
#pragma unroll
    for (int d = 0; d < DIM; ++d)
#pragma unroll
      for (int v = 1; v < NV; ++v) own[d][v - 1] = vf[((e * DIM + d) * NV + v) * NN + a];
#pragma unroll
    for (int d = 0; d < DIM; ++d)
#pragma unroll
      for (int v = 1; v < NV; ++v) s_vf[(d * (NV - 1) + v - 1) * PN + pa] = own[d][v - 1];
  }
  __syncthreads();
  if (vf) {
    auto vterm = [&](int d, int xd, int m, int pb) {
      const double w = s_Dh[xd * DS + m];
      const double* g = s_vf + d * ((NV - 1) * PN) + pb;
#pragma unroll
      for (int v = 1; v < NV; ++v) {
#pragma clang fp contract(off)
        acc[v] = acc[v] + w * g[(v - 1) * PN];
      }
    };
    if constexpr (DIM == 3) {
#pragma unroll 1
      for (int m = 0; m < iz; ++m) vterm(2, iz, m, zb + m * PZ);
    }
    // y below, x up to the node, the node's own y and z, the rest of x and y:
    // the same terms as above with the node itself among them
#pragma unroll 1
    for (int t = 0; t <= iy + ix; ++t) {
      const bool dy = t < iy;
      const int m = dy ? t : t - iy;
      vterm(dy ? 1 : 0, dy ? iy : ix, m, dy ? yb + m * PY : xb + m);
    }
    vterm(1, iy, iy, pa);
    if constexpr (DIM == 3) vterm(2, iz, iz, pa);
#pragma unroll 1
    for (int t = 0; t < 2 * N - ix - iy; ++t) {
      const bool dy = t >= N - ix;
      const int m = dy ? iy + 1 + t - (N - ix) : ix + 1 + t;
      vterm(dy ? 1 : 0, dy ? iy : ix, m, dy ? yb + m * PY : xb + m);
    }
    if constexpr (DIM == 3) {
#pragma unroll 1
      for (int m = iz + 1; m <= N; ++m) vterm(2, iz, m, zb + m * PZ);
    }
    // 3c. the viscous interface terms in direction order
    // (structured_solver.hpp:359-360 with the one-sided flux of
    // parabolic_viscous.hpp:318-334 / :570-585): the lower face takes the
    // node's own (-F_v) . (sign(J) Ja^d), the upper face the upper
    // neighbour's at its node with index 0.
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const bool lower = idx[d] == 0, upper = idx[d] == N;
      if (lower || upper) {
        int64_t lo, hi;
        face_neighbours<DIM, false>(p, eid, e, d, lo, hi);
        const int64_t ve = lower ? e : hi;
        const int vn = lower ? a : a - N * stride[d];
        const double vij = lower ? ij : (NODAL ? p.invJ[ve * NN + vn] : p.invJ[ve]);
        const double sg = vij >= 0.0 ? 1.0 : -1.0;
#pragma unroll
        for (int v = 1; v < NV; ++v) {
#pragma clang fp contract(off)
          const double fp = sg * vf[((ve * DIM + d) * NV + v) * NN + vn];
          acc[v] = lower ? acc[v] - fp * p.lhat0 : acc[v] + fp * p.lhatN;
        }
      }
    }
  }
  // 4b. the face fluxes, lifted in direction order
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const bool lower = idx[d] == 0, upper = idx[d] == N;
    if (lower || upper) {
      // line of the node in direction d
      const int line = DIM == 2 ? idx[1 - d]
                                : idx[d == 2 ? 1 : 2] * n + idx[d == 0 ? 1 : 0];
      const double* f = s_face + (d * 2 + (lower ? 0 : 1)) * (NV * FN) + line;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
#pragma clang fp contract(off)
        acc[v] = lower ? acc[v] - f[v * FN] * p.lhat0 : acc[v] + f[v * FN] * p.lhatN;
      }
    }
  }
  const double* tot = acc;

  // 5. -1/J and the stage combination.  1/J, the base
  // state and the result are touched once per launch: non-temporal accesses
  // keep them from displacing the neighbours' face traces in the L2.
  const int64_t g = e * NV * NN + a;
  const double fac = -ij;
  // the base state's loads go out together (a select between the stage
  // kinds inside the variable loop would serialise them)
  const bool with_base = p.mode == kModeStage3;
  double ub[NV];
  if (with_base) {
#pragma unroll
    for (int v = 0; v < NV; ++v) ub[v] = __builtin_nontemporal_load(&p.u_base[g + v * NN]);
  }
  double uk[NV];  // the stage input, reloaded (an L2 hit) rather than held
#pragma unroll
  for (int v = 0; v < NV; ++v) uk[v] = p.u[g + v * NN];
  double r[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) r[v] = tot[v] * fac;
  if (p.mode == kModeRhs) {
#pragma unroll
    for (int v = 0; v < NV; ++v) __builtin_nontemporal_store(r[v], &p.out[g + v * NN]);
  } else {
    // the stage combinations of SSPRK3.hpp:12-143, rounded term by term
    double s[NV];
    if (with_base) {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
#pragma clang fp contract(off)
        s[v] = p.c1 * ub[v] + p.c2 * uk[v] + p.c3 * r[v];
      }
    } else {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
#pragma clang fp contract(off)
        s[v] = p.c1 * uk[v] + p.c2 * r[v];
      }
    }
    if (p.floor_value > 0.0) {
      if (s[0] < p.floor_value) s[0] = p.floor_value;
      double m2 = 0.0;
      for (int k = 0; k < DIM; ++k) m2 += s[k + 1] * s[k + 1];
      const double kin = 0.5 * m2 / s[0];
      if ((p.gamma - 1.0) * (s[NV - 1] - kin) < p.floor_value)
        s[NV - 1] = p.floor_value / (p.gamma - 1.0) + kin;
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) __builtin_nontemporal_store(s[v], &p.out[g + v * NN]);
  }
}

template <int DIM, int N, bool NODAL, int SF>
hipError_t launch_node_kernel(const KParams& p, hipStream_t stream) {
  constexpr int NN = Shape<DIM, N>::NN;
  if (p.E <= 0) return hipSuccess;
  if (p.E > INT32_MAX) return hipErrorInvalidValue;
  hipLaunchKernelGGL((rhs_node_kernel<DIM, N, NODAL, SF>), dim3((unsigned)p.E), dim3(NN), 0, stream,
                     p);
  return hipGetLastError();
}

}  // namespace detail
}  // namespace dgsem
