// BR1 parabolic terms of the compressible Navier-Stokes RHS on the GPU.
//
// One kernel before the inviscid one forms the contravariant viscous flux
// Ja^d . (-F_v) at every node: q = (rho, v, T); along each line the weak
// derivative D_hat q, the BR1 face value q_hat = (q_L + q_R)/2 lifted with
// l_hat; the physical gradient sum_d Ja^d (.) / J; the flux.  The gradient
// itself never goes to memory, nor does anything of rho, which the viscous
// flux does not differentiate, nor the flux's zero mass component.  Reference:
// GradientVolumeIntegralFunctor, GradientPhysicalTransformFunctor,
// GradientInterfaceFluxFunctor, GradientSurfaceIntegralFunctor,
// GradientJacobianProjFunctor (parabolic_gradient.hpp:17-478 3D, :480-818 2D)
// and ViscousFluxFunctor (parabolic_viscous.hpp:39-66 3D, :367-386 2D).
//   * viscous_flux_kernel: line threads, for the line kernels (rhs_kernel),
//     whose line threads form the flux's D_hat divergence and the interface
//     flux, the upper ("primary") element's (-F_v).n only
//     (parabolic_viscous.hpp:318-334 3D, :570-585 2D), beside the pair fluxes.
//     Layout [E][d][var][line * n + k]: node k of line `line` of direction d,
//     so that a line thread reads contiguous runs.
//   * gradient_node_kernel: for the elements of the node-parallel RHS kernel
//     (node_kernel_for), rounded as the reference; layout [E][d][var][dof].
// The tangent and adjoint kernels (adjoint_impl.hpp) form the gradient they
// linearise at themselves, with line_gradient.
// BCS (2D): some face is not periodic; face_neighbours gives -1 there and the
// face values come from the boundary condition (wall_gradient_value and
// rhs_kernel's wall branch).
#pragma once

#include <hip/hip_runtime.h>

#include "kernels.hpp"
#include "physics.hpp"
#include "rhs_kernel_impl.hpp"

namespace dgsem {
namespace detail {

// grad_vars and viscous_flux_dir (the pointwise gradient variables and
// viscous flux) live in physics.hpp, shared with the host-side traits.

template <bool NODAL, int DIM, int NN>
__device__ __forceinline__ double metric(const KParams& p, int64_t e, int r, int c, int dof) {
  if constexpr (NODAL)
    return p.Ja[((e * DIM + r) * DIM + c) * NN + dof];
  else
    return p.Ja[(e * DIM + r) * DIM + c];
}

template <bool NODAL, int NN>
__device__ __forceinline__ double inv_jac(const KParams& p, int64_t e, int dof) {
  if constexpr (NODAL)
    return p.invJ[e * NN + dof];
  else
    return p.invJ[e];
}

// Gradient face value at a boundary node: the adiabatic walls take the inner
// gradient variables q with the velocity set to zero (no slip,
// navier_stokes_wall_boundary.hpp:81-114) or with its component along the
// normal nrm = sign(J) Ja^dir removed (slip, :163-197 and :28-36).
// Dirichlet faces take the outer state's variables (computed by the caller,
// dirichlet_boundary.hpp:122-162).  Kinds without a gradient hook
// (boundary_set.hpp:16-33) leave the face value at zero, as the reference's
// cleared face array does.
template <int DIM>
__device__ __forceinline__ void wall_gradient_value(int kind, const double* q, const double* nrm,
                                                    double* qw) {
  constexpr int NV = DIM + 2;
  static_assert(DIM == 2, "non-periodic boundaries are built for 2D meshes");
  if (kind == kBcNsNoSlipWall) {
    qw[0] = q[0];
    qw[1] = 0.0;
    qw[2] = 0.0;
    qw[3] = q[3];
  } else if (kind == kBcNsSlipWall) {
    const double nn = nrm[0] * nrm[0] + nrm[1] * nrm[1];
    const double vn = (q[1] * nrm[0] + q[2] * nrm[1]) / nn;
    qw[0] = q[0];
    qw[1] = q[1] - vn * nrm[0];
    qw[2] = q[2] - vn * nrm[1];
    qw[3] = q[3];
  } else {
#pragma unroll
    for (int v = 0; v < NV; ++v) qw[v] = 0.0;
  }
}

// Position of node `dof` in the direction-d rows line * n + k (LineNodes).
template <int DIM, int N>
__device__ __forceinline__ int row_pos(int d, int dof) {
  constexpr int n = N + 1;
  if (d == 0) return dof;
  const int ix = dof % n, iy = (dof / n) % n, iz = dof / (n * n);
  if constexpr (DIM == 2) return ix * n + iy;
  return d == 1 ? (iz * n + ix) * n + iy : (iy * n + ix) * n + iz;
}

// Metric terms Ja^d_c of a node, from the box table (rows of halved terms) or
// the per-node arrays.
template <int DIM, int N, bool NODAL, bool BOX>
__device__ __forceinline__ void node_metric(const KParams& p, int64_t e, const int* eid, int dof,
                                            double ja[DIM][DIM]) {
  constexpr int NN = Shape<DIM, N>::NN;
#pragma unroll
  for (int d = 0; d < DIM; ++d)
#pragma unroll
    for (int c = 0; c < DIM; ++c)
      ja[d][c] = BOX ? 2.0 * box_row<DIM, N>(p, eid, c, d, 0)[row_pos<DIM, N>(d, dof)]
                     : metric<NODAL, DIM, NN>(p, e, d, c, dof);
}

// The weak derivative of the variables v, T along one line, with the BR1 face
// values lifted: acc = D_hat x -+ l_hat sign(J) q_hat, q_hat = (q_L + q_R) / 2 on
// both line ends.  x[k][v - 1]: the line's variables; q_lo, q_hi: the
// neighbours' (NV values, from grad_vars; overwritten); blo, bhi: the end is a
// boundary face, whose value comes from the boundary condition; sg_*: sign(J) at
// the line's end nodes (the face terms use the element's own normal).
template <int DIM, int N, bool NODAL, bool BCS, class Ops>
__device__ __forceinline__ void line_gradient(const KParams& p, const Ops& op, int64_t el,
                                              const int* eid, int dl, int line, int first, int last,
                                              const double (&x)[N + 1][DIM + 1], double* q_lo,
                                              double* q_hi, bool blo, bool bhi, double sg_lo,
                                              double sg_hi, double (&acc)[N + 1][DIM + 1]) {
  constexpr int n = N + 1, NV = DIM + 2, ND = NV - 1, NN = Shape<DIM, N>::NN;
#pragma unroll
  for (int k = 0; k < n; ++k)
#pragma unroll
    for (int v = 0; v < ND; ++v) {
      double r = 0.0;
#pragma unroll
      for (int i = 0; i < n; ++i) r += op.Dhat(k, i) * x[i][v];
      acc[k][v] = r;
    }
#pragma unroll
  for (int v = 1; v < NV; ++v) {
    q_lo[v] = 0.5 * (q_lo[v] + x[0][v - 1]);
    q_hi[v] = 0.5 * (x[n - 1][v - 1] + q_hi[v]);
  }
  if constexpr (BCS) {
    auto wall = [&](int side, int dof, double sg, const double* xn, double* out) {
      const int face = 2 * dl + side;
      if (p.bc[face] == kBcDirichlet) {
        const int64_t bnode = (int64_t)(dl == 0 ? eid[1] : eid[0]) * n + line;
        const double* vals = p.bc_values[face];
        double so[NV];
        for (int v = 0; v < NV; ++v) so[v] = vals ? vals[bnode * NV + v] : p.bc_state[face][v];
        grad_vars<DIM>(p.gamma, so, out);
      } else {
        double own[NV], nrm[DIM];
        own[0] = 0.0;  // rho: not differentiated
        for (int v = 1; v < NV; ++v) own[v] = xn[v - 1];
        for (int c = 0; c < DIM; ++c) nrm[c] = sg * metric<NODAL, DIM, NN>(p, el, dl, c, dof);
        wall_gradient_value<DIM>(p.bc[face], own, nrm, out);
      }
    };
    if (blo) wall(0, first, sg_lo, x[0], q_lo);
    if (bhi) wall(1, last, sg_hi, x[n - 1], q_hi);
  }
#pragma unroll
  for (int v = 1; v < NV; ++v) {
    acc[0][v - 1] -= sg_lo * p.lhat0 * q_lo[v];
    acc[n - 1][v - 1] += sg_hi * p.lhatN * q_hi[v];
  }
}

// The nodes' viscous fluxes into p.visc_out (see the top of the file).  Memory
// bound: a node reads its state (and, off a box mesh, its metric terms) and
// writes DIM (DIM + 1) fluxes.  Whole-node staging, line threads and LDS planes
// as in rhs_kernel; the line derivatives take the place of q in LDS, so that
// five blocks of the 3D N = 3 kernel fit a CU.  Storing the fluxes instead of
// the gradient, with the divergence in rhs_kernel, replaced a gradient and a
// viscous-divergence kernel (85 -> 46 doubles of traffic per node and stage on a
// box mesh): SSPRK3 step at 32^3 N = 3 1.10 -> 0.57 ms, 2D shock tube 200 x 100
// N = 3 with walls, 12 stages, 468 -> 316 us.
template <int DIM, int N, int EPW, bool NODAL, bool BCS, bool BOX>
__global__ void __launch_bounds__((EPW * Shape<DIM, N>::LINES)) viscous_flux_kernel(const KParams p) {
  using S = Shape<DIM, N>;
  constexpr int n = S::n, NV = S::NV, NN = S::NN, FN = S::FN, PN = S::PN;
  constexpr int ND = NV - 1;  // differentiated variables v, T: planes v - 1
  constexpr int BLOCK = EPW * S::LINES, NODES = EPW * NN, PASSES = (NODES + BLOCK - 1) / BLOCK;
  constexpr int SG = DIM * ND * PN + S::slot_pad(DIM * ND * PN);
  __shared__ double s_g[EPW * SG];  // q [var], later D_hat q + lift [dir][var]
  const int tid = threadIdx.x;
  const int64_t e0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * EPW;
  const int nvalid = (int)((p.E - e0) < EPW ? (p.E - e0) : EPW);
  auto has_node = [&](int k) { return (k + 1) * BLOCK <= NODES || tid + k * BLOCK < NODES; };

  // node states; slots past the last valid element take a copy of it
  double q[PASSES][NV];
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (has_node(k)) {
      const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN;
      const double* src = p.u + (e0 + (sl < nvalid ? sl : nvalid - 1)) * (NV * NN) + node;
#pragma unroll
      for (int v = 0; v < NV; ++v) q[k][v] = src[v * NN];
    }
  }
  // the line and its neighbours' traces, threads ordered (dir, slot, line)
  const int dir = tid / (EPW * FN), rem = tid % (EPW * FN), slot = rem / FN, line = rem % FN;
  const bool valid = slot < nvalid && dir < DIM;
  const int64_t el = valid ? e0 + slot : e0;
  const int dl = dir < DIM ? dir : DIM - 1;
  const LineNodes<DIM, N> ln(dl, line);
  const int first = ln.base, last = ln.base + N * ln.stride;
  int eid[3];
  element_indices<DIM>(p, (int)el, eid);
  int64_t nb_lo, nb_hi;
  face_neighbours<DIM, BCS>(p, eid, el, dl, nb_lo, nb_hi);
  const bool blo = BCS && nb_lo < 0, bhi = BCS && nb_hi < 0;
  double t_lo[NV], t_hi[NV];
  {
    const double* ulo = p.u + (blo ? el : nb_lo) * (NV * NN) + last;
    const double* uhi = p.u + (bhi ? el : nb_hi) * (NV * NN) + first;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      t_lo[v] = ulo[v * NN];
      t_hi[v] = uhi[v * NN];
    }
  }
  const double sg_lo = BOX || inv_jac<NODAL, NN>(p, el, first) >= 0.0 ? 1.0 : -1.0;
  const double sg_hi = BOX || inv_jac<NODAL, NN>(p, el, last) >= 0.0 ? 1.0 : -1.0;
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (has_node(k)) {
      const int i = tid + k * BLOCK, sl = i / NN, pn = lds_pos<N>(i - sl * NN);
      double u[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) u[v] = q[k][v];
      grad_vars<DIM>(p.gamma, u, q[k]);
#pragma unroll
      for (int v = 1; v < NV; ++v) s_g[sl * SG + (v - 1) * PN + pn] = q[k][v];
    }
  }
  __syncthreads();
  double acc[n][ND];
  {
    double x[n][ND];
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) x[k][v] = s_g[slot * SG + v * PN + ln.pbase + k * ln.pstride];
    double q_lo[NV], q_hi[NV];
    grad_vars<DIM>(p.gamma, t_lo, q_lo);
    grad_vars<DIM>(p.gamma, t_hi, q_hi);
    line_gradient<DIM, N, NODAL, BCS>(p, Operators<N>(p), el, eid, dl, line, first, last, x, q_lo,
                                      q_hi, blo, bhi, sg_lo, sg_hi, acc);
  }
  __syncthreads();  // every line has read its q
  if (dir < DIM) {
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v)
        s_g[slot * SG + (dir * ND + v) * PN + ln.pbase + k * ln.pstride] = acc[k][v];
  }
  __syncthreads();
  // physical gradient g_c = (sum_d Ja^d_c G_d) / J and the fluxes
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (!has_node(k)) continue;
    const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN, pn = lds_pos<N>(node);
    if (sl >= nvalid) continue;
    const int64_t e = e0 + sl;
    int id[3];
    element_indices<DIM>(p, (int)e, id);
    double ja[DIM][DIM], g[DIM][NV], fv[DIM][NV];
    node_metric<DIM, N, NODAL, BOX>(p, e, id, node, ja);
    const double ij = inv_jac<NODAL, NN>(p, e, node);
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
      g[c][0] = 0.0;  // not used by the flux
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        double t = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) t += ja[d][c] * s_g[sl * SG + (d * ND + v - 1) * PN + pn];
        g[c][v] = t * ij;
      }
    }
#pragma unroll
    for (int c = 0; c < DIM; ++c) viscous_flux_dir<DIM>(p.mu, p.kappa, q[k], g, c, fv[c]);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      double* out = p.visc_out + (e * DIM + d) * (NV * NN) + row_pos<DIM, N>(d, node);
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        double r = 0.0;
#pragma unroll
        for (int c = 0; c < DIM; ++c) r += ja[d][c] * -fv[c][v];
        out[v * NN] = r;
      }
    }
  }
}

// Viscous fluxes for the node-parallel RHS kernel: at node `node` of
// element e the contravariant flux Ja^d . (-F_v) of each direction d, into
// p.visc_out [E][d][var][dof], rounded as ViscousFluxFunctor and the viscous
// volume integral's fref (parabolic_viscous.hpp:39-66 and :103-163 3D,
// :367-386 and :412-447 2D): -F_v of each physical direction, then
// Ja^d_0 f_0 + Ja^d_1 f_1 (+ Ja^d_2 f_2) from left to right, with no fused
// multiply-adds.  The interface value (-F_v) . (sign(J) Ja^d) of a face node
// is sign(J) times this sum to the bit (scaling by a sign is exact), so the
// RHS kernel needs nothing more.  The mass component is zero: not stored.
template <int DIM, int N, bool NODAL>
__device__ __forceinline__ void store_viscous_fluxes(const KParams& p, int64_t e, int node,
                                                     const double* q, const double g[DIM][DIM + 2]) {
  constexpr int NV = DIM + 2, NN = Shape<DIM, N>::NN;
  double fv[DIM][NV];
#pragma unroll
  for (int c = 0; c < DIM; ++c) viscous_flux_dir<DIM>(p.mu, p.kappa, q, g, c, fv[c]);
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    double ja[DIM];
#pragma unroll
    for (int c = 0; c < DIM; ++c) ja[c] = metric<NODAL, DIM, NN>(p, e, d, c, node);
#pragma unroll
    for (int v = 1; v < NV; ++v) {
#pragma clang fp contract(off)
      double r = ja[0] * -fv[0][v];
#pragma unroll
      for (int c = 1; c < DIM; ++c) r = r + ja[c] * -fv[c][v];
      p.visc_out[((e * DIM + d) * NV + v) * NN + node] = r;
    }
  }
}

// BR1 gradient for the node-parallel RHS kernel's elements (periodic, no
// shock capturing, N >= 7), one workgroup per element and one thread per
// node, rounded as the reference's scalar functors round it: the weak
// derivative sum_m D_hat(x_d, m) q(m) of each direction d from left to right
// (GradientVolumeIntegralFunctor, parabolic_gradient.hpp:40-79 3D,
// :502-527 2D), the physical transform Ja^0_c r_0 + Ja^1_c r_1 (+ Ja^2_c r_2)
// (:121-150 / :567-584), the lifted face values (-l_0 or l_N) q_hat times
// sign(J) Ja^d_c, q_hat = (q_lower + q_upper) / 2, in direction order
// (:186-291 and :348-430 / :628-685 and :737-788), then 1/J (:462-474 /
// :806-815); no fused multiply-adds.  The derivative of T = p / rho cancels
// terms some thousand times its size at N = 7, so these roundings show in
// the viscous terms at the 1e-12 level.  Writes the node's viscous fluxes
// (store_viscous_fluxes), not the gradient.
template <int DIM, int N, bool NODAL>
__global__ void __launch_bounds__((Shape<DIM, N>::NN)) gradient_node_kernel(const KParams p) {
  constexpr int n = N + 1, NV = DIM + 2, NN = Shape<DIM, N>::NN;
  __shared__ double s_q[NV * NN];
  __shared__ double s_Dh[n * n];
  const int a = threadIdx.x;
  const int64_t e = xcd_block(blockIdx.x, gridDim.x);
  const int idx[3] = {a % n, (a / n) % n, DIM == 3 ? a / (n * n) : 0};
  constexpr int stride[3] = {1, n, n * n};
  int eid[3];
  element_indices<DIM>(p, (int)e, eid);
  double u[NV], q[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) u[v] = p.u[(e * NV + v) * NN + a];
  grad_vars<DIM>(p.gamma, u, q);
#pragma unroll
  for (int v = 0; v < NV; ++v) s_q[v * NN + a] = q[v];
  if (a < n * n) s_Dh[a] = p.basis[n * n + a];
  __syncthreads();
  double r[DIM][NV];
#pragma unroll
  for (int d = 0; d < DIM; ++d)
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      double t = 0.0;
#pragma unroll
      for (int m = 0; m < n; ++m) {
#pragma clang fp contract(off)
        t = t + s_Dh[idx[d] * n + m] * s_q[v * NN + a + (m - idx[d]) * stride[d]];
      }
      r[d][v] = t;
    }
  double g[DIM][NV];
#pragma unroll
  for (int c = 0; c < DIM; ++c) {
    double ja[DIM];
#pragma unroll
    for (int d = 0; d < DIM; ++d) ja[d] = metric<NODAL, DIM, NN>(p, e, d, c, a);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
#pragma clang fp contract(off)
      double t = ja[0] * r[0][v];
#pragma unroll
      for (int d = 1; d < DIM; ++d) t = t + ja[d] * r[d][v];
      g[c][v] = t;
    }
  }
  const double ij = inv_jac<NODAL, NN>(p, e, a);
  const double sg = ij >= 0.0 ? 1.0 : -1.0;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const bool lower = idx[d] == 0, upper = idx[d] == N;
    if (lower || upper) {
      int64_t lo, hi;
      face_neighbours<DIM, false>(p, eid, e, d, lo, hi);
      const int64_t ne = lower ? lo : hi;
      const int nn = lower ? a + N * stride[d] : a - N * stride[d];
      double un[NV], qn[NV], nrm[DIM];
#pragma unroll
      for (int v = 0; v < NV; ++v) un[v] = p.u[(ne * NV + v) * NN + nn];
      grad_vars<DIM>(p.gamma, un, qn);
#pragma unroll
      for (int c = 0; c < DIM; ++c) nrm[c] = sg * metric<NODAL, DIM, NN>(p, e, d, c, a);
      const double factor = lower ? -p.lhat0 : p.lhatN;
#pragma unroll
      for (int v = 0; v < NV; ++v) {
#pragma clang fp contract(off)
        const double fq = factor * (0.5 * (qn[v] + q[v]));
#pragma unroll
        for (int c = 0; c < DIM; ++c) g[c][v] = g[c][v] + fq * nrm[c];
      }
    }
  }
#pragma unroll
  for (int c = 0; c < DIM; ++c)
#pragma unroll
    for (int v = 0; v < NV; ++v) g[c][v] = g[c][v] * ij;
  // the node's gradient is complete: its viscous fluxes follow here, so the
  // gradient itself never goes to memory
  store_viscous_fluxes<DIM, N, NODAL>(p, e, a, q, g);
}

template <int DIM, int N>
constexpr int parabolic_elems_per_block() {
  constexpr int e = (DIM == 2 ? 64 : 192) / Shape<DIM, N>::LINES;  // as elems_per_block
  return e < 1 ? 1 : e;
}

template <int DIM, int N, bool NODAL, bool BCS>
hipError_t launch_parabolic_t(bool sc, const KParams& p, hipStream_t s) {
  constexpr int EPW = parabolic_elems_per_block<DIM, N>();
  constexpr int BLOCK = EPW * Shape<DIM, N>::LINES;
  const int64_t nb = (p.E + EPW - 1) / EPW;
  if (nb <= 0) return hipSuccess;
  if constexpr (node_kernel_for(N, false, BCS)) {
    if (!sc) {
      hipLaunchKernelGGL((gradient_node_kernel<DIM, N, NODAL>), dim3((unsigned)p.E),
                         dim3(Shape<DIM, N>::NN), 0, s, p);
      return hipGetLastError();
    }
  }
  if constexpr (NODAL) {
    if (p.ja_box && box_table_for<DIM, N>(p.E, p.cus)) {
      hipLaunchKernelGGL((viscous_flux_kernel<DIM, N, EPW, NODAL, BCS, true>), dim3((unsigned)nb),
                         dim3(BLOCK), 0, s, p);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((viscous_flux_kernel<DIM, N, EPW, NODAL, BCS, false>), dim3((unsigned)nb),
                     dim3(BLOCK), 0, s, p);
  return hipGetLastError();
}

}  // namespace detail
}  // namespace dgsem
