// Tangent (JVP) and discrete adjoint (VJP) kernels of the DGSEM right-hand
// side L(u) = -(1/J) (A(u) + R(u)): A the split-form volume integral (under
// shock capturing blended with the subcell finite volumes, alpha frozen)
// plus the LLF or HLLC surface flux lifted with l_hat, R the BR1 viscous part
// (Navier-Stokes).  On 2D meshes a face may be a boundary face: the outer
// state, the wall gradient value and the wall viscous flux are functions of
// the own element's nodes, differentiated with them.  They differentiate what
// rhs_kernel and viscous_flux_kernel compute, with the pointwise derivatives
// of physics_ad.hpp.
//
// Two kernels each (one for Euler), laid out as the forward's: whole-node
// staging into padded LDS planes, line threads in (dir, slot, line) order, box
// meshes' metric rows from the table, per-direction sums.
// Tangent:
//   jvp_viscous_kernel  the gradient and its tangent at every node, the
//                       viscous fluxes' tangent Ja^d . (-dF_v)   -> a.dgrad
//   jvp_rhs_kernel      dA and the divergence of those, then -(1/J) and the
//                       output combination
// Adjoint, with r = -(1/J) w the cotangent of A + R:
//   vjp_viscous_kernel  r -> Hbar (transposed D_hat and interface lifting)
//                       -> Fbar -> (qbar direct, gbar) -> Gbar -> a.qbar, a.dgrad
//   vjp_rhs_kernel      pairs and faces -> primitive / conservative cotangents;
//                       Gbar -> qbar (transposed D_hat and BR1 face averages,
//                       gathered from the neighbours) -> conservative; the
//                       output combination
// One MI355X, a tangent and an adjoint of a viscous TGV step (16^3, N = 3): 753 us
// with separate gradient and viscous kernels (21 launches), 323 us in these 12.
// a.dgrad is [E][d][var][line * n + k] (no mass component).  Every kernel
// gathers what it needs from the neighbours (no atomics), so results do not
// depend on scheduling.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "kernels.hpp"
#include "parabolic_impl.hpp"
#include "physics_ad.hpp"

namespace dgsem {
namespace detail {

// Elements per workgroup, as elems_per_block: one wave in 2D (a tangent plus an
// adjoint of a step, 192 threads -> one wave: split form N = 3 80 x 80 94 -> 80 us,
// HLLC channel N = 3 128 x 128 209 -> 171 us, viscous N = 5 160 x 160 822 -> 725
// us; 8% on the average of 8 x 8 to 224 x 224).  A few sizes whose last round of
// 192-thread blocks happens to be full are 1-2.5% slower (split form N = 3 160 x 160
// 212 -> 218 us, N = 5 128 x 128 360 -> 365; before the two-kernel form 367 and 700).
template <int DIM, int N>
constexpr int ad_elems_per_block() {
  constexpr int e = (DIM == 2 ? 64 : 192) / Shape<DIM, N>::LINES;
  return e < 1 ? 1 : e;
}

__device__ __forceinline__ double combine(const AdParams& a, int64_t g, double r) {
  double o = a.c * r;
  if (a.b != 0.0) o += a.b * a.v[g];
  if (a.x1) o += a.a1 * a.x1[g];
  if (a.x2) o += a.a2 * a.x2[g];
  return o;
}

// The basis operators among the kernel's arguments.  The derivative kernels use
// them right after their first loads, where the table of Operators would put its
// pointer's load in front (1.5% of a tangent plus adjoint at 16^3, N = 3).
struct AdOperators {
  const AdParams& a;
  __device__ __forceinline__ double Ds(int i, int j) const { return a.Ds[i][j]; }
  __device__ __forceinline__ double Dhat(int i, int j) const { return a.Dhat[i][j]; }
  __device__ __forceinline__ double inv_w(int i) const { return a.inv_w[i]; }
};

template <int DIM, int NN>
__device__ __forceinline__ void load_state(const double* u, int64_t e, int node, double* s) {
  for (int v = 0; v < DIM + 2; ++v) s[v] = u[(e * (DIM + 2) + v) * NN + node];
}

template <bool NODAL, int DIM, int NN>
__device__ __forceinline__ double sign_j(const KParams& p, int64_t e, int node) {
  return inv_jac<NODAL, NN>(p, e, node) >= 0.0 ? 1.0 : -1.0;
}

// Minimum waves per SIMD of the RHS derivative kernels: up to N = 3 the LLF
// split-form ones are held to three (168 VGPRs; with nodal metrics at 3D N = 3 the
// adjoint spills 14 registers, 31 with viscous terms, the tangent 83 with viscous
// terms); the HLLC and subcell derivatives would spill hundreds.
template <int N, bool SC, int SF>
constexpr int ad_waves() {
  return N <= 3 && !SC && SF == kFluxLLF ? 3 : 1;
}

// Normal of subcell interface f (between nodes f and f + 1) on line `line`
// of direction dir: the nodal subcell normals, or the element's metric row
// (affine), as the forward's subcell flux uses them.
template <int DIM, int N, bool NODAL>
__device__ __forceinline__ void subcell_normal(const KParams& p, int64_t e, int dir, int line, int f,
                                               double* nrm) {
  constexpr int FN = Shape<DIM, N>::FN;
  for (int c = 0; c < DIM; ++c)
    nrm[c] = NODAL ? p.sn[((((e * DIM + dir) * FN) + line) * N + f) * DIM + c]
                   : p.Ja[(e * DIM + dir) * DIM + c];
}

// Frozen blending factor of element e (shock capturing): the split-form
// weight coef = 1 - alpha and the subcell weight alpha of a troubled
// element, coef = 1 and no subcell terms otherwise
// (volume_flux.hpp:843-869 with the atol test of :772-773).
template <bool SC>
__device__ __forceinline__ bool frozen_blend(const KParams& p, int64_t e, double& coef, double& alpha) {
  coef = 1.0;
  alpha = 0.0;
  if constexpr (SC) {
    alpha = p.alpha_in[e];
    if (fabs(alpha - 0.0) > p.atol) {
      coef = 1.0 - alpha;
      return true;
    }
  }
  return false;
}

// Non-periodic faces (2D meshes; face_neighbours gives -1 there).  The
// outer state of face `face` (2 dir + upper) at boundary node bnode is the
// one the forward's boundary_state forms (rhs_kernel_impl.hpp), with the
// line's states read from memory.  As a map of the state it is one of
// three kinds: a slip wall (and the inviscid part of the Navier-Stokes
// walls) mirrors the momentum about the face, linear and symmetric in the
// momentum; outflow takes the mean of the line's n nodes; a Dirichlet state
// (constant or per node) does not depend on the state.
enum class BcMap { kConstant, kMirror, kMean };

template <int DIM>
__device__ __forceinline__ BcMap bc_map(const KParams& p, int face, int64_t bnode) {
  constexpr int NV = DIM + 2;
  const int kind = p.bc[face];
  if (kind == kBcMixedDirichletSlipWall && p.bc_values[face][bnode * (NV + 1) + NV] != 0.0)
    return BcMap::kConstant;
  if (kind == kBcSlipWall || kind == kBcNsNoSlipWall || kind == kBcNsSlipWall ||
      kind == kBcMixedDirichletSlipWall)
    return BcMap::kMirror;
  return kind == kBcOutflow ? BcMap::kMean : BcMap::kConstant;
}

// Boundary node of line `line` of element e on a face of direction dir
// (2D, elements numbered e = ie * ny + je), as the forward numbers it.
template <int DIM, int N>
__device__ __forceinline__ int64_t boundary_node(const KParams& p, int64_t e, int dir, int line) {
  const int64_t along = dir == 0 ? e % p.cells[1] : e / p.cells[1];
  return along * (N + 1) + line;
}

// The outer state; ue: the element's states in memory ([var][node]).
template <int DIM, int N, int NN>
__device__ void bc_outer_state(const KParams& p, int face, int64_t bnode, BcMap m, const double* ue,
                               const int* dofs, const double* uin, const double* nrm, double* uout) {
  constexpr int n = N + 1, NV = DIM + 2;
  if (m == BcMap::kMirror) {
    const double rho = uin[0];
    double v[DIM], vn = 0.0, nn = 0.0;
    for (int c = 0; c < DIM; ++c) v[c] = uin[1 + c] / rho;
    for (int c = 0; c < DIM; ++c) nn += nrm[c] * nrm[c];
    for (int c = 0; c < DIM; ++c) vn += v[c] * nrm[c];
    vn = vn / nn;
    uout[0] = rho;
    for (int c = 0; c < DIM; ++c) uout[1 + c] = rho * (v[c] - 2.0 * vn * nrm[c]);
    uout[NV - 1] = uin[NV - 1];
  } else if (m == BcMap::kMean) {
    for (int v = 0; v < NV; ++v) {
      double acc = 0.0;
      for (int k = 0; k < n; ++k) acc += ue[v * NN + dofs[k]];
      uout[v] = acc / (double)n;
    }
  } else {
    const double* vals = p.bc_values[face];
    if (p.bc[face] == kBcMixedDirichletSlipWall) {
      for (int v = 0; v < NV; ++v) uout[v] = vals[bnode * (NV + 1) + v];
    } else {
      for (int v = 0; v < NV; ++v) uout[v] = vals ? vals[bnode * NV + v] : p.bc_state[face][v];
    }
  }
}

// Its tangent: dve the tangent's states of the element, duin the tangent at
// the boundary node.
template <int DIM, int N, int NN>
__device__ void bc_outer_tangent(BcMap m, const double* dve, const int* dofs, const double* duin,
                                 const double* nrm, double* duout) {
  constexpr int n = N + 1, NV = DIM + 2;
  if (m == BcMap::kMirror) {
    double mn = 0.0, nn = 0.0;
    for (int c = 0; c < DIM; ++c) {
      mn += duin[1 + c] * nrm[c];
      nn += nrm[c] * nrm[c];
    }
    mn = mn / nn;
    duout[0] = duin[0];
    for (int c = 0; c < DIM; ++c) duout[1 + c] = duin[1 + c] - 2.0 * mn * nrm[c];
    duout[NV - 1] = duin[NV - 1];
  } else if (m == BcMap::kMean) {
    for (int v = 0; v < NV; ++v) {
      double acc = 0.0;
      for (int k = 0; k < n; ++k) acc += dve[v * NN + dofs[k]];
      duout[v] = acc / (double)n;
    }
  } else {
    for (int v = 0; v < NV; ++v) duout[v] = 0.0;
  }
}

// Navier-Stokes faces of bounded meshes (parabolic_impl.hpp).  The gradient's
// face value is the wall map of the own node's gradient variables
// (wall_gradient_value: no slip zeroes the velocity, slip removes its normal
// part; both linear in q and symmetric) or a Dirichlet state's, which is
// constant; this applies the map's derivative (which is its transpose) to x.
template <int DIM>
__device__ __forceinline__ void wall_gradient_linear(int kind, const double* x, const double* nrm,
                                                     double* y) {
  if (kind == kBcDirichlet) {
    for (int v = 0; v < DIM + 2; ++v) y[v] = 0.0;
  } else {
    wall_gradient_value<DIM>(kind, x, nrm, y);
  }
}

// The variables [lo, hi) of the own node's viscous flux a boundary face
// carries: all at a Dirichlet face, the momentum at a no-slip wall, none
// otherwise.
__device__ __forceinline__ void wall_viscous_range(int kind, int nv, int& lo, int& hi) {
  lo = kind == kBcDirichlet ? 0 : 1;
  hi = kind == kBcDirichlet ? nv : (kind == kBcNsNoSlipWall ? nv - 1 : 0);
}

// A thread's line in the derivative kernels: direction, element slot and line
// number (threads ordered (dir, slot, line)), the line's nodes, the element's
// indices and its face neighbours.  Threads whose slot is past the last valid
// element take element e0 and are not `valid`.  blo, bhi: the lower or upper end
// is a boundary face (2D), whose neighbour index is then the own element.
template <int DIM, int N, int EPW>
struct AdLine {
  int dir, slot, line, eid[3];
  bool valid, blo, bhi;
  int64_t e, lo, hi;
  LineNodes<DIM, N> ln;
  __device__ __forceinline__ AdLine(const KParams& p, int tid, int64_t e0, int nvalid)
      : dir(tid / (EPW * Shape<DIM, N>::FN)),
        slot(tid % (EPW * Shape<DIM, N>::FN) / Shape<DIM, N>::FN),
        line(tid % Shape<DIM, N>::FN),
        ln(dir, line) {
    valid = slot < nvalid;
    e = valid ? e0 + slot : e0;
    element_indices<DIM>(p, (int)e, eid);
    face_neighbours<DIM, DIM == 2>(p, eid, e, dir, lo, hi);
    blo = DIM == 2 && lo < 0;
    bhi = DIM == 2 && hi < 0;
    if (blo) lo = e;
    if (bhi) hi = e;
  }
  __device__ __forceinline__ int dof(int k) const { return ln.base + k * ln.stride; }
  __device__ __forceinline__ int pos(int k) const { return ln.pbase + k * ln.pstride; }
  __device__ __forceinline__ int first() const { return ln.base; }
  __device__ __forceinline__ int last() const { return ln.base + N * ln.stride; }
};

// The line's metric rows, halved (NODAL), or the element's row in ja[0].
template <int DIM, int N, int EPW, bool NODAL>
__device__ __forceinline__ void line_metric(const KParams& p, const AdLine<DIM, N, EPW>& l,
                                            double (&ja)[NODAL ? N + 1 : 1][DIM]) {
  constexpr int NN = Shape<DIM, N>::NN;
  if constexpr (NODAL) {
    if (p.ja_box) {
#pragma unroll
      for (int c = 0; c < DIM; ++c) {
        const double* row = box_row<DIM, N>(p, l.eid, c, l.dir, l.line);
#pragma unroll
        for (int k = 0; k <= N; ++k) ja[k][c] = row[k];
      }
    } else {
      const double* row = p.Ja + (l.e * DIM + l.dir) * (DIM * NN);
#pragma unroll
      for (int k = 0; k <= N; ++k)
#pragma unroll
        for (int c = 0; c < DIM; ++c) ja[k][c] = 0.5 * row[c * NN + l.dof(k)];
    }
  } else {
#pragma unroll
    for (int c = 0; c < DIM; ++c) ja[0][c] = p.Ja[(l.e * DIM + l.dir) * DIM + c];
  }
}

// A node's metric terms, from the table on a box mesh.
template <int DIM, int N, bool NODAL>
__device__ __forceinline__ void ad_node_metric(const KParams& p, int64_t e, int dof,
                                               double ja[DIM][DIM]) {
  int eid[3];
  element_indices<DIM>(p, (int)e, eid);
  if (NODAL && p.ja_box)
    node_metric<DIM, N, NODAL, true>(p, e, eid, dof, ja);
  else
    node_metric<DIM, N, NODAL, false>(p, e, eid, dof, ja);
}

// Keeps values where they are computed (see `pin` in element_body.inc): with
// it the divergent branch of the logarithmic means does not multiply the
// registers of the unrolled pairs.
template <int K>
__device__ __forceinline__ void pin_values(double* x) {
#pragma unroll
  for (int i = 0; i < K; ++i) asm volatile("" : "+v"(x[i]));
}

// ---------------------------------------------------------------------------
// Tangent
// ---------------------------------------------------------------------------

// The tangent's viscous fluxes Ja^d . (-dF_v) into a.dgrad.  The gradient's and
// the tangent's line derivatives pass through the same LDS planes one after
// the other: of the gradient a node keeps its stress only.
template <int DIM, int N, int EPW, bool NODAL>
__global__ void __launch_bounds__((EPW * Shape<DIM, N>::LINES)) jvp_viscous_kernel(const AdParams a) {
  using S = Shape<DIM, N>;
  constexpr int n = S::n, NV = S::NV, NN = S::NN, PN = S::PN;
  constexpr int ND = NV - 1;  // differentiated variables v, T: planes v - 1
  constexpr int BLOCK = EPW * S::LINES, NODES = EPW * NN, PASSES = (NODES + BLOCK - 1) / BLOCK;
  constexpr int SG = DIM * ND * PN + S::slot_pad(DIM * ND * PN);
  static_assert(DIM >= 2, "q and dq fit the planes of the line derivatives");
  const KParams& p = a.k;
  const AdOperators op{a};
  __shared__ double s_g[EPW * SG];  // q and dq [var], then the derivatives [dir][var]
  const int tid = threadIdx.x;
  const int64_t e0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * EPW;
  const int nvalid = (int)((p.E - e0) < EPW ? (p.E - e0) : EPW);
  auto has_node = [&](int k) { return (k + 1) * BLOCK <= NODES || tid + k * BLOCK < NODES; };
  double q[PASSES][NV], dq[PASSES][NV];
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (has_node(k)) {
      const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN;
      const int64_t e = e0 + (sl < nvalid ? sl : nvalid - 1);
      load_state<DIM, NN>(p.u, e, node, q[k]);
      load_state<DIM, NN>(a.v, e, node, dq[k]);
    }
  }
  const AdLine<DIM, N, EPW> l(p, tid, e0, nvalid);
  double t_lo[NV], t_hi[NV], dt_lo[NV], dt_hi[NV];
  load_state<DIM, NN>(p.u, l.lo, l.last(), t_lo);
  load_state<DIM, NN>(p.u, l.hi, l.first(), t_hi);
  load_state<DIM, NN>(a.v, l.lo, l.last(), dt_lo);
  load_state<DIM, NN>(a.v, l.hi, l.first(), dt_hi);
  const double sg_lo = sign_j<NODAL, DIM, NN>(p, l.e, l.first());
  const double sg_hi = sign_j<NODAL, DIM, NN>(p, l.e, l.last());
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (has_node(k)) {
      const int i = tid + k * BLOCK, sl = i / NN, pn = lds_pos<N>(i - sl * NN);
      double u[NV], du[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        u[v] = q[k][v];
        du[v] = dq[k][v];
      }
      grad_vars<DIM>(p.gamma, u, q[k]);
      grad_vars_jvp<DIM>(p.gamma, u, du, dq[k]);
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        s_g[sl * SG + (v - 1) * PN + pn] = q[k][v];
        s_g[sl * SG + (ND + v - 1) * PN + pn] = dq[k][v];
      }
    }
  }
  __syncthreads();
  double acc[n][ND], dacc[n][ND];
  {
    double x[n][ND], q_lo[NV], q_hi[NV], dq_lo[NV], dq_hi[NV];
    grad_vars<DIM>(p.gamma, t_lo, q_lo);
    grad_vars<DIM>(p.gamma, t_hi, q_hi);
    grad_vars_jvp<DIM>(p.gamma, t_lo, dt_lo, dq_lo);
    grad_vars_jvp<DIM>(p.gamma, t_hi, dt_hi, dq_hi);
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) x[k][v] = s_g[l.slot * SG + v * PN + l.pos(k)];
    line_gradient<DIM, N, NODAL, DIM == 2>(p, op, l.e, l.eid, l.dir, l.line, l.first(), l.last(), x,
                                           q_lo, q_hi, l.blo, l.bhi, sg_lo, sg_hi, acc);
    double dx[n][ND];
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) dx[k][v] = s_g[l.slot * SG + (ND + v) * PN + l.pos(k)];
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) {
        double r = 0.0;
#pragma unroll
        for (int i = 0; i < n; ++i) r += op.Dhat(k, i) * dx[i][v];
        dacc[k][v] = r;
      }
#pragma unroll
    for (int v = 1; v < NV; ++v) {
      dq_lo[v] = 0.5 * (dq_lo[v] + dx[0][v - 1]);
      dq_hi[v] = 0.5 * (dx[n - 1][v - 1] + dq_hi[v]);
    }
    if constexpr (DIM == 2) {
      // a boundary face: the wall map of the own node's variables
      auto wall = [&](int side, int dof, double sg, const double* xn, double* out) {
        double own[NV], nrm[DIM];
        own[0] = 0.0;
        for (int v = 1; v < NV; ++v) own[v] = xn[v - 1];
        for (int c = 0; c < DIM; ++c) nrm[c] = sg * metric<NODAL, DIM, NN>(p, l.e, l.dir, c, dof);
        wall_gradient_linear<DIM>(p.bc[2 * l.dir + side], own, nrm, out);
      };
      if (l.blo) wall(0, l.first(), sg_lo, dx[0], dq_lo);
      if (l.bhi) wall(1, l.last(), sg_hi, dx[n - 1], dq_hi);
    }
#pragma unroll
    for (int v = 1; v < NV; ++v) {
      dacc[0][v - 1] -= sg_lo * p.lhat0 * dq_lo[v];
      dacc[n - 1][v - 1] += sg_hi * p.lhatN * dq_hi[v];
    }
  }
  auto store = [&](const double (&x)[n][ND]) {
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) s_g[l.slot * SG + (l.dir * ND + v) * PN + l.pos(k)] = x[k][v];
  };
  // physical gradient g_c = (sum_d Ja^d_c G_d) / J of node pass k
  auto gradient = [&](int sl, int node, const double (&ja)[DIM][DIM], double (&g)[DIM][NV]) {
    const int pn = lds_pos<N>(node);
    const double ij = inv_jac<NODAL, NN>(p, e0 + sl, node);
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
  };
  __syncthreads();  // every line has read its q and dq
  store(acc);
  __syncthreads();
  double tau[PASSES][DIM][DIM];
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (!has_node(k)) continue;
    const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN;
    if (sl >= nvalid) continue;
    double ja[DIM][DIM], g[DIM][NV];
    ad_node_metric<DIM, N, NODAL>(p, e0 + sl, node, ja);
    gradient(sl, node, ja, g);
    stress<DIM>(g, tau[k]);
  }
  __syncthreads();
  store(dacc);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (!has_node(k)) continue;
    const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN;
    if (sl >= nvalid) continue;
    double ja[DIM][DIM], dg[DIM][NV], df[DIM][NV];
    ad_node_metric<DIM, N, NODAL>(p, e0 + sl, node, ja);
    gradient(sl, node, ja, dg);
    viscous_flux_jvp_stress<DIM>(p.mu, p.kappa, q[k], tau[k], dq[k], dg, df);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      double* out = a.dgrad + ((e0 + sl) * DIM + d) * (NV * NN) + row_pos<DIM, N>(d, node);
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        double r = 0.0;
#pragma unroll
        for (int c = 0; c < DIM; ++c) r += ja[d][c] * -df[c][v];
        out[v * NN] = r;
      }
    }
  }
}

template <int DIM, int N, int EPW, bool NODAL, bool NS, bool SC, int SF, int FF>
__global__ void __launch_bounds__((EPW * Shape<DIM, N>::LINES))
    __attribute__((amdgpu_waves_per_eu((ad_waves<N, SC, SF>())))) jvp_rhs_kernel(const AdParams a) {
  using S = Shape<DIM, N>;
  constexpr int n = S::n, NV = S::NV, NN = S::NN, PN = S::PN;
  constexpr int NQ = DIM + 2;  // rho, v[DIM], beta
  constexpr int BLOCK = EPW * S::LINES, NODES = EPW * NN, PASSES = (NODES + BLOCK - 1) / BLOCK;
  constexpr int SQ = NQ * PN + S::slot_pad(NQ * PN);
  const KParams& p = a.k;
  const AdOperators op{a};
  __shared__ double s_p[EPW * SQ];   // rho, v, beta; later the per-direction sums
  __shared__ double s_dq[EPW * SQ];  // their tangents
  double* const s_acc = s_p;
  const int tid = threadIdx.x;
  const int64_t e0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * EPW;
  const int nvalid = (int)((p.E - e0) < EPW ? (p.E - e0) : EPW);
  auto has_node = [&](int k) { return (k + 1) * BLOCK <= NODES || tid + k * BLOCK < NODES; };
  {
    double u[PASSES][NV], du[PASSES][NV];
#pragma unroll
    for (int k = 0; k < PASSES; ++k) {
      if (has_node(k)) {
        const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN;
        const int64_t e = e0 + (sl < nvalid ? sl : nvalid - 1);
        load_state<DIM, NN>(p.u, e, node, u[k]);
        load_state<DIM, NN>(a.v, e, node, du[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < PASSES; ++k) {
      if (has_node(k)) {
        const int i = tid + k * BLOCK, sl = i / NN, pn = lds_pos<N>(i - sl * NN);
        const NodePrims<DIM> q = node_prims<DIM>(p.gamma, u[k]);
        PrimTangent<DIM> dq;
        prims_jvp<DIM>(p.gamma, u[k], q, du[k], dq);
        double* d = s_p + sl * SQ + pn;
        double* t = s_dq + sl * SQ + pn;
        d[0] = q.rho;
        t[0] = dq.rho;
#pragma unroll
        for (int c = 0; c < DIM; ++c) {
          d[(1 + c) * PN] = q.v[c];
          t[(1 + c) * PN] = dq.v[c];
        }
        d[(DIM + 1) * PN] = q.beta;
        t[(DIM + 1) * PN] = dq.beta;
      }
    }
  }
  const AdLine<DIM, N, EPW> l(p, tid, e0, nvalid);
  double ja[NODAL ? n : 1][DIM];
  line_metric<DIM, N, EPW, NODAL>(p, l, ja);
  __syncthreads();

  double acc[n][NV];
#pragma unroll
  for (int k = 0; k < n; ++k)
#pragma unroll
    for (int v = 0; v < NV; ++v) acc[k][v] = 0.0;
  if (l.valid) {
    // faces, both states and their tangents from memory
#pragma unroll 1
    for (int side = 0; side < 2; ++side) {
      const bool lower = side == 0;
      const int od = lower ? l.first() : l.last(), nd = lower ? l.last() : l.first();
      const int64_t nb = lower ? l.lo : l.hi;
      double uo[NV], duo[NV], un[NV], dun[NV], nrm[DIM], df[NV];
      load_state<DIM, NN>(p.u, l.e, od, uo);
      load_state<DIM, NN>(a.v, l.e, od, duo);
      bool boundary = false;
      if constexpr (DIM == 2) boundary = lower ? l.blo : l.bhi;
      // the normal of the face's upper element at its first node; at a
      // boundary face, of the own element at its node
      const int64_t en = lower || boundary ? l.e : nb;
      const int nn = boundary ? od : l.first();
      const double sg = sign_j<NODAL, DIM, NN>(p, en, nn);
#pragma unroll
      for (int c = 0; c < DIM; ++c) nrm[c] = sg * metric<NODAL, DIM, NN>(p, en, l.dir, c, nn);
      if (boundary) {
        if constexpr (DIM == 2) {
          int dofs[n];
          for (int k = 0; k < n; ++k) dofs[k] = l.dof(k);
          const int face = 2 * l.dir + side;
          const int64_t bnode = boundary_node<DIM, N>(p, l.e, l.dir, l.line);
          const BcMap m = bc_map<DIM>(p, face, bnode);
          bc_outer_state<DIM, N, NN>(p, face, bnode, m, p.u + l.e * NV * NN, dofs, uo, nrm, un);
          bc_outer_tangent<DIM, N, NN>(m, a.v + l.e * NV * NN, dofs, duo, nrm, dun);
        }
      } else {
        load_state<DIM, NN>(p.u, nb, nd, un);
        load_state<DIM, NN>(a.v, nb, nd, dun);
      }
      double ul[NV], ur[NV], dul[NV], dur[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        ul[v] = lower ? un[v] : uo[v];
        dul[v] = lower ? dun[v] : duo[v];
        ur[v] = lower ? uo[v] : un[v];
        dur[v] = lower ? duo[v] : dun[v];
      }
      if constexpr (SF == kFluxHLLC)
        hllc_jvp<DIM>(p.gamma, ul, ur, dul, dur, nrm, df);
      else
        llf_jvp<DIM>(p.gamma, ul, node_prims<DIM>(p.gamma, ul), ur, node_prims<DIM>(p.gamma, ur), dul,
                     dur, nrm, df);
      if (lower) {
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[0][v] -= df[v] * p.lhat0;
      } else {
#pragma unroll
        for (int v = 0; v < NV; ++v) acc[n - 1][v] += df[v] * p.lhatN;
      }
    }
    pin_values<NV>(acc[0]);
    pin_values<NV>(acc[n - 1]);

    double coef, alpha;
    const bool troubled = frozen_blend<SC>(p, l.e, coef, alpha);
    const double* pr = s_p + l.slot * SQ;
    const double* tq = s_dq + l.slot * SQ;
    auto prims = [&](int pos) {
      NodePrims<DIM> q;
      q.rho = pr[pos];
#pragma unroll
      for (int c = 0; c < DIM; ++c) q.v[c] = pr[(1 + c) * PN + pos];
      q.beta = pr[(DIM + 1) * PN + pos];
      q.kin = q.p = q.c = 0.0;
      return q;
    };
    auto tangent = [&](int pos) {
      PrimTangent<DIM> t;
      t.rho = tq[pos];
#pragma unroll
      for (int c = 0; c < DIM; ++c) t.v[c] = tq[(1 + c) * PN + pos];
      t.beta = tq[(DIM + 1) * PN + pos];
      t.kin = 0.0;
      return t;
    };
#pragma unroll
    for (int ia = 0; ia < n - 1; ++ia) {
      const NodePrims<DIM> qa = prims(l.pos(ia));
      const PrimTangent<DIM> ta = tangent(l.pos(ia));
#pragma unroll
      for (int ib = ia + 1; ib < n; ++ib) {
        const NodePrims<DIM> qb = prims(l.pos(ib));
        const PrimTangent<DIM> tb = tangent(l.pos(ib));
        double nrm[DIM], df[NV];
#pragma unroll
        for (int c = 0; c < DIM; ++c) nrm[c] = NODAL ? ja[NODAL ? ia : 0][c] + ja[NODAL ? ib : 0][c] : ja[0][c];
        chandrashekar_jvp<DIM>(p.inv_gm1, qa, qb, ta, tb, nrm, df);
        const double wa = coef * op.Ds(ia, ib), wb = coef * op.Ds(ib, ia);
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          acc[ia][v] += wa * df[v];
          acc[ib][v] += wb * df[v];
        }
        pin_values<NV>(acc[ia]);
        pin_values<NV>(acc[ib]);
      }
    }
    // first-order subcell fluxes of a troubled element, weighted by the
    // frozen alpha as the forward's blend weights them.  With LLF and up to
    // N = 5 the loop is unrolled: a run-time index would put the accumulators
    // in scratch memory (at 3D N = 3 the tangent took 667 instead of 757 us
    // with every element troubled at 32^3).  The HLLC tangent measured 1.5%
    // slower unrolled, and at N = 7 the unrolled fluxes spill more.
    if constexpr (SC) {
      if (troubled) {
        constexpr int FV_UNROLL = N <= 5 && FF != kFluxHLLC ? N : 1;
#pragma unroll FV_UNROLL
        for (int fi = 1; fi < n; ++fi) {
          double ul[NV], ur[NV], dul[NV], dur[NV], nrm[DIM], df[NV];
          load_state<DIM, NN>(p.u, l.e, l.dof(fi - 1), ul);
          load_state<DIM, NN>(p.u, l.e, l.dof(fi), ur);
          load_state<DIM, NN>(a.v, l.e, l.dof(fi - 1), dul);
          load_state<DIM, NN>(a.v, l.e, l.dof(fi), dur);
          subcell_normal<DIM, N, NODAL>(p, l.e, l.dir, l.line, fi - 1, nrm);
          if constexpr (FF == kFluxHLLC)
            hllc_jvp<DIM>(p.gamma, ul, ur, dul, dur, nrm, df);
          else
            llf_jvp<DIM>(p.gamma, ul, node_prims<DIM>(p.gamma, ul), ur, node_prims<DIM>(p.gamma, ur),
                         dul, dur, nrm, df);
          const double wl = alpha * op.inv_w(fi - 1), wr = alpha * op.inv_w(fi);
          for (int v = 0; v < NV; ++v) {
            acc[fi - 1][v] += wl * df[v];
            acc[fi][v] -= wr * df[v];
          }
          if constexpr (FV_UNROLL > 1) {
            pin_values<NV>(acc[fi - 1]);
            pin_values<NV>(acc[fi]);
          }
        }
      }
    }
    // the divergence of the viscous fluxes' tangent and its interface terms
    // (rhs_kernel's Navier-Stokes part)
    if constexpr (NS) {
      int lo_end = NV, hi_end = NV;  // variables [1, end) carried, per side
      if constexpr (DIM == 2) {
        int lo0, hi0;
        if (l.blo) wall_viscous_range(p.bc[2 * l.dir], NV, lo0, lo_end);
        if (l.bhi) wall_viscous_range(p.bc[2 * l.dir + 1], NV, hi0, hi_end);
      }
      const double sg_lo = sign_j<NODAL, DIM, NN>(p, l.e, l.first());
      const double sg_hi = l.bhi ? sign_j<NODAL, DIM, NN>(p, l.e, l.last())
                                 : sign_j<NODAL, DIM, NN>(p, l.hi, l.first());
      const double* h = a.dgrad + (l.e * DIM + l.dir) * (NV * NN) + l.line * n;
      const double* hu = l.bhi ? h + N : a.dgrad + (l.hi * DIM + l.dir) * (NV * NN) + l.line * n;
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        double x[n];
#pragma unroll
        for (int k = 0; k < n; ++k) x[k] = h[v * NN + k];
        const double up = hu[v * NN];
#pragma unroll
        for (int k = 0; k < n; ++k) {
          double r = 0.0;
#pragma unroll
          for (int i = 0; i < n; ++i) r += op.Dhat(k, i) * x[i];
          if (k == 0 && v < lo_end) r -= sg_lo * x[0] * p.lhat0;
          if (k == n - 1 && v < hi_end) r += sg_hi * up * p.lhatN;
          acc[k][v] += r;
        }
      }
    }
  }
  __syncthreads();  // s_acc aliases the primitives
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    if (l.valid && l.dir == d) {
#pragma unroll
      for (int k = 0; k < n; ++k)
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          const int idx = l.slot * SQ + v * PN + l.pos(k);
          s_acc[idx] = d == 0 ? acc[k][v] : s_acc[idx] + acc[k][v];
        }
    }
    __syncthreads();
  }
  for (int i = tid; i < NODES; i += BLOCK) {
    const int sl = i / NN, node = i - sl * NN, pn = lds_pos<N>(node);
    if (sl >= nvalid) continue;
    const int64_t e = e0 + sl;
    const double fac = -inv_jac<NODAL, NN>(p, e, node);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int64_t g = (e * NV + v) * NN + node;
      a.out[g] = combine(a, g, s_acc[sl * SQ + v * PN + pn] * fac);
    }
  }
}

// ---------------------------------------------------------------------------
// Adjoint
// ---------------------------------------------------------------------------

// r = -(1/J) w of element e at node: the cotangent of A + R.
template <int DIM, int NN, bool NODAL>
__device__ __forceinline__ void load_r(const AdParams& a, int64_t e, int node, double* r) {
  const double f = -inv_jac<NODAL, NN>(a.k, e, node);
  for (int v = 0; v < DIM + 2; ++v) r[v] = f * a.v[(e * (DIM + 2) + v) * NN + node];
}

// The viscous flux's adjoint at every node: Gbar into a.dgrad, the direct
// cotangent of the velocities into a.qbar.  As in jvp_viscous_kernel the
// gradient's line derivatives and Hbar share the LDS planes in turn.
template <int DIM, int N, int EPW, bool NODAL>
__global__ void __launch_bounds__((EPW * Shape<DIM, N>::LINES)) vjp_viscous_kernel(const AdParams a) {
  using S = Shape<DIM, N>;
  constexpr int n = S::n, NV = S::NV, NN = S::NN, PN = S::PN;
  constexpr int ND = NV - 1;  // variables v, T (and momentum, energy): planes v - 1
  constexpr int BLOCK = EPW * S::LINES, NODES = EPW * NN, PASSES = (NODES + BLOCK - 1) / BLOCK;
  constexpr int SG = DIM * ND * PN + S::slot_pad(DIM * ND * PN);
  const KParams& p = a.k;
  const AdOperators op{a};
  __shared__ double s_g[EPW * SG];  // q and r [var], then G and Hbar [dir][var]
  const int tid = threadIdx.x;
  const int64_t e0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * EPW;
  const int nvalid = (int)((p.E - e0) < EPW ? (p.E - e0) : EPW);
  auto has_node = [&](int k) { return (k + 1) * BLOCK <= NODES || tid + k * BLOCK < NODES; };
  double q[PASSES][NV], r[PASSES][NV];
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (has_node(k)) {
      const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN;
      const int64_t e = e0 + (sl < nvalid ? sl : nvalid - 1);
      load_state<DIM, NN>(p.u, e, node, q[k]);
      load_r<DIM, NN, NODAL>(a, e, node, r[k]);
    }
  }
  const AdLine<DIM, N, EPW> l(p, tid, e0, nvalid);
  double t_lo[NV], t_hi[NV], r_lo[NV];
  load_state<DIM, NN>(p.u, l.lo, l.last(), t_lo);
  load_state<DIM, NN>(p.u, l.hi, l.first(), t_hi);
  load_r<DIM, NN, NODAL>(a, l.lo, l.last(), r_lo);
  const double sg_lo = sign_j<NODAL, DIM, NN>(p, l.e, l.first());
  const double sg_hi = sign_j<NODAL, DIM, NN>(p, l.e, l.last());
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (has_node(k)) {
      const int i = tid + k * BLOCK, sl = i / NN, pn = lds_pos<N>(i - sl * NN);
      double u[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) u[v] = q[k][v];
      grad_vars<DIM>(p.gamma, u, q[k]);
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        s_g[sl * SG + (v - 1) * PN + pn] = q[k][v];
        s_g[sl * SG + (ND + v - 1) * PN + pn] = r[k][v];
      }
    }
  }
  __syncthreads();
  double acc[n][ND], hb[n][ND];
  {
    double x[n][ND], q_lo[NV], q_hi[NV];
    grad_vars<DIM>(p.gamma, t_lo, q_lo);
    grad_vars<DIM>(p.gamma, t_hi, q_hi);
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) x[k][v] = s_g[l.slot * SG + v * PN + l.pos(k)];
    line_gradient<DIM, N, NODAL, DIM == 2>(p, op, l.e, l.eid, l.dir, l.line, l.first(), l.last(), x,
                                           q_lo, q_hi, l.blo, l.bhi, sg_lo, sg_hi, acc);
    double rx[n][ND];
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) rx[k][v] = s_g[l.slot * SG + (ND + v) * PN + l.pos(k)];
    // Hbar_k = sum_k' Dhat[k'][k] r_k'  (transpose of the weak divergence)
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) {
        double h = 0.0;
#pragma unroll
        for (int i = 0; i < n; ++i) h += op.Dhat(i, k) * rx[i][v];
        hb[k][v] = h;
      }
    // the first node's value is lifted by this element (-l_hat0, lower face)
    // and by the lower neighbour (+l_hatN, its upper face, whose primary
    // element this is); a boundary lower face lifts the variables its
    // condition carries, a boundary upper face the own last node's flux
    if (!l.blo) {
#pragma unroll
      for (int v = 0; v < ND; ++v) hb[0][v] += sg_lo * (p.lhatN * r_lo[v + 1] - p.lhat0 * rx[0][v]);
    }
    if constexpr (DIM == 2) {
      int vlo, vhi;
      if (l.blo) {
        wall_viscous_range(p.bc[2 * l.dir], NV, vlo, vhi);
#pragma unroll
        for (int v = 1; v < NV; ++v)
          if (v >= vlo && v < vhi) hb[0][v - 1] -= sg_lo * p.lhat0 * rx[0][v - 1];
      }
      if (l.bhi) {
        wall_viscous_range(p.bc[2 * l.dir + 1], NV, vlo, vhi);
#pragma unroll
        for (int v = 1; v < NV; ++v)
          if (v >= vlo && v < vhi) hb[n - 1][v - 1] += sg_hi * p.lhatN * rx[n - 1][v - 1];
      }
    }
  }
  auto store = [&](const double (&x)[n][ND]) {
#pragma unroll
    for (int k = 0; k < n; ++k)
#pragma unroll
      for (int v = 0; v < ND; ++v) s_g[l.slot * SG + (l.dir * ND + v) * PN + l.pos(k)] = x[k][v];
  };
  __syncthreads();  // every line has read its q and r
  store(acc);
  __syncthreads();
  double tau[PASSES][DIM][DIM];
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (!has_node(k)) continue;
    const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN, pn = lds_pos<N>(node);
    if (sl >= nvalid) continue;
    double ja[DIM][DIM], g[DIM][NV];
    ad_node_metric<DIM, N, NODAL>(p, e0 + sl, node, ja);
    const double ij = inv_jac<NODAL, NN>(p, e0 + sl, node);
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
      g[c][0] = 0.0;
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        double t = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) t += ja[d][c] * s_g[sl * SG + (d * ND + v - 1) * PN + pn];
        g[c][v] = t * ij;
      }
    }
    stress<DIM>(g, tau[k]);
  }
  __syncthreads();
  store(hb);
  __syncthreads();
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    if (!has_node(k)) continue;
    const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN, pn = lds_pos<N>(node);
    if (sl >= nvalid) continue;
    const int64_t e = e0 + sl;
    double ja[DIM][DIM], fb[DIM][NV], qb[NV], gb[DIM][NV];
    ad_node_metric<DIM, N, NODAL>(p, e, node, ja);
    const double ij = inv_jac<NODAL, NN>(p, e, node);
#pragma unroll
    for (int c = 0; c < DIM; ++c) {
      fb[c][0] = gb[c][0] = 0.0;
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        gb[c][v] = 0.0;
        double f = 0.0;
#pragma unroll
        for (int d = 0; d < DIM; ++d) f -= ja[d][c] * s_g[sl * SG + (d * ND + v - 1) * PN + pn];
        fb[c][v] = f;
      }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) qb[v] = 0.0;
    viscous_flux_vjp_stress<DIM>(p.mu, p.kappa, q[k], tau[k], fb, qb, gb);
#pragma unroll
    for (int c = 0; c < DIM; ++c) a.qbar[(e * NV + c + 1) * NN + node] = qb[c + 1];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      double* out = a.dgrad + (e * DIM + d) * (NV * NN) + row_pos<DIM, N>(d, node);
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        double G = 0.0;
#pragma unroll
        for (int c = 0; c < DIM; ++c) G += ja[d][c] * gb[c][v];
        out[v * NN] = ij * G;
      }
    }
  }
}

// Whether the adjoint kernel forms the subcell cotangents of all directions at
// once: in 3D up to N = 3, where a line's n NV cotangents fit the registers its
// other sums have left.  They wait there for their direction's turn to be added, so
// the LDS (40 KB a block at N = 3) holds nothing for them.  32^3, N = 3, one
// direction at a time -> all at once, us an adjoint right-hand side with every
// element troubled: LLF 382 -> 282, HLLC 600 -> 430, viscous 571 -> 477 and 1175 ->
// 630; with none troubled 195 -> 195, 286 -> 287, 394 -> 396 and 655 -> 492 (the
// serial pass took the viscous HLLC kernel past 256 registers).  16^3: 13-40% less.
template <int DIM, int N>
constexpr bool par_subcell_adjoint() {
  return DIM == 3 && N <= 3;
}

template <int DIM, int N, int EPW, bool NODAL, bool NS, bool SC, int SF, int FF>
__global__ void __launch_bounds__((EPW * Shape<DIM, N>::LINES))
    __attribute__((amdgpu_waves_per_eu((ad_waves<N, SC, SF>())))) vjp_rhs_kernel(const AdParams a) {
  using S = Shape<DIM, N>;
  constexpr int n = S::n, NV = S::NV, NN = S::NN, PN = S::PN;
  constexpr int NQ = DIM + 2;  // rho, v[DIM], beta
  constexpr int ND = NV - 1;   // viscous cotangents of v, T
  constexpr int BLOCK = EPW * S::LINES, NODES = EPW * NN, PASSES = (NODES + BLOCK - 1) / BLOCK;
  constexpr int SQ = NQ * PN + S::slot_pad(NQ * PN), SU = S::SU;
  constexpr int SD = NS ? ND * PN + S::slot_pad(ND * PN) : 0;
  const KParams& p = a.k;
  const AdOperators op{a};
  __shared__ double s_p[EPW * SQ];  // rho, v, beta; later their cotangents' sums
  __shared__ double s_r[EPW * SU];
  // conservative cotangents of the faces and subcells; without the subcells'
  // reads of r they take its planes
  __shared__ double s_ub_own[SC ? EPW * SU : 1];
  __shared__ double s_qv[NS ? EPW * SD : 1];
  double* const s_qb = s_p;
  double* const s_ub = SC ? s_ub_own : s_r;
  // PAR_FV: the troubled elements' subcell cotangents are formed by all
  // directions' lines at once instead of one direction at a time.
  constexpr bool PAR_FV = SC && par_subcell_adjoint<DIM, N>();
  const int tid = threadIdx.x;
  const int64_t e0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * EPW;
  const int nvalid = (int)((p.E - e0) < EPW ? (p.E - e0) : EPW);
  auto has_node = [&](int k) { return (k + 1) * BLOCK <= NODES || tid + k * BLOCK < NODES; };
  {
    double u[PASSES][NV], r[PASSES][NV];
#pragma unroll
    for (int k = 0; k < PASSES; ++k) {
      if (has_node(k)) {
        const int i = tid + k * BLOCK, sl = i / NN, node = i - sl * NN;
        const int64_t e = e0 + (sl < nvalid ? sl : nvalid - 1);
        load_state<DIM, NN>(p.u, e, node, u[k]);
        load_r<DIM, NN, NODAL>(a, e, node, r[k]);
      }
    }
#pragma unroll
    for (int k = 0; k < PASSES; ++k) {
      if (has_node(k)) {
        const int i = tid + k * BLOCK, sl = i / NN, pn = lds_pos<N>(i - sl * NN);
        const NodePrims<DIM> q = node_prims<DIM>(p.gamma, u[k]);
        double* d = s_p + sl * SQ + pn;
        d[0] = q.rho;
#pragma unroll
        for (int c = 0; c < DIM; ++c) d[(1 + c) * PN] = q.v[c];
        d[(DIM + 1) * PN] = q.beta;
#pragma unroll
        for (int v = 0; v < NV; ++v) s_r[sl * SU + v * PN + pn] = r[k][v];
      }
    }
  }
  const AdLine<DIM, N, EPW> l(p, tid, e0, nvalid);
  double ja[NODAL ? n : 1][DIM];
  line_metric<DIM, N, EPW, NODAL>(p, l, ja);
  __syncthreads();

  double ub_lo[NV], ub_hi[NV];
#pragma unroll
  for (int v = 0; v < NV; ++v) ub_lo[v] = ub_hi[v] = 0.0;
  // an outflow face's outer state is the mean of the line: its cotangent
  // goes to every node of the line
  double ub_line[NV];
  bool line_mean = false;
#pragma unroll
  for (int v = 0; v < NV; ++v) ub_line[v] = 0.0;
  double qb[n][NQ];  // cotangents of rho, v, beta
#pragma unroll
  for (int k = 0; k < n; ++k)
#pragma unroll
    for (int i = 0; i < NQ; ++i) qb[k][i] = 0.0;
  double qv[NS ? n : 1][ND];
  double coef = 1.0, alpha = 0.0;
  const bool troubled = l.valid && frozen_blend<SC>(p, l.e, coef, alpha);
  bool any = false;  // an element of the block is troubled (uniform)
  if constexpr (PAR_FV) {
#pragma unroll
    for (int sl = 0; sl < EPW; ++sl) {
      double cf, al;
      any = frozen_blend<SC>(p, e0 + (sl < nvalid ? sl : nvalid - 1), cf, al) || any;
    }
  }
  if (l.valid) {
    const double* rr = s_r + l.slot * SU;
    // faces: this element's share of each face flux's adjoint
#pragma unroll 1
    for (int side = 0; side < 2; ++side) {
      const bool lower = side == 0;
      const int od = lower ? l.first() : l.last(), nd = lower ? l.last() : l.first();
      const int64_t nb = lower ? l.lo : l.hi;
      double uo[NV], un[NV], ro[NV], rn[NV], nrm[DIM], g[NV];
      load_state<DIM, NN>(p.u, l.e, od, uo);
      const int po = lower ? l.pos(0) : l.pos(n - 1);
#pragma unroll
      for (int v = 0; v < NV; ++v) ro[v] = rr[v * PN + po];
      bool boundary = false;
      if constexpr (DIM == 2) boundary = lower ? l.blo : l.bhi;
      const int64_t en = lower || boundary ? l.e : nb;
      const int nn = boundary ? od : l.first();
      const double sg = sign_j<NODAL, DIM, NN>(p, en, nn);
#pragma unroll
      for (int c = 0; c < DIM; ++c) nrm[c] = sg * metric<NODAL, DIM, NN>(p, en, l.dir, c, nn);
      if (boundary) {
        if constexpr (DIM == 2) {
          // a non-periodic face: the flux enters this element alone, and the
          // outer state's cotangent maps back through the boundary condition
          int dofs[n];
          for (int k = 0; k < n; ++k) dofs[k] = l.dof(k);
          const int face = 2 * l.dir + side;
          const int64_t bnode = boundary_node<DIM, N>(p, l.e, l.dir, l.line);
          const BcMap m = bc_map<DIM>(p, face, bnode);
          double ul[NV], ur[NV], ubl[NV], ubr[NV];
          bc_outer_state<DIM, N, NN>(p, face, bnode, m, p.u + l.e * NV * NN, dofs, uo, nrm, un);
          for (int v = 0; v < NV; ++v) {
            g[v] = lower ? -p.lhat0 * ro[v] : p.lhatN * ro[v];
            ul[v] = lower ? un[v] : uo[v];
            ur[v] = lower ? uo[v] : un[v];
            ubl[v] = ubr[v] = 0.0;
          }
          if constexpr (SF == kFluxHLLC) {
            hllc_vjp<DIM>(p.gamma, ul, ur, nrm, g, true, true, ubl, ubr);
          } else {
            const NodePrims<DIM> ql = node_prims<DIM>(p.gamma, ul), qr = node_prims<DIM>(p.gamma, ur);
            llf_vjp_side<DIM>(p.gamma, ul, ql, ur, qr, nrm, g, true, ubl);
            llf_vjp_side<DIM>(p.gamma, ul, ql, ur, qr, nrm, g, false, ubr);
          }
          double own[NV], outer[NV];
          for (int v = 0; v < NV; ++v) {
            own[v] = lower ? ubr[v] : ubl[v];
            outer[v] = lower ? ubl[v] : ubr[v];
          }
          if (m == BcMap::kMirror) {
            // the mirror is symmetric: its transpose is itself
            double mn = 0.0, n2 = 0.0;
            for (int c = 0; c < DIM; ++c) {
              mn += outer[1 + c] * nrm[c];
              n2 += nrm[c] * nrm[c];
            }
            mn = mn / n2;
            own[0] += outer[0];
            for (int c = 0; c < DIM; ++c) own[1 + c] += outer[1 + c] - 2.0 * mn * nrm[c];
            own[NV - 1] += outer[NV - 1];
          } else if (m == BcMap::kMean) {
            line_mean = true;
            for (int v = 0; v < NV; ++v) ub_line[v] += outer[v] / (double)n;
          }
          for (int v = 0; v < NV; ++v) {
            ub_lo[v] = lower ? own[v] : ub_lo[v];
            ub_hi[v] = lower ? ub_hi[v] : own[v];
          }
        }
        continue;
      }
      load_state<DIM, NN>(p.u, nb, nd, un);
      load_r<DIM, NN, NODAL>(a, nb, nd, rn);
      double ul[NV], ur[NV], ubf[NV];
      // the face flux enters the upper element's first node with -l_hat0
      // and the lower element's last node with +l_hatN
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        g[v] = lower ? p.lhatN * rn[v] - p.lhat0 * ro[v] : p.lhatN * ro[v] - p.lhat0 * rn[v];
        ul[v] = lower ? un[v] : uo[v];
        ur[v] = lower ? uo[v] : un[v];
        ubf[v] = 0.0;
      }
      // this element is the face's right state at its lower face
      if constexpr (SF == kFluxHLLC)
        hllc_vjp<DIM>(p.gamma, ul, ur, nrm, g, !lower, lower, ubf, ubf);
      else
        llf_vjp_side<DIM>(p.gamma, ul, node_prims<DIM>(p.gamma, ul), ur, node_prims<DIM>(p.gamma, ur),
                          nrm, g, !lower, ubf);
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        ub_lo[v] = lower ? ubf[v] : ub_lo[v];
        ub_hi[v] = lower ? ub_hi[v] : ubf[v];
      }
    }
    pin_values<NV>(ub_lo);
    pin_values<NV>(ub_hi);

    const double* pr = s_p + l.slot * SQ;
    auto prims = [&](int pos) {
      NodePrims<DIM> q;
      q.rho = pr[pos];
#pragma unroll
      for (int c = 0; c < DIM; ++c) q.v[c] = pr[(1 + c) * PN + pos];
      q.beta = pr[(DIM + 1) * PN + pos];
      q.kin = q.p = q.c = 0.0;
      return q;
    };
    auto add = [](double* t, const PrimTangent<DIM>& x) {
      t[0] += x.rho;
#pragma unroll
      for (int c = 0; c < DIM; ++c) t[1 + c] += x.v[c];
      t[DIM + 1] += x.beta;
      pin_values<NQ>(t);
    };
#pragma unroll
    for (int ia = 0; ia < n - 1; ++ia) {
      const NodePrims<DIM> qa = prims(l.pos(ia));
#pragma unroll
      for (int ib = ia + 1; ib < n; ++ib) {
        const NodePrims<DIM> qbn = prims(l.pos(ib));
        double nrm[DIM], g[NV];
#pragma unroll
        for (int c = 0; c < DIM; ++c) nrm[c] = NODAL ? ja[NODAL ? ia : 0][c] + ja[NODAL ? ib : 0][c] : ja[0][c];
        const double wa = coef * op.Ds(ia, ib), wb = coef * op.Ds(ib, ia);
#pragma unroll
        for (int v = 0; v < NV; ++v) g[v] = wa * rr[v * PN + l.pos(ia)] + wb * rr[v * PN + l.pos(ib)];
        PrimTangent<DIM> xa{}, xb{};
        chandrashekar_vjp<DIM>(p.inv_gm1, qa, qbn, nrm, g, xa, xb);
        add(qb[ia], xa);
        add(qb[ib], xb);
      }
    }
    // Navier-Stokes: the transposed D_hat of Gbar, and the BR1 averages q_hat =
    // (q_L + q_R)/2 on this element's faces and on the neighbours' faces that
    // used this element's face values
    if constexpr (NS) {
      const double sg_lo = sign_j<NODAL, DIM, NN>(p, l.e, l.first());
      const double sg_hi = sign_j<NODAL, DIM, NN>(p, l.e, l.last());
      const double nsg_lo = sign_j<NODAL, DIM, NN>(p, l.lo, l.last());
      const double nsg_hi = sign_j<NODAL, DIM, NN>(p, l.hi, l.first());
      const double* G = a.dgrad + (l.e * DIM + l.dir) * (NV * NN) + l.line * n;
      const double* Glo = a.dgrad + (l.lo * DIM + l.dir) * (NV * NN) + l.line * n + N;
      const double* Ghi = a.dgrad + (l.hi * DIM + l.dir) * (NV * NN) + l.line * n;
      double x_lo[NV], x_hi[NV];  // the faces' own terms
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        double x[n];
#pragma unroll
        for (int k = 0; k < n; ++k) x[k] = G[v * NN + k];
#pragma unroll
        for (int k = 0; k < n; ++k) {
          double h = 0.0;
#pragma unroll
          for (int i = 0; i < n; ++i) h += op.Dhat(i, k) * x[i];
          qv[k][v - 1] = h;
        }
        x_lo[v] = -sg_lo * p.lhat0 * x[0];
        x_hi[v] = sg_hi * p.lhatN * x[n - 1];
        if (!l.blo) qv[0][v - 1] += 0.5 * (nsg_lo * p.lhatN * Glo[v * NN] + x_lo[v]);
        if (!l.bhi) qv[n - 1][v - 1] += 0.5 * (x_hi[v] - nsg_hi * p.lhat0 * Ghi[v * NN]);
      }
      // a boundary face's value is the wall map of the own node's variables:
      // its transpose (the map itself) takes the face term's cotangent back
      if constexpr (DIM == 2) {
        auto wall = [&](int side, int dof, double sg, double* x, double* out) {
          double nrm[DIM], y[NV];
          x[0] = 0.0;
          for (int c = 0; c < DIM; ++c) nrm[c] = sg * metric<NODAL, DIM, NN>(p, l.e, l.dir, c, dof);
          wall_gradient_linear<DIM>(p.bc[2 * l.dir + side], x, nrm, y);
          for (int v = 1; v < NV; ++v) out[v - 1] += y[v];
        };
        if (l.blo) wall(0, l.first(), sg_lo, x_lo, qv[0]);
        if (l.bhi) wall(1, l.last(), sg_hi, x_hi, qv[n - 1]);
      }
    }
  }
  __syncthreads();  // the sums take the planes of the primitives (and of r)
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    if (l.valid && l.dir == d) {
#pragma unroll
      for (int k = 0; k < n; ++k) {
        double* t = s_qb + l.slot * SQ + l.pos(k);
#pragma unroll
        for (int i = 0; i < NQ; ++i) t[i * PN] = d == 0 ? qb[k][i] : t[i * PN] + qb[k][i];
        if constexpr (NS) {
          double* w = s_qv + l.slot * SD + l.pos(k);
#pragma unroll
          for (int i = 0; i < ND; ++i) w[i * PN] = d == 0 ? qv[k][i] : w[i * PN] + qv[k][i];
        }
        // the conservative cotangents touch the line's end nodes (and, with
        // an outflow face, all of them); the first direction sets every node
        double* x = s_ub + l.slot * SU + l.pos(k);
        if (d == 0 || k == 0 || k == n - 1 || (DIM == 2 && line_mean)) {
#pragma unroll
          for (int v = 0; v < NV; ++v) {
            double o = k == 0 ? ub_lo[v] : (k == n - 1 ? ub_hi[v] : 0.0);
            if constexpr (DIM == 2) o += ub_line[v];
            x[v * PN] = d == 0 ? o : x[v * PN] + o;
          }
        }
      }
      // subcell fluxes of a troubled element: flux fi enters node fi - 1
      // with alpha w_inv(fi - 1) and node fi with -alpha w_inv(fi); each line
      // owns its nodes within this direction, so the sums need no atomics
      if constexpr (SC && !PAR_FV) {
        if (troubled) {
          const double* rr = s_r + l.slot * SU;
#pragma unroll 1
          for (int fi = 1; fi < n; ++fi) {
            double ul[NV], ur[NV], nrm[DIM], g[NV], ubl[NV], ubr[NV];
            load_state<DIM, NN>(p.u, l.e, l.dof(fi - 1), ul);
            load_state<DIM, NN>(p.u, l.e, l.dof(fi), ur);
            subcell_normal<DIM, N, NODAL>(p, l.e, l.dir, l.line, fi - 1, nrm);
            const double wl = alpha * op.inv_w(fi - 1), wr = alpha * op.inv_w(fi);
            for (int v = 0; v < NV; ++v) {
              g[v] = wl * rr[v * PN + l.pos(fi - 1)] - wr * rr[v * PN + l.pos(fi)];
              ubl[v] = ubr[v] = 0.0;
            }
            if constexpr (FF == kFluxHLLC) {
              hllc_vjp<DIM>(p.gamma, ul, ur, nrm, g, true, true, ubl, ubr);
            } else {
              const NodePrims<DIM> ql = node_prims<DIM>(p.gamma, ul), qr = node_prims<DIM>(p.gamma, ur);
              llf_vjp_side<DIM>(p.gamma, ul, ql, ur, qr, nrm, g, true, ubl);
              llf_vjp_side<DIM>(p.gamma, ul, ql, ur, qr, nrm, g, false, ubr);
            }
            for (int v = 0; v < NV; ++v) {
              s_ub[l.slot * SU + v * PN + l.pos(fi - 1)] += ubl[v];
              s_ub[l.slot * SU + v * PN + l.pos(fi)] += ubr[v];
            }
          }
        }
      }
    }
    __syncthreads();
  }
  // PAR_FV: the same subcell terms, formed by all directions' lines at once now
  // that the line's other sums are in LDS (and their registers free), then added
  // one direction at a time.
  if constexpr (PAR_FV) {
    if (any) {
      double fv[n][NV];
#pragma unroll
      for (int k = 0; k < n; ++k)
#pragma unroll
        for (int v = 0; v < NV; ++v) fv[k][v] = 0.0;
      if (troubled) {
        const double* rr = s_r + l.slot * SU;
#pragma unroll
        for (int fi = 1; fi < n; ++fi) {
          double ul[NV], ur[NV], nrm[DIM], g[NV];
          load_state<DIM, NN>(p.u, l.e, l.dof(fi - 1), ul);
          load_state<DIM, NN>(p.u, l.e, l.dof(fi), ur);
          subcell_normal<DIM, N, NODAL>(p, l.e, l.dir, l.line, fi - 1, nrm);
          const double wl = alpha * op.inv_w(fi - 1), wr = alpha * op.inv_w(fi);
#pragma unroll
          for (int v = 0; v < NV; ++v)
            g[v] = wl * rr[v * PN + l.pos(fi - 1)] - wr * rr[v * PN + l.pos(fi)];
          if constexpr (FF == kFluxHLLC) {
            hllc_vjp<DIM>(p.gamma, ul, ur, nrm, g, true, true, fv[fi - 1], fv[fi]);
          } else {
            const NodePrims<DIM> ql = node_prims<DIM>(p.gamma, ul), qr = node_prims<DIM>(p.gamma, ur);
            llf_vjp_side<DIM>(p.gamma, ul, ql, ur, qr, nrm, g, true, fv[fi - 1]);
            llf_vjp_side<DIM>(p.gamma, ul, ql, ur, qr, nrm, g, false, fv[fi]);
          }
          pin_values<NV>(fv[fi - 1]);
          pin_values<NV>(fv[fi]);
        }
      }
#pragma unroll
      for (int d = 0; d < DIM; ++d) {
        if (troubled && l.dir == d) {
#pragma unroll
          for (int k = 0; k < n; ++k)
#pragma unroll
            for (int v = 0; v < NV; ++v) s_ub[l.slot * SU + v * PN + l.pos(k)] += fv[k][v];
        }
        __syncthreads();
      }
    }
  }
  for (int i = tid; i < NODES; i += BLOCK) {
    const int sl = i / NN, node = i - sl * NN, pn = lds_pos<N>(node);
    if (sl >= nvalid) continue;
    const int64_t e = e0 + sl;
    double u[NV], ub[NV];
    load_state<DIM, NN>(p.u, e, node, u);
    const NodePrims<DIM> q = node_prims<DIM>(p.gamma, u);
    const double* t = s_qb + sl * SQ + pn;
    PrimTangent<DIM> qbar;
    qbar.rho = t[0];
#pragma unroll
    for (int c = 0; c < DIM; ++c) qbar.v[c] = t[(1 + c) * PN];
    qbar.beta = t[(DIM + 1) * PN];
    qbar.kin = 0.0;  // the pair flux does not take it
#pragma unroll
    for (int v = 0; v < NV; ++v) ub[v] = s_ub[sl * SU + v * PN + pn];
    prims_vjp<DIM>(p.gamma, q, qbar, 0.0, ub);
    if constexpr (NS) {
      double x[NV];
      x[0] = 0.0;  // the gradient does not differentiate rho
#pragma unroll
      for (int v = 1; v < NV; ++v) x[v] = s_qv[sl * SD + (v - 1) * PN + pn];
#pragma unroll
      for (int c = 0; c < DIM; ++c) x[1 + c] += a.qbar[(e * NV + c + 1) * NN + node];
      grad_vars_vjp<DIM>(p.gamma, u, x, ub);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      const int64_t g = (e * NV + v) * NN + node;
      a.out[g] = combine(a, g, ub[v]);
    }
  }
}

// The Navier-Stokes derivatives run the viscous kernel first (it fills a.dgrad,
// which the RHS kernel takes); every RHS kernel takes the flux kinds as template
// arguments.
template <int DIM, int N, bool NODAL, bool SC, bool ADJ>
hipError_t launch_ad_t(bool ns, const AdParams& a, hipStream_t s) {
  constexpr int EPW = ad_elems_per_block<DIM, N>();
  constexpr int BLOCK = EPW * Shape<DIM, N>::LINES;
  const int64_t nb = (a.k.E + EPW - 1) / EPW;
  if (nb <= 0) return hipSuccess;
  const dim3 grid((unsigned)nb), block(BLOCK);
  if (ns) {
    // its launch is checked with the RHS kernel's
    if constexpr (ADJ) {
      hipLaunchKernelGGL((vjp_viscous_kernel<DIM, N, EPW, NODAL>), grid, block, 0, s, a);
    } else {
      hipLaunchKernelGGL((jvp_viscous_kernel<DIM, N, EPW, NODAL>), grid, block, 0, s, a);
    }
  }
  const bool shllc = a.k.surface_flux == kFluxHLLC, fhllc = SC && a.k.fv_flux == kFluxHLLC;
  auto go = [&](auto nsv, auto sf, auto ff) {
    constexpr bool NSv = decltype(nsv)::value;
    constexpr int SFv = decltype(sf)::value, FFv = decltype(ff)::value;
    if constexpr (ADJ)
      hipLaunchKernelGGL((vjp_rhs_kernel<DIM, N, EPW, NODAL, NSv, SC, SFv, FFv>), grid, block, 0, s,
                         a);
    else
      hipLaunchKernelGGL((jvp_rhs_kernel<DIM, N, EPW, NODAL, NSv, SC, SFv, FFv>), grid, block, 0, s,
                         a);
    return hipGetLastError();
  };
  auto flux = [&](auto nsv) {
    using LLF = std::integral_constant<int, kFluxLLF>;
    using HLLC = std::integral_constant<int, kFluxHLLC>;
    if constexpr (SC) {
      if (shllc) return fhllc ? go(nsv, HLLC{}, HLLC{}) : go(nsv, HLLC{}, LLF{});
      return fhllc ? go(nsv, LLF{}, HLLC{}) : go(nsv, LLF{}, LLF{});
    } else {
      return shllc ? go(nsv, HLLC{}, LLF{}) : go(nsv, LLF{}, LLF{});
    }
  };
  return ns ? flux(std::true_type{}) : flux(std::false_type{});
}

template <int DIM, int N, bool NODAL, bool SC>
hipError_t launch_jvp_t(bool ns, const AdParams& a, hipStream_t s) {
  return launch_ad_t<DIM, N, NODAL, SC, false>(ns, a, s);
}

template <int DIM, int N, bool NODAL, bool SC>
hipError_t launch_vjp_t(bool ns, const AdParams& a, hipStream_t s) {
  return launch_ad_t<DIM, N, NODAL, SC, true>(ns, a, s);
}

}  // namespace detail
}  // namespace dgsem
