// Kernel parameter block and launch entry points shared by the ABI layer
// and the kernel translation unit.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace dgsem {

constexpr int kMaxN1 = 8;  // max nodes per direction (N <= 7)

#ifndef DGSEM_NODE_KERNEL_MIN_N
#define DGSEM_NODE_KERNEL_MIN_N 7
#endif

// Split-form elements of degree N >= 7 on periodic meshes run the
// node-parallel kernel, in 2D and 3D.
__host__ __device__ constexpr bool node_kernel_for(int N, bool shock_capturing, bool boundaries) {
  return !shock_capturing && !boundaries && N >= DGSEM_NODE_KERNEL_MIN_N;
}

enum StageMode : int {
  kModeRhs = 0,     // out = L(u)
  kModeStage2 = 1,  // out = c1 u + c2 L(u)                (parallel_ma2)
  kModeStage3 = 2,  // out = c1 u_base + c2 u + c3 L(u)    (parallel_ma3)
};

// Boundary condition kinds per face (values of DGSEM_BC_* in the C header).
enum BoundaryKind : int {
  kBcPeriodic = 0,
  kBcSlipWall = 1,
  kBcOutflow = 2,
  kBcDirichlet = 3,
  kBcNsNoSlipWall = 4,  // Navier-Stokes adiabatic walls
  kBcNsSlipWall = 5,
  kBcMixedDirichletSlipWall = 6,  // per-node choice, states [node][NV + 1]
};

// Division of 0 <= x < 2^31 by a constant d >= 1 as a multiply-high and a
// shift: with s = ceil(log2 d) and mul = floor(2^(31+s) / d) + 1, x / d is
// x mul >> (31 + s): mul d = 2^(31+s) + r with 0 < r <= d <= 2^s, and x r <
// 2^(31+s) keeps the excess below 1 / d.  A division by a run-time value takes
// some twenty instructions otherwise.
struct FastDiv {
  uint32_t mul;
  int32_t shift;
  __host__ __device__ static FastDiv by(uint32_t d) {
    int s = 0;
    while ((1ull << s) < d) ++s;
    return {(uint32_t)((1ull << (31 + s)) / d + 1), s};
  }
  __host__ __device__ int operator()(int x) const {
    return (int)((uint32_t)((((uint64_t)(uint32_t)x << 1) * mul) >> 32) >> shift);
  }
};

// Ordered by use: what a kernel's first loads need comes first, so that it
// arrives with the first scalar load.
struct KParams {
  const double* u;       // stage input, [E][NV][NN]
  const double* basis;   // operators of the 1D basis (Operators below)
  int64_t E;
  int cells[3];
  int mode;
  FastDiv div_y, div_z;  // by cells[1] and cells[2]
  // Box meshes (the linear mapping of a Cartesian box, nodal geometry): the
  // halved metric terms Ja^r_c / 2 of a node depend on its element only through the
  // element's indices in the directions other than c, so each distinct row
  // is stored once: ja_box[ja_box_off[c] + (pair * DIM + r) * NN + line * n + k]
  // with pair = i_m * cells[l] + i_l (3D; m = c+1, l = c+2 mod 3) or i_m (2D;
  // m = 1-c), for node k of line `line` of direction r: the row a line thread
  // reads is contiguous.  Null unless the mesh is such a box, whose 1/J is
  // then positive at every node.
  const double* ja_box;
  int64_t ja_box_off[3];
  const double* Ja;      // nodal: [E][dim][dim][NN]; affine: [E][dim][dim]
  const double* invJ;    // nodal: [E][NN]; affine: [E]
  double gamma, inv_gm1;
  double lhat0, lhatN;
  const double* visc;    // Navier-Stokes: viscous fluxes (parabolic_impl.hpp)
  double* visc_out;      // written by the viscous kernel
  double mu, kappa;      // viscosity and gamma / ((gamma - 1) Pr)
  const double* sn;      // nodal subcell normals [E][dim][FN][N][dim]
  const double* alpha_in;  // [E] frozen blending factor to use instead of the
                           // indicator's (shock capturing), or null
  double* alpha;         // [E] blending factor (shock capturing), written
  double alpha_max, alpha_min, atol, threshold, sfac;
  int surface_flux, fv_flux;  // FluxKind
  int volume_flux;            // VolumeFluxKind (read by the run-time flux kernels only)
  const double* u_base;  // base state for kModeStage3
  double* out;           // L(u) or the stage result
  double c1, c2, c3;
  double floor_value;
  // boundary conditions (2D): kind per face (-x, +x, -y, +y; 0 = periodic),
  // constant Dirichlet states and optional per-node Dirichlet states
  int bc[6];
  double bc_state[6][5];
  const double* bc_values[6];
  int cus;               // compute units of the device, for the launchers' choice of kernel
};

// The basis operators of N + 1 = n nodes at KParams::basis: D_split, D_hat and
// the inverse Legendre Vandermonde matrix, n x n each, then the n inverse
// weights.  They sit in device memory rather than among the kernel's arguments:
// a launch's arguments are new to every cache, the table is not (a kernel that
// only sums 52 of 208 values takes 5.0 us a launch from arguments, 2.5 from a
// table).  The table is constant while kernels run, so its loads are scalar
// (address space 4).  One MI355X, with the arguments in the order of their use:
// Sedov blast 32^3, N = 3, 313 -> 293 us a step; 2D Riemann problem 101 x 97,
// N = 5, 261 -> 255 us for four; an ensemble of 64 2D cases 425 -> 404 us for two.
template <int N>
struct Operators {
  static constexpr int n = N + 1;
#if defined(__HIP_DEVICE_COMPILE__)
  using Table = const __attribute__((address_space(4))) double*;
#else
  using Table = const double*;
#endif
  Table t;
  __host__ __device__ explicit Operators(const KParams& p) : t((Table)p.basis) {}
  __host__ __device__ double Ds(int i, int j) const { return t[i * n + j]; }
  __host__ __device__ double Dhat(int i, int j) const { return t[n * n + i * n + j]; }
  __host__ __device__ double Vinv(int i, int j) const { return t[2 * n * n + i * n + j]; }
  __host__ __device__ double inv_w(int i) const { return t[3 * n * n + i]; }
};

// Per-(dim, N) launchers, explicitly specialised in rhs_inst.hip.
// boundaries: some face is not periodic (2D only)
template <int DIM, int N>
hipError_t launch_rhs_dn(bool shock_capturing, bool nodal, bool boundaries, const KParams& p,
                         hipStream_t stream);
template <int DIM, int N>
hipError_t launch_parabolic_dn(bool shock_capturing, bool nodal, bool boundaries, const KParams& p,
                               hipStream_t stream);

// The Navier-Stokes terms: the viscous fluxes of p.u into p.visc_out, in the
// layout the RHS kernel of the configuration reads (parabolic_impl.hpp).
hipError_t launch_parabolic(int dim, int N, bool shock_capturing, bool nodal, bool boundaries,
                            const KParams& p, hipStream_t stream);

// Launches the fused RHS / stage kernel for the configuration; returns
// hipErrorInvalidValue when (dim, N, shock capturing, nodal) is not built.
hipError_t launch_rhs(int dim, int N, bool shock_capturing, bool nodal, bool boundaries,
                      const KParams& p, hipStream_t stream);

// Layout conversion between the reference layout [e][dof][v] and the
// internal layout [e][v][dof]; to_internal selects the direction.
hipError_t launch_pack(const double* src, double* dst, int64_t E, int nn, int nv,
                       bool to_internal, hipStream_t stream);

// Same between a column-major (LayoutLeft) reference view u(ie, je[, ke],
// dof, var) over cells[0] x cells[1] x cells[2] elements and the internal
// layout.
hipError_t launch_pack_left(const double* src, double* dst, const int cells[3], int nn, int nv,
                            bool to_internal, hipStream_t stream);

// Tangent (JVP) and adjoint (VJP) of the right-hand side at the state k.u
// (adjoint_impl.hpp).  Op is J = dL/du (tangent) or J^T (adjoint) and the
// kernels write
//     out = a1 x1 + a2 x2 + b v + c Op(v)
// (x1, x2 may be null), which covers the tangent and adjoint of every SSPRK3
// stage.  Navier-Stokes needs the scratch arrays dgrad [E][dim][NV][NN] (null
// for Euler) and qbar [E][NV][NN].
struct AdParams {
  KParams k;
  double Ds[kMaxN1][kMaxN1], Dhat[kMaxN1][kMaxN1], inv_w[kMaxN1];  // as Operators
  const double* v;  // tangent direction or cotangent
  const double* x1;
  const double* x2;
  double a1, a2, b, c;
  double* out;
  double* dgrad;
  double* qbar;
};

template <int DIM, int N>
hipError_t launch_jvp_dn(bool nodal, const AdParams& a, hipStream_t stream);
template <int DIM, int N>
hipError_t launch_vjp_dn(bool nodal, const AdParams& a, hipStream_t stream);
// Launch the tangent or adjoint kernels for (dim, N).
hipError_t launch_jvp(int dim, int N, bool nodal, bool navier_stokes, const AdParams& a,
                      hipStream_t stream);
hipError_t launch_vjp(int dim, int N, bool nodal, bool navier_stokes, const AdParams& a,
                      hipStream_t stream);
// Kinetic energy sum_e sum_i w_i / |1/J_i| |m_i|^2 / (2 rho_i) into *result
// (device), and its gradient: grad += scale * dKE/du.  partial: scratch of
// ke_partials(E) doubles.
int64_t ke_partials(int64_t E);
hipError_t launch_kinetic_energy(int dim, int nn, const double* w_nodes, bool nodal,
                                 const KParams& p, double* partial, double* result,
                                 hipStream_t stream);
hipError_t launch_kinetic_energy_grad(int dim, int nn, const double* w_nodes, bool nodal,
                                      const KParams& p, double scale, double* grad,
                                      hipStream_t stream);

// Batched ensembles of 2D cases (batch_impl.hpp).  A tile is up to
// batch_slots(block, N) consecutive elements of one case.
struct BatchTile {
  int32_t case_id;
  int16_t polydeg;
  int16_t nvalid;  // elements in this tile
  int64_t e0;      // first element of the tile within its case
};

// The tile list is sorted by degree, highest first: the tiles of degree N
// are [begin[N], begin[N - 1]), and begin[0] is the number of tiles.
struct BatchRanges {
  int begin[8];
};

struct BatchLaunch {
  const BatchTile* tiles;
  int ntiles;
  BatchRanges ranges;
  const KParams* params;  // one per case
  int grid;               // persistent workgroups
  size_t lds_bytes;       // dynamic LDS: the largest tile footprint in the batch
  bool shock_capturing, nodal;
  int surface_flux, fv_flux;
  int* probe;  // non-null: store the resident workgroups per CU instead of launching
};

// Workgroup sizes the batch kernel is built for.
constexpr int kBatchBlocks[] = {128, 256};

// Workgroups of a batch launch: as many as wanted, but no more than there are tiles
// (the kernel strides by the grid) and than fit the 2^32 - 1 work-items of a launch.
constexpr int batch_grid(int64_t wanted, int64_t ntiles, int block) {
  const int64_t most = 0xffffffffll / block, g = wanted < ntiles ? wanted : ntiles;
  return (int)(g < 1 ? 1 : (g < most ? g : most));
}

template <int BLOCK>
hipError_t launch_batch_bs(const BatchLaunch& b, hipStream_t stream);
hipError_t launch_batch(int block, const BatchLaunch& b, hipStream_t stream);
// Element slots of one tile and its LDS bytes, for a 2D tile of degree N;
// 0 when (block, N) is not built.
int batch_slots(int block, int polydeg);
size_t batch_lds_bytes(int block, int polydeg);

}  // namespace dgsem
