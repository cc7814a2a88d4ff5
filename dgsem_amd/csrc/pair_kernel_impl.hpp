// RHS / stage kernel of small 2D grids: one thread per two-point flux.
//
// The line kernel (rhs_kernel) gives a thread a whole line: N (N + 1) / 2 pair
// fluxes, two face fluxes and N subcell fluxes, one after the other.  On a grid
// that leaves the chip's SIMDs empty that chain is the run time (2D, 16 x 16
// elements, N = 3, Kelvin-Helmholtz with the indicator: 5 of 12 us a launch are
// pair fluxes, 2.3 the indicator and the subcells, and an empty launch takes 1.7).
// Here the fluxes of a line go to different threads and meet in LDS:
//   wave 0             one thread per node: state, metric rows and primitives into
//                      LDS; the blending factors while the other waves form
//                      fluxes; at the end the sums of the node's fluxes and the
//                      stage combination
//   the next waves     one thread per pair flux
//   the last waves     one thread per face flux (line end), whose neighbour trace
//                      they load while wave 0 stages
// then all of them the subcell fluxes, in blocks with a troubled element.  A
// block takes the EPW elements whose nodes fit wave 0.
//
// The sums run in the line kernel's order on the same operations (surface terms,
// pairs by the other node, subcell faces, viscous terms; then direction 0 +
// direction 1), so both kernels give the same bits and the choice between them
// (pair_kernel_for) cannot be seen in the results.  Bounded by latency: of the 6.4
// us a launch takes at 16 x 16, N = 3 (11.7 in the line kernel), 1.7 are an empty
// launch's and 0.7 a copy's; then come one flux, the indicator and the sums, each
// behind a barrier.
#pragma once

namespace dgsem {
namespace detail {

template <int N>
struct PairShape {
  static constexpr int n = N + 1, NN = n * n, PN = Shape<2, N>::PN;
  static constexpr int EPW = 64 / NN;                 // elements per block
  static constexpr int LINES = 2 * n, LP = n * N / 2;  // lines per element, pairs per line
  static constexpr int NODES = EPW * NN, PAIRS = EPW * LINES * LP;
  static constexpr int FACES = EPW * LINES * 2, SUBS = EPW * LINES * N;
  static constexpr int INTER = EPW * LINES * (n + 1);  // interfaces: line ends and subcell faces
  static constexpr int PAIR_WAVES = (PAIRS + 63) / 64, FACE_WAVES = (FACES + 63) / 64;
  static constexpr int BLOCK = 64 * (1 + PAIR_WAVES + FACE_WAVES);
};

// Waves per SIMD the registers are held to: with LLF fluxes six, so that four
// blocks of five waves find their places on a CU (at five per SIMD the 64 x 64 grid
// of N = 3 took 8.6 us a launch instead of 7.1); nine-wave blocks (N = 7) and the
// HLLC and run-time kinds would spill.
template <int N, int SF, int FF>
constexpr int pair_waves_per_simd() {
  return SF == kFluxLLF && FF == kFluxLLF && N != 7 ? 6 : 5;
}

// The pair kernel serves grids whose blocks all fit the device's CUs at once (N = 7:
// twice over): beyond that its waves queue, while the line kernel, with fewer
// instructions per flux, still fits.  The HLLC kinds fill five waves per SIMD
// badly, and with viscous terms the viscous kernel takes a share of the gain:
// 16 waves per CU for both.  Times per launch at the sides of the line on 256 CUs,
// line kernel -> this one (us; Kelvin-Helmholtz with the indicator, LLF):
//   N = 1 (24576 elements)  128 x 128: 7.1 -> 6.6    160 x 160:  8.5 ->  9.0
//   N = 2 (7168)              64 x 64: 8.4 -> 7.8      96 x 96:  9.8 -> 11.0
//   N = 3 (4096)              64 x 64: 9.1 -> 7.5      96 x 96: 10.6 -> 14.2
//   N = 4 (2048)            32 x 32: 13.5 -> 7.8       64 x 64: 12.6 -> 15.9
//   N = 5 (1024)            32 x 32: 15.9 -> 8.9       48 x 48: 15.0 -> 15.8
//   N = 7 (1024)            32 x 32: 23.8 -> 15.9      48 x 48: 22.5 -> 26.9
// HLLC without the indicator, N = 3 (3072): 48 x 48 8.5 -> 7.2, 64 x 64 8.8 -> 9.3;
// viscous, N = 5 (768): 16 x 16 16.6 -> 12.1, 32 x 32 15.8 -> 13.8 (more at N = 3:
// 64 x 64 11.0 -> 12.2).
template <int N, int SF, int FF>
constexpr bool pair_kernel_for(int64_t E, bool viscous, int cus) {
  constexpr bool llf = SF == kFluxLLF && FF == kFluxLLF;
  constexpr int waves = PairShape<N>::BLOCK / 64, rounds = N == 7 ? 2 : 1;
  const int per_cu = viscous || !(llf || N == 7) ? 16 : 4 * pair_waves_per_simd<N, SF, FF>();
  return E <= (int64_t)PairShape<N>::EPW * cus * (per_cu / waves) * rounds;
}

// Orders the LDS accesses of one wave among its lanes.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Blending factors of the block's elements by one wave, block_alpha's sweeps and
// sums with a lane per node: w is the lane's indicator variable, s_w a plane per
// element, V the inverse Vandermonde matrix.  The three energy sums of an element run in three lanes.
template <int N>
__device__ __forceinline__ void wave_alpha(const KParams& p, double w, const double* V, int lane,
                                           double* s_w, double* s_alpha) {
  using W = PairShape<N>;
  constexpr int n = W::n, NN = W::NN, PN = W::PN;
  const bool node = lane < W::NODES;
  const int slot = node ? lane / NN : 0, dof = node ? lane % NN : 0, i = dof % n, j = dof / n;
  double* const A = s_w + slot * PN;
  if (node) A[lds_pos<N>(dof)] = w;
  wave_sync();
  double r = 0.0;
#pragma unroll
  for (int ii = 0; ii < n; ++ii) r += V[i * n + ii] * A[j * (n + 1) + ii];
  wave_sync();
  if (node) A[lds_pos<N>(dof)] = r;
  wave_sync();
  r = 0.0;
#pragma unroll
  for (int jj = 0; jj < n; ++jj) r += V[j * n + jj] * A[jj * (n + 1) + i];
  wave_sync();
  if (node) A[lds_pos<N>(dof)] = r;
  wave_sync();
  // lane = 3 element + q: the modes below n - q in both directions
  const int el = lane / 3 < W::EPW ? lane / 3 : 0, lim = n - lane % 3;
  double sum = 0.0;
#pragma unroll
  for (int jj = 0; jj < n; ++jj)
#pragma unroll
    for (int ii = 0; ii < n; ++ii) {
      const double m = s_w[el * PN + jj * (n + 1) + ii];
      const double t = sum + m * m;
      sum = jj < lim && ii < lim ? t : sum;
    }
  const int src = lane < W::EPW ? 3 * lane : 0;
  const double total = __shfl(sum, src), clip1 = __shfl(sum, src + 1), clip2 = __shfl(sum, src + 2);
  if (lane < W::EPW) s_alpha[lane] = blending_factor(p, total, clip1, clip2);
}

// The metric terms come from the full arrays on box meshes too: at these sizes
// the table of the larger grids (box_table_for) saves no time on memory and its
// addresses cost 2%.
template <int N, bool SC, bool NODAL, int SF, int FF, bool BCS>
__global__ void __launch_bounds__(PairShape<N>::BLOCK)
    __attribute__((amdgpu_waves_per_eu(pair_waves_per_simd<N, SF, FF>())))
    rhs_pair_kernel(const KParams p) {
  using W = PairShape<N>;
  constexpr int n = W::n, NV = 4, NN = W::NN, PN = W::PN, EPW = W::EPW, LP = W::LP;
  __shared__ double s_u[EPW * NV * PN];   // [slot][var][node]
  __shared__ double s_p[EPW * 3 * PN];    // [slot][v, beta][node]
  __shared__ double s_ja[NODAL ? EPW * 4 * PN : 1];  // [slot][dir * 2 + c][node], halved
  __shared__ double s_w[SC ? EPW * PN : 1];
  __shared__ double s_alpha[EPW];
  __shared__ double s_f[NV * W::PAIRS];   // pair fluxes, [var][slot, dir, line, pair]
  __shared__ double s_i[NV * W::INTER];   // interface fluxes, [var][slot, dir, line, interface]
  __shared__ double s_v[6 * W::NODES];    // viscous terms, [dir][var - 1][node]
  __shared__ double s_op[3 * NN + n];     // the basis operators

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t e0 = (int64_t)xcd_block(blockIdx.x, gridDim.x) * EPW;
  const int nvalid = (int)((p.E - e0) < EPW ? (p.E - e0) : EPW);
  // slots past the last valid element work on a copy of it
  auto element = [&](int slot) { return e0 + (slot < nvalid ? slot : nvalid - 1); };

  // 1. loads.  Wave 0: the node's state, metric rows and what the sums need at
  // the end; the face waves: the far trace and the metric at the face node.
  const int nslot = lane < W::NODES ? lane / NN : 0, node = lane < W::NODES ? lane % NN : 0;
  const int ni = node % n, nj = node / n, npos = nslot * NV * PN + lds_pos<N>(node);
  const bool with_base = p.mode == kModeStage3;
  double u[NV], ub[NV], fac = 0.0;
  const int ft = (wave - 1 - W::PAIR_WAVES) * 64 + lane;  // face item [slot][dir][side][line]
  const bool face = wave > W::PAIR_WAVES && ft < W::FACES;
  const int fline = ft % n, fside = ft / n % 2, fdir = ft / (2 * n) % 2, fslot = ft / (4 * n);
  double far[NV], nrm_f[2];
  int fid[3];
  bool boundary = false;
  int64_t fe = 0;
  if (wave == 0) {
    const int64_t e = element(nslot);
    const double* src = p.u + e * (NV * NN) + node;
#pragma unroll
    for (int v = 0; v < NV; ++v) u[v] = src[v * NN];
    double ja[4];
    if constexpr (NODAL) {
#pragma unroll
      for (int k = 0; k < 4; ++k) ja[k] = 0.5 * p.Ja[(e * 4 + k) * NN + node];
    }
    fac = NODAL ? -p.invJ[e * NN + node] : -p.invJ[e];
    if (with_base) {
#pragma unroll
      for (int v = 0; v < NV; ++v) ub[v] = p.u_base[e * (NV * NN) + node + v * NN];
    }
    if (lane < W::NODES) {
      const NodePrims<2> q = node_prims<2>(p.gamma, u);
#pragma unroll
      for (int v = 0; v < NV; ++v) s_u[npos + v * PN] = u[v];
      double* d = s_p + nslot * 3 * PN + lds_pos<N>(node);
      d[0] = q.v[0];
      d[PN] = q.v[1];
      d[2 * PN] = q.beta;
      if constexpr (NODAL) {
#pragma unroll
        for (int k = 0; k < 4; ++k) s_ja[npos + k * PN] = ja[k];
      }
    }
  } else if (face) {
    // the flux takes the upper element's metric at its first node; at a
    // boundary face, whose far state follows below, the own element's
    fe = element(fslot);
    element_indices<2>(p, (int)fe, fid);
    int64_t lo, hi;
    face_neighbours<2, BCS>(p, fid, fe, fdir, lo, hi);
    const int64_t nb = fside ? hi : lo;
    boundary = BCS && nb < 0;
    const LineNodes<2, N> ln(fdir, fline);
    const int first = ln.base, last = ln.base + N * ln.stride;
    const int64_t ue = fside && !boundary ? hi : fe;  // whose metric, and where
    const int at = fside && boundary ? last : first;
    const double* src = p.u + (boundary ? fe : nb) * (NV * NN) + (fside ? first : last);
#pragma unroll
    for (int v = 0; v < NV; ++v) far[v] = src[v * NN];
    const double sg = p.invJ[NODAL ? ue * NN + at : ue] >= 0.0 ? 1.0 : -1.0;
#pragma unroll
    for (int c = 0; c < 2; ++c)
      nrm_f[c] = sg * p.Ja[NODAL ? ((ue * 2 + fdir) * 2 + c) * NN + at : (ue * 2 + fdir) * 2 + c];
  }
  if (wave > 0 && wave <= W::PAIR_WAVES)
    for (int t = tid - 64; t < 3 * NN + n; t += 64 * W::PAIR_WAVES) s_op[t] = p.basis[t];
  // Navier-Stokes: the D_hat divergence and the face terms of the viscous
  // fluxes (element_body.inc), by the pair waves while wave 0 stages
  if (p.visc && wave > 0 && wave <= W::PAIR_WAVES) {
    for (int t = tid - 64; t < 2 * W::NODES; t += 64 * W::PAIR_WAVES) {
      const int k = t % n, line = t / n % n, dir = t / NN % 2, slot = t / (2 * NN);
      const int64_t e = element(slot);
      int eid[3];
      element_indices<2>(p, (int)e, eid);
      int64_t lo, hi;
      face_neighbours<2, BCS>(p, eid, e, dir, lo, hi);
      int lo_end = NV, hi_end = NV;
      const bool own_hi = BCS && hi < 0;
      if constexpr (BCS) {
        auto carried = [&](int f) {
          const int kind = p.bc[f];
          return kind == kBcDirichlet ? NV : (kind == kBcNsNoSlipWall ? NV - 1 : 0);
        };
        if (lo < 0) lo_end = carried(2 * dir);
        if (own_hi) hi_end = carried(2 * dir + 1);
      }
      const LineNodes<2, N> ln(dir, line);
      const int64_t ue = own_hi ? e : hi;
      const int at = ln.base + (own_hi ? N * ln.stride : 0);
      const double sg_lo = p.invJ[NODAL ? e * NN + ln.base : e] >= 0.0 ? 1.0 : -1.0;
      const double sg_hi = p.invJ[NODAL ? ue * NN + at : ue] >= 0.0 ? 1.0 : -1.0;
      const double* h = p.visc + (e * 2 + dir) * (NV * NN) + line * n;
      const double* hu = own_hi ? h + N : p.visc + (hi * 2 + dir) * (NV * NN) + line * n;
      double dh[n];
#pragma unroll
      for (int i = 0; i < n; ++i) dh[i] = p.basis[NN + k * n + i];
#pragma unroll
      for (int v = 1; v < NV; ++v) {
        double r = 0.0;
#pragma unroll
        for (int i = 0; i < n; ++i) r += dh[i] * h[v * NN + i];
        if (k == 0 && v < lo_end) r -= sg_lo * h[v * NN] * p.lhat0;
        if (k == n - 1 && v < hi_end) r += sg_hi * hu[v * NN] * p.lhatN;
        s_v[(dir * 3 + v - 1) * W::NODES + slot * NN + ln.base + k * ln.stride] = r;
      }
    }
  }
  __syncthreads();

  // 2. pair fluxes, face fluxes and blending factors, wave by wave
  if (wave == 0) {
    if constexpr (SC) {
      if (p.alpha_in) {
        if (lane < nvalid) s_alpha[lane] = p.alpha_in[e0 + lane];
      } else {
        wave_alpha<N>(p, indicator_variable<2>(u), s_op + 2 * NN, lane, s_w, s_alpha);
      }
    }
  } else if (wave <= W::PAIR_WAVES) {
    const int t = (wave - 1) * 64 + lane;
    if (t < W::PAIRS) {
      const int q = t % LP, line = t / LP % n, dir = t / (LP * n) % 2, slot = t / (LP * n * 2);
      // pair q = (a, b), a < b, in the order of the line's two loops
      int a = 0;
#pragma unroll
      for (int k = 1; k < N; ++k) a += q >= k * n - k * (k + 1) / 2 ? 1 : 0;
      const int b = q - (a * n - a * (a + 1) / 2) + a + 1;
      const LineNodes<2, N> ln(dir, line);
      const int pa = ln.pbase + a * ln.pstride, pb = ln.pbase + b * ln.pstride;
      const double* su = s_u + slot * NV * PN;
      const double* pr = s_p + slot * 3 * PN;
      double nrm[2], f[NV];
      if constexpr (NODAL) {
        const double* row = s_ja + (slot * 4 + dir * 2) * PN;
#pragma unroll
        for (int c = 0; c < 2; ++c) nrm[c] = row[c * PN + pa] + row[c * PN + pb];
      } else {
#pragma unroll
        for (int c = 0; c < 2; ++c) nrm[c] = p.Ja[(element(slot) * 2 + dir) * 2 + c];
      }
      if (SF == kFluxAny && p.volume_flux == kVolumeCentral) {
        double ua[NV], uc[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          ua[v] = su[v * PN + pa];
          uc[v] = su[v * PN + pb];
        }
        flux_central<2>(p.gamma, ua, uc, nrm, f);
      } else {
        NodePrims<2> qa{}, qb{};
        qa.rho = su[pa];
        qb.rho = su[pb];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          qa.v[c] = pr[c * PN + pa];
          qb.v[c] = pr[c * PN + pb];
        }
        qa.beta = pr[2 * PN + pa];
        qb.beta = pr[2 * PN + pb];
        flux_chandrashekar<2>(p.inv_gm1, qa, qb, nrm, f);
      }
#pragma unroll
      for (int v = 0; v < NV; ++v) s_f[v * W::PAIRS + t] = f[v];
    }
  } else if (face) {
    const LineNodes<2, N> ln(fdir, fline);
    const double* su = s_u + fslot * NV * PN;
    const int at = ln.pbase + (fside ? N * ln.pstride : 0);
    double own[NV], f[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) own[v] = su[v * PN + at];
    if constexpr (BCS) {
      if (boundary) {
        int pdofs[n];
#pragma unroll
        for (int k = 0; k < n; ++k) pdofs[k] = ln.pbase + k * ln.pstride;
        const int64_t bnode = (int64_t)(fdir == 0 ? fid[1] : fid[0]) * n + fline;
        boundary_state<2, N>(p, 2 * fdir + fside, bnode, su, pdofs, own, nrm_f, far);
      }
    }
    double ul[NV], ur[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      ul[v] = fside ? own[v] : far[v];
      ur[v] = fside ? far[v] : own[v];
    }
    surface_flux<2>(SF == kFluxAny ? p.surface_flux : SF, p.gamma, ul, ur, nrm_f, f);
    const int at_i = ((fslot * 2 + fdir) * n + fline) * (n + 1) + (fside ? n : 0);
#pragma unroll
    for (int v = 0; v < NV; ++v) s_i[v * W::INTER + at_i] = f[v];
  }
  __syncthreads();

  // 3. subcell fluxes of the troubled elements
  if constexpr (SC) {
    bool any = false;
#pragma unroll
    for (int sl = 0; sl < EPW; ++sl) any = any || (sl < nvalid && fabs(s_alpha[sl] - 0.0) > p.atol);
    if (any) {
      for (int t = tid; t < W::SUBS; t += W::BLOCK) {
        const int fi = t % N + 1, l = t / N, line = l % n, dir = l / n % 2, slot = l / (2 * n);
        if (slot >= nvalid || !(fabs(s_alpha[slot] - 0.0) > p.atol)) continue;
        const int64_t e = e0 + slot;
        const LineNodes<2, N> ln(dir, line);
        const double* su = s_u + slot * NV * PN + ln.pbase + fi * ln.pstride;
        double ul[NV], ur[NV], nrm[2], f[NV];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          ul[v] = su[v * PN - ln.pstride];
          ur[v] = su[v * PN];
        }
#pragma unroll
        for (int c = 0; c < 2; ++c)
          nrm[c] = NODAL ? p.sn[(((e * 2 + dir) * n + line) * N + (fi - 1)) * 2 + c]
                         : p.Ja[(e * 2 + dir) * 2 + c];
        surface_flux<2>(FF == kFluxAny ? p.fv_flux : FF, p.gamma, ul, ur, nrm, f);
#pragma unroll
        for (int v = 0; v < NV; ++v) s_i[v * W::INTER + l * (n + 1) + fi] = f[v];
      }
      __syncthreads();
    }
  }

  // 4. the node's sums, -1/J and the stage combination
  if (wave == 0 && lane < W::NODES && nslot < nvalid) {
    double alpha = 0.0, coef = 1.0;
    bool troubled = false;
    if constexpr (SC) {
      alpha = s_alpha[nslot];
      troubled = fabs(alpha - 0.0) > p.atol;
      if (troubled) coef = 1.0 - alpha;
    }
    double du[NV];
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
      const int k = dir == 0 ? ni : nj, line = dir == 0 ? nj : ni, l = (nslot * 2 + dir) * n + line;
      const double* inter = s_i + l * (n + 1);
      const double* pair = s_f + l * LP;
      double acc[NV];
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        acc[v] = 0.0;
        if (k == 0) acc[v] = -(inter[v * W::INTER] * p.lhat0);
        if (k == n - 1) acc[v] = inter[v * W::INTER + n] * p.lhatN;
      }
#pragma unroll
      for (int m = 0; m < n; ++m) {
        const int a = m < k ? m : k, b = m < k ? k : m;
        const double* f = pair + (a * n - a * (a + 1) / 2 + (m == k ? 0 : b - a - 1));
        const double w = coef * s_op[k * n + m];
#pragma unroll
        for (int v = 0; v < NV; ++v) {
          const double s = acc[v] + w * (m == k ? pair : f)[v * W::PAIRS];
          acc[v] = m == k ? acc[v] : s;
        }
      }
      if constexpr (SC) {
        if (troubled) {
          const double wn = alpha * s_op[3 * NN + k];
          if (k > 0) {
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] -= wn * inter[v * W::INTER + k];
          }
          if (k < n - 1) {
#pragma unroll
            for (int v = 0; v < NV; ++v) acc[v] += wn * inter[v * W::INTER + k + 1];
          }
        }
      }
      if (p.visc) {
#pragma unroll
        for (int v = 1; v < NV; ++v) acc[v] += s_v[(dir * 3 + v - 1) * W::NODES + lane];
      }
#pragma unroll
      for (int v = 0; v < NV; ++v) du[v] = dir == 0 ? acc[v] : du[v] + acc[v];
    }
    double r[NV];
#pragma unroll
    for (int v = 0; v < NV; ++v) r[v] = du[v] * fac;
    double* out = p.out + (e0 + nslot) * (NV * NN) + node;
    if (p.mode != kModeRhs) stage_combine<2>(p, with_base, u, ub, r);
#pragma unroll
    for (int v = 0; v < NV; ++v) out[v * NN] = r[v];
  }
  if constexpr (SC) {
    if (tid < nvalid) p.alpha[e0 + tid] = s_alpha[tid];
  }
}

template <int N, bool SC, bool NODAL, int SF, int FF, bool BCS>
hipError_t launch_pair_kernel(const KParams& p, hipStream_t stream) {
  using W = PairShape<N>;
  const int64_t nb = (p.E + W::EPW - 1) / W::EPW;
  if (nb <= 0) return hipSuccess;
  hipLaunchKernelGGL((rhs_pair_kernel<N, SC, NODAL, SF, FF, BCS>), dim3((unsigned)nb), dim3(W::BLOCK),
                     0, stream, p);
  return hipGetLastError();
}

}  // namespace detail
}  // namespace dgsem
