// The tangent and adjoint of the LLF flux (physics_ad.hpp) against the forward
// function the kernels run, flux_llf: tangent against central finite differences,
// adjoint by the dot-product identity, at random states and near equal ones.
// Prints the largest relative errors.
#include <cmath>
#include <cstdio>
#include <random>

#include "../../dgsem_amd/csrc/physics_ad.hpp"

using namespace dgsem;

static std::mt19937_64 rng(7);
static double uni(double a, double b) { return std::uniform_real_distribution<double>(a, b)(rng); }

template <int DIM>
static void check(double& fd, double& dot) {
  constexpr int NV = DIM + 2;
  for (int trial = 0; trial < 400; ++trial) {
    double u[2][NV], d[2][NV], n[DIM], g[NV], p[2];
    for (int s = 0; s < 2; ++s) {
      double v2 = 0.0;
      u[s][0] = uni(0.5, 2.0);
      p[s] = uni(0.5, 2.0);
      for (int k = 0; k < DIM; ++k) {
        const double v = uni(-1.0, 1.0);
        u[s][k + 1] = u[s][0] * v;
        v2 += v * v;
      }
      u[s][NV - 1] = p[s] / 0.4 + 0.5 * u[s][0] * v2;
    }
    if (trial % 2)
      for (int i = 0; i < NV; ++i) u[1][i] = u[0][i] * (1.0 + 1e-3 * uni(-1.0, 1.0));
    for (int i = 0; i < NV; ++i) {
      g[i] = uni(-1.0, 1.0);
      for (int s = 0; s < 2; ++s) d[s][i] = uni(-1.0, 1.0);
    }
    for (int k = 0; k < DIM; ++k) n[k] = uni(-1.0, 1.0);
    const NodePrims<DIM> ql = node_prims<DIM>(1.4, u[0]), qr = node_prims<DIM>(1.4, u[1]);
    double df[NV], f[2][NV], w[2][NV], scale = 0.0;
    llf_jvp<DIM>(1.4, u[0], ql, u[1], qr, d[0], d[1], n, df);
    const double h = 1e-7;
    for (int side = 0; side < 2; ++side) {
      for (int s = 0; s < 2; ++s)
        for (int i = 0; i < NV; ++i) w[s][i] = u[s][i] + (side ? -h : h) * d[s][i];
      flux_llf<DIM>(1.4, w[0], w[1], n, f[side]);
    }
    for (int i = 0; i < NV; ++i) scale = std::fmax(scale, std::fabs(df[i]));
    for (int i = 0; i < NV; ++i)
      fd = std::fmax(fd, std::fabs((f[0][i] - f[1][i]) / (2.0 * h) - df[i]) / scale);
    double b[2][NV] = {}, lhs = 0.0, rhs = 0.0, mag = 0.0;
    llf_vjp_side<DIM>(1.4, u[0], ql, u[1], qr, n, g, true, b[0]);
    llf_vjp_side<DIM>(1.4, u[0], ql, u[1], qr, n, g, false, b[1]);
    for (int i = 0; i < NV; ++i) {
      lhs += g[i] * df[i];
      for (int s = 0; s < 2; ++s) {
        rhs += b[s][i] * d[s][i];
        mag += std::fabs(b[s][i] * d[s][i]);
      }
    }
    dot = std::fmax(dot, std::fabs(lhs - rhs) / mag);
  }
}

int main() {
  double fd = 0.0, dot = 0.0;
  check<2>(fd, dot);
  check<3>(fd, dot);
  std::printf("fd %.3e dot %.3e\n", fd, dot);
  return 0;
}
