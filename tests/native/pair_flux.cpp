// The logarithmic means and the Chandrashekar flux of physics.hpp against long
// double evaluations of their definitions, at the edges of the branches (f2
// around 1e-4 and kSeriesMax, ratios around sqrt(2) 2^k) and across the range.
// Prints the largest relative errors in units of the double epsilon.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <limits>
#include <random>
#include <vector>

#include "../../dgsem_amd/csrc/physics.hpp"

using namespace dgsem;
using L = long double;

static const double eps = std::numeric_limits<double>::epsilon();

// artanh(xi) / xi, xi = (x - y) / (x + y), from log1p, or from the logarithm of
// the ratio where 1 - |xi| cancels
static L exact_ratio(double x, double y) {
  const L d = (L)x - y, s = (L)x + y, xi = d / s;
  if (fabsl(xi) < 1e-9L) return 1 + xi * xi / 3;
  if (fabsl(xi) > 0.25L) return 0.5L * logl((L)x / y) / xi;
  return 0.5L * (log1pl(xi) - log1pl(-xi)) / xi;
}

template <int DIM>
static double flux_error(std::mt19937_64& g, double spread, bool& symmetric) {
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  auto state = [&](double r0, double b0) {
    NodePrims<DIM> q{};
    q.rho = r0 * std::exp(spread * u(g));
    q.beta = b0 * std::exp(spread * u(g));
    for (int k = 0; k < DIM; ++k) q.v[k] = u(g);
    for (int k = 0; k < DIM; ++k) q.kin += 0.5 * q.v[k] * q.v[k];
    return q;
  };
  double worst = 0.0;
  for (int i = 0; i < 20000; ++i) {
    const double r0 = std::exp(6.0 * u(g)), b0 = std::exp(6.0 * u(g));
    const NodePrims<DIM> a = state(r0, b0), b = state(r0, b0);
    double n[DIM], f[DIM + 2], h[DIM + 2];
    for (int k = 0; k < DIM; ++k) n[k] = u(g);
    flux_chandrashekar<DIM>(2.5, a, b, n, f);
    flux_chandrashekar<DIM>(2.5, b, a, n, h);
    symmetric = symmetric && std::memcmp(f, h, sizeof f) == 0;
    // numerical_flux.hpp:520-594, and the sum of magnitudes each component
    // is rounded against
    const L rm = ((L)a.rho + b.rho) / 2 / exact_ratio(a.rho, b.rho);
    const L bm = ((L)a.beta + b.beta) / 2 / exact_ratio(a.beta, b.beta);
    const L p = 0.5L * ((L)a.rho + b.rho) / ((L)a.beta + b.beta);
    L vn = 0, vabs = 0, sq = 0, sum = 0, mag = 0;
    for (int k = 0; k < DIM; ++k) {
      const L v = 0.5L * ((L)a.v[k] + b.v[k]);
      vn += v * n[k];
      vabs += fabsl(0.5L * a.v[k] * n[k]) + fabsl(0.5L * b.v[k] * n[k]);
      sq += 0.5L * ((L)a.v[k] * a.v[k] + (L)b.v[k] * b.v[k]);
    }
    const L f1 = rm * vn, m1 = rm * vabs;
    worst = std::max(worst, (double)(fabsl(f[0] - f1) / m1));
    for (int k = 0; k < DIM; ++k) {
      const L v = 0.5L * ((L)a.v[k] + b.v[k]), va = 0.5L * (fabsl((L)a.v[k]) + fabsl((L)b.v[k]));
      const L fk = f1 * v + p * n[k];
      worst = std::max(worst, (double)(fabsl(f[k + 1] - fk) / (m1 * va + p * fabsl((L)n[k]))));
      sum += fk * v;
      mag += (m1 * va + p * fabsl((L)n[k])) * va;
    }
    const L fe = f1 * 0.5L * (2.5L / bm - sq) + sum;
    worst = std::max(worst, (double)(fabsl(f[DIM + 1] - fe) / (m1 * 0.5L * (2.5L / bm + sq) + mag)));
  }
  return worst / eps;
}

int main() {
  std::mt19937_64 g(5);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  std::vector<double> ratios = {1.0};
  // xi at the branch edges, from both sides
  for (double f2 : {1.0e-4, kSeriesMax})
    for (double s : {1.0 - 1e-12, 1.0, 1.0 + 1e-12, 0.999, 1.001}) {
      const double xi = std::sqrt(f2 * s);
      ratios.push_back((1.0 + xi) / (1.0 - xi));
    }
  for (int k = -40; k <= 40; ++k)
    for (double r : {1.0, 1.4142135623730949, 1.4142135623730951, 1.4142135623730954, 1.1})
      ratios.push_back(std::ldexp(r, k));
  for (int i = 0; i < 100000; ++i) ratios.push_back(std::exp(30.0 * (u(g) - 0.5) * (i % 2 ? 1.0 : 0.02)));
  double worst = 0.0;
  bool symmetric = true;
  for (double r : ratios) {
    const double y = std::exp(10.0 * (u(g) - 0.5)), x = r * y, xi = (x - y) / (x + y);
    const double q = artanh_ratio(x, y, xi * xi), t = artanh_ratio(y, x, xi * xi);
    symmetric = symmetric && q == t;
    worst = std::max(worst, (double)fabsl(q / exact_ratio(x, y) - 1) / eps);
  }
  const bool nan_signs = std::isnan(artanh_ratio(1.0, -2.0, 9.0)) && std::isnan(artanh_ratio(-1.0, 2.0, 9.0));
  double flux = 0.0;
  for (double spread : {1e-4, 0.01, 0.1, 0.17, 0.5, 2.0, 8.0})
    flux = std::max({flux, flux_error<2>(g, spread, symmetric), flux_error<3>(g, spread, symmetric)});
  std::printf("ratio %.3f flux %.3f symmetric %d nan %d\n", worst, flux, symmetric, nan_signs);
  return 0;
}
