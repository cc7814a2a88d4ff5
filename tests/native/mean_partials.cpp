// The partial derivatives of the Chandrashekar flux's means (physics_ad.hpp)
// against long double, at the edges of the branches and across the range.
// Prints the largest error of a partial relative to its mean over its argument,
// in units of the double epsilon.
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <limits>
#include <random>
#include <vector>

#include "../../dgsem_amd/csrc/physics_ad.hpp"

using namespace dgsem;
using L = long double;

// Logarithmic mean M = (x - y) / log(x / y) = s / (2 Q), Q = artanh(xi) / xi, and
// its derivative by x: for f2 = xi^2 < 1/4 from the series of Q summed to
// convergence, beyond as (1 - M / x) / log(x / y) (nearer, that difference loses
// 1 / log^2 of long double's digits).
static void exact(double x, double y, L& M, L& Mx) {
  const L s = (L)x + y, xi = ((L)x - y) / s, f = xi * xi;
  if (f < 0.25L) {
    L Q = 0, dQ = 0;
    for (int k = 60; k >= 0; --k) Q = 1 / (2 * k + 1.0L) + f * Q;
    for (int k = 60; k >= 1; --k) dQ = k / (2 * k + 1.0L) + f * dQ;
    M = s / (2 * Q);
    Mx = 1 / (2 * Q) - 2 * (L)y * xi * dQ / (Q * Q * s);
    return;
  }
  const L d = logl((L)x / y);
  M = ((L)x - y) / d;
  Mx = (1 - M / x) / d;
}

int main() {
  const double eps = std::numeric_limits<double>::epsilon();
  std::mt19937_64 g(11);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  std::vector<double> ratios = {1.0, 1.0 + 1e-12, 1.0 + 1e-8};
  for (double f2 : {1.0e-4, kSeriesMax})
    for (double s : {1.0 - 1e-12, 1.0, 1.0 + 1e-12, 0.99, 1.01}) {
      const double xi = std::sqrt(f2 * s);
      ratios.push_back((1.0 + xi) / (1.0 - xi));
    }
  for (int k = 1; k <= 12; ++k) ratios.push_back(std::ldexp(1.4142135623730951, k));
  for (int i = 0; i < 20000; ++i) ratios.push_back(std::exp((i % 2 ? 8.0 : 0.1) * u(g)));
  double worst = 0.0;
  for (double ratio : ratios)
    for (int swap = 0; swap < 2; ++swap) {
      const double y = std::exp(6.0 * (u(g) - 0.5));
      NodePrims<3> a{}, b{};
      a.rho = a.beta = swap ? y : ratio * y;
      b.rho = b.beta = swap ? ratio * y : y;
      const ChandrashekarMeans m = chandrashekar_means<3>(a, b);
      L M, Ma, Mb, t;
      exact(a.rho, b.rho, M, Ma);
      exact(b.rho, a.rho, t, Mb);
      auto err = [&](double got, L want, L scale) {
        worst = std::max(worst, (double)(fabsl(got - want) / scale) / eps);
      };
      err(m.rho, M, M);
      err(m.rho_a, Ma, M / a.rho);
      err(m.rho_b, Mb, M / b.rho);
      err(m.B, 1 / M, 1 / M);
      err(m.B_a, -Ma / (M * M), 1 / (M * a.beta));
      err(m.B_b, -Mb / (M * M), 1 / (M * b.beta));
    }
  std::printf("worst %.3f\n", worst);
  return 0;
}
