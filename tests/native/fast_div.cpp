// FastDiv (kernels.hpp) against the integer division: every divisor up to 2^10
// and divisors around the powers of two, at the ends of the range [0, 2^31) and
// around the multiples of the divisor.
#include <cstdint>
#include <cstdio>
#include <vector>

#include "../../dgsem_amd/csrc/kernels.hpp"

int main() {
  std::vector<uint32_t> divisors;
  for (uint32_t d = 1; d <= 1024; ++d) divisors.push_back(d);
  for (int s = 11; s < 31; ++s)
    for (int k = -2; k <= 2; ++k) divisors.push_back((1u << s) + k);
  divisors.push_back(INT32_MAX);
  long checked = 0;
  for (uint32_t d : divisors) {
    const dgsem::FastDiv f = dgsem::FastDiv::by(d);
    auto check = [&](int64_t x) {
      if (x < 0 || x > INT32_MAX) return true;
      ++checked;
      if (f((int)x) == (int)(x / d)) return true;
      std::printf("%lld / %u: %d\n", (long long)x, d, f((int)x));
      return false;
    };
    const int64_t top = INT32_MAX / d;
    for (int64_t q = 0; q <= top; q += q < 200 ? 1 : (top / 500 + 1))
      for (int k = -1; k <= 1; ++k)
        if (!check(q * d + k)) return 1;
    for (int64_t q = top; q >= 0 && q > top - 100; --q)
      for (int k = -1; k <= 1; ++k)
        if (!check(q * d + k)) return 1;
    if (!check(INT32_MAX)) return 1;
  }
  std::printf("ok %ld\n", checked);
  return 0;
}
