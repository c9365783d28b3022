// Checks the roots and quotients without range handling (root64.hpp) on the host
// against the IEEE operations, with seeds of 1/sqrt(x) that are off by up to
// 2^-23.  Built and run by tests/test_root64.py; prints "ok" or the first
// violation.
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "../mumfim_amd/csrc/root64.hpp"

static uint64_t s = 1;
static uint64_t next() {
  uint64_t z = (s += 0x9E3779B97F4A7C15ULL);
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
  return z ^ (z >> 31);
}
static double uniform() { return (double)(next() >> 11) * 0x1p-53; }

int main(int argc, char **argv) {
  const int n = argc > 1 ? std::atoi(argv[1]) : 1000000;
  double worst = 0;
  for (int i = 0; i < n; ++i) {
    // squared lengths over the whole declared range, forces over half of it
    const double x = std::ldexp(1.0 + uniform(), (int)(next() % 1201) - 600);
    const double f = std::ldexp(1.0 + uniform(), (int)(next() % 601) - 300);
    const double e = (i & 3) == 0 ? 0x1p-23 : (i & 3) == 1 ? -0x1p-23 : (2 * uniform() - 1) * 0x1p-23;
    const double y = (double)((1.0L + e) / std::sqrt((long double)x));
    double l, rl;
    mf::kern::root64(x, y, l, rl);
    if (l != std::sqrt(x)) {
      std::printf("FAIL root of %a with seed error %g: %a\n", x, e, l);
      return 1;
    }
    // div64 wants a reciprocal good to 1.25 ulp (an ulp: 2^-52 of it): half an ulp of
    // the root's rounding, half of h's own, a quarter of g's through r
    const double off = (double)std::fabs((long double)rl * l - 1.0L);
    worst = off > worst ? off : worst;
    if (off > 1.25 * 0x1p-52) {
      std::printf("FAIL reciprocal of the root of %a, seed error %g: off by %g ulp\n", x, e,
                  off * 0x1p52);
      return 1;
    }
    for (const double a : {f, -f, f * uniform()})
      if (mf::kern::div64(a, l, rl) != a / l) {
        std::printf("FAIL %a / %a\n", a, l);
        return 1;
      }
    // quotients by a length, a mass or a step count: an IEEE reciprocal
    const double b = std::ldexp(1.0 + uniform(), (int)(next() % 601) - 300), rb = 1.0 / b;
    if (mf::kern::div64(l, b, rb) != l / b || mf::kern::div64(f, b, rb) != f / b) {
      std::printf("FAIL quotient by %a\n", b);
      return 1;
    }
  }
  std::printf("ok, reciprocal within %.3f ulp\n", worst * 0x1p52);
  return 0;
}
