// The rule between the two ways of a measurement's environments against times measured on MI355X (ms, complex128,
// bonds min(2^k, 2^(n - k), chi)): the way it takes may be 20% slower than the other one.
#include "../../tnqvm_amd/csrc/chain_rule.h"

#include <algorithm>
#include <cstdio>

namespace {
enum Op { NORM, Z, ZZ_NEXT, ZZ_ONE, ZZ_FAR, ZZ_ALL, OUTCOMES };
struct Case {
  int n, chi, kap;
  size_t m;  // diagonals
  Op op;
  double products, chain;
};
const Case cases[] = {
    {10, 4, 1, 1, NORM, 0.098, 0.037},
    {10, 32, 1, 11, Z, 0.185, 0.051},
    {40, 1, 1, 41, Z, 0.551, 0.098},
    {40, 8, 1, 780, ZZ_ALL, 1.205, 0.477},
    {40, 24, 1, 780, ZZ_ALL, 1.308, 0.819},
    {40, 32, 1, 1, NORM, 0.382, 0.322},
    {40, 32, 1, 41, Z, 0.531, 0.337},
    {40, 32, 2, 1, NORM, 0.425, 0.576},
    {40, 32, 2, 780, ZZ_ALL, 1.437, 2.507},
    {40, 32, 4, 1, NORM, 0.503, 1.100},
    {40, 32, 4, 41, Z, 0.699, 1.135},
    {40, 32, 4, 39, ZZ_NEXT, 0.743, 1.125},
    {40, 32, 4, 780, ZZ_ALL, 1.662, 4.685},
    {40, 32, 4, 16, OUTCOMES, 8.098, 1.109},
    {40, 16, 4, 1, NORM, 0.372, 0.261},
    {40, 16, 4, 41, Z, 0.568, 0.276},
    {40, 8, 4, 1, ZZ_ONE, 0.557, 0.135},
    {200, 2, 1, 201, Z, 2.432, 0.419},
    {200, 32, 1, 199, ZZ_NEXT, 2.860, 1.994},
    {200, 32, 1, 1, ZZ_FAR, 4.542, 1.841},
    {200, 16, 2, 199, ZZ_NEXT, 2.720, 0.940},
    {200, 32, 2, 201, Z, 2.842, 3.861},
    {200, 32, 4, 2, OUTCOMES, 5.418, 6.628},
    {200, 32, 4, 1, ZZ_ONE, 3.382, 6.528},
    {600, 8, 1, 601, Z, 7.086, 4.555},
    {600, 24, 1, 601, Z, 7.036, 9.728},
    {600, 28, 1, 599, ZZ_NEXT, 7.356, 15.288},
    {1000, 4, 1, 1001, Z, 11.845, 5.894},
    {1000, 8, 1, 999, ZZ_NEXT, 12.328, 9.632},
    {1000, 16, 1, 1001, Z, 11.589, 13.780},
    {1000, 24, 1, 999, ZZ_NEXT, 12.357, 19.216},
    {1000, 32, 1, 1001, Z, 12.453, 35.803},
    {1000, 32, 1, 1, NORM, 10.161, 9.391},
    {2000, 1, 1, 1999, ZZ_NEXT, 24.549, 21.213},
    {2000, 8, 1, 2001, Z, 23.135, 38.058},
    {2000, 16, 1, 2001, Z, 23.035, 54.919},
    {2000, 32, 1, 1999, ZZ_NEXT, 26.020, 143.959},
    {2000, 8, 1, 1, NORM, 12.679, 6.165},
    {4000, 1, 1, 4001, Z, 46.586, 82.228},
    {4000, 4, 1, 3999, ZZ_NEXT, 48.635, 94.408},
    {4000, 16, 1, 4001, Z, 46.142, 217.061},
    {4000, 16, 1, 3999, ZZ_NEXT, 48.028, 217.685},
    {4000, 16, 1, 1, NORM, 31.935, 16.705},
};

// the s of a site that k_env_chain takes side by side (chain_slots in kernels.h)
int slots(int cl, int cr) {
  const int w = cl > cr ? cl * cr : cr * cr;
  return w > 512 ? 1 : std::min(1024 / w, 16);
}
int bond(const Case& c, int k) { return (int)std::min<long long>(1ll << std::min({k, c.n - k, 12}), c.chi); }
}  // namespace

int main() {
  using namespace hipmps;
  int bad = 0;
  for (const Case& c : cases) {
    double sites = 0.0;
    for (int k = 0; k < c.n; ++k) {
      const int s = slots(bond(c, k), bond(c, k + 1));
      sites += chain_site_us(bond(c, k), (2 * c.kap + s - 1) / s);
    }
    const int cmax = bond(c, c.n / 2);
    const size_t n = c.n;
    double products = 0.0;
    switch (c.op) {
      case NORM: products = sweep_us(c.n, cmax); break;
      case Z: products = both_sweeps_us(c.n); break;
      case ZZ_NEXT: products = zz_us(c.n, 1, n - 1); break;
      case ZZ_ONE: products = zz_us(c.n, 1, 1); break;
      case ZZ_FAR: products = zz_us(c.n, n - 1, n - 1); break;
      case ZZ_ALL: products = zz_us(c.n, n - 1, n * (n - 1) / 2); break;
      case OUTCOMES: products = (double)c.m * sweep_us(c.n, cmax); break;
    }
    const bool chain = chain_us(sites, cmax, c.m, c.n) < products;
    const double taken = chain ? c.chain : c.products, best = std::min(c.chain, c.products);
    if (taken > 1.2 * best) {
      std::printf("n %d bond %d kap %d, %zu diagonals, op %d: %s takes %.3f ms, the other %.3f\n", c.n, c.chi, c.kap, c.m,
                  (int)c.op, chain ? "one launch" : "products", taken, best);
      ++bad;
    }
  }
  std::puts(bad ? "failed" : "ok");
  return bad != 0;
}
