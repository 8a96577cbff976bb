// chain_rule.h -- which way the environments of a measurement go (internal): products of one site launched one by one,
// or every diagonal a workgroup of one launch (k_env_chain).  Estimates in us, from times on MI355X at bonds 1 to 32,
// Kraus legs 1 to 4 and 10 to 4000 qubits; in 755 of them the way taken is at most 16% slower than the other one.
#pragma once
#include <cstddef>

namespace hipmps {

// A site of k_env_chain, whose s go `steps` at a time: 1.8 at bond 1, 3.1 at 8, 4.2 at 16, 9.3 at 32 (two steps), 33
// at 32 with a Kraus leg of 4 (eight steps)
inline double chain_site_us(int cl, int steps) { return 1.3 + steps * (0.5 + 0.12 * cl); }

// m diagonals of n sites, `sites` being the sum over the sites: 512 workgroups run at a time, two a CU, which at
// bond 32 slow each other nearly twofold; their 2n values each are written and copied at 5.7 GB/s
inline double chain_us(double sites, int cmax, size_t m, int n) {
  return sites * (double)((m + 511) / 512) * (m > 256 ? 1.0 + 0.025 * cmax : 1.0) + 0.0028 * (double)m * n;
}

// One sweep of products: two launches a site, 6 at small bonds, 8 at 16 and 10 at 32
inline double sweep_us(int n, int cmax) { return n * (6.0 + 0.12 * cmax); }

// Both sweeps at once and a dot product a site
inline double both_sweeps_us(int n) { return 12.0 * n; }

// <ZZ>: the two sweeps, then chains advanced together, `longest` steps in all and `steps` of single chains
inline double zz_us(int n, size_t longest, size_t steps) { return both_sweeps_us(n) + 6.0 * longest + 0.6 * steps; }

}  // namespace hipmps
