// Prints what the FP64 Coulomb table gives: for each "kappa r_off r2" read from
// standard input, g and f of FP64 systems and g of mixed precision's energies as
// hexadecimal floats (coulomb_table.hpp).
#include <cstdio>

#include "coulomb_table.hpp"

int main() {
  double kappa, roff, r2, k0 = -1, o0 = -1;
  std::vector<apo::CoefPair> cf, ce;
  while (std::scanf("%la %la %la", &kappa, &roff, &r2) == 3) {
    const double per = apo::erfc_intervals(kappa, roff);
    if (kappa != k0 || roff != o0) {
      cf = apo::erfc_table(kappa * roff, per, true);
      ce = apo::erfc_table(kappa * roff, per, false);
    }
    k0 = kappa;
    o0 = roff;
    double g, f, ge, unused;
    apo::erfc_factors<true>(cf.data(), r2, 1.0 / std::sqrt(r2), per * kappa, g, f);
    apo::erfc_factors<false>(ce.data(), r2, 1.0 / std::sqrt(r2), per * kappa, ge, unused);
    std::printf("%a %a %a %zu\n", g, f, ge, ce.size() / apo::erfc_stride(false) - 1);
  }
}
