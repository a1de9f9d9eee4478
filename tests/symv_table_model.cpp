// Reads nb and 5 nb times (option by option) and prints the rows of symv_choose: the fixed counts,
// then the table to install.
#include <cstdio>

#include "symv_table.h"

int main() {
  int nb = 0;
  if (std::scanf("%d", &nb) != 1 || nb < 1) return 2;
  std::vector<double> t((dftbhip::kTuneFixed + 1) * (size_t)nb);
  for (double& x : t)
    if (std::scanf("%lf", &x) != 1) return 2;
  dftbhip::TileTable fixed, install;
  dftbhip::symv_choose(t, nb, &fixed, &install);
  for (const auto* rows : {&fixed, &install}) {
    for (const auto& r : *rows) std::printf("%d %d ", r.first, r.second);
    std::printf("\n");
  }
  return 0;
}
