// Host check of the row blocks of the M -> G workgroups (turned_row in csrc/g4acc_kernels.hpp): every row once per
// plane, and the needed ones (w1 + w2 >= nwE - 1) spread over the eight XCDs that take the workgroups in turn.
// Prints "OK" and exits 0.
#include <algorithm>
#include <cstdio>
#include <vector>

#include "../../dca_amd/csrc/g4acc_kernels.hpp"

using namespace g4acc;

int main() {
  int bad = 0;
  // Columns as planes: row block b of n holds w1 up to (b + 1) nwE / n; column w2 needs it from nwE - 1 - w1 on.
  for (int n = 8; n <= 80; ++n)
    for (int nwE : {32, 66, 129}) {
      double load[8] = {}, mean = 0;
      for (int w2 = 0; w2 < nwE; ++w2) {
        std::vector<int> seen(n, 0);
        for (int x = 0; x < n; ++x) {
          const int b = turned_row(x, w2, n, n);
          bad += b < 0 || b >= n || seen[b]++;
          if ((b + 1) * nwE / n + w2 >= nwE - 1) {
            load[(x + n * w2) % 8] += 1;
            mean += 1. / 8;
          }
        }
      }
      // Eight columns in a row put each row on each XCD once: up to 8 of nwE are left over, twice for the wrap.
      const double most = *std::max_element(load, load + 8) / mean;
      if (most > 1 + 0.5 * 16 / nwE) {
        std::printf("FAIL n=%d nwE=%d: %.3f of the mean\n", n, nwE, most);
        ++bad;
      }
    }
  // Slots as planes of c columns; every column of a row is as much work as its row (b + 1 of n).
  for (int n = 8; n <= 80; ++n)
    for (int c = 1; c <= 9; ++c) {
      const int slots = 64;
      double load[8] = {}, mean = 0;
      for (int z = 0; z < slots; ++z)
        for (int y = 0; y < c; ++y)
          for (int x = 0; x < n; ++x) {
            const int b = turned_row(x, z, n * c, n);
            load[(x + n * (y + static_cast<long>(c) * z)) % 8] += b + 1;
            mean += (b + 1) / 8.;
          }
      const double most = *std::max_element(load, load + 8) / mean;
      if (most > 1 + 8. / slots) {
        std::printf("FAIL n=%d c=%d: %.3f of the mean\n", n, c, most);
        ++bad;
      }
    }
  if (bad == 0)
    std::printf("OK\n");
  return bad != 0;
}
