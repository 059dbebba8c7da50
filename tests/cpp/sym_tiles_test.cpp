// Host check of the symmetric G4 tile sets (csrc/g4acc_kernels.hpp): for every frequency count,
// exchange frequency and channel kind, the computed tiles and their images by the rule of the tile
// kernel write every (w1, w2) of a channel exactly once. Prints "OK" and exits 0.
#include <cstdio>
#include <vector>

#include "../../dca_amd/csrc/g4acc_kernels.hpp"

using namespace g4acc;

static int check(int nw, int nu, bool ph, bool pp, int sym) {
  std::vector<int> n_ph(nw * nw, 0), n_pp(nw * nw, 0);
  auto in = [&](int a, int b) { return a >= 0 && a < nw && b >= 0 && b < nw; };
  auto used = [&](int a, int b) { return sym_tile_computed(nw, nu, a, b, ph, pp, sym); };
  for (int w1 = 0; w1 < nw; ++w1)
    for (int w2 = 0; w2 < nw; ++w2) {
      if (!used(w1, w2))
        continue;
      const int c1 = nw - 1 - nu - w2, c2 = nw - 1 - nu - w1, p1 = nw - 1 + nu - w1, p2 = nw - 1 + nu - w2;
      const bool t = sym == SYM_CONJ_TRANSPOSE && w1 != w2;
      const bool c = sym == SYM_CONJ ? in(c1, c2) && !used(c1, c2) : w1 + w2 != nw - 1;
      ++n_ph[w1 + nw * w2];
      ++n_pp[w1 + nw * w2];
      if (t)
        ++n_ph[w2 + nw * w1];
      if (c)
        ++n_ph[c1 + nw * c2];
      if (t && c)
        ++n_ph[c2 + nw * c1];
      if (sym == SYM_CONJ && in(p1, p2) && !used(p1, p2))
        ++n_pp[p1 + nw * p2];
    }
  int bad = 0;
  for (int i = 0; i < nw * nw; ++i)
    bad += (ph && n_ph[i] != 1) + (pp && n_pp[i] != 1);
  if (bad)
    std::printf("FAIL nw=%d nu=%d ph=%d pp=%d sym=%d: %d tiles\n", nw, nu, ph, pp, sym, bad);
  return bad;
}

int main() {
  int bad = 0;
  for (int nw = 2; nw <= 12; nw += 2) {
    for (int nu = -nw - 2; nu <= nw + 2; ++nu)
      for (int kind = 1; kind < 4; ++kind)
        bad += check(nw, nu, kind & 1, kind & 2, SYM_CONJ);
    bad += check(nw, 0, true, false, SYM_CONJ_TRANSPOSE);
  }
  if (!bad)
    std::printf("OK\n");
  return bad != 0;
}
