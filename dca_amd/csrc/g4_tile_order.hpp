// Dispatch order of the single-band G4 tiles (host).
#ifndef G4ACC_G4_TILE_ORDER_HPP
#define G4ACC_G4_TILE_ORDER_HPP

#include <algorithm>
#include <utility>
#include <vector>

#include "g4acc_kernels.hpp"

namespace g4acc {

// Tile (w1, w2) of G4 reads the G blocks X = (w1, w2), Y = (w2 + v, w1 + v) and
// Z = (v + nw - 1 - w1, v + nw - 1 - w2) (extended frequencies). The transpose of a tile holds its
// Y block as X, its mirror (w -> nw - 1 - w) its Z block, and the neighbour along the diagonal
// the next v. Schedule 2, (w1 | w2 << 16) for all nw^2 frequency pairs: a group is `strip` consecutive positions on the diagonals w1 - w2 = +d and -d
// together with their mirror images; the workgroups resident on one XCD at a time cover a few
// groups and find most of their blocks in its L2.
inline std::vector<int> diagonal_tile_order(int nw, int strip) {
  std::vector<int> out;
  out.reserve(static_cast<size_t>(nw) * nw);
  std::vector<char> seen(static_cast<size_t>(nw) * nw, 0);
  for (int d = 0; d < nw; ++d)
    for (int p0 = 0; p0 < nw - d; p0 += strip)
      for (int sgn = 0; sgn < 2; ++sgn) {
        if (d == 0 && sgn == 1)
          continue;
        for (int p = p0; p < std::min(p0 + strip, nw - d); ++p)
          for (int mir = 0; mir < 2; ++mir) {
            int w2 = p, w1 = p + d;
            if (sgn)
              std::swap(w1, w2);
            if (mir) {
              w1 = nw - 1 - w1;
              w2 = nw - 1 - w2;
            }
            char& s = seen[w1 + static_cast<size_t>(nw) * w2];
            if (s)
              continue;
            s = 1;
            out.push_back(w1 | (w2 << 16));
          }
      }
  return out;
}

// The tiles computed for any of the exchange frequencies under sym >= SYM_CONJ, by schedule: 0 w1 fastest, 1
// super-tiles of 8 x 8, 2 diagonal strips.
inline std::vector<int> symmetric_tile_order(int nw, int schedule, int strip, const std::vector<int>& w_ex, bool has_ph,
                                             bool has_pp, int sym) {
  std::vector<int> out;
  auto add = [&](int w1, int w2) {
    for (int nu : w_ex)
      if (sym_tile_computed(nw, nu, w1, w2, has_ph, has_pp, sym)) {
        out.push_back(w1 | (w2 << 16));
        return;
      }
  };
  if (schedule < 2) {
    const int side = schedule == 0 ? nw : 8;
    for (int b2 = 0; b2 < nw; b2 += side)
      for (int b1 = 0; b1 < nw; b1 += side)
        for (int w2 = b2; w2 < std::min(b2 + side, nw); ++w2)
          for (int w1 = b1; w1 < std::min(b1 + side, nw); ++w1)
            add(w1, w2);
    return out;
  }
  // A tile's X block lies on the diagonal w1 - w2 = d, its Y block on -d and the conjugate of its Z
  // block on d again, each shifted along it by v: strips of both diagonals together.
  for (int d = 0; d < nw; ++d)
    for (int p0 = 0; p0 < nw - d; p0 += strip)
      for (int sgn = 0; sgn < (d == 0 ? 1 : 2); ++sgn)
        for (int p = p0; p < std::min(p0 + strip, nw - d); ++p)
          add(sgn ? p : p + d, sgn ? p + d : p);
  return out;
}

}  // namespace g4acc

#endif
