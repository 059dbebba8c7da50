// Host check of the G4 images (csrc/g4acc_kernels.hpp, csrc/g4_tile_order.hpp), with the kernel's own rules: on small clusters and
// a random G with G(-p1, -p2) = conj G(p1, p2), every G4 entry formed by the definition equals the one that
// the computed tiles and their images give, and every tile is needed by the table once. Prints "OK", exits 0.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>

#include "../../dca_amd/csrc/g4_tile_order.hpp"

using namespace g4acc;
using cd = std::complex<double>;

// The momenta of an Lx x Ly torus, k = x + Lx y.
struct Torus {
  int nc;
  std::vector<int> add, sub, neg;
  Torus(int lx, int ly) : nc(lx * ly), add(nc * nc), sub(nc * nc), neg(nc) {
    for (int a = 0; a < nc; ++a)
      for (int b = 0; b < nc; ++b) {
        const int ax = a % lx, ay = a / lx, bx = b % lx, by = b / lx;
        add[a + nc * b] = (ax + bx) % lx + lx * ((ay + by) % ly);
        sub[a + nc * b] = (bx - ax + lx) % lx + lx * ((by - ay + ly) % ly);  // k_b - k_a
      }
    for (int a = 0; a < nc; ++a)
      neg[a] = (lx - a % lx) % lx + lx * ((ly - a / lx) % ly);
  }
};

static int check(const Torus& t, int nw, const std::vector<int>& w_ex, int q, bool ph, bool pp, int sym) {
  const int nc = t.nc;
  int ext = 0;
  for (int nu : w_ex)
    ext = std::max(ext, std::abs(nu));
  const int nwe = nw + 2 * ext, D = nc * nwe;
  // Two spins of G over extended pairs p = k + nc w, conjugate symmetric.
  std::mt19937 rng(nc + 31 * nw + q);
  std::uniform_real_distribution<double> u(-1, 1);
  std::vector<cd> G[2];
  auto inv = [&](int p) { return t.neg[p % nc] + nc * (nwe - 1 - p / nc); };
  for (auto& g : G) {
    g.resize(static_cast<size_t>(D) * D);
    for (int a = 0; a < D; ++a)
      for (int b = 0; b < D; ++b)
        g[a + static_cast<size_t>(D) * b] = cd(u(rng), u(rng));
    for (int a = 0; a < D; ++a)
      for (int b = 0; b < D; ++b) {
        const int ia = inv(a), ib = inv(b);
        if (ia + static_cast<size_t>(D) * ib > a + static_cast<size_t>(D) * b)
          g[ia + static_cast<size_t>(D) * ib] = std::conj(g[a + static_cast<size_t>(D) * b]);
        else if (ia == a && ib == b)
          g[a + static_cast<size_t>(D) * b] = g[a + static_cast<size_t>(D) * b].real();
      }
  }
  const std::vector<int> order0 = symmetric_tile_order(nw, 0, 2, w_ex, ph, pp, sym);
  int bad = 0;
  for (auto [schedule, strip] : {std::pair<int, int>{0, 2}, {1, 2}, {2, 1}, {2, 2}, {2, 5}}) {
    std::vector<int> o = symmetric_tile_order(nw, schedule, strip, w_ex, ph, pp, sym), r = order0;
    std::sort(o.begin(), o.end());
    std::sort(r.begin(), r.end());
    bad += o != r || std::unique(o.begin(), o.end()) != o.end();
  }
  for (int nu : w_ex) {
    auto g = [&](int s, int ka, int wa, int kb, int wb) {  // compact frequencies, possibly shifted
      return G[s][ka + nc * (wa + ext) + static_cast<size_t>(D) * (kb + nc * (wb + ext))];
    };
    auto add = [&](int a, int b) { return t.add[a + nc * b]; };
    auto sub = [&](int a, int b) { return t.sub[a + nc * b]; };
    auto value = [&](int kind, int k1, int w1, int k2, int w2) {  // 0 charge, 1 transverse, 2 pp
      const int k1q = add(k1, q), k2q = add(k2, q);
      auto y = [&](int s) { return g(s, k2q, w2 + nu, k1q, w1 + nu); };
      auto z = [&](int s) { return g(s, sub(k1, q), nu + nw - 1 - w1, sub(k2, q), nu + nw - 1 - w2); };
      auto x = [&](int s) { return g(s, k1, w1, k2, w2); };
      if (kind == 2)
        return x(0) * z(1) + x(1) * z(0);
      if (kind == 1)
        return -(x(0) * y(1) + x(1) * y(0));
      const cd a = g(0, k1, w1, k1q, w1 + nu) + g(1, k1, w1, k1q, w1 + nu);
      const cd b = g(0, k2q, w2 + nu, k2, w2) + g(1, k2q, w2 + nu, k2, w2);
      return a * b - (x(0) * y(0) + x(1) * y(1));
    };
    for (int kind = 0; kind < 3; ++kind) {
      if (kind == 2 ? !pp : !ph)
        continue;
      const size_t P = static_cast<size_t>(nc) * nw;
      std::vector<cd> got(P * P, 0);
      auto at = [&](int k1, int w1, int k2, int w2) -> cd& { return got[k1 + nc * w1 + P * (k2 + nc * w2)]; };
      for (int packed : order0) {
        const int w1 = packed & 0xffff, w2 = packed >> 16;
        if (!sym_tile_computed(nw, nu, w1, w2, ph, pp, sym))
          continue;
        const TileImages m = tile_images(nw, nu, w1, w2, ph, pp, sym);
        for (int k1 = 0; k1 < nc; ++k1)
          for (int k2 = 0; k2 < nc; ++k2) {
            at(k1, w1, k2, w2) += value(kind, k1, w1, k2, w2);
            if (kind == 2) {
              if (m.p)
                at(swap_momentum(nc, t.sub.data(), q, k1), m.p1, swap_momentum(nc, t.sub.data(), q, k2), m.p2) +=
                    value(kind, k1, w1, k2, w2);
              continue;
            }
            for (int im = 0; im < 3; ++im) {
              if (!(im == 0 ? m.t : im == 1 ? m.c : m.t && m.c))
                continue;
              int s1, s2;
              image_source(im, nc, t.add.data(), t.sub.data(), t.neg.data(), q, k1, k2, s1, s2);
              const cd v = value(kind, s1, w1, s2, w2);
              const int wa = im == 0 ? w2 : im == 1 ? m.c1 : m.c2, wb = im == 0 ? w1 : im == 1 ? m.c2 : m.c1;
              at(k1, wa, k2, wb) += im == 0 ? v : std::conj(v);
            }
          }
      }
      double err = 0;
      for (int w1 = 0; w1 < nw; ++w1)
        for (int w2 = 0; w2 < nw; ++w2)
          for (int k1 = 0; k1 < nc; ++k1)
            for (int k2 = 0; k2 < nc; ++k2)
              err = std::max(err, std::abs(at(k1, w1, k2, w2) - value(kind, k1, w1, k2, w2)));
      if (err > 1e-13) {
        std::printf("FAIL nc=%d nw=%d nu=%d q=%d ph=%d pp=%d sym=%d kind=%d: %g\n", nc, nw, nu, q, ph, pp, sym, kind, err);
        ++bad;
      }
    }
  }
  return bad;
}

int main() {
  int bad = 0;
  for (const Torus& t : {Torus(2, 2), Torus(3, 1), Torus(4, 2), Torus(3, 3)})
    for (int q = 0; q < t.nc; ++q) {
      for (int kind = 1; kind < 4; ++kind)
        for (const std::vector<int>& w_ex : {std::vector<int>{0}, {0, 1, 2}, {-2, 1}, {3}, {-5}, {6}})
          bad += check(t, 4, w_ex, q, kind & 1, kind & 2, SYM_CONJ);
      if (t.neg[q] == q)
        for (int nw : {2, 6})
          bad += check(t, nw, {0}, q, true, false, SYM_CONJ_TRANSPOSE);
    }
  // Each schedule and strip is an order of its own, over the same tiles.
  std::vector<std::vector<int>> orders;
  for (auto [schedule, strip] : {std::pair<int, int>{0, 2}, {1, 2}, {2, 1}, {2, 2}, {2, 5}}) {
    orders.push_back(symmetric_tile_order(24, schedule, strip, {0, 1}, true, true, SYM_CONJ));
    for (size_t i = 0; i + 1 < orders.size(); ++i)
      bad += orders[i] == orders.back() || orders[i].size() != orders.back().size();
  }
  if (!bad)
    std::printf("OK\n");
  return bad != 0;
}
