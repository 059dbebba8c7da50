// M -> G for the single-band clusters of 4, 8 and 16 sites on the matrix cores, complex64 and
// complex128 (the 16-site one for a 4x4 torus):
//
//   left   A[(k, w), j] = sum_r e^{i k.r} sum_{i in site r} T[w, i] M[i, j]
//   right  G[p1, (k2, w2)] = -G0(p1) / Nc sum_r e^{-i k2.r} (sum_{j in site r} A[p1, j] conj(T[w2, j])) G0(k2, w2)
//                            + beta G0(p1) delta
//
// Both walk the vertices, sorted by site, in steps of four of one site (the last step of a site padded
// with zeros): a step is a 16 x 16 x 4 matrix-core product, real or complex, accumulated in one
// register tile that moves to the site's slot behind a branch taken once per site. SPLIT waves share
// a tile and take NC / SPLIT sites each, so that the site sums fit 64 registers in either
// precision; they then exchange the sums through LDS, one component at a time (32 KiB), and each wave
// ends up with all sites for 4 / SPLIT of the tile's rows per lane, where the site transform is
// lane-local. Operands are loaded PF steps ahead, the ring of loads indexed statically.
//
// M is real, so A(-k, -w) = conj A(k, w): where the momenta have their inverses (kneg) the left
// kernel forms the upper half of the frequencies and writes both.
//
// What bounds them is latency and the writes of A and G, not the products: one thread per (w, j)
// walking a column of M through two dependent loads took 236 us and the vector right kernel 599 us
// for 32 FP64 measurements (4x4, 64 frequencies, N ~ U[64, 256]); these take 101 and 300 us. One FP64
// measurement (32 frequencies): 98 -> 29 us. 256 complex64 ones: 1.25 + 1.50 -> 0.87 + 1.57 ms.
#include <algorithm>
#include <type_traits>

#include "g4acc_common.hpp"
#include "g4acc_kernels.hpp"
#include "mfma16.hpp"
#include "site_fft.hpp"

namespace g4acc {

namespace {

// Side of the torus whose site transform runs as two L-point passes (0: dense).
template <int NC>
constexpr int torus_side() {
  return NC == 4 ? 2 : NC == 16 ? 4 : 0;
}

template <typename Real, int NC>
struct Tile {
  static constexpr int SPLIT = sizeof(Real) == 8 ? NC / 4 : NC == 16 ? 2 : 1;  // waves per tile
  static constexpr int NH = NC / SPLIT;                                        // sites per wave
  static constexpr int NI = 4 / SPLIT;   // tile rows per lane after the exchange
  static constexpr int TPW = 4 / SPLIT;  // tiles per workgroup of four waves
  static constexpr int X_REALS = SPLIT > 1 ? 4 * NH * 4 * 64 : 1;
};

// Steps of four sorted vertices a slot may need (sum over sites of ceil(n_r / 4)).
constexpr int kMaxSteps = 128;

// The slot's steps: site vertex ranges So, first step Sp of each site, and per step its first vertex
// and vertex count (bits 20..22).
template <int NC>
struct Steps {
  int So[NC + 1], Sp[NC + 1], Sb[kMaxSteps];
};

template <int NC>
__device__ __forceinline__ void build_steps(Steps<NC>& S, const int* __restrict__ O) {
  if (threadIdx.x <= NC)
    S.So[threadIdx.x] = O[threadIdx.x];
  __syncthreads();
  if (threadIdx.x <= NC) {
    int acc = 0;
    for (int r = 0; r < static_cast<int>(threadIdx.x); ++r)
      acc += (S.So[r + 1] - S.So[r] + 3) >> 2;
    S.Sp[threadIdx.x] = acc;
  }
  __syncthreads();
  if (threadIdx.x < kMaxSteps && static_cast<int>(threadIdx.x) < S.Sp[NC]) {
    const int q = threadIdx.x;
    int r = 0;
    while (S.Sp[r + 1] <= q)
      ++r;
    const int base = S.So[r] + 4 * (q - S.Sp[r]);
    S.Sb[q] = base | (min(4, S.So[r + 1] - base) << 20);
  }
  __syncthreads();
}

// This wave's step table across its lanes: step q_lo + q (q = lane + 64 h) is entry h of lane q % 64,
// packed as in Sb with, for the last step of a site, 1 + (site - r_lo) in bits 24..28.
template <int NC>
struct StepTable {
  int tab[kMaxSteps / 64];
  int n;
  __device__ __forceinline__ StepTable(const Steps<NC>& S, int r_lo, int nh, int lane) {
    const int q_lo = S.Sp[r_lo];
    n = __builtin_amdgcn_readfirstlane(S.Sp[r_lo + nh] - q_lo);
#pragma unroll
    for (int h = 0; h < kMaxSteps / 64; ++h) {
      const int q = lane + 64 * h;
      int e = 0;
      if (q < n) {
        int r = r_lo;
        while (S.Sp[r + 1] <= q_lo + q)
          ++r;
        e = S.Sb[q_lo + q] | (q_lo + q == S.Sp[r + 1] - 1 ? (r - r_lo + 1) << 24 : 0);
      }
      tab[h] = e;
    }
  }
  __device__ __forceinline__ int operator()(int q) const {  // q wave-uniform
    int e = 0;
#pragma unroll
    for (int h = 0; h < kMaxSteps / 64; ++h) {
      const int v = __builtin_amdgcn_readlane(tab[h], q & 63);
      e = (q >> 6) == h ? v : e;
    }
    return q < n ? e : 0;
  }
};

// Moves the current site's tile (cr, ci) to the slot of site fs - 1 and clears it.
template <int NH, typename V>
__device__ __forceinline__ void site_store(int fs, V (&er)[NH], V (&ei)[NH], V& cr, V& ci) {
  switch (fs - 1) {  // a branch, not per-site selects on every step
#define MTOG_SITE_STORE(R)  \
  case R:                   \
    if constexpr (R < NH) { \
      er[R] = cr;           \
      ei[R] = ci;           \
    }                       \
    break;
    MTOG_SITE_STORE(0) MTOG_SITE_STORE(1) MTOG_SITE_STORE(2) MTOG_SITE_STORE(3)
    MTOG_SITE_STORE(4) MTOG_SITE_STORE(5) MTOG_SITE_STORE(6) MTOG_SITE_STORE(7)
#undef MTOG_SITE_STORE
    default: break;
  }
  cr = ci = V{0, 0, 0, 0};
}

// Gathers all sites' sums for this lane's NI rows i = NI part + ii of the tile.
template <typename Real, int NC, typename V>
__device__ __forceinline__ void exchange(const V (&er)[Tile<Real, NC>::NH], const V (&ei)[Tile<Real, NC>::NH],
                                         Real* __restrict__ X, int wave, int part, int lane,
                                         Cplx<Real> (&x)[Tile<Real, NC>::NI][NC]) {
  using TL = Tile<Real, NC>;
  if constexpr (TL::SPLIT == 1) {
#pragma unroll
    for (int r = 0; r < NC; ++r)
#pragma unroll
      for (int ii = 0; ii < TL::NI; ++ii)
        x[ii][r] = Cplx<Real>{er[r][ii], ei[r][ii]};
  }
  else {
    Real* mine = X + wave * (TL::NH * 4 * 64) + lane;
    const Real* tile = X + (wave - part) * (TL::NH * 4 * 64) + lane;  // of the tile's first wave
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      __syncthreads();
#pragma unroll
      for (int r = 0; r < TL::NH; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          mine[(r * 4 + i) * 64] = c == 0 ? er[r][i] : ei[r][i];
      __syncthreads();
#pragma unroll
      for (int r = 0; r < NC; ++r)
#pragma unroll
        for (int ii = 0; ii < TL::NI; ++ii) {
          const Real v = tile[(r * 4 + TL::NI * part + ii) * 64];
          if (c == 0)
            x[ii][r].x = v;
          else
            x[ii][r].y = v;
        }
    }
  }
}

// Site transform of one row: e^{+-i k.r} over the sites; entry kk is the caller's momentum Kl[kk]
// (torus) or kk (dense, Dl[k + NC r] = e^{i k.r}).
template <typename Real, int NC, bool SEP, int SGN>
__device__ __forceinline__ void site_sum(Cplx<Real> (&e)[NC], const Cplx<Real>* __restrict__ Dl) {
  if constexpr (SEP)
    site_transform_2d<torus_side<NC>(), SGN, Real>(e);
  else {
    Cplx<Real> f[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      Cplx<Real> acc{0, 0};
#pragma unroll
      for (int r = 0; r < NC; ++r) {
        if (SGN > 0)
          cfma(acc, e[r], Dl[k + NC * r]);
        else
          cfmac(acc, e[r], Dl[k + NC * r]);
      }
      f[k] = acc;
    }
#pragma unroll
    for (int k = 0; k < NC; ++k)
      e[k] = f[k];
  }
}

constexpr int PF = 4;  // steps in flight

}  // namespace

// A workgroup owns 16 columns j, whose M entries it stages once in LDS (sorted rows, padded per site,
// e^V applied), and walks the frequency tiles of 16, TPW at a time. Lane l supplies M[i0 + l/16][j0 +
// l%16] and T[w0 + l%16][i0 + l/16] and holds rows j0 + row(l/16, i) of column w0 + l%16.
template <typename Real, int NC, bool SEP>
__global__ void __launch_bounds__(256) mtog_left_small(const SlotDesc* __restrict__ desc, Geo g, int n_max,
                                                       int slot0, const int* __restrict__ perm,
                                                       const int* __restrict__ off,
                                                       const Cplx<Real>* __restrict__ T,
                                                       const Cplx<Real>* __restrict__ dft,
                                                       const int* __restrict__ kmap,
                                                       const int* __restrict__ kneg, Cplx<Real>* __restrict__ A) {
  using C = Cplx<Real>;
  using TL = Tile<Real, NC>;
  using V = typename Mfma16<Real>::acc_t;
  __shared__ Steps<NC> S;
  __shared__ Real X[TL::X_REALS];
  __shared__ C Dl[SEP ? 1 : NC * NC];
  __shared__ int Kl[NC], Nl[NC];  // caller momentum of each transform entry, and its inverse
  extern __shared__ unsigned char smem_raw[];
  Real* Ml = reinterpret_cast<Real*>(smem_raw);  // [step][4][16]
  const int slot = slot0 + blockIdx.z;
  const SlotDesc d = desc[slot];
  const int n = d.n, j0 = blockIdx.x * 16;
  if (j0 >= n)
    return;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wave % TL::SPLIT, tile = wave / TL::SPLIT;
  const int* P = perm + static_cast<size_t>(slot) * n_max;
  const C* Ts = T + static_cast<size_t>(slot) * g.nwE * n_max;
  if constexpr (!SEP)
    for (int i = threadIdx.x; i < NC * NC; i += 256)
      Dl[i] = dft[i];
  if (threadIdx.x < NC) {
    const int k = SEP ? kmap[threadIdx.x] : threadIdx.x;
    Kl[threadIdx.x] = k;
    Nl[threadIdx.x] = kneg ? kneg[k] : 0;
  }
  build_steps(S, off + static_cast<size_t>(slot) * (NC + 1));
  const int total = S.Sp[NC] * 64;
#pragma unroll 4
  for (int e = threadIdx.x; e < total; e += 256) {
    const int sb = S.Sb[e >> 6], row = (e >> 4) & 3, col = e & 15;
    const bool live = row < (sb >> 20) && j0 + col < n;
    const int i = P[live ? (sb & 0xfffff) + row : 0], j = P[live ? j0 + col : 0];
    double m = d.m[i + static_cast<size_t>(d.ld) * j];
    if (d.expv)  // N and exp(V): M_ij = (exp(V_i) - 1) N_ij, formed in FP64
      m = (d.expv[i] - 1.0) * m;
    Ml[e] = live ? static_cast<Real>(m) : 0;
  }
  const StepTable<NC> step(S, part * TL::NH, TL::NH, lane);
  const int q_lo = S.Sp[part * TL::NH];
  __syncthreads();
  const int jl = lane >> 4;
  const Real* Mq = Ml + q_lo * 64 + lane;
  // With inverses: the upper half of the frequencies, tiled from nwE / 2 (nwE is even).
  const int w_lo = kneg ? g.nwE / 2 : 0;
  const int n_wt = (g.nwE - w_lo + 15) / 16;
  for (int wt0 = blockIdx.y * TL::TPW; wt0 < n_wt; wt0 += gridDim.y * TL::TPW) {
    const int wl = w_lo + (wt0 + tile) * 16 + (lane & 15);
    const int wc = wl < g.nwE ? wl : g.nwE - 1;
    V er[TL::NH], ei[TL::NH];
#pragma unroll
    for (int r = 0; r < TL::NH; ++r)
      er[r] = ei[r] = V{0, 0, 0, 0};
    V cr{0, 0, 0, 0}, ci{0, 0, 0, 0};
    C qt[PF];
    Real qm[PF];
    int qe[PF];
    auto load = [&](int k, int q) {
      qe[k] = step(q);
      // Past the step's vertices: the padded rows of M are zero; the phase read is a valid one.
      const int v = (qe[k] & 0xfffff) + (jl < ((qe[k] >> 20) & 7) ? jl : 0);
      qt[k] = Ts[wc + static_cast<size_t>(g.nwE) * v];
      qm[k] = Mq[64 * (q < step.n ? q : 0)];
    };
#pragma unroll
    for (int k = 0; k < PF; ++k)
      load(k, k);
    for (int g0 = 0; g0 < step.n; g0 += PF) {
#pragma unroll
      for (int k = 0; k < PF; ++k) {
        if (g0 + k >= step.n)
          break;
        const int fs = qe[k] >> 24;
        const C t = qt[k];
        const Real m = qm[k];
        load(k, g0 + k + PF);
        cr = Mfma16<Real>::mma(m, t.x, cr);
        ci = Mfma16<Real>::mma(m, t.y, ci);
        if (fs != 0)
          site_store<TL::NH>(fs, er, ei, cr, ci);
      }
    }
    C x[TL::NI][NC];
    exchange<Real, NC>(er, ei, X, wave, part, lane, x);
    if (wl >= g.nwE)
      continue;  // every wave walks the same tiles (barriers above)
#pragma unroll
    for (int ii = 0; ii < TL::NI; ++ii) {
      const int jj = j0 + Mfma16<Real>::row(jl, TL::NI * part + ii);
      if (jj >= n)
        continue;
      site_sum<Real, NC, SEP, 1>(x[ii], Dl);
      C* Aj = A + static_cast<size_t>(blockIdx.z) * g.D * n_max + static_cast<size_t>(g.D) * jj;
#pragma unroll
      for (int kk = 0; kk < NC; ++kk)
        Aj[Kl[kk] + NC * wl] = x[ii][kk];
      if (kneg)
#pragma unroll
        for (int kk = 0; kk < NC; ++kk)
          Aj[Nl[kk] + NC * (g.nwE - 1 - wl)] = C{x[ii][kk].x, -x[ii][kk].y};
    }
  }
}

// A workgroup owns TPW tiles of 16 rows p1 and walks the frequency tiles w2 of its y block. Lane l
// supplies conj-T[w0 + l%16][j0 + l/16] and A[p0 + l%16][j0 + l/16] and holds E_r[w0 + row(l/16,
// i)][p0 + l%16]; after the exchange a store of one (i, k2) writes 16 consecutive rows of G.
template <typename Real, int NC, bool SEP>
__global__ void __launch_bounds__(256) mtog_right_small(Geo g, int n_max, int slot0, int w_sum_min,
                                                        const int* __restrict__ off,
                                                        const Cplx<Real>* __restrict__ T,
                                                        const Cplx<Real>* __restrict__ A,
                                                        const Cplx<Real>* __restrict__ dft,
                                                        const double2* __restrict__ bphase,
                                                        const double2* __restrict__ G0,
                                                        const int* __restrict__ kmap,
                                                        Cplx<Real>* __restrict__ G) {
  using C = Cplx<Real>;
  using TL = Tile<Real, NC>;
  using V = typename Mfma16<Real>::acc_t;
  __shared__ Steps<NC> S;
  __shared__ Real X[TL::X_REALS];
  __shared__ C Dl[SEP ? 1 : NC * NC];
  __shared__ double2 G0l[NC * 16];
  __shared__ int Kl[NC];
  const int slot = slot0 + blockIdx.z;
  const int s = slot & 1;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int part = wave % TL::SPLIT;
  const int bx = turned_row(blockIdx.x, blockIdx.z, gridDim.x * gridDim.y, gridDim.x);
  const int p0 = (bx * TL::TPW + wave / TL::SPLIT) * 16;
  const int n_wt = (g.nwE + 15) / 16;
  // The first frequency tile that reaches w_sum_min with the workgroup's highest row.
  const int w_first = w_sum_min - 15 - ((bx + 1) * (16 * TL::TPW) - 1) / NC;
  const int wt_first = w_first > 0 ? (w_first + 15) / 16 : 0;
  if (wt_first + static_cast<int>(blockIdx.y) >= n_wt)
    return;
  const C* Ts = T + static_cast<size_t>(slot) * g.nwE * n_max;
  const C* Ab = A + static_cast<size_t>(blockIdx.z) * g.D * n_max;
  if constexpr (!SEP)
    for (int i = threadIdx.x; i < NC * NC; i += 256)
      Dl[i] = dft[i];
  if (threadIdx.x < NC)
    Kl[threadIdx.x] = SEP ? kmap[threadIdx.x] : threadIdx.x;
  build_steps(S, off + static_cast<size_t>(slot) * (NC + 1));
  const StepTable<NC> step(S, part * TL::NH, TL::NH, lane);
  const int jl = lane >> 4, pl = p0 + (lane & 15);
  const bool p_ok = pl < g.D;
  const int pc = p_ok ? pl : g.D - 1;
  const int k1 = pc % NC, w1 = pc / NC;
  const double2 ga = G0[s + 2 * (k1 + static_cast<size_t>(NC) * w1)];
  const double inv_nc = 1.0 / NC;
  const double2 gneg{-ga.x * inv_nc, -ga.y * inv_nc};  // -G0(p1) / Nc, folded once per row
  C* Gs = G + static_cast<size_t>(slot) * g.D * g.D + pl;

  for (int wt = wt_first + blockIdx.y; wt < n_wt; wt += gridDim.y) {
    const int w0 = wt * 16;
    __syncthreads();  // the previous tile's epilogue has read G0l
    for (int i = threadIdx.x; i < NC * 16; i += 256) {
      const int k = i % NC, w = w0 + i / NC;
      G0l[i] = w < g.nwE ? G0[s + 2 * (k + static_cast<size_t>(NC) * w)] : double2{0, 0};
    }
    const int wc = min(w0 + (lane & 15), g.nwE - 1);
    V er[TL::NH], ei[TL::NH];
#pragma unroll
    for (int r = 0; r < TL::NH; ++r)
      er[r] = ei[r] = V{0, 0, 0, 0};
    V cr{0, 0, 0, 0}, ci{0, 0, 0, 0};
    C qt[PF], qa[PF];
    int qe[PF];
    auto load = [&](int k, int q) {  // branch-free, clamped to valid entries
      qe[k] = step(q);
      const int v = (qe[k] & 0xfffff) + (jl < ((qe[k] >> 20) & 7) ? jl : 0);
      qt[k] = Ts[wc + static_cast<size_t>(g.nwE) * v];
      qa[k] = Ab[pc + static_cast<size_t>(g.D) * v];
    };
#pragma unroll
    for (int k = 0; k < PF; ++k)
      load(k, k);
    for (int g0 = 0; g0 < step.n; g0 += PF) {
#pragma unroll
      for (int k = 0; k < PF; ++k) {
        if (g0 + k >= step.n)
          break;
        const int ce = qe[k];
        const bool live = jl < ((ce >> 20) & 7);
        const C ct = qt[k], ca{live ? qa[k].x : 0, live ? qa[k].y : 0};
        load(k, g0 + k + PF);
        // E += conj(T) A = (Tx Ax + Ty Ay) + i (Tx Ay - Ty Ax)
        cr = Mfma16<Real>::mma(ct.x, ca.x, cr);
        ci = Mfma16<Real>::mma(ct.x, ca.y, ci);
        cr = Mfma16<Real>::mma(ct.y, ca.y, cr);
        ci = Mfma16<Real>::mma(-ct.y, ca.x, ci);
        if (ce >> 24)
          site_store<TL::NH>(ce >> 24, er, ei, cr, ci);
      }
    }
    C x[TL::NI][NC];
    exchange<Real, NC>(er, ei, X, wave, part, lane, x);
    if constexpr (TL::SPLIT == 1)
      __syncthreads();  // G0l (the exchange has barriers of its own)
    if (!p_ok)
      continue;  // every wave walks the same tiles (barriers above)
#pragma unroll
    for (int ii = 0; ii < TL::NI; ++ii) {
      const int wr = Mfma16<Real>::row(jl, TL::NI * part + ii), w2 = w0 + wr;
      if (w2 >= g.nwE)
        continue;
      site_sum<Real, NC, SEP, -1>(x[ii], Dl);
#pragma unroll
      for (int kk = 0; kk < NC; ++kk) {
        const int k2 = Kl[kk];
        double2 m = to_d(x[ii][kk]);
        if (bphase)
          m = cmulc(cmul(m, bphase[k1]), bphase[k2]);
        double2 v = cmul(cmul(gneg, m), G0l[k2 + NC * wr]);
        const int p2 = k2 + NC * w2;
        if (pl == p2) {
          v.x = fma(ga.x, g.beta, v.x);
          v.y = fma(ga.y, g.beta, v.y);
        }
        Gs[static_cast<size_t>(g.D) * p2] = from_d<C>(v);
      }
    }
  }
}

int mtog_small_max_vertices(int nc) { return 4 * (kMaxSteps - nc); }

namespace {

template <typename Real, int NC, bool SEP>
void launch_small(const MtoGArgs<Real>& a, int s0, int ns, hipStream_t st) {
  using TL = Tile<Real, NC>;
  const Geo& g = a.g;
  // Few slots: the frequency tiles are dealt over the grid as well, up to two workgroups per CU.
  auto spread = [&](int blocks, int tiles) { return std::max(1, std::min(tiles, 512 / std::max(1, blocks))); };
  const int steps = std::min(kMaxSteps, a.n_max / 4 + NC) + 1;  // a wave without sites reads one past the last
  const size_t lds = sizeof(Real) * 64 * steps;
  const int cols = (a.n_max + 15) / 16;
  const int w_tiles = ((a.kneg ? g.nwE / 2 : g.nwE) + 15) / 16;
  hipLaunchKernelGGL((mtog_left_small<Real, NC, SEP>),
                     dim3(cols, spread(cols * ns, (w_tiles + TL::TPW - 1) / TL::TPW), ns), dim3(256), lds, st, a.desc, g,
                     a.n_max, s0, a.perm, a.off, a.T, a.dft, a.kmap, a.kneg, a.A);
  const int rows = (g.D + 16 * TL::TPW - 1) / (16 * TL::TPW);
  hipLaunchKernelGGL((mtog_right_small<Real, NC, SEP>), dim3(rows, spread(rows * ns, (g.nwE + 15) / 16), ns), dim3(256),
                     0, st, g, a.n_max, s0, a.w_sum_min, a.off, a.T, a.A, a.dft, a.bphase, a.G0, a.kmap, a.G);
}

}  // namespace

namespace {

// Vertices up to which the register-fused kernels are the faster ones: there the products are few and the
// time is the writing of G, which they do with less per tile. Each against the other at that count, M -> G:
// 8 sites, complex128, 64 frequencies, 8 walkers: 8 vertices 1.5, 48 1.05; 32 frequencies, 48 walkers: 8
// 1.44, 48 1.06; with little G to write (8 frequencies, 8 walkers) 8 1.05, 16 1.0, 48 0.65.
template <typename Real>
int mtog_small_min_vertices(const Geo& g, int ns) {
  constexpr bool dp = sizeof(Real) == 8;
  const bool writes = static_cast<size_t>(g.D) * g.D * ns * sizeof(Cplx<Real>) >= size_t(32) << 20;
  switch (g.nc) {
    case 4: return writes ? 24 : 8;
    case 8: return writes ? (dp ? 80 : 40) : (dp ? 12 : 0);
    default: return writes ? (dp ? 24 : 32) : (dp ? 8 : 0);
  }
}

}  // namespace

template <typename Real>
bool launch_mtog_small(const MtoGArgs<Real>& a, int s0, int ns, hipStream_t st) {
  if (a.n_max <= mtog_small_min_vertices<Real>(a.g, ns) || a.n_max > mtog_small_max_vertices(a.g.nc))
    return false;
  const bool torus = a.kmap && a.grid_L * a.grid_L == a.g.nc;
  switch (a.g.nc) {
    case 4:
      torus ? launch_small<Real, 4, true>(a, s0, ns, st) : launch_small<Real, 4, false>(a, s0, ns, st);
      return true;
    case 8:
      launch_small<Real, 8, false>(a, s0, ns, st);
      return true;
    case 16:
      if (torus)
        launch_small<Real, 16, true>(a, s0, ns, st);
      return torus;
    default:
      return false;
  }
}

template bool launch_mtog_small<float>(const MtoGArgs<float>&, int, int, hipStream_t);
template bool launch_mtog_small<double>(const MtoGArgs<double>&, int, int, hipStream_t);

}  // namespace g4acc
