// Host-side declarations of the g4acc kernel launchers.
#pragma once

#include "g4acc_common.hpp"

namespace g4acc {

template <typename Real>
struct MtoGArgs {
  Geo g;
  const SlotDesc* desc;   // n_slots device descriptors
  int n_slots;            // 2 * walkers
  int n_max;              // vertex capacity per slot
  int chunk;              // slots whose S1..S4 workspaces exist at once
  bool fused;             // use the register-fused single-band kernels
  int tw;                 // frequencies per thread in the fused right kernel (0: default)
  int mfma;               // 4, 8 and 16 sites: the matrix-core kernels of mtog_small.hip
  // 6x6 and 8x8 clusters: the whole M -> G on the matrix cores with the B, E and Ms workspaces
  // (mtog_large.hip), instead of the register-fused kernels.
  bool large = false;
  // FP32 only: S3, the right site transform and the epilogue in one kernel, E kept in registers
  // and LDS (no E workspace).
  bool right_fused = false;
  void* Ms = nullptr;     // [chunk][n_max][n_max] M in sorted order, working precision
  const int* perm;        // [n_slots][n_max]  rows of M, sorted by the vertices' right labels
  const int* off;         // [n_slots][n_orb + 1]
  Cplx<Real>* T;          // [n_slots][n_max][nwE]
  // Columns of M, sorted by the vertices' left labels, and their phases: the same arrays as
  // perm / off / T unless the vertices are non-density-density (four-stage kernels only).
  const int* perm2;
  const int* off2;
  Cplx<Real>* T2;
  Cplx<Real>* B;          // [chunk][n_max][D]
  Cplx<Real>* A;          // [chunk][n_max][D]
  Cplx<Real>* E;          // [chunk][D][D]
  Cplx<Real>* G;          // [n_slots][D][D]
  const Cplx<Real>* dft;  // [Nc][Nc] (k fastest)
  const double2* bphase;  // [Nc][nb] or nullptr
  const double2* G0;      // (b1, b2, s, k, wE)
  // Square L x L clusters (L = 2, 4, 6, 8): sites are relabelled x + L y and the right site DFT
  // runs as two L-point passes; kmap[kx + L ky] is the caller's momentum index. L = 0: dense DFT.
  int grid_L;
  const int* kmap;
  bool real_m = true;         // no slot holds complex M
  const int* kneg = nullptr;  // real M: index(-k), where dft(-k, r) = conj dft(k, r): A(-k, -w) = conj A(k, w)
  // Smallest w1 + w2 (extended frequencies) the consumer reads: nwE - 1 where G is conjugate
  // symmetric and the tile kernel reads that half only, else 0. Blocks of G wholly below it are
  // neither computed nor written.
  int w_sum_min = 0;
};

// M = diag(exp_v - 1) N for one n x n matrix (column-major, leading dimensions ldn, ldm).
void launch_compute_m(int n, const double* exp_v, const double* N, int ldn, double* M, int ldm,
                      hipStream_t st);

// site_map (or nullptr): the internal label of each caller site (sites sorted by it).
// left = true sorts by the vertices' left labels (where a descriptor has them).
void launch_sort(const SlotDesc* desc, const Geo& g, int n_slots, int n_max, const int* site_map,
                 int* perm, int* off, int* err_flag, hipStream_t st, bool left = false);
// Phases T[slot][w + nwE ii] = exp(i w_w tau_{perm ii}) of the vertices in the order of perm.
template <typename Real>
void launch_phases(const SlotDesc* desc, const Geo& g, int n_slots, int n_max, const int* perm,
                   Cplx<Real>* T, hipStream_t st);

template <typename Real>
void launch_mtog(const MtoGArgs<Real>& a, hipStream_t st);
// Register-fused single-band M -> G (mtog_fused.hip); false if the geometry is not covered.
template <typename Real>
bool launch_mtog_fused(const MtoGArgs<Real>& a, hipStream_t st);
bool mtog_fused_covers(const Geo& g);
// Matrix-core M -> G of the 4-, 8- and 16-site clusters (mtog_small.hip) on slots [s0, s0 + ns); false
// where it does not apply (the register-fused kernels then run).
template <typename Real>
bool launch_mtog_small(const MtoGArgs<Real>& a, int s0, int ns, hipStream_t st);
// M -> G for single-band 6x6 (NC = 36) and 8x8 (NC = 64) clusters with site labels x + L y, on
// slots [s0, s0 + ns) of a chunk (needs the Ms, B and E workspaces).
template <typename Real, int NC>
void launch_mtog_large(const MtoGArgs<Real>& a, int s0, int ns, hipStream_t st);

enum SumMode { SUM_FP64 = 0, SUM_FP32_KAHAN = 1 };

template <typename Real>
struct G4Args {
  Geo g;
  int channel;                 // FourPointType value
  const Cplx<Real>* G;         // [n_slots][D][D]
  const SlotDesc* desc;        // signs
  int n_walkers;
  const int* k_add;            // device [Nc][Nc]
  const int* k_sub;
  const int* k_ex;             // device [nq]
  const int* w_ex;             // device [nv]
  int sum_mode;
  void* g4;                    // double2[size] (FP64) or float4[size] (value, compensation)
  // false: the updateG4 branch of models that are not spin symmetric (pp and magnetic, spin
  // sector 0 only, tp_accumulator_cpu.hpp:668-757)
  bool spin_symmetric = true;
};

template <typename Real>
void launch_g4(const G4Args<Real>& a, hipStream_t st);

// Row block of the M -> G workgroup at place x of its plane (a column or slot) of n row blocks; planes start
// `stride` workgroups apart. Over half of the pairs higher rows have more to do, and workgroups go to the eight
// XCDs round-robin: with an even stride a row keeps to half of them or fewer (with a multiple of eight to one: 6x6,
// complex128, 56 frequencies, 14 slots of 7..42 vertices: the last had 1.22 of the mean, 588 us before the halves,
// 672 with them, 530 with the rows turned by one per plane). An odd stride spreads the rows by itself; turned as
// well, they stayed (3 bands, 8 sites, 64 frequencies, 2 slots, complex128: S4 52.6 us, turned 69.9).
__host__ __device__ inline int turned_row(unsigned x, unsigned plane, unsigned stride, unsigned n) {
  return static_cast<int>((x + (stride % 2 ? 0 : plane)) % n);
}

// Symmetries of the single-band G4 over the pairs p = (k, w), with Q = (q, v) the transfer:
//   transpose    T: (p1, p2) -> (p2 + Q, p1 + Q): for particle-hole channels X and Y, and the two
//                   rank-one factors, swap. Needs 2 Q = 0 (v = 0, q its own inverse).
//   conjugate    C: (p1, p2) -> (-p2 - Q, -p1 - Q), value conjugated: the same swap when
//                   G(-p1, -p2) = conj G(p1, p2), i.e. for real M and G0(-p) = conj G0(p).
//   pair swap    P: (p1, p2) -> (Q - p1, Q - p2): X and Z of the pp channel swap.
// SYM_TRANSPOSE uses T alone (one q = 0, one v = 0, no pp channel); SYM_CONJ uses C for the
// particle-hole channels and P for pp; SYM_CONJ_TRANSPOSE C and T (no pp channel).
enum G4Sym { SYM_NONE = 0, SYM_TRANSPOSE = 1, SYM_CONJ = 2, SYM_CONJ_TRANSPOSE = 3 };

// Whether tile (w1, w2) of exchange frequency index nu is computed, for sym >= SYM_CONJ: the
// tiles on or above the anti-diagonals about which C and P reflect (w1 + w2 = nw - 1 - nu and
// nw - 1 + nu; the lower of the two bounds both, so every tile left out has its image in), and
// those whose image of a channel in use lies outside the compact frequencies.
__host__ __device__ inline bool sym_tile_computed(int nw, int nu, int w1, int w2, bool has_ph, bool has_pp, int sym) {
  const int an = nu < 0 ? -nu : nu;
  if (w1 + w2 >= nw - 1 - an)
    return sym != SYM_CONJ_TRANSPOSE || w1 <= w2;
  const int hi = w1 > w2 ? w1 : w2, lo = w1 > w2 ? w2 : w1;
  return (has_ph && (nw - 1 - nu - hi < 0 || nw - 1 - nu - lo >= nw)) ||
         (has_pp && (nw - 1 + nu - hi < 0 || nw - 1 + nu - lo >= nw));
}

// The images that a computed tile (w1, w2) writes, and their tiles: t (w2, w1), c (c1, c2) and both
// (c2, c1) of the particle-hole channels, p (p1, p2) of the pp channel.
struct TileImages {
  int c1, c2, p1, p2;
  bool t, c, p;
};
__host__ __device__ inline TileImages tile_images(int nw, int nu, int w1, int w2, bool has_ph, bool has_pp, int sym) {
  TileImages m{nw - 1 - nu - w2, nw - 1 - nu - w1, nw - 1 + nu - w1, nw - 1 + nu - w2, false, false, false};
  auto left_out = [&](int a, int b) {
    return a >= 0 && a < nw && b >= 0 && b < nw && !sym_tile_computed(nw, nu, a, b, has_ph, has_pp, sym);
  };
  m.t = (sym & 1) && w1 != w2;
  m.c = sym == SYM_CONJ ? left_out(m.c1, m.c2) : sym == SYM_CONJ_TRANSPOSE && w1 + w2 != nw - 1;
  m.p = has_pp && sym == SYM_CONJ && left_out(m.p1, m.p2);
  return m;
}

// The pair (s1, s2) of the tile that entry (k1, k2) of an image holds, kind 0: T, 1: C (conjugated),
// 2: both (conjugated); q is the exchange momentum.
__host__ __device__ inline void image_source(int kind, int nc, const int* k_add, const int* k_sub, const int* k_neg,
                                             int q, int k1, int k2, int& s1, int& s2) {
  if (kind == 0) {
    s1 = k_sub[q + nc * k2];
    s2 = k_sub[q + nc * k1];
  }
  else if (kind == 1) {
    s1 = k_neg[k_add[k2 + nc * q]];
    s2 = k_neg[k_add[k1 + nc * q]];
  }
  else {
    s1 = k_neg[k1];
    s2 = k_neg[k2];
  }
}

// The momentum of the pair-swap image that momentum k of the tile moves to.
__host__ __device__ inline int swap_momentum(int nc, const int* k_sub, int q, int k) { return k_sub[k + nc * q]; }

// Single-band, all channels in one launch (g4_tiled.hip). Returns false when the geometry is
// outside what the tiled kernel handles (the caller then uses launch_g4 per channel).
template <typename Real>
struct TiledArgs {
  Geo g;
  const Cplx<Real>* G;         // [n_slots][D][D]
  Cplx<Real>* UV;              // [walkers][4][nq*nv][Nc*nw] rank-one factors
  const SlotDesc* desc;
  int n_walkers;
  int n_ch;
  int ch[4];                   // channel types in G4 order
  void* g4[4];
  const int* k_add;
  const int* k_sub;
  const int* k_ex;
  const int* w_ex;
  int nqg;                     // momentum groups per exchange frequency (set by the launcher)
  int tile_order;              // 0: natural, 1: XCD-aware super-tiles
  int qg_cap;                  // largest momentum group (0: as many as registers allow)
  int super_tile, n_super, n_xcd;  // tile schedule (set by the launcher)
  const int* tile_perm;        // schedule 2: (w1 | w2 << 16) in dispatch order, nw * nw entries
  int sum_mode;
  bool need_y, need_z;         // particle-hole channels, pp
  // Symmetries of G4 used to compute a part of the tiles and write their images (G4Sym).
  int sym = 0, sym_few = 0;  // sym_few: where the launch has few tiles
  // G is conjugate symmetric: only its half wa + wb >= nwE - 1 (extended frequencies) is read.
  bool half_g = false;
  const int* k_neg = nullptr;       // device [Nc], index(-k); half_g only
  const int* sym_tiles = nullptr;   // computed tiles (w1 | w2 << 16) for sym >= SYM_CONJ, in dispatch order
  int n_sym_tiles = 0;
  int qg = 0;                       // momenta per workgroup (set by the launcher)
  bool rank_one = false;            // magnetic or charge among the channels (set by the launcher)
  int uv_lds = -1;                  // few walkers: place of their rank-one factors in LDS (set by the launcher)
};

template <typename Real>
bool launch_g4_tiled(TiledArgs<Real> a, hipStream_t st);
// Multiband LDS-tiled G4 update (g4_band.hip); false if the band count, cluster or channel set
// is not covered (the generic kernel then runs).
template <typename Real>
bool launch_g4_band(TiledArgs<Real> a, hipStream_t st);
int tiled_pairs_per_thread(int nc);
// LDS of one tile workgroup with momentum groups of qg and n_ph particle-hole channels.
size_t tiled_lds_bytes(const Geo& g, int n_ph, bool need_z, size_t cplx_bytes, int qg);

// Single-particle accumulator (sp_acc.hip): exact FP64 M_r_w of the batch's slots added to acc
// (and M_ij^2's to acc_sqr when squared_too), acc laid out [s][(b1 + nb (b2 + nb r)) n_w + w].
struct SpArgs {
  Geo g;
  const SlotDesc* desc;
  int n_slots, n_max, n_w;     // n_w = 2 * single-particle frequencies
  const int* perm;             // sort of the slots' vertices by caller orbital b + nb r
  const int* off;
  double2* T;                  // [n_slots][n_max][n_w / 2] phases (upper half of the frequencies)
  double2* C;                  // [n_slots][n_orb][n_orb][n_w / 2] orbital-pair sums
  const int* rsub;             // [Nc][Nc], rsub[a + Nc b] = index(r_b - r_a)
  double2* acc;
  double2* acc_sqr;
  bool squared_too;
};
void launch_sp_accumulate(const SpArgs& a, hipStream_t st);

// dst += src over n complex entries of a G4 buffer in the given sum mode.
void launch_g4_add(void* dst, const void* src, size_t n, int sum_mode, hipStream_t st);
// G4 buffer (any sum mode) -> complex double.
void launch_g4_export(const void* src, double2* dst, size_t n, int sum_mode, hipStream_t st);
// Fill n 16-byte entries with zeros (a kernel, not hipMemsetAsync, so it is safe to capture).
void launch_zero16(void* dst, size_t n, hipStream_t st);
// Reference-layout G (b1,b2,s,k1,k2,w1E,w2E) complex double -> per-slot device layout of one walker.
template <typename Real>
void launch_import_G(const double2* ref, Cplx<Real>* G, const Geo& g, hipStream_t st);
template <typename Real>
void launch_export_G(const Cplx<Real>* G, double2* ref, const Geo& g, hipStream_t st);

}  // namespace g4acc
