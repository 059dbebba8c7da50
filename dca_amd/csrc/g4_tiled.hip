// Single-band G4 update, LDS-tiled: all channels of a batch of walkers in one launch.
//
// Same sums as g4_kernels.hip (tp_accumulator_cpu.hpp:407-666) for n_bands == 1, organised around
// what the entries of one tile share. A workgroup owns the tile
//     { (k1, w1, k2, w2, q, v) : all k1, k2;  w1, w2 fixed;  v fixed;  q in a group of QG }
// and, per walker and spin, reads
//   X(k1,k2) = G[(k1, w1), (k2, w2)]            in registers: the thread's own pairs
//   Yb(a,b)  = G[(a, w2+v), (b, w1+v)]          into LDS: Y^q(k1,k2) = Yb(k2+q, k1+q)
//   Zb(a,b)  = G[(a, v-w1), (b, v-w2)]          into LDS: Z^q(k1,k2) = Zb(q-k1, q-k2)
// so every G element a tile needs is fetched once per walker and reused by the QG momenta. Of the
// walker loop's products
//   xs = a (X_0 Y_0 + X_1 Y_1),  pz = a (X_0 Z_1 + X_1 Z_0),  tr = a (X_0 Y_1 + X_1 Y_0)
// MAGNETIC and CHARGE share xs: MAGNETIC = R_m - xs, CHARGE = R_c - xs, PP_UP_DOWN = pz,
// TRANSVERSE = -tr. The rank-one terms R_c(k1,k2) = sum_m U_c[m](k1) V_c[m](k2), with
//   U = a (u_0 -+ u_1), u_s = G_s[(k1,w1), (k1+q, w1+v)],  V = v_0 -+ v_1, v_s = G_s[(k2+q,w2+v), (k2,w2)]
// precomputed by uv_kernel, are a matrix product over the batch's walkers: each tile forms its own
// 16 x 16 blocks of it on the matrix cores after the walker loop, so they cost no vector
// instructions per walker and no buffer of G4's size.
//
// What bounds it: the blocks read from L2 and beyond, with the vector ALUs half busy beside it (4x4, three
// channels, 256 walkers, 64 frequencies, 4 q, 3 v: 2.88 ms, 24.6 GB asked of L2, 13.3 GB of that from
// beyond it, vector ALUs 52 %). So each block is read once per walker for all the momenta whose
// totals fit the registers. The next walkers' loads are in flight during a walker's products; every
// load is issued (idle slots and walkers past the batch re-read valid elements).
// Per batch (256 walkers) the stage went from 3.64 ms, with the rank-one terms in a buffer of G4's
// size, to 2.9 ms; 6x6 (64 walkers, 64 frequencies, 4 q, 2 v) from 10.6 to 4.6 ms.
// Launches of few walkers (few_walkers) are the G4 read-modify-write with little before it (FEW): all tiles,
// without images, the rank-one factors staged in LDS beside the blocks, and one entry (complex128 G in small
// tiles: four) loaded before it is stored. With the code for many walkers (images, factors read from memory in
// the tail, twelve entries in flight) a launch of one walker took, 4x4, three channels, 64 frequencies, 4 q,
// 3 v: FP64 340 against 279 us, FP32 336 against 257; of three, FP32 445 against 303.
// Products are formed in the G precision; with complex64 G, tiles of up to 256 threads sum eight walkers in
// FP32 before the FP64 totals, larger tiles (whose registers hold the totals) add every walker.
// G4 is read and written once per launch (FP64, or FP32 value + Kahan compensation).
// Compiled once per precision: complex64 through g4_tiled32.hip.
#include <algorithm>
#include <type_traits>

#include "g4_tile_common.hpp"
#include "mfma16.hpp"

namespace g4acc {

namespace {

// Two values read together from LDS (one 16-byte read for complex64).
template <typename C>
struct alignas(2 * sizeof(C)) CPair {
  C a, b;
};

// A 16-byte pair is stored whole (one ds_write_b128); a 32-byte one member by member, since a
// 32-byte aligned temporary goes through scratch memory.
template <typename C>
__device__ __forceinline__ void store_pair(CPair<C>& dst, C a, C b) {
  if constexpr (sizeof(C) == 8) {
    dst = CPair<C>{a, b};
  }
  else {
    dst.a = a;
    dst.b = b;
  }
}

// Terms formed by the walker loop.
constexpr int HAS_X = 1, HAS_Z = 2, HAS_T = 4;

// Registers of a workgroup's threads (waves per SIMD that must fit: 64 registers for eight, 128 for four,
// 168 for three, 256 for two). 704 threads hold 33..37-site clusters with two pairs each: eleven waves
// leave 168 registers, enough for the totals of four momenta (6x6, magnetic and pp, 64 walkers, 64
// frequencies: 2.4 ms per batch; two momenta 3.0, one 4.9, since each group of momenta reads the blocks
// again). 256 threads take what their totals need: held to 128, two pairs of complex128 G spilled 147
// registers (20 sites, magnetic and pp, 16 walkers, 48 frequencies: 1.41 ms against 0.32).
// 1024 threads with few totals fit 64 registers or nearly so: two workgroups per CU instead of one (25
// sites, magnetic, complex64, 8 walkers: 60 -> 51 us). Without images and matrix-core tail (FEW) small shapes
// take less.
template <typename Real, int TT, int PPT, int QG, int SET, bool FEW>
struct PairShape {
  static constexpr bool fp32 = sizeof(Real) == 4;
  static constexpr int TERMS = (SET & 1) + (SET >> 1 & 1) + (SET >> 2 & 1);
  static constexpr int TOTALS = PPT * QG * TERMS;  // complex FP64, per thread
  // Fits 64 registers.
  static constexpr bool SMALL = PPT == 1 && TOTALS <= 2 && (fp32 || (FEW && TERMS == 1));
  static constexpr int FLUSH = fp32 && TT <= 256 ? 8 : 1;
  // Walkers in flight: two where one workgroup fills a CU and its registers allow it (complex128, magnetic, 32
  // sites, 32 walkers, 48 frequencies: 881 -> 809 us).
  static constexpr int DEPTH = !fp32 && !FEW && TT == 1024 && PPT == 1 && TERMS == 1 ? 2 : 1;
  static constexpr int WAVES =
      TT == 704    ? 3
      : TT == 1024 ? (SMALL ? 8 : 4)
      : FEW        ? (SMALL ? 8 : PPT == 1 && TOTALS <= 8 ? 4 : 2)
      : PPT == 1   ? (TOTALS >= (fp32 ? 12 : 8) ? 3 : 4)
      : fp32       ? (TOTALS >= 8 ? 3 : 4)
                   : (TOTALS <= 2 ? 4 : TOTALS <= 4 ? 3 : 2);
  // The compiler sinks the loads to their use, behind the products they are to overlap; kept in place
  // they must fit beside everything else, which complex128 G in large tiles does not.
  static constexpr bool HOLD = fp32 || TT <= 256 || (PPT == 1 && TOTALS <= 4);
  // FEW: no loads past the last walker, where a branch around them costs no registers.
  static constexpr bool EXACT = FEW && (fp32 || TT <= 256 || PPT == 1);
};

// G4[i] += v in two steps, so that a thread's loads are issued ahead of its stores.
__device__ __forceinline__ void g4_put(void* g4, size_t i, float4 old, double2 acc, int sum_mode) {
  if (sum_mode == SUM_FP64) {
    static_cast<double2*>(g4)[i] = double2{__hiloint2double(__float_as_int(old.y), __float_as_int(old.x)) + acc.x,
                                           __hiloint2double(__float_as_int(old.w), __float_as_int(old.z)) + acc.y};
  }
  else {
    float4 v = old;
    const float hx = static_cast<float>(acc.x), hy = static_cast<float>(acc.y);
    const float lx = static_cast<float>(acc.x - hx), ly = static_cast<float>(acc.y - hy);
    const float yx = hx - v.z, yy = hy - v.w;
    const float tx = v.x + yx, ty = v.y + yy;
    v.z = ((tx - v.x) - yx) - lx;
    v.w = ((ty - v.y) - yy) - ly;
    v.x = tx;
    v.y = ty;
    static_cast<float4*>(g4)[i] = v;
  }
}

}  // namespace

// UV[((m * 4 + plane) * nqv + qv) * P + p], planes: a(u0-u1), a(u0+u1), v0-v1, v0+v1.
template <typename Real>
__global__ void __launch_bounds__(256) uv_kernel(TiledArgs<Real> a) {
  using C = Cplx<Real>;
  const Geo& g = a.g;
  const int P = g.nc * g.nw;
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= P)
    return;
  const int qv = blockIdx.y, m = blockIdx.z;
  const int nqv = g.nq * g.nv;
  const int q = a.k_ex[qv % g.nq], nu = a.w_ex[qv / g.nq];
  const int k = p % g.nc, w = p / g.nc;
  const int kq = a.k_add[k + g.nc * q];
  const size_t D = g.D;
  const C* G0 = a.G + (2 * static_cast<size_t>(m)) * D * D;
  const C* G1 = G0 + D * D;
  const int we = w + g.ext, wq = w + nu + g.ext;
  const C u0 = g_upper(a, G0, k, we, kq, wq), u1 = g_upper(a, G1, k, we, kq, wq);
  const C v0 = g_upper(a, G0, kq, wq, k, we), v1 = g_upper(a, G1, kq, wq, k, we);
  const Real alpha = static_cast<Real>(0.5 * a.desc[2 * m].sign);
  C* out = a.UV + (static_cast<size_t>(m) * 4 * nqv + qv) * P + p;
  const size_t plane = static_cast<size_t>(nqv) * P;
  out[0] = C{alpha * (u0.x - u1.x), alpha * (u0.y - u1.y)};
  out[plane] = C{alpha * (u0.x + u1.x), alpha * (u0.y + u1.y)};
  out[2 * plane] = C{v0.x - v1.x, v0.y - v1.y};
  out[3 * plane] = C{v0.x + v1.x, v0.y + v1.y};
}

template <typename Real, int TT, int PPT, int QG, int SET, bool FEW>
__global__ void __launch_bounds__(TT, (PairShape<Real, TT, PPT, QG, SET, FEW>::WAVES)) g4_pair_kernel(TiledArgs<Real> a) {
  using C = Cplx<Real>;
  using P2 = CPair<C>;
  using Shape = PairShape<Real, TT, PPT, QG, SET, FEW>;
  constexpr bool HX = (SET & HAS_X) != 0, HZ = (SET & HAS_Z) != 0, HT = (SET & HAS_T) != 0, HY = HX || HT;
  constexpr int DEPTH = Shape::DEPTH, FLUSH = Shape::FLUSH;
  extern __shared__ unsigned char smem_raw[];
  const Geo& g = a.g;
  const int nc = g.nc, nw = g.nw, e = g.ext, P = nc * nw;
  const size_t D = g.D, DD = D * D;
  int w1, w2, z;
  if (!tile_coords(a, w1, w2, z))
    return;
  // Channel tables by select: a run-time index would put the arguments in scratch memory, whose loads
  // wait behind the G4 loads and stores in flight.
  auto ch_of = [&](int c) { return c == 0 ? a.ch[0] : c == 1 ? a.ch[1] : c == 2 ? a.ch[2] : a.ch[3]; };
  auto g4_of = [&](int c) { return c == 0 ? a.g4[0] : c == 1 ? a.g4[1] : c == 2 ? a.g4[2] : a.g4[3]; };
  const int iv = z / a.nqg, q0 = (z % a.nqg) * QG;
  const int nu = a.w_ex[iv];
  const int ld = nc + 1, bs = nc * ld, ncc = nc * nc;
  P2* Yl = reinterpret_cast<P2*>(smem_raw);  // [b][a] (a fastest): {spin 0, spin 1}
  P2* Zl = Yl + (HY ? bs : 0);
  C* const Fl = reinterpret_cast<C*>(smem_raw + a.uv_lds);  // FEW: rank-one factors [walker][plane][momentum][k]
  // Blocks (wa, wb) of G (extended frequencies). Of a conjugate symmetric G only the half
  // wa + wb >= nwE - 1 is read: another block is the conjugate of (-wa, -wb) at (-ka, -kb); its sign
  // is applied where the block is staged (Y, Z) or scaled by alpha (X).
  auto mirrored = [&](int wa, int wb) { return a.half_g && wa + wb < g.nwE - 1; };
  auto block = [&](int wa, int wb) {
    const bool m = mirrored(wa, wb);
    return nc * static_cast<size_t>(m ? g.nwE - 1 - wa : wa) + D * (nc * static_cast<size_t>(m ? g.nwE - 1 - wb : wb));
  };
  const int wy = nu + e, wz = nu + nw - 1 + e;
  const bool xm = mirrored(w1 + e, w2 + e), ym = mirrored(w2 + wy, w1 + wy), zm = mirrored(wz - w1, wz - w2);
  // Wave-uniform block bases and, per thread, element offsets within a block (below nc D < 2^32).
  const C* Xg = a.G + block(w1 + e, w2 + e);
  const C* Yg = a.G + block(w2 + wy, w1 + wy);
  const C* Zg = a.G + block(wz - w1, wz - w2);
  const Real xs_im = xm ? -1 : 1, ys_im = ym ? -1 : 1, zs_im = zm ? -1 : 1;
  auto element = [&](int ka, int kb, bool m) {
    return static_cast<unsigned>(m ? a.k_neg[ka] : ka) + static_cast<unsigned>(D) * static_cast<unsigned>(m ? a.k_neg[kb] : kb);
  };

  // The thread's pairs: element j is idx = tid + TT j of the block, (k1, k2) = (idx % nc, idx / nc)
  // (pair 0 for idle ones). It loads X, Y and Z at the same idx.
  bool ok[PPT];
  unsigned xo[PPT], yo[PPT], zo[PPT];
  int li[PPT], kk[PPT];  // LDS place; k1 | k2 << 16
  int yz[PPT][QG];  // LDS places of Y^q and Z^q, 16 bits each (bs <= 64 * 65)
#pragma unroll
  for (int j = 0; j < PPT; ++j) {
    const int idx = threadIdx.x + TT * j;
    ok[j] = idx < ncc;
    const int k1 = ok[j] ? idx % nc : 0, k2 = ok[j] ? idx / nc : 0;
    xo[j] = element(k1, k2, xm);
    yo[j] = element(k1, k2, ym);
    zo[j] = element(k1, k2, zm);
    li[j] = k2 * ld + k1;
    kk[j] = k1 | (k2 << 16);
#pragma unroll
    for (int qi = 0; qi < QG; ++qi) {
      const int q = a.k_ex[q0 + qi < g.nq ? q0 + qi : 0];
      yz[j][qi] = (a.k_add[k1 + nc * q] * ld + a.k_add[k2 + nc * q]) |
                  ((a.k_sub[k2 + nc * q] * ld + a.k_sub[k1 + nc * q]) << 16);
    }
  }

  double2 tx[PPT][QG], tz[PPT][QG], tt[PPT][QG];  // FP64 totals
  C fx[PPT][QG], fz[PPT][QG], ft[PPT][QG];         // partial sums (FLUSH > 1)
#pragma unroll
  for (int j = 0; j < PPT; ++j)
#pragma unroll
    for (int qi = 0; qi < QG; ++qi) {
      tx[j][qi] = tz[j][qi] = tt[j][qi] = double2{0, 0};
      fx[j][qi] = fz[j][qi] = ft[j][qi] = C{0, 0};
    }
  const int n_walk = a.n_walkers;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const size_t uv_row = static_cast<size_t>(g.nq) * g.nv * P;  // between the planes of one walker
  C px[DEPTH][PPT][2], py[DEPTH][PPT][2], pz[DEPTH][PPT][2];  // the next walkers'
  double sign[DEPTH];
  auto fetch = [&](int m, int d) {
    const int mc = m < n_walk ? m : n_walk - 1;
    const size_t mo = 2 * static_cast<size_t>(mc) * DD;
    sign[d] = a.desc[2 * mc].sign;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const C* X = Xg + mo + s * DD;
      const C* Y = Yg + mo + s * DD;
      const C* Z = Zg + mo + s * DD;
#pragma unroll
      for (int j = 0; j < PPT; ++j) {
        if (HY)
          py[d][j][s] = Y[yo[j]];
        if (HZ)
          pz[d][j][s] = Z[zo[j]];
      }
#pragma unroll
      for (int j = 0; j < PPT; ++j)
        px[d][j][s] = X[xo[j]];
    }
  };
  auto flush = [&]() {
    auto add = [](double2& t, C f) {
      if constexpr (FEW && FLUSH > 1)
        t = to_d(f);  // the one sum of the launch
      else
        t = double2{t.x + static_cast<double>(f.x), t.y + static_cast<double>(f.y)};
    };
#pragma unroll
    for (int j = 0; j < PPT; ++j)
#pragma unroll
      for (int qi = 0; qi < QG; ++qi) {
        if (HX)
          add(tx[j][qi], fx[j][qi]);
        if (HZ)
          add(tz[j][qi], fz[j][qi]);
        if (HT)
          add(tt[j][qi], ft[j][qi]);
        fx[j][qi] = fz[j][qi] = ft[j][qi] = C{0, 0};
      }
  };
  auto walker = [&](int m, int d) {
    __syncthreads();  // the previous walker's blocks have been read
#pragma unroll
    for (int j = 0; j < PPT; ++j)
      if (ok[j]) {
        if (HY)
          store_pair(Yl[li[j]], C{py[d][j][0].x, py[d][j][0].y * ys_im}, C{py[d][j][1].x, py[d][j][1].y * ys_im});
        if (HZ)
          store_pair(Zl[li[j]], C{pz[d][j][0].x, pz[d][j][0].y * zs_im}, C{pz[d][j][1].x, pz[d][j][1].y * zs_im});
      }
    const Real al = static_cast<Real>(0.5 * sign[d]), ali = al * xs_im;
    C x0[PPT], x1[PPT];
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
      x0[j] = C{al * px[d][j][0].x, ali * px[d][j][0].y};
      x1[j] = C{al * px[d][j][1].x, ali * px[d][j][1].y};
    }
    __syncthreads();
    if constexpr (Shape::EXACT) {
      if (m + 1 < n_walk)
        fetch(m + 1, d);
    }
    else {
      fetch(m + DEPTH, d);
      if constexpr (Shape::HOLD)
        asm volatile("" ::: "memory");
    }
#pragma unroll
    for (int j = 0; j < PPT; ++j) {
#pragma unroll
      for (int qi = 0; qi < QG; ++qi) {
        if (HY) {
          const P2& yy = Yl[yz[j][qi] & 0xffff];
          const C y0 = yy.a, y1 = yy.b;
          if (HX) {
            cfma(fx[j][qi], x0[j], y0);
            cfma(fx[j][qi], x1[j], y1);
          }
          if (HT) {
            cfma(ft[j][qi], x0[j], y1);
            cfma(ft[j][qi], x1[j], y0);
          }
        }
        if (HZ) {
          const P2& zz = Zl[static_cast<unsigned>(yz[j][qi]) >> 16];
          const C z0 = zz.a, z1 = zz.b;
          cfma(fz[j][qi], x0[j], z1);
          cfma(fz[j][qi], x1[j], z0);
        }
      }
    }
    if (FLUSH == 1 || (!FEW && (m + 1) % FLUSH == 0))
      flush();
  };
  if (n_walk > 0) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
      fetch(d, d);
    if constexpr (FEW && HX)
      for (int i = threadIdx.x; i < (a.rank_one ? n_walk * 4 * QG * nc : 0); i += TT) {
        const int k = i % nc, r = i / nc, qi = r % QG, row = r / QG;  // row: plane + 4 walker
        const int qc = q0 + qi < g.nq ? q0 + qi : q0;
        Fl[i] = a.UV[uv_row * row + static_cast<size_t>(qc + g.nq * iv) * P + nc * static_cast<size_t>((row & 2) ? w2 : w1) + k];
      }
    if (wave * 64 >= ncc) {  // a wave without pairs
      for (int m = 0; m < n_walk; ++m) {
        __syncthreads();
        __syncthreads();
      }
    }
    else {
      int m = 0;
      for (; m + DEPTH <= n_walk; m += DEPTH)
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
          walker(m + d, d);
      if constexpr (DEPTH > 1)
        if (m < n_walk)
          walker(m, 0);
    }
    if (FLUSH > 1)
      flush();
  }

  // Rank-one terms, totals and G4, for RB momenta at a time: rank-one blocks of both channels into
  // LDS, then each thread's channel totals, its G4 entries and the images (G4Sym) that no workgroup
  // computes. P keeps the order of k1 up to a permutation of its Nc entries and is stored directly;
  // T, C and both together (v = 0) go through LDS, so that the stores run along k1 of the image:
  // thread (k1, k2) of an image takes the tile's pair below.
  // LDS holds the particle-hole channels of those momenta together, or one channel at a time where a
  // plane is large (PPT = 4: up to 66.5 KB).
  constexpr int RB = TT <= 256 && PPT == 1 ? QG : 1;
  constexpr bool kOneCh = PPT == 4;
  const TileImages im = tile_images(nw, nu, w1, w2, HY, HZ, a.sym);
  double2* Rl = reinterpret_cast<double2*>(smem_raw);  // [momentum][particle-hole channel][k2][k1]
  auto g4_index = [&](int ka, int wa, int kb, int wb, int qv) {
    return ka + static_cast<size_t>(nc) *
                    (wa + static_cast<size_t>(nw) * (kb + static_cast<size_t>(nc) * (wb + static_cast<size_t>(nw) * qv)));
  };
  // Index arithmetic below starts from an opaque copy of k1 and k2 per group of entries: held for all
  // entries at once it would not fit beside the totals.
  auto own_index = [&](int kp, int qv) { return g4_index(kp & 0xffff, w1, kp >> 16, w2, qv); };
  auto swap_index = [&](int kp, int qv, int q) {
    return g4_index(swap_momentum(nc, a.k_sub, q, kp & 0xffff), im.p1, swap_momentum(nc, a.k_sub, q, kp >> 16), im.p2,
                    qv);
  };
  auto opaque = [](int v) {
    asm volatile("" : "+v"(v));
    return v;
  };
  // FEW: a matrix-core step would be mostly padding; each thread forms its entries' rank-one terms.
  auto rank_one = [&](int j, int qi, int pl) {
    double2 r{0, 0};
    for (int m = 0; m < n_walk; ++m)
      cfma(r, to_d(Fl[((4 * m + pl + 2) * QG + qi) * nc + (kk[j] >> 16)]),
           to_d(Fl[((4 * m + pl) * QG + qi) * nc + (kk[j] & 0xffff)]));
    return r;
  };
  // G4 entries per channel in flight, and channels whose entries are in flight together (one where four
  // groups of momenta are unrolled: the loop over them must unroll for the totals to stay in registers).
  constexpr int GS = RB * PPT >= 4 && !(FEW && Shape::fp32) ? 4 : RB * PPT >= 2 && !FEW ? 2 : 1;
  constexpr int CG = FEW || kOneCh || QG / RB > 2 ? 1 : 3;
#pragma unroll
  for (int r0 = 0; r0 < QG; r0 += RB) {
    if (q0 + r0 >= g.nq)
      break;
    const int nr = min(RB, g.nq - q0 - r0);
    for (int c_lo = 0; c_lo < a.n_ch; c_lo += kOneCh ? 1 : a.n_ch) {
    const int c_hi = kOneCh ? c_lo + 1 : a.n_ch;
    int n_ph = 0, n_r = 0;  // particle-hole channels, and those of them with a rank-one term
    for (int c = c_lo; c < c_hi; ++c) {
      n_ph += ch_of(c) != PP_UP_DOWN;
      n_r += ch_of(c) == PH_MAGNETIC || ch_of(c) == PH_CHARGE;
    }
    if constexpr (!FEW)
      __syncthreads();
    if (!FEW && HX && n_r > 0) {
      // R(k2, k1) blocks of 16 x 16: lane l supplies V[m0 + l/16][k2] and U[m0 + l/16][k1] and holds
      // rows k2 = 4 (l/16) + i (FP32) or l/16 + 4 i (FP64) of column k1 = l % 16.
      // complex64 G: tiles of up to 256 threads add eight walkers' FP32 products to FP64 sums, as their walker
      // loop does; larger tiles, whose walker loop adds every walker, multiply in FP64.
      constexpr bool kR32 = Shape::fp32 && TT <= 256;
      using RT = std::conditional_t<kR32, float, double>;
      using V4 = typename Mfma16<RT>::acc_t;
      const int nt = (nc + 15) / 16, n_items = nr * n_r * nt * nt;
      const size_t row = uv_row;
      for (int it = wave; it < n_items; it += TT / 64) {
        const int ta = it % nt, tb = (it / nt) % nt, cr = (it / (nt * nt)) % n_r, rq = it / (nt * nt * n_r);
        int c = c_lo, ph = 0;  // the cr-th channel with a rank-one term
        for (int left = cr;; ++c) {
          const bool has = ch_of(c) == PH_MAGNETIC || ch_of(c) == PH_CHARGE;
          if (has && left-- == 0)
            break;
          ph += ch_of(c) != PP_UP_DOWN;
        }
        const int k1 = ta * 16 + (lane & 15), k2 = tb * 16 + (lane & 15), kl = lane >> 4;
        const int pl = ch_of(c) == PH_MAGNETIC ? 0 : 1;
        const C* U = a.UV + pl * row + static_cast<size_t>(q0 + r0 + rq + g.nq * iv) * P +
                     nc * static_cast<size_t>(w1) + (k1 < nc ? k1 : 0);
        const C* V = a.UV + (pl + 2) * row + static_cast<size_t>(q0 + r0 + rq + g.nq * iv) * P +
                     nc * static_cast<size_t>(w2) + (k2 < nc ? k2 : 0);
        V4 fr{0, 0, 0, 0}, fi{0, 0, 0, 0};
        double dr[4] = {0, 0, 0, 0}, di[4] = {0, 0, 0, 0};
        constexpr int RU = 4;  // steps of four walkers loaded together
        for (int m0 = 0; m0 < n_walk; m0 += 4 * RU) {
          C u[RU], v[RU];
          bool live[RU];
#pragma unroll
          for (int i = 0; i < RU; ++i) {
            const int m = m0 + 4 * i + kl;
            live[i] = m < n_walk;
            const size_t mo = 4 * row * static_cast<size_t>(m < n_walk ? m : n_walk - 1);
            u[i] = U[mo];
            v[i] = V[mo];
          }
#pragma unroll
          for (int i = 0; i < RU; ++i) {
            if (m0 + 4 * i >= n_walk)
              break;
            // R += V U = (Vx Ux - Vy Uy) + i (Vy Ux + Vx Uy)
            const C vv = live[i] ? v[i] : C{0, 0}, uu = live[i] ? u[i] : C{0, 0};
            const RT vr = vv.x, vi = vv.y, ur = uu.x, ui = uu.y;
            fr = Mfma16<RT>::mma(vr, ur, fr);
            fi = Mfma16<RT>::mma(vi, ur, fi);
            fr = Mfma16<RT>::mma(-vi, ui, fr);
            fi = Mfma16<RT>::mma(vr, ui, fi);
            if (kR32 && (i % 2 == 1 || m0 + 4 * i + 4 >= n_walk)) {  // eight walkers per FP32 sum
#pragma unroll
              for (int h = 0; h < 4; ++h) {
                dr[h] += static_cast<double>(fr[h]);
                di[h] += static_cast<double>(fi[h]);
              }
              fr = fi = V4{0, 0, 0, 0};
            }
          }
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const int kr = tb * 16 + (kR32 ? 4 * kl + h : kl + 4 * h);
          if (k1 < nc && kr < nc)
            Rl[(rq * n_ph + ph) * bs + kr * ld + k1] =
                kR32 ? double2{dr[h], di[h]} : double2{static_cast<double>(fr[h]), static_cast<double>(fi[h])};
        }
      }
      __syncthreads();
    }
    // The tile's own entries, CG channels' loads in flight before their stores.
    int ph0 = 0;
    for (int c0 = c_lo; c0 < c_hi; c0 += CG) {
#pragma unroll
      for (int i0 = 0; i0 < RB * PPT; i0 += GS) {
        int kp[GS];
#pragma unroll
        for (int i = 0; i < GS; ++i)
          kp[i] = opaque(kk[(i0 + i) % PPT]);
        float4 old[CG][GS], oldp[HZ ? GS : 1];  // at most one pp channel
#pragma unroll
        for (int k = 0; k < CG; ++k)
          if (c0 + k < c_hi)
#pragma unroll
            for (int i = 0; i < GS; ++i) {
              const int r = (i0 + i) / PPT, j = (i0 + i) % PPT;
              if (r >= nr || !ok[j])
                continue;
              const int qv = q0 + r0 + r + g.nq * iv;
              old[k][i] = static_cast<const float4*>(g4_of(c0 + k))[own_index(kp[i], qv)];
              if (!FEW && im.p && ch_of(c0 + k) == PP_UP_DOWN)
                oldp[HZ ? i : 0] =
                    static_cast<const float4*>(g4_of(c0 + k))[swap_index(kp[i], qv, a.k_ex[q0 + r0 + r])];
            }
        int ph = ph0;
#pragma unroll
        for (int k = 0; k < CG; ++k)
          if (c0 + k < c_hi) {
            const int type = ch_of(c0 + k);
            const bool is_pp = HZ && type == PP_UP_DOWN;
            void* g4 = g4_of(c0 + k);
#pragma unroll
            for (int i = 0; i < GS; ++i) {
              const int r = (i0 + i) / PPT, j = (i0 + i) % PPT;
              if (r >= nr || !ok[j])
                continue;
              const int qv = q0 + r0 + r + g.nq * iv;
              double2 v;
              if (is_pp)
                v = tz[j][r0 + r];
              else if (HX && (type == PH_MAGNETIC || type == PH_CHARGE)) {
                if constexpr (FEW)
                  v = rank_one(j, r0 + r, type == PH_MAGNETIC ? 0 : 1);
                else
                  v = Rl[(r * n_ph + ph) * bs + li[j]];
                v.x -= tx[j][r0 + r].x;
                v.y -= tx[j][r0 + r].y;
              }
              else
                v = double2{-tt[j][r0 + r].x, -tt[j][r0 + r].y};
              g4_put(g4, own_index(kp[i], qv), old[k][i], v, a.sum_mode);
              if (!FEW && !is_pp && (im.t || im.c))
                Rl[(r * n_ph + ph) * bs + li[j]] = v;
              if (!FEW && is_pp && im.p)
                g4_put(g4, swap_index(kp[i], qv, a.k_ex[q0 + r0 + r]), oldp[HZ ? i : 0], v, a.sum_mode);
            }
            ph += !is_pp;
          }
      }
      for (int k = 0; k < CG && c0 + k < c_hi; ++k)
        ph0 += ch_of(c0 + k) != PP_UP_DOWN;
    }
    if (FEW || n_ph == 0 || (!im.t && !im.c))
      continue;
    __syncthreads();
    // Images of the particle-hole channels.
    for (int kind = 0; kind < 3; ++kind) {  // T, C, both
      if (!(kind == 0 ? im.t : kind == 1 ? im.c : im.t && im.c))
        continue;
      const int wa = kind == 0 ? w2 : kind == 1 ? im.c1 : im.c2, wb = kind == 0 ? w1 : kind == 1 ? im.c2 : im.c1;
      int ph0 = 0;
      for (int c0 = c_lo; c0 < c_hi; c0 += CG) {
#pragma unroll
        for (int i0 = 0; i0 < RB * PPT; i0 += GS) {
          int kp[GS];
#pragma unroll
          for (int i = 0; i < GS; ++i)
            kp[i] = opaque(kk[(i0 + i) % PPT]);
          float4 old[CG][GS];
#pragma unroll
          for (int k = 0; k < CG; ++k)
            if (c0 + k < c_hi && ch_of(c0 + k) != PP_UP_DOWN)
#pragma unroll
              for (int i = 0; i < GS; ++i) {
                const int r = (i0 + i) / PPT, j = (i0 + i) % PPT;
                if (r < nr && ok[j])
                  old[k][i] = static_cast<const float4*>(g4_of(c0 + k))[g4_index(kp[i] & 0xffff, wa, kp[i] >> 16, wb, q0 + r0 + r + g.nq * iv)];
              }
          int ph = ph0;
#pragma unroll
          for (int k = 0; k < CG; ++k)
            if (c0 + k < c_hi && ch_of(c0 + k) != PP_UP_DOWN) {
#pragma unroll
              for (int i = 0; i < GS; ++i) {
                const int r = (i0 + i) / PPT, j = (i0 + i) % PPT;
                if (r >= nr || !ok[j])
                  continue;
                const int k1 = kp[i] & 0xffff, k2 = kp[i] >> 16;
                int s1, s2;
                image_source(kind, nc, a.k_add, a.k_sub, a.k_neg, a.k_ex[q0 + r0 + r], k1, k2, s1, s2);
                double2 v = Rl[(r * n_ph + ph) * bs + s2 * ld + s1];
                if (kind != 0)
                  v.y = -v.y;
                g4_put(g4_of(c0 + k), g4_index(k1, wa, k2, wb, q0 + r0 + r + g.nq * iv), old[k][i], v, a.sum_mode);
              }
              ++ph;
            }
        }
        for (int k = 0; k < CG && c0 + k < c_hi; ++k)
          ph0 += ch_of(c0 + k) != PP_UP_DOWN;
      }
    }
    }
  }
}

namespace {

// Complex totals (pairs x momenta x terms, four registers each) that a thread may hold: 16; 8 where the loads
// in flight need the others (complex128 G, or several pairs per thread, in a 1024-thread workgroup's 128
// registers: 40 sites, magnetic and pp, complex64, 32 walkers, 32 frequencies, four momenta with 16
// totals 1.13 ms, two with 8 0.58). With few walkers fewer groups save less reading: 12 or 8, and 2 where two
// workgroups then share a CU (complex128, magnetic, 32 sites, four momenta: 1.16 of the time of two).
constexpr int totals_limit(bool fp32, int threads, int ppt, int terms, bool few) {
  if (few)
    return threads == 1024 && ppt == 1 && terms == 1 ? 2 : threads == 704 || (ppt == 1 && (fp32 || threads < 1024)) ? 12 : 8;
  return threads == 1024 && (!fp32 || ppt > 1) ? 8 : 16;
}

// Launches of fewer walkers than this take the FEW kernel, up to two pairs per thread (its registers hold no
// more). It computes every tile. Where all of them are resident at once, or nearly so, the other kernel gains
// little from computing half; with many it does (`many`, 2048 frequency tiles, for tiles of more than 256
// threads), and the more walkers the sooner. Each against the other, G4 stage with four momenta, over the channel
// sets (one term; two):
//   8 to 16 sites  complex64 three walkers 0.9 - 1.05; 0.6 - 0.97, five 1.0 - 1.1; 0.7 - 1.04. complex128 two
//                  0.9 - 1.0, three 0.9 - 1.1; 0.7 - 1.0, five 0.9 - 1.4; 0.9 - 1.3
//   18, 20 sites   four walkers 0.9 - 1.1; 0.75 - 1.05
//   25, 32 sites   few tiles: five 0.8 - 1.0; 0.8 - 1.1. Many: three 0.8 - 0.9; 0.95 - 1.06, five 0.8 - 1.04; 0.93 - 1.1
//   36 sites       few tiles: five 0.9; 0.8 - 0.97. Many: complex64 one 0.9 - 1.03; 0.9 - 1.06, two 1.03;
//                  1.01 - 1.05; complex128 five 0.95; one 1.02 - 1.1
//   40, 45 sites   complex64 few tiles: three 0.9 - 1.0; two 0.92 - 1.0, three 0.98 - 1.1. Many: one 0.91 - 0.98, two
//                  1.0; one 0.97 - 1.09. complex128 five 0.93 - 0.97; one 1.05 - 1.33
constexpr int few_walkers(bool fp32, int threads, int ppt, int terms, bool many) {
  const bool one = terms == 1;
  if (ppt == 4)
    return 0;
  if (threads <= 256)
    return ppt == 2 ? 8 : fp32 ? (one ? 4 : 6) : (one ? 3 : 4);
  if (ppt == 1)
    return !many ? 9 : !one ? 3 : fp32 ? 6 : 4;
  if (threads == 704)
    return !many ? 6 : fp32 ? 2 : one ? 6 : 0;
  return !fp32 ? (one ? 6 : 0) : !many ? (one ? 4 : 3) : one ? 2 : 0;
}
constexpr size_t kLdsBytes = 160 * 1024;  // of a CU

template <typename Real, int TT, int PPT, int QG, int SET, bool FEW>
void launch_pair_kernel(TiledArgs<Real> a, size_t lds, hipStream_t st) {
  constexpr int terms = (SET & 1) + (SET >> 1 & 1) + (SET >> 2 & 1);
  if constexpr (QG == 1 || PPT * QG * terms <= totals_limit(sizeof(Real) == 4, TT, PPT, terms, FEW)) {  // others are never chosen
    const unsigned tiles = tile_schedule(a);
    hipLaunchKernelGGL((g4_pair_kernel<Real, TT, PPT, QG, SET, FEW>), dim3(tiles), dim3(TT), lds, st, a);
  }
}

template <typename Real, int TT, int PPT, int QG, int SET>
void launch_pair_set(const TiledArgs<Real>& a, size_t lds, hipStream_t st) {
  constexpr int terms = (SET & 1) + (SET >> 1 & 1) + (SET >> 2 & 1);
  if constexpr (few_walkers(sizeof(Real) == 4, TT, PPT, terms, false) > 0)
    if (a.uv_lds >= 0)
      return launch_pair_kernel<Real, TT, PPT, QG, SET, true>(a, lds, st);
  launch_pair_kernel<Real, TT, PPT, QG, SET, false>(a, lds, st);
}

template <typename Real, int TT, int PPT, int QG>
void launch_pair_shape(const TiledArgs<Real>& a, int set, size_t lds, hipStream_t st) {
  switch (set) {
    case HAS_X: launch_pair_set<Real, TT, PPT, QG, HAS_X>(a, lds, st); break;
    case HAS_Z: launch_pair_set<Real, TT, PPT, QG, HAS_Z>(a, lds, st); break;
    case HAS_X | HAS_Z: launch_pair_set<Real, TT, PPT, QG, HAS_X | HAS_Z>(a, lds, st); break;
    case HAS_T:
    case HAS_X | HAS_T: launch_pair_set<Real, TT, PPT, QG, HAS_X | HAS_T>(a, lds, st); break;
    default: launch_pair_set<Real, TT, PPT, QG, HAS_X | HAS_Z | HAS_T>(a, lds, st); break;
  }
}

// Workgroup shape: up to 256 threads while a thread owns at most 2 of the nc^2 (k1, k2) pairs, as few as
// hold the pairs (8 sites in 256 threads, three waves of four idle: 1.6 times the time of 64), 1024 threads
// (at most 4 pairs each) for larger clusters.
struct TileShape {
  int threads, ppt;
};
TileShape tile_shape(int nc) {
  const int pairs = nc * nc;
  if (pairs <= 64)
    return {64, 1};
  if (pairs <= 128)
    return {128, 1};
  if (pairs <= 256)
    return {256, 1};
  if (pairs <= 512)
    return {256, 2};
  if (pairs <= 1024)
    return {1024, 1};
  if (pairs <= 1408)
    return {704, 2};
  if (pairs <= 2048)
    return {1024, 2};
  if (pairs <= 4096)
    return {1024, 4};
  return {0, 0};
}

}  // namespace

#ifndef G4_TILED_FLOAT
int tiled_pairs_per_thread(int nc) { return tile_shape(nc).ppt; }

// LDS of a workgroup: the staged blocks (both spins), or the rank-one planes of the particle-hole
// channels that are finished together.
size_t tiled_lds_bytes(const Geo& g, int n_ph, bool need_z, size_t cplx_bytes, int qg) {
  const size_t bs = static_cast<size_t>(g.nc) * (g.nc + 1);
  const TileShape ts = tile_shape(g.nc);
  const int planes = (ts.threads <= 256 && ts.ppt == 1 ? qg : 1) * (ts.ppt == 4 ? std::min(n_ph, 1) : n_ph);
  return bs * std::max(cplx_bytes * 2 * ((n_ph > 0 ? 1 : 0) + (need_z ? 1 : 0)), sizeof(double2) * planes);
}
#endif

template <typename Real>
bool launch_g4_tiled(TiledArgs<Real> a, hipStream_t st) {
  const Geo& g = a.g;
  const TileShape ts = tile_shape(g.nc);
  const int ppt = ts.ppt;
  if (g.nb != 1 || ppt == 0 || a.n_ch < 1 || a.n_ch > 4)
    return false;
  int set = 0, n_ph = 0;
  for (int c = 0; c < a.n_ch; ++c) {
    set |= a.ch[c] == PP_UP_DOWN ? HAS_Z : a.ch[c] == PH_MAGNETIC || a.ch[c] == PH_CHARGE ? HAS_X : HAS_T;
    n_ph += a.ch[c] != PP_UP_DOWN;
  }
  a.rank_one = (set & HAS_X) != 0;
  const int terms = set == (HAS_X | HAS_Z) ? 2 : set == HAS_X || set == HAS_Z ? 1 : set & HAS_Z ? 3 : 2;
  auto plan = [&](bool few) {  // LDS of the launch
    // Momenta per workgroup: as many as the totals allow.
    int qg = g.nq >= 3 ? 4 : g.nq;
    while (qg > 1 && ppt * qg * terms > totals_limit(sizeof(Real) == 4, ts.threads, ppt, terms, few))
      qg /= 2;
    while (a.qg_cap > 0 && qg > a.qg_cap)
      qg /= 2;
    a.nqg = (g.nq + qg - 1) / qg;
    a.qg = qg;
    if (!few) {
      a.uv_lds = -1;
      return tiled_lds_bytes(g, n_ph, a.need_z, sizeof(Cplx<Real>), qg);
    }
    const size_t block = static_cast<size_t>(g.nc) * (g.nc + 1) * 2 * sizeof(Cplx<Real>);  // Y or Z, both spins
    a.uv_lds = static_cast<int>(block * ((n_ph > 0 ? 1 : 0) + (a.need_z ? 1 : 0)));
    return a.uv_lds + (a.rank_one ? sizeof(Cplx<Real>) * a.n_walkers * 4 * qg * g.nc : 0);
  };
  const bool many = static_cast<size_t>(g.nw) * g.nw * g.nv > 2048;
  bool few = a.n_walkers < few_walkers(sizeof(Real) == 4, ts.threads, ppt, terms, many);
  size_t lds = plan(few);
  if (few && lds > kLdsBytes) {
    few = false;
    lds = plan(few);
  }
  // Where every tile is resident at once (four workgroups of up to 256 threads per CU, one of 1024), half of
  // them take as long as all, and writing the images comes on top: 6x6, 16 walkers, 16 frequencies
  // (256 tiles) 183 us against 179; 24 frequencies 305 against 329.
  if (few)
    a.sym = SYM_NONE;
  else if (a.sym >= SYM_CONJ &&
           static_cast<size_t>(g.nw) * g.nw * g.nv * a.nqg <= (ts.threads <= 256 ? size_t(1024) : size_t(256)))
    a.sym = a.sym_few;
  if (a.rank_one) {
    const dim3 ug((g.nc * g.nw + 255) / 256, g.nq * g.nv, a.n_walkers);
    hipLaunchKernelGGL(uv_kernel<Real>, ug, dim3(256), 0, st, a);
  }
  auto by_qg = [&](auto tt, auto pp) {
    constexpr int TT = decltype(tt)::value, PP = decltype(pp)::value;
    if (a.qg == 4)
      launch_pair_shape<Real, TT, PP, (PP <= 2 ? 4 : 2)>(a, set, lds, st);
    else if (a.qg == 2)
      launch_pair_shape<Real, TT, PP, 2>(a, set, lds, st);
    else
      launch_pair_shape<Real, TT, PP, 1>(a, set, lds, st);
  };
  using I256 = std::integral_constant<int, 256>;
  using I704 = std::integral_constant<int, 704>;
  using I1024 = std::integral_constant<int, 1024>;
  if (ts.threads == 64)
    by_qg(std::integral_constant<int, 64>{}, std::integral_constant<int, 1>{});
  else if (ts.threads == 128)
    by_qg(std::integral_constant<int, 128>{}, std::integral_constant<int, 1>{});
  else if (ts.threads == 256 && ppt == 1)
    by_qg(I256{}, std::integral_constant<int, 1>{});
  else if (ts.threads == 256)
    by_qg(I256{}, std::integral_constant<int, 2>{});
  else if (ts.threads == 704)
    by_qg(I704{}, std::integral_constant<int, 2>{});
  else if (ppt == 1)
    by_qg(I1024{}, std::integral_constant<int, 1>{});
  else if (ppt == 2)
    by_qg(I1024{}, std::integral_constant<int, 2>{});
  else
    by_qg(I1024{}, std::integral_constant<int, 4>{});
  return true;
}

#ifdef G4_TILED_FLOAT
template bool launch_g4_tiled<float>(TiledArgs<float>, hipStream_t);
#else
template bool launch_g4_tiled<double>(TiledArgs<double>, hipStream_t);
#endif

}  // namespace g4acc
