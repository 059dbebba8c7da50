// Single-particle accumulator: M_r_w of every measurement, summed over measurements in FP64.
//
// The reference measures (SpAccumulator, sp_accumulator.hpp:160-221; GPU sp_accumulator_gpu.hpp)
//     M_r_w(b1, s, b2, s, r, w) += sign / Nc sum_{i, j} M_s(i, j) exp(i w (tau_i - tau_j))
//                                   [b_i = b1, b_j = b2, r_i - r_j = r]
// over the single-particle Matsubara frequencies, through a delayed NFFT (a Kaiser-Bessel window
// convolved onto an oversampled time grid, one FFT at finalize; dnfft_1d.hpp). Here the same sum
// is evaluated exactly in FP64, as the orbital-resolved NDFT at equal frequencies:
//     C(o1, o2; w) = sum_{i in o1} T(w, i) sum_{j in o2} M_ij conj(T(w, j)),  T(w, i) = e^{i w tau_i}
//     M_r_w(b1, b2, r, w) = 1/Nc sum over orbital pairs o1 = (b1, r1), o2 = (b2, r2), r1 - r2 = r
// with the vertices of a slot sorted by orbital (sort_kernel). M is real, so C(w') = conj C(w) at the
// opposite frequency w' = n_w - 1 - w: only the upper half of the frequencies is formed and the
// reduction writes both.
//
// The work is small (2.5 FP64 FMAs per pair of vertices and frequency) and was all latency while one
// wave walked every column for eight orbitals: 7.8 ms per 16 measurements of N ~ U[60, 180], 8
// orbitals, 128 frequencies. One wave per orbital pair and 64 frequencies gives n_orb^2 waves per
// slot; the pair's M block is loaded 64 entries at a time, one per lane, and broadcast by readlane.
// Those 64 measurements through M -> G, G4 and M_r_w: 31.3 -> 1.26 ms.
#include "g4acc_common.hpp"
#include "g4acc_kernels.hpp"

namespace g4acc {

// T_sp[slot][h + nh * ii] = exp(i w_h tau_{perm ii}), w_h = (2h + 1) pi / beta for the upper half
// h < nh = n_w / 2 (frequency_domain.cpp:29-49), reduced exactly: (2h + 1) tau / beta taken modulo
// 2, sincospi.
__global__ void __launch_bounds__(256) sp_phase_kernel(const SlotDesc* __restrict__ desc, Geo g, int nh,
                                                       int n_max, const int* __restrict__ perm,
                                                       double2* __restrict__ T) {
  const int slot = blockIdx.y;
  const SlotDesc d = desc[slot];
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= nh * d.n)
    return;
  const int h = idx % nh, ii = idx / nh;
  const int v = perm[static_cast<size_t>(slot) * n_max + ii];
  double x = static_cast<double>(2 * h + 1) * (d.tau[v] / g.beta);
  x -= 2.0 * rint(0.5 * x);
  double s, c;
  sincospi(x, &s, &c);
  T[static_cast<size_t>(slot) * nh * n_max + idx] = double2{c, s};
}

__device__ __forceinline__ double lane_value(double v, int lane) {
  const long long b = __double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane(static_cast<int>(b), lane);
  const unsigned hi = __builtin_amdgcn_readlane(static_cast<int>(b >> 32), lane);
  return __longlong_as_double(static_cast<long long>((static_cast<unsigned long long>(hi) << 32) | lo));
}

// C[slot][(o1 * n_orb + o2) * nh + h]: one wave per (o1, o2) and 64 frequencies. Per step lane l
// holds M of row i0 + l / 4 and column j0 + l % 4 (zero past the orbitals' ranges); the four columns'
// conj phases stay in registers while the sixteen rows pass.
__global__ void __launch_bounds__(256) sp_ndft_kernel(const SlotDesc* __restrict__ desc, Geo g, int nh,
                                                      int n_max, bool squared,
                                                      const int* __restrict__ perm,
                                                      const int* __restrict__ off,
                                                      const double2* __restrict__ T,
                                                      double2* __restrict__ Cout) {
  const int slot = blockIdx.y;
  const int n_orb = g.n_orb;
  const int nhb = (nh + 63) / 64;
  const int pair = __builtin_amdgcn_readfirstlane(blockIdx.x / nhb * 4 + (threadIdx.x >> 6));
  if (pair >= n_orb * n_orb)
    return;
  const SlotDesc d = desc[slot];
  const int lane = threadIdx.x & 63;
  const int o1 = pair / n_orb, o2 = pair % n_orb;
  const int h = blockIdx.x % nhb * 64 + lane;
  const int hc = h < nh ? h : nh - 1;
  const int* P = perm + static_cast<size_t>(slot) * n_max;
  const int* O = off + static_cast<size_t>(slot) * (n_orb + 1);
  const double2* Ts = T + static_cast<size_t>(slot) * nh * n_max + hc;
  const int i_lo = O[o1], i_hi = O[o1 + 1], j_lo = O[o2], j_hi = O[o2 + 1];
  double2 acc{0, 0};
  for (int j0 = j_lo; j0 < j_hi; j0 += 4) {
    double2 tj[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      tj[k] = Ts[static_cast<size_t>(nh) * (j0 + k < j_hi ? j0 + k : j_lo)];
    const int jl = j0 + (lane & 3);
    for (int i0 = i_lo; i0 < i_hi; i0 += 16) {
      const int il = i0 + (lane >> 2);
      double m = 0;
      if (il < i_hi && jl < j_hi) {
        const int i = P[il];
        m = d.m[i + static_cast<size_t>(d.ld) * P[jl]];
        if (d.expv)
          m *= d.expv[i] - 1.0;
        if (squared)
          m *= m;
      }
      const int rows = i_hi - i0 < 16 ? i_hi - i0 : 16;
#pragma unroll 4
      for (int r = 0; r < rows; ++r) {
        const double2 ti = Ts[static_cast<size_t>(nh) * (i0 + r)];
        double2 b{0, 0};  // sum over the four columns of M_ij conj(T(w, j))
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double mk = lane_value(m, 4 * r + k);
          b.x = fma(mk, tj[k].x, b.x);
          b.y = fma(-mk, tj[k].y, b.y);
        }
        cfma(acc, ti, b);
      }
    }
  }
  if (h < nh)
    Cout[(static_cast<size_t>(slot) * n_orb * n_orb + pair) * nh + h] = acc;
}

// acc[s][(b1 + nb (b2 + nb r)) * n_w + w] += sign / Nc sum over the slots of spin s and the
// orbital pairs (b1, r1), (b2, r2) with index(r1 - r2) = r, and the conjugate at the opposite
// frequency. Four waves share a label and 64 frequencies, each taking every fourth slot; their sums
// are added in wave order (deterministic).
__global__ void __launch_bounds__(256) sp_reduce_kernel(const SlotDesc* __restrict__ desc, Geo g, int nh,
                                                        int n_slots, const int* __restrict__ rsub,
                                                        const double2* __restrict__ Cin,
                                                        double2* __restrict__ acc) {
  __shared__ double2 part[4][64];
  const int nb = g.nb, nc = g.nc, n_orb = g.n_orb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int s = blockIdx.z;
  const int lab = blockIdx.y;
  const int h = blockIdx.x * 64 + lane;
  const int hc = h < nh ? h : nh - 1;
  const int b1 = lab % nb, b2 = (lab / nb) % nb, r = lab / (nb * nb);
  const double inv_nc = 1.0 / nc;
  double2 sum{0, 0};
  for (int slot = s + 2 * wave; slot < n_slots; slot += 8) {
    if (desc[slot].n == 0)
      continue;
    const double f = desc[slot].sign * inv_nc;
    const double2* C = Cin + static_cast<size_t>(slot) * n_orb * n_orb * nh + hc;
#pragma unroll 8
    for (int r1 = 0; r1 < nc; ++r1) {
      // the site r2 with r1 - r2 = r: r2 = index(r1 - r) (rsub[a + nc b] = index(r_b - r_a))
      const int r2 = rsub[r + nc * r1];
      const double2 c = C[(static_cast<size_t>(b1 + nb * r1) * n_orb + (b2 + nb * r2)) * nh];
      sum.x = fma(f, c.x, sum.x);
      sum.y = fma(f, c.y, sum.y);
    }
  }
  part[wave][lane] = sum;
  __syncthreads();
  if (wave != 0 || h >= nh)
    return;
  for (int k = 1; k < 4; ++k)
    sum = cadd(sum, part[k][lane]);
  double2* a = acc + (static_cast<size_t>(s) * gridDim.y + lab) * 2 * nh;
  double2 up = a[nh + h], lo = a[nh - 1 - h];
  up = cadd(up, sum);
  lo = cadd(lo, double2{sum.x, -sum.y});
  a[nh + h] = up;
  a[nh - 1 - h] = lo;
}

void launch_sp_accumulate(const SpArgs& a, hipStream_t st) {
  const Geo& g = a.g;
  const int nh = a.n_w / 2;
  hipLaunchKernelGGL(sp_phase_kernel, dim3((nh * a.n_max + 255) / 256, a.n_slots), dim3(256), 0, st, a.desc,
                     g, nh, a.n_max, a.perm, a.T);
  const dim3 grid((nh + 63) / 64 * ((g.n_orb * g.n_orb + 3) / 4), a.n_slots);
  const dim3 rgrid((nh + 63) / 64, g.nb * g.nb * g.nc, 2);
  for (int q = 0; q < (a.squared_too ? 2 : 1); ++q) {
    hipLaunchKernelGGL(sp_ndft_kernel, grid, dim3(256), 0, st, a.desc, g, nh, a.n_max, q == 1, a.perm, a.off,
                       a.T, a.C);
    hipLaunchKernelGGL(sp_reduce_kernel, rgrid, dim3(256), 0, st, a.desc, g, nh, a.n_slots, a.rsub, a.C,
                       q == 0 ? a.acc : a.acc_sqr);
  }
}

}  // namespace g4acc
