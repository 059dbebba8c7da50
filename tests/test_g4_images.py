"""G4 images of the symmetric tiles: the kernel's index maps on the CPU, and on the GPU at sizes whose tiles are
more than the card holds at once (below that every tile is computed): each cluster shape, transverse and pp
alone, self-inverse transfers (conjugate and transpose images together), negative exchange frequencies and one
beyond half of the window, FP64, FP32 and compensated sums.

Tolerances as in test_gpu_parity.py: 1e-12 (FP64) and 1e-6 (FP32), l_inf over the largest sum of the terms' sizes.
"""
import math
import os
import subprocess

import numpy as np
import pytest

from dca_amd import geometry as geo
from dca_amd import g4acc, synth

HERE = os.path.dirname(os.path.abspath(__file__))
TR, MAG, CHG, PP = (geo.PARTICLE_HOLE_TRANSVERSE, geo.PARTICLE_HOLE_MAGNETIC, geo.PARTICLE_HOLE_CHARGE,
                    geo.PARTICLE_PARTICLE_UP_DOWN)
P0, PPI, PX, PH = (0.0, 0.0), (math.pi, math.pi), (math.pi, 0.0), (math.pi / 2, math.pi / 2)
SQ = lambda L: ((L, 0), (0, L))

# name: (cluster, n_freq, w_ex, k_ex, channels)
CASES = {
    "4x4_all": (SQ(4), 34, (0,), (P0, PH), (TR, MAG, CHG, PP)),
    "4x4_self_inverse": (SQ(4), 34, (0,), (PPI, PX), (TR, MAG)),
    "4x4_pp_only": (SQ(4), 24, (0, 2), (P0, PH), (PP,)),
    "4x4_negative_wex": (SQ(4), 24, (-2, 1), (PH,), (TR, MAG, PP)),
    "4x4_wex_beyond_half": (SQ(4), 34, (20,), (P0,), (CHG, PP)),
    "4x4_wex_beyond_half_ph": (SQ(4), 34, (20,), (P0,), (CHG,)),
    "8site": (((2, 2), (2, -2)), 24, (0, 1), (P0, PH), (MAG, CHG, PP)),
    "3x3": (SQ(3), 34, (1,), (P0, (2 * math.pi / 3, 0.0)), (MAG, PP)),
    "18site": (((3, 3), (3, -3)), 34, (0,), (P0, PPI), (MAG, PP)),
    "25site": (SQ(5), 18, (1,), (P0,), (CHG, PP)),
    "6x6": (SQ(6), 18, (1,), (P0, PX, (2 * math.pi / 3, 0.0)), (MAG, PP)),
    "6x6_self_inverse": (SQ(6), 18, (0,), (PX,), (CHG,)),
    "8x8": (SQ(8), 18, (0,), (P0, (math.pi / 4, 0.0)), (CHG,)),
}
WALKERS = 9  # fewer take every tile


def _inverse(cl):
    return [int(np.flatnonzero(cl.add[k] == cl.k_index((0.0, 0.0)))[0]) for k in range(cl.nc)]


def _workload(name):
    vec, nf, wex, kex, channels = CASES[name]
    wl = synth.tiny_workload(cluster=geo.cluster_2d(*vec), n_freq=nf, w_ex=wex, k_ex=kex, channels=list(channels),
                             n_range=(4, 16), seed_cfg=960 + list(CASES).index(name), zeeman=0.37)
    # Exactly conjugate symmetric G0 and phases, whatever the rounding of the momenta.
    g, neg = wl.geometry, _inverse(wl.geometry.cluster)
    half = g.n_ext // 2
    for w in range(half):
        for k in range(g.nc):
            g.g0[:, :, :, neg[k], w] = np.conj(g.g0[:, :, :, k, g.n_ext - 1 - w])
    for k in range(g.nc):
        if neg[k] == k:
            g.cluster.dft[k] = g.cluster.dft[k].real
        elif neg[k] < k:
            g.cluster.dft[k] = np.conj(g.cluster.dft[neg[k]])
    return wl, neg


def _computed(nw, nu, ph, pp):
    """[w1, w2]: whether the tile is computed where images are in use (sym_tile_computed, csrc/g4acc_kernels.hpp)."""
    w1, w2 = np.meshgrid(np.arange(nw), np.arange(nw), indexing="ij")
    hi, lo = np.maximum(w1, w2), np.minimum(w1, w2)
    outside = lambda n: (n - hi < 0) | (n - lo >= nw)
    return (w1 + w2 >= nw - 1 - abs(nu)) | (ph & outside(nw - 1 - nu)) | (pp & outside(nw - 1 + nu))


def _exact_images(g, neg, g4, channel):
    """Tiles left out, if every entry of them equals its source bit for bit (conjugate for particle-hole, pair
    swap for pp), else None."""
    nc, nw = g.nc, g.n_freq
    ph, pp = any(c != PP for c in g.channels), PP in g.channels
    a = g4.reshape((nc, nw, nc, nw, len(g.k_ex), len(g.w_ex)), order="F")
    left_out = 0
    for iv, nu in enumerate(g.w_ex):
        done = _computed(nw, nu, ph, pp)
        for iq, q in enumerate(g.k_ex):
            x = a[..., iq, iv]
            if channel == PP:  # (k1, w1, k2, w2) -> (q - k1, ., q - k2, .)
                k = g.cluster.sub[:, q]
                f = lambda w1, w2: (nw - 1 + nu - w1, nw - 1 + nu - w2)
            else:              # (1, 2) -> (-(2 + Q), -(1 + Q)), conjugated
                k = np.array(neg)[g.cluster.add[:, q]]
                f = lambda w1, w2: (nw - 1 - nu - w2, nw - 1 - nu - w1)
            for w1, w2 in zip(*np.nonzero(~done)):
                v1, v2 = f(w1, w2)
                own, src = x[:, w1, :, w2], x[:, v1, :, v2][np.ix_(k, k)]
                left_out += 1
                if not np.array_equal(own, src if channel == PP else np.conj(src.T)):
                    return None
    return left_out


def test_index_maps_on_the_cpu():
    exe = os.path.join(HERE, "cpp", "_build", "sym_images_test")
    if not os.path.exists(exe):
        os.makedirs(os.path.dirname(exe), exist_ok=True)
        subprocess.run(["g++", "-std=c++17", "-O2", "-Wno-unknown-pragmas", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", os.path.join(HERE, "cpp", "sym_images_test.cpp"), "-o", exe],
                       check=True)
    out = subprocess.run([exe], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout.strip() == "OK", out.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_images_match_oracle(oracle_lib, name):
    wl, neg = _workload(name)
    g = wl.geometry
    ms = wl.draw(WALKERS)
    ref = size = None
    for m in ms:
        acc = oracle_lib.OracleAccumulator(g)
        acc.accumulate(m)
        one = acc.get_G4()
        ref = one if ref is None else [a + b for a, b in zip(ref, one)]
        size = [np.abs(b) for b in one] if size is None else [a + np.abs(b) for a, b in zip(size, one)]
    for precision, sum_mode, tol in (("fp64", "fp64", 1e-12), ("fp32", "fp64", 1e-6), ("fp32", "fp32_kahan", 1e-6)):
        acc = g4acc.TpAccumulator(g, precision=precision, sum_mode=sum_mode, max_walkers=WALKERS,
                                  max_vertices=wl.n_max, tuned=False)
        acc.resetAccumulation()
        acc.accumulate_batch(ms)
        got = acc.get_G4()
        for ch, r, s, x in zip(g.channels, ref, size, got):
            err = np.abs(x - r).max() / s.max()
            print(f"{name} {precision}/{sum_mode} channel {ch}: {err:.3e}", flush=True)
            assert err < tol
            images = _exact_images(g, neg, x, ch)
            # With pp no tile has both its images inside the window beyond half of it.
            assert images == 0 if name == "4x4_wex_beyond_half" else images > 0
        acc.set_tuning(g4_sym=0)
        acc.resetAccumulation()
        acc.accumulate_batch(ms)
        for ch, r, s, x in zip(g.channels, ref, size, acc.get_G4()):
            assert np.abs(x - r).max() / s.max() < tol
        acc.close()
