"""The four-stage M -> G at batches whose right site transform runs from LDS over half of the frequency pairs (16
frequencies and more, enough walkers), and at the first sizes below, through G4 against the oracle.

Tolerances as in test_gpu_parity.py: 1e-12 (FP64) and 1e-6 (FP32), l_inf over the largest sum of the terms' sizes.
"""
import math

import numpy as np
import pytest

from dca_amd import geometry as geo
from dca_amd import g4acc, synth

pytestmark = pytest.mark.gpu

MAG, PP = geo.PARTICLE_HOLE_MAGNETIC, geo.PARTICLE_PARTICLE_UP_DOWN
CLUSTERS = {8: ((2, 2), (2, -2)), 9: ((3, 0), (0, 3)), 10: ((3, 1), (-1, 3))}


# bands, sites, frequencies, walkers: blocks of 64 (k, w) x frequencies x slots at 512 and above, and below
@pytest.mark.parametrize("nb,nc,nf,walkers", [(3, 8, 16, 8), (3, 8, 16, 7), (3, 8, 14, 12), (2, 8, 18, 10), (1, 9, 16, 6),
                                              (1, 9, 18, 5), (1, 10, 22, 8)])
def test_batches_match_oracle(oracle_lib, nb, nc, nf, walkers):
    wl = synth.tiny_workload(nb=nb, cluster=geo.cluster_2d(*CLUSTERS[nc]), n_freq=nf, w_ex=(0,), channels=[MAG, PP],
                             n_range=(3, 30), seed_cfg=1000 + nb + nc, zeeman=0.2)
    g = wl.geometry
    ms = wl.draw(walkers)
    ref = size = None
    for m in ms:
        acc = oracle_lib.OracleAccumulator(g)
        acc.accumulate(m)
        one = acc.get_G4()
        ref = one if ref is None else [a + b for a, b in zip(ref, one)]
        size = [np.abs(b) for b in one] if size is None else [a + np.abs(b) for a, b in zip(size, one)]
    for precision, tol in (("fp64", 1e-12), ("fp32", 1e-6)):
        acc = g4acc.TpAccumulator(g, precision=precision, max_walkers=walkers, max_vertices=wl.n_max)
        acc.resetAccumulation()
        acc.accumulate_batch(ms)
        for ch, r, s, x in zip(g.channels, ref, size, acc.get_G4()):
            err = np.abs(x - r).max() / s.max()
            print(f"nb={nb} nc={nc} nf={nf} W={walkers} {precision} channel {ch}: {err:.3e}", flush=True)
            assert err < tol
        acc.close()


CLUSTERS[4] = ((2, 0), (0, 2))


# 3 bands, complex128: from 512 blocks on with 64 pairs (k, w), 256 with 256 pairs, and below
@pytest.mark.parametrize("nc,nf,walkers", [(8, 32, 1), (8, 30, 1), (8, 8, 32), (8, 8, 31), (4, 32, 4), (4, 14, 20)])
def test_three_bands_match_oracle(oracle_lib, nc, nf, walkers):
    test_batches_match_oracle(oracle_lib, 3, nc, nf, walkers)
