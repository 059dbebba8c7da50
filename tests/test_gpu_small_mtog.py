"""The matrix-core M -> G of the 4-, 8- and 16-site clusters against the oracle at the edges of its
tiles: 16 columns, 16 frequencies, 16 rows, four vertices per step, the step table's capacity.

G tolerances as in test_gpu_parity.py: 1e-12 (FP64), 1e-6 (FP32), max-normalised l_inf.
"""
import math

import numpy as np
import pytest

from dca_amd import geometry as geo
from dca_amd import g4acc, synth
from oracle import bruteforce as bf

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cluster,n_max_table", [("2x2", 496), ("8site", 480), ("4x4", 448)])
@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
@pytest.mark.parametrize("n_freq", [2, 16, 34])
@pytest.mark.parametrize("n", [(1, 0), (3, 4), (16, 17), (33, 5)])
def test_small_cluster_g(oracle_lib, cluster, n_max_table, precision, tol, n_freq, n):
    cl = geo.cluster_2d((2, 2), (2, -2)) if cluster == "8site" else geo.square_cluster(int(cluster[0]))
    g = geo.make_geometry(1, cl, 5.0, n_freq, [0], [0], [geo.PARTICLE_HOLE_MAGNETIC], zeeman=0.2)
    sizes = iter(n)
    meas = synth.draw_measurement(synth.Stream(900 + n_freq + n[0]), 1, g.nc, g.beta, lambda rs: next(sizes), False)
    ora = oracle_lib.OracleAccumulator(g)
    ora.compute_G(meas)
    ref = ora.get_G()
    # The step table's capacity, and one vertex above it (the register-fused kernels).
    for n_max in (max(n), n_max_table, n_max_table + 1):
        acc = g4acc.TpAccumulator(g, precision=precision, max_vertices=n_max, tuned=False)
        err = bf.difference(ref, acc.compute_G(meas))["l_inf"]
        print(f"{cluster} {precision} nf={n_freq} n={n} n_max={n_max}: {err:.3e}", flush=True)
        assert err < tol
        acc.close()


@pytest.mark.parametrize("precision,tol", [("fp64", 1e-12), ("fp32", 1e-6)])
@pytest.mark.parametrize("n", [(448, 447), (440, 1)])
def test_full_step_table(oracle_lib, precision, tol, n):
    """All vertices a table of 128 steps may hold, most of them on one site and the rest one per site."""
    g = geo.make_geometry(1, geo.square_cluster(4), 5.0, 6, [0], [0], [geo.PARTICLE_HOLE_MAGNETIC])
    sizes = iter(n)
    meas = synth.draw_measurement(synth.Stream(77), 1, g.nc, g.beta, lambda rs: next(sizes), False)
    for s in range(2):
        meas.site[s][:] = 5
        meas.site[s][:min(16, n[s])] = np.arange(min(16, n[s]))
    ora = oracle_lib.OracleAccumulator(g)
    ora.compute_G(meas)
    acc = g4acc.TpAccumulator(g, precision=precision, max_vertices=448)
    assert bf.difference(ora.get_G(), acc.compute_G(meas))["l_inf"] < tol
