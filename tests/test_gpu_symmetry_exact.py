"""FP64: a conjugate stands for an entry only where it is that entry to the last bit of what formed it."""
import numpy as np
import pytest

from dca_amd import geometry as geo
from dca_amd import g4acc, synth

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def test_g0_off_by_a_few_roundings_takes_every_tile(monkeypatch):
    """4x4 with one entry of G0 four roundings off its conjugate partner: the same G4, bit for bit, as without
    the use of symmetries."""
    wl = synth.tiny_workload(L=4, n_freq=24, w_ex=(0, 1), channels=[geo.PARTICLE_HOLE_MAGNETIC], n_range=(4, 20),
                             seed_cfg=995)
    wl.geometry.g0[0, 0, 1, 1, 2] *= 1.0 + 4 * EPS
    ms = wl.draw(9)
    out = []
    for no_sym in (False, True):
        if no_sym:
            monkeypatch.setenv("G4ACC_NO_SYM", "1")
        acc = g4acc.TpAccumulator(wl.geometry, max_walkers=9, max_vertices=wl.n_max)
        acc.resetAccumulation()
        acc.accumulate_batch(ms)
        out.append(acc.get_G4())
        acc.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("nb", [1, 2])
def test_phases_from_rounded_angles_are_used_as_given(oracle_lib, nb):
    """3x3 with the phases of one momentum turned by 50 eps: G of it and of its inverse each from its own.
    Off-diagonal G over their largest: sums of 16 vertices and twice 9 sites, 34 roundings of eps / 2 at most."""
    wl = synth.tiny_workload(nb=nb, L=3, n_freq=4, channels=[geo.PARTICLE_HOLE_MAGNETIC], n_range=(16, 16),
                             seed_cfg=996 + nb)
    g = wl.geometry
    cl = g.cluster
    zero = cl.k_index((0.0, 0.0))
    neg = [int(np.flatnonzero(cl.add[k] == zero)[0]) for k in range(cl.nc)]
    for k in range(cl.nc):  # exact partners first
        if neg[k] < k:
            cl.dft[k] = np.conj(cl.dft[neg[k]])
        elif neg[k] == k:
            cl.dft[k] = cl.dft[k].real
    k = next(k for k in range(cl.nc) if neg[k] != k)
    cl.dft[k] *= 1.0 + 50j * EPS
    meas = wl.draw(1)[0]
    ora = oracle_lib.OracleAccumulator(g)
    ora.compute_G(meas)
    ref = ora.get_G()
    acc = g4acc.TpAccumulator(g, precision="fp64", max_vertices=wl.n_max)
    got = acc.compute_G(meas)
    acc.close()
    off = np.ones(ref.shape, bool)
    for k1 in range(g.nc):
        for w in range(g.n_ext):
            off[:, :, :, k1, k1, w, w] = False
    assert np.abs(got - ref)[off].max() / np.abs(ref[off]).max() < 34 * EPS / 2
