"""Tuning keys that change what is computed: switching them back gives the first results again."""
import math

import numpy as np
import pytest

from dca_amd import geometry as geo
from dca_amd import g4acc, synth

pytestmark = pytest.mark.gpu

MAG, CHG, PP = (geo.PARTICLE_HOLE_MAGNETIC, geo.PARTICLE_HOLE_CHARGE, geo.PARTICLE_PARTICLE_UP_DOWN)


def _workload():
    """4x4 at a size whose tiles are more than the card holds (24 frequencies, two exchange frequencies); only the
    conjugate symmetry applies (two transfers, pp among the channels)."""
    return synth.tiny_workload(L=4, n_freq=24, w_ex=(0, 1), k_ex=((0.0, 0.0), (math.pi, math.pi)),
                               channels=[MAG, CHG, PP], n_range=(4, 20), seed_cfg=990, zeeman=0.3)


def _run(acc, ms):
    acc.resetAccumulation()
    acc.accumulate_batch(ms)
    return acc.get_G4()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_g4_sym_off_and_on_again(precision):
    wl = _workload()
    ms = wl.draw(12)
    acc = g4acc.TpAccumulator(wl.geometry, precision=precision, max_walkers=12, max_vertices=wl.n_max, tuned=False)
    first = _run(acc, ms)
    acc.set_tuning(g4_sym=0)
    full = _run(acc, ms)
    assert any(not np.array_equal(a, b) for a, b in zip(first, full))  # the other tiles round by themselves
    acc.set_tuning(g4_sym=1)
    for a, b in zip(first, _run(acc, ms)):
        assert np.array_equal(a, b)
    acc.close()


def test_g4_sym_is_refused_without_a_symmetry():
    wl = _workload()
    wl.geometry.g0[0, 0, 1, 1, 2] *= 1.3
    acc = g4acc.TpAccumulator(wl.geometry, max_walkers=2, max_vertices=wl.n_max)
    with pytest.raises(g4acc.LogicError, match="g4_sym"):
        acc.set_tuning(g4_sym=1)
    acc.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_tile_schedules_and_strips_of_the_symmetric_tiles(precision):
    """Every schedule and strip, set between batches of one handle: each tile sums the same products in the same
    order wherever it runs, so the results are equal bit for bit."""
    wl = _workload()
    ms = wl.draw(12)
    acc = g4acc.TpAccumulator(wl.geometry, precision=precision, max_walkers=12, max_vertices=wl.n_max, tuned=False)
    first = _run(acc, ms)
    for order, strip in ((0, 2), (1, 2), (2, 1), (2, 5), (2, 16), (-1, 2)):
        acc.set_tuning(g4_tile_strip=strip, g4_tile_order=order)
        for a, b in zip(first, _run(acc, ms)):
            assert np.array_equal(a, b)
    acc.close()
