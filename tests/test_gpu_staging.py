"""Host inputs through the handle's staging blocks: the queue's block beside other calls' ones.

The queue packs a measurement when it is handed over and copies the block when it runs; calls that
stage in between (batches, compute_G, accumulate_G) use the other block. Results equal the same
measurements batched (bit for bit), errors appear when the queue runs and drop it, as documented.
"""
import numpy as np
import pytest

from dca_amd import geometry as geo
from dca_amd import g4acc, synth

pytestmark = pytest.mark.gpu


def _workload(nb):
    return synth.tiny_workload(nb=nb, L=2, n_freq=4, w_ex=(0, 1), n_range=(1, 19), seed_cfg=860 + nb)


@pytest.mark.parametrize("nb", [1, 2])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_queue_beside_other_calls(nb, precision):
    wl = _workload(nb)
    g = wl.geometry
    ms = wl.draw(10)
    ref = g4acc.TpAccumulator(g, precision=precision, max_walkers=3, max_vertices=wl.n_max)
    ref.resetAccumulation()
    # compute_G waits for the handle's work, which runs the queue: ms[3] alone.
    for part in (ms[0:3], ms[8:10], ms[3:4], ms[4:7], ms[7:8]):
        ref.accumulate_batch(part)
    G = ref.compute_G(ms[0])
    acc = g4acc.TpAccumulator(g, precision=precision, max_walkers=3, max_vertices=wl.n_max)
    acc.resetAccumulation()
    for i, m in enumerate(ms[:8]):
        acc.accumulate_queued(m)
        if i == 3:
            acc.accumulate_batch(ms[8:10])  # one measurement waits in the queue
            assert np.array_equal(acc.compute_G(ms[0]), G)
        if i == 4:
            zero = np.zeros((g.nb, g.nb, 2, g.nc, g.nc, g.n_ext, g.n_ext), np.complex128)
            acc.accumulate_G(zero, 1.0)
    for a, b in zip(ref.get_G4(), acc.get_G4()):
        assert np.array_equal(a, b)


def test_queue_error_and_reset():
    wl = _workload(1)
    g = wl.geometry
    ms = wl.draw(6)
    acc = g4acc.TpAccumulator(g, max_walkers=3, max_vertices=wl.n_max)
    acc.resetAccumulation()
    bad = ms[1]
    bad.site[0] = bad.site[0].copy()
    bad.site[0][0] = g.nc
    acc.accumulate_queued(ms[0])
    acc.accumulate_queued(bad)
    with pytest.raises(g4acc.LogicError, match="out of range"):
        acc.flush()
    assert all(np.all(x == 0) for x in acc.get_G4())  # the queue was dropped
    acc.accumulate_queued(ms[2])
    acc.resetAccumulation()  # discards it
    acc.accumulate_queued(ms[3])
    one = g4acc.TpAccumulator(g, max_walkers=3, max_vertices=wl.n_max)
    one.resetAccumulation()
    one.accumulate_batch([ms[3]])
    for a, b in zip(one.get_G4(), acc.get_G4()):
        assert np.array_equal(a, b)


def test_device_index_error_is_reported_once():
    import torch
    from dca_amd.devpool import DevicePool
    wl = _workload(1)
    ms = wl.draw(2)
    ms[0].band[1] = ms[0].band[1] + 7
    pool = DevicePool(torch, ms)
    acc = g4acc.TpAccumulator(wl.geometry, max_walkers=2, max_vertices=wl.n_max)
    acc.resetAccumulation()
    acc.accumulate_device(pool.walkers)
    with pytest.raises(g4acc.LogicError, match="out of range"):
        acc.finalize()
    acc.finalize()
    acc.resetAccumulation()
    acc.accumulate_device(pool.walkers[1:])
    acc.finalize()
