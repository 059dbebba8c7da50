"""Host batches larger than one page-locked piece: the queue and direct calls through two pieces.

A handle of three walkers with up to 320 vertices packs into two pieces of 2 MiB that hold two or three of
a batch's six slots each, so that a batch takes several pieces and a device block, and a direct call sends
one piece several times while the queue holds the other. The same measurements from device memory give
the same G4 bit for bit.
"""
import numpy as np
import pytest

from dca_amd import geometry as geo
from dca_amd import g4acc, synth

pytestmark = pytest.mark.gpu

W, LO, HI = 3, 280, 320


def _workload(nb=1):
    return synth.tiny_workload(nb=nb, L=2, n_freq=2, w_ex=(0,), n_range=(LO, HI), seed_cfg=870 + nb,
                               channels=[geo.PARTICLE_HOLE_MAGNETIC, geo.PARTICLE_PARTICLE_UP_DOWN])


def _handle(wl, **kw):
    acc = g4acc.TpAccumulator(wl.geometry, max_walkers=W, max_vertices=wl.n_max, **kw)
    acc.resetAccumulation()
    return acc


def _device_batches(wl, parts):
    """G4 of the parts as device batches, one launch each."""
    import torch
    from dca_amd.devpool import DevicePool
    acc = _handle(wl)
    pools = [DevicePool(torch, p) for p in parts]
    for p in pools:
        acc.accumulate_device(p.walkers)
    g4 = acc.get_G4()
    acc.close()
    return g4


def _equal(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


@pytest.mark.parametrize("walkers,n", [(W, HI), (8, 700)])
def test_page_locked_memory_is_two_pieces_allocated_at_creation(walkers, n):
    """A queue's first phase allocates no page-locked memory; a handle holds two pieces, of a slot or
    2 MiB each, whatever its batch."""
    wl = synth.tiny_workload(n_freq=2, n_range=(n - 40, n), seed_cfg=880)
    acc = g4acc.TpAccumulator(wl.geometry, max_walkers=walkers, max_vertices=n)
    acc.resetAccumulation()
    held = acc.lib.g4acc_host_bytes(acc._h)
    slot = 8 * n * n + 24 * n
    assert 2 * max(slot, 2 << 20) <= held <= 2 * max(slot, 2 << 20) + 1024 * walkers
    assert held < 2 * walkers * slot  # less than one batch
    for m in wl.draw(walkers + 1):
        acc.accumulate_queued(m)
    acc.finalize()
    assert acc.lib.g4acc_host_bytes(acc._h) == held
    acc.close()


@pytest.mark.parametrize("nb", [1, 2])
def test_queue_over_several_batches(nb):
    wl = _workload(nb)
    ms = wl.draw(4 * W + 2)
    parts = [ms[i:i + W] for i in range(0, len(ms), W)]
    acc = _handle(wl)
    for m in ms:
        acc.accumulate_queued(m)
    assert _equal(_device_batches(wl, parts), acc.get_G4())
    acc.resetAccumulation()
    for p in parts:
        acc.accumulate_batch(p)
    assert _equal(_device_batches(wl, parts), acc.get_G4())
    acc.close()


@pytest.mark.parametrize("queued", [1, 2])  # the queue holds its first piece, or its second and a block
def test_direct_calls_beside_a_held_piece(queued):
    wl = _workload()
    ms = wl.draw(queued + 2 * W + 1)
    wait, rest = ms[:queued], ms[queued:]
    acc = _handle(wl)
    ref = _handle(wl)
    G = ref.compute_G(rest[0])
    ref.close()
    for m in wait:
        acc.accumulate_queued(m)
    acc.accumulate_batch(rest)  # chunks of W, W and one, all through the other piece
    got = acc.get_G4()
    assert _equal(_device_batches(wl, [rest[:W], rest[W:2 * W], rest[2 * W:], wait]), got)
    acc.resetAccumulation()
    acc.accumulate_queued(wait[0])
    assert np.array_equal(acc.compute_G(rest[0]), G)
    acc.close()


def test_error_after_a_piece_was_sent():
    """The third measurement of a batch is bad: its batch is dropped, the next one is whole."""
    wl = _workload()
    ms = wl.draw(2 * W)
    bad = wl.draw(1)[0]
    bad.site[1] = bad.site[1].copy()
    bad.site[1][5] = wl.geometry.nc
    acc = _handle(wl)
    for m in ms[:W - 1]:
        acc.accumulate_queued(m)
    with pytest.raises(g4acc.LogicError, match="out of range"):
        acc.accumulate_queued(bad)
    for m in ms[W:]:
        acc.accumulate_queued(m)
    assert _equal(_device_batches(wl, [ms[W:]]), acc.get_G4())
    with pytest.raises(g4acc.LogicError, match="out of range"):
        acc.accumulate_batch([ms[0], ms[1], bad])
    acc.close()


def test_hand_off_and_padded_columns_through_two_pieces():
    """N with exp V, and M with a leading dimension above n, over several pieces."""
    wl = _workload()
    ms = wl.draw(W)
    rng = np.random.default_rng(5)
    exp_v = [[np.exp(rng.choice([-0.6, 0.6], m.n[s])) for s in range(2)] for m in ms]
    formed = []
    for m, x in zip(ms, exp_v):
        formed.append(synth.Measurement(n=m.n, M=[(x[s] - 1.0)[:, None] * m.M[s] for s in range(2)], tau=m.tau,
                                        site=m.site, band=m.band, sign=m.sign))
    ref, acc = _handle(wl), _handle(wl)
    ref.accumulate_batch(formed)
    acc.accumulate_batch_n(ms, exp_v)
    for a, b in zip(ref.get_G4(), acc.get_G4()):
        # M formed on the host and on the device rounds alike (one product in FP64)
        assert np.array_equal(a, b)
    padded = [synth.Measurement(n=m.n, M=[np.asfortranarray(np.vstack([m.M[s], np.full((3, m.n[s]), np.nan)]))
                                          for s in range(2)], tau=m.tau, site=m.site, band=m.band, sign=m.sign)
              for m in ms]
    acc.resetAccumulation()
    for m in padded:
        acc.accumulate_queued(m)
    assert _equal(_device_batches(wl, [ms]), acc.get_G4())
    ref.close()
    acc.close()
