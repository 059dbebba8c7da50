"""G4 launches of few walkers (their own tile kernel) and of the first counts above, against the oracle: every
workgroup shape, momentum groups with a remainder, each set of terms, transverse alone (no rank-one terms).

Tolerances as in test_gpu_parity.py: 1e-12 (FP64) and 1e-6 (FP32), l_inf over the largest sum of the terms' sizes.
"""
import numpy as np
import pytest

from dca_amd import geometry as geo
from dca_amd import g4acc, synth
from oracle import bruteforce as bf

pytestmark = pytest.mark.gpu

TR, MAG, CHG, PP = (geo.PARTICLE_HOLE_TRANSVERSE, geo.PARTICLE_HOLE_MAGNETIC, geo.PARTICLE_HOLE_CHARGE,
                    geo.PARTICLE_PARTICLE_UP_DOWN)
# cluster vectors: 64, 128, 256, 2 x 256, 1024, 704, 2 x 1024 and 4 x 1024 threads' pairs
CLUSTERS = {8: ((2, 2), (2, -2)), 9: ((3, 0), (0, 3)), 10: ((3, 1), (-1, 3)), 16: ((4, 0), (0, 4)),
            18: ((3, 3), (3, -3)), 25: ((5, 0), (0, 5)), 36: ((6, 0), (0, 6)), 40: ((6, 2), (-2, 6)),
            64: ((8, 0), (0, 8))}
SETS = [(MAG,), (PP,), (TR,), (CHG, PP), (TR, CHG), (TR, PP), (TR, MAG, CHG, PP)]


@pytest.mark.parametrize("nc", list(CLUSTERS))
@pytest.mark.parametrize("channels", SETS, ids=lambda c: "-".join(map(str, c)))
def test_few_walkers_match_oracle(oracle_lib, nc, channels):
    wl = synth.tiny_workload(cluster=geo.cluster_2d(*CLUSTERS[nc]), n_freq=4 if nc < 25 else 2, w_ex=(0, 1) if nc < 25 else (1,),
                             channels=list(channels), n_range=(3, 20), seed_cfg=900 + nc, zeeman=0.2)
    g = wl.geometry
    g.k_ex = [0, nc // 2, 1, nc - 1, 2][:3 if nc > 16 else 5]
    ms = wl.draw(9)
    refs = []
    for m in ms:
        acc = oracle_lib.OracleAccumulator(g)
        acc.accumulate(m)
        refs.append(acc.get_G4())
    for precision, tol in (("fp64", 1e-12), ("fp32", 1e-6)):
        acc = g4acc.TpAccumulator(g, precision=precision, max_walkers=9, max_vertices=wl.n_max, tuned=False)
        for walkers in (1, 2, 5, 6, 8, 9):
            acc.resetAccumulation()
            acc.accumulate_batch(ms[:walkers])
            for c, x in enumerate(acc.get_G4()):
                part = [r[c] for r in refs[:walkers]]
                # Signs differ, so a sum may be much smaller than its terms: their size is what is rounded.
                err = np.abs(x - sum(part)).max() / sum(map(np.abs, part)).max()
                print(f"nc={nc} {precision} W={walkers} channel {g.channels[c]}: {err:.3e}", flush=True)
                assert err < tol
        acc.close()


@pytest.mark.parametrize("nc", [16, 36])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_few_walkers_over_launches_equal_one_batch(nc, precision):
    """One walker at a time, in pairs and in fives against all seventeen in one launch (the matrix-core rank-one
    tail, two passes of sixteen): the forms differ by the order of sums only."""
    wl = synth.tiny_workload(cluster=geo.cluster_2d(*CLUSTERS[nc]), n_freq=4, w_ex=(0, 2), channels=[MAG, CHG, PP],
                             n_range=(3, 20), seed_cfg=930 + nc, zeeman=0.2)
    wl.geometry.k_ex = [0, 5, nc - 1]
    ms = wl.draw(17)
    acc = g4acc.TpAccumulator(wl.geometry, precision=precision, max_walkers=17, max_vertices=wl.n_max, tuned=False)
    acc.resetAccumulation()
    acc.accumulate_batch(ms)
    ref = acc.get_G4()
    for step in (1, 2, 5):
        acc.resetAccumulation()
        for i in range(0, 17, step):
            acc.accumulate_batch(ms[i:i + step])
        for a, b in zip(ref, acc.get_G4()):
            # 17 sums of FP64 products; complex64: products of eight walkers in FP32 before FP64
            assert bf.difference(a, b)["l_inf"] < (1e-14 if precision == "fp64" else 1e-6)
    acc.close()


@pytest.mark.parametrize("nc", [25, 36, 40])
@pytest.mark.parametrize("n_freq", [44, 46])
def test_few_walkers_around_the_tile_count(monkeypatch, nc, n_freq):
    """Tiles of more than 256 threads: the count of walkers below which the form for few is taken falls at 2048
    frequency tiles (46 squared is more, 44 squared less). Both sides against the per-entry kernel."""
    channels = [MAG, PP] if nc > 25 else [MAG]
    wl = synth.tiny_workload(cluster=geo.cluster_2d(*CLUSTERS[nc]), n_freq=n_freq, w_ex=(1,), channels=channels,
                             n_range=(3, 20), seed_cfg=960 + nc)
    g = wl.geometry
    g.k_ex = [0, nc // 2]
    ms = wl.draw(6)
    make = lambda p: g4acc.TpAccumulator(g, precision=p, max_walkers=6, max_vertices=wl.n_max, tuned=False)
    monkeypatch.setenv("G4ACC_GENERIC_G4", "1")
    ref = make("fp64")
    monkeypatch.delenv("G4ACC_GENERIC_G4")
    accs = {p: make(p) for p in ("fp64", "fp32")}
    ref.resetAccumulation()
    total, size, done = [0.0] * len(channels), [0.0] * len(channels), 0
    for m in ms:
        ref.resetAccumulation()
        ref.accumulate_batch([m])
        for c, x in enumerate(ref.get_G4()):
            total[c] = total[c] + x
            size[c] = size[c] + np.abs(x)
        done += 1
        for p, tol in (("fp64", 1e-12), ("fp32", 1e-6)):
            accs[p].resetAccumulation()
            accs[p].accumulate_batch(ms[:done])
            for c, x in enumerate(accs[p].get_G4()):
                err = np.abs(x - total[c]).max() / size[c].max()
                print(f"nc={nc} freq={n_freq} {p} W={done} channel {channels[c]}: {err:.3e}", flush=True)
                assert err < tol
    for a in (ref, *accs.values()):
        a.close()
