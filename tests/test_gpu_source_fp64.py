"""The FP64 source at the edges of its tiles: nodes and directions about 64 and
about multiples of 4 and 16, lanes about 128, output groups about 64, bands that
start and end inside a 16-group chunk, against the oracle's factorised sum.
Tolerance: sums of at most (Ng + nang) terms of one sign structure, rounded at
2^-53 each: 1e-12 of the largest result.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Ng,nyz,nang", [(5, 1, 1), (16, 3, 4), (17, 65, 7), (63, 9, 15), (64, 2, 64),
                                         (65, 33, 12), (130, 5, 65), (40, 64, 18), (33, 129, 3)])
def test_source_tiles(gpu, oracle_mod, Ng, nyz, nang):
    rng = np.random.default_rng(Ng)
    Fp, fp = rng.standard_normal(Ng * nyz * nang), rng.standard_normal(Ng * nyz * nang)
    ke1, ke2 = np.zeros((Ng, Ng)), np.zeros((Ng, Ng))
    beg, end = np.zeros(Ng, np.int32), np.zeros(Ng, np.int32)
    for g in range(Ng - 1):
        if g % 7 == 5:
            continue  # no band
        beg[g] = g + 1 + rng.integers(0, 1 + (Ng - g - 2) // 2)
        end[g] = rng.integers(beg[g] + 1, Ng + 1)
        ke1[g, beg[g]:end[g]] = rng.random(end[g] - beg[g])
        ke2[g, beg[g]:end[g]] = rng.standard_normal(end[g] - beg[g])
    kv = rng.random((Ng, nang, nang)) * (rng.random((Ng, nang, nang)) < 0.4)
    want = oracle_mod.secondary_source_factorized(Fp, fp, ke1, ke2, kv, beg, end, Ng, nyz, nang, 0.5)
    dev = [gpu.DeviceArray(a) for a in (Fp, fp, np.full(Ng * nyz * nang, np.nan))]
    gpu.ops.secondary_source(*dev, *(gpu.DeviceArray(a) for a in (ke1, ke2, kv, beg, end)), Ng, nyz,
                             nang, 0.5)
    assert np.abs(dev[2].numpy() - want).max() <= 1e-12 * max(np.abs(want).max(), 1e-300)
