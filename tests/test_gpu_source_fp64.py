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


@pytest.mark.parametrize("low,high", [(24, 30), (32, 48), (19, 33), (47, 49)])
def test_a_band_reads_its_own_groups_only(gpu, low, high):
    """Output tiles of 16 groups with the same band [low, high) each, between
    tiles whose bands are wider: infinite values in the source groups beside the
    narrow band, and weights there that are no numbers, leave those tiles as
    they are."""
    Ng, nyz, nang = 80, 3, 5
    rng = np.random.default_rng(low)
    Fp, fp = rng.random((Ng, nyz * nang)), rng.standard_normal((Ng, nyz * nang))
    kv = rng.random((Ng, nang, nang))
    beg, end = np.full(Ng, 17, np.int32), np.full(Ng, 60, np.int32)
    narrow = np.zeros(Ng, bool)
    narrow[:16] = narrow[48:64] = True
    beg[narrow], end[narrow] = low, high
    inside = (np.arange(Ng) >= beg[:, None]) & (np.arange(Ng) < end[:, None])
    ke1, ke2 = (np.where(inside, rng.random((Ng, Ng)), 0.0) for _ in range(2))
    out = []
    for spoil in (False, True):
        X, e1, e2 = Fp.copy(), ke1.copy(), ke2.copy()
        if spoil:
            X[low - 1, 2] = X[high, 4] = np.inf
            e1[~inside] = e2[~inside] = np.nan
        dev = [gpu.DeviceArray(a.ravel()) for a in (X, fp, np.zeros((Ng, nyz * nang)))]
        gpu.ops.secondary_source(*dev, *(gpu.DeviceArray(a) for a in (e1, e2, kv, beg, end)), Ng, nyz,
                                 nang, 0.5)
        out.append(dev[2].numpy().reshape(Ng, -1))
    np.testing.assert_array_equal(out[1][narrow], out[0][narrow])
    assert np.abs(out[0][narrow]).min() > 0.0
    assert not np.isfinite(out[1][~narrow]).all()
