"""The DST over direction planes of every packing: planes that share a tile,
ragged rows, planes of one and two tiles, tiles that hold planes of two energy
groups or end a run part full.

Each plane is checked against its own maximum, over magnitudes from 1e-25 to
1e20: planes that share a tile keep their own scale.  Tolerance: the products
carry about 2^-22 (three FP16 products) and sums are FP32; on random 20 x 20
planes that makes 2.3e-7 of the maximum, and 1e-5 leaves the factor 40 by
which single planes of a few values may exceed it.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("Nmu,Nom", [(1, 1), (2, 3), (4, 4), (5, 8), (8, 5), (8, 8), (7, 7), (8, 9),
                                     (9, 8), (3, 16), (16, 2), (11, 11), (12, 12), (16, 16),
                                     (9, 13), (17, 3), (17, 6), (20, 17), (5, 19), (16, 18),
                                     (32, 31)])
@pytest.mark.parametrize("nyz,Ng", [(1, 7), (3, 5), (6, 4), (25, 2)])
def test_planes_against_the_oracle(gpu, oracle_mod, Nmu, Nom, nyz, Ng):
    rng = np.random.default_rng(1000 * Nmu + 10 * Nom + nyz)
    scale = 10.0 ** rng.uniform(-25, 20, (Ng, nyz, 1, 1))
    F = (rng.standard_normal((Ng, nyz, Nmu, Nom)) * scale).astype(np.float32)
    F[0, 0] = 0.0  # an empty plane stays empty beside others
    sig = rng.uniform(0.0, 4.0, Ng)
    args = (nyz, Ng, Nmu, Nom, 0.2, 0.13, 0.05, 1.2)
    want = F.astype(np.float64).ravel()
    oracle_mod.angle_full(want, sig, *args)
    want = want.reshape(F.shape)
    d = gpu.DeviceArray(F)
    gpu.ops.angle_full(d, sig, *args)
    got = d.numpy().reshape(F.shape).astype(np.float64)
    top = np.abs(F).max(axis=(2, 3), keepdims=True).astype(np.float64)
    assert np.all(np.abs(got - want) <= 1e-5 * top)
    assert np.all(got[0, 0] == 0.0)


@pytest.mark.parametrize("Nmu,Nom", [(7, 7), (4, 12), (12, 5), (11, 11), (20, 20)])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_a_plane_that_is_not_finite_spoils_itself_only(gpu, Nmu, Nom, bad):
    nyz, Ng = 5, 4
    rng = np.random.default_rng(3)
    F = rng.standard_normal((Ng, nyz, Nmu, Nom)).astype(np.float32)
    sig = rng.uniform(0.0, 4.0, Ng)
    out = []
    for spoil in (False, True):
        G = F.copy()
        if spoil:
            G[1, 2, 0, 0] = G[3, 0, Nmu - 1, Nom - 1] = bad
        d = gpu.DeviceArray(G)
        gpu.ops.angle_full(d, sig, nyz, Ng, Nmu, Nom, 0.2, 0.13, 0.05, 1.2)
        out.append(d.numpy().reshape(F.shape))
    spoiled = np.zeros((Ng, nyz), bool)
    spoiled[1, 2] = spoiled[3, 0] = True
    np.testing.assert_array_equal(out[1][~spoiled], out[0][~spoiled])
    assert np.all(np.isnan(out[1][spoiled]))


@pytest.mark.parametrize("Nmu,Nom", [(1, 1), (3, 2), (8, 8), (9, 8), (5, 20), (13, 13), (20, 20),
                                     (21, 3), (20, 17), (32, 32), (33, 31)])
@pytest.mark.parametrize("nyz,Ng", [(1, 3), (7, 5), (40, 2)])
def test_fp64_planes_against_the_oracle(gpu, oracle_mod, Nmu, Nom, nyz, Ng):
    """Lines padded to the kernel's sizes, work-groups part full; 1e-12 of the
    plane's maximum: four sums of at most 32 products, rounded at 2^-53."""
    rng = np.random.default_rng(1000 * Nmu + 10 * Nom + nyz)
    scale = 10.0 ** rng.uniform(-200, 200, (Ng, nyz, 1, 1))
    F = rng.standard_normal((Ng, nyz, Nmu, Nom)) * scale
    sig = rng.uniform(0.0, 4.0, Ng)
    args = (nyz, Ng, Nmu, Nom, 0.2, 0.13, 0.05, 1.2)
    want = F.ravel().copy()
    oracle_mod.angle_full(want, sig, *args)
    d = gpu.DeviceArray(F)
    gpu.ops.angle_full(d, sig, *args)
    err = np.abs(d.numpy().reshape(F.shape) - want.reshape(F.shape))
    assert np.all(err <= 1e-12 * np.abs(F).max(axis=(2, 3), keepdims=True))


@pytest.mark.parametrize("Nmu,Nom", [(1, 1), (1, 2), (2, 1), (2, 2), (4, 6), (1, 12), (12, 1), (10, 4),
                                     (22, 2), (30, 28)])
@pytest.mark.parametrize("at", [(0, 0), (-1, -1)])
def test_fp64_planes_with_an_infinity(gpu, oracle_mod, Nmu, Nom, at):
    """The lines are padded, the sums are not: infinities and NaNs come out where
    the plane's own values make them, and the other planes are untouched.  (Sizes
    whose bases hold no zero: the sign of a rounded one would be arbitrary.)"""
    nyz, Ng = 3, 2
    rng = np.random.default_rng(10 * Nmu + Nom)
    F = rng.standard_normal((Ng, nyz, Nmu, Nom))
    F[1, 1][at] = np.inf
    sig = rng.uniform(0.0, 4.0, Ng)
    args = (nyz, Ng, Nmu, Nom, 0.2, 0.13, 0.05, 1.2)
    want = F.ravel().copy()
    with np.errstate(invalid="ignore"):
        oracle_mod.angle_full(want, sig, *args)
    d = gpu.DeviceArray(F)
    gpu.ops.angle_full(d, sig, *args)
    got = d.numpy().ravel()
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    ok = np.isfinite(want)
    assert ok.sum() >= F.size - Nmu * Nom
    assert np.abs(got[ok] - want[ok]).max() <= 1e-12 * np.abs(F[np.isfinite(F)]).max()


@pytest.mark.parametrize("Nmu,Nom", [(1, 4), (1, 5), (5, 1), (1, 8), (1, 16), (17, 1), (2, 8), (2, 9),
                                     (9, 2), (2, 16), (24, 2), (24, 3), (25, 3), (3, 25), (31, 3),
                                     (32, 3), (4, 29), (23, 24), (28, 27)])
def test_fp64_thin_planes_and_every_padding(gpu, oracle_mod, Nmu, Nom):
    """Both sides of the line between a thread per line and a thread per value,
    exact and padded lines; the bound of the planes above."""
    nyz, Ng = 37, 3
    rng = np.random.default_rng(100 * Nmu + Nom)
    F = rng.standard_normal((Ng, nyz, Nmu, Nom))
    sig = rng.uniform(0.0, 4.0, Ng)
    args = (nyz, Ng, Nmu, Nom, 0.2, 0.13, 0.05, 1.2)
    want = F.ravel().copy()
    oracle_mod.angle_full(want, sig, *args)
    d = gpu.DeviceArray(F)
    gpu.ops.angle_full(d, sig, *args)
    err = np.abs(d.numpy().reshape(F.shape) - want.reshape(F.shape))
    assert np.all(err <= 1e-12 * np.abs(F).max(axis=(2, 3), keepdims=True))


@pytest.mark.parametrize("Nmu,Nom", [(1, 1), (3, 3), (5, 5), (8, 8), (7, 16), (16, 7), (12, 6), (11, 11),
                                     (16, 16), (20, 20)])
def test_a_plane_has_the_same_bits_wherever_it_sits(gpu, Nmu, Nom):
    """Alone in a tile, and at every place of a tile that it shares with planes of
    its own and of the next energy group."""
    nyz, Ng = 5, 6
    rng = np.random.default_rng(Nmu + 50 * Nom)
    F = (rng.standard_normal((Ng, nyz, Nmu, Nom)) * 10.0 ** rng.uniform(-6, 6, (Ng, nyz, 1, 1)))
    F = F.astype(np.float32)
    sig = rng.uniform(0.0, 4.0, Ng)
    d = gpu.DeviceArray(F)
    gpu.ops.angle_full(d, sig, nyz, Ng, Nmu, Nom, 0.2, 0.13, 0.05, 1.2)
    together = d.numpy().reshape(F.shape)
    for g in range(Ng):
        for s in range(nyz):
            one = gpu.DeviceArray(np.ascontiguousarray(F[g, s]))
            gpu.ops.angle_full(one, sig[g:g + 1], 1, 1, Nmu, Nom, 0.2, 0.13, 0.05, 1.2)
            np.testing.assert_array_equal(one.numpy().reshape(Nmu, Nom), together[g, s])
