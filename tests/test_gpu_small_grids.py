"""Grids of few lanes: the energy sweeps that share a lane between two threads.

At the edges of that kernel (one lane, a ragged last wave, fewer groups than
its ring and its coefficient chunks) against the sweeps of wide grids and the
oracle.
"""
import numpy as np
import pytest

from gpu_cases import small_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("straggling,with_source", [(False, False), (True, False), (False, True),
                                                     (True, True)])
@pytest.mark.parametrize("lanes,Ng", [(1, 1), (31, 2), (32, 15), (33, 16), (97, 17), (64, 31),
                                      (130, 32), (63, 50)])
def test_half_sweep_equals_the_wide_grid_sweep(gpu, dtype, straggling, with_source, lanes, Ng):
    """The same lanes alone and as the first columns of a grid of 2^16 lanes
    and more (one thread per lane): the same operations on every value, so the
    same bits."""
    rng = np.random.default_rng(100 * lanes + Ng)
    wide = (1 << 16) + 32
    h, dg, rho = 0.01, 0.518, 1.1
    S = 5.0 + 100.0 * rng.random(Ng + 1)
    sig, T = 0.02 * rng.random(Ng), 0.01 * rng.random(Ng)
    F = rng.standard_normal((Ng, wide)).astype(dtype)
    f = (0.3 * rng.standard_normal((Ng, wide))).astype(dtype)
    Q = rng.random((Ng, wide)).astype(dtype) if with_source else None
    tabs = [gpu.DeviceArray(a) for a in (S, sig, T)]

    def run(cols):
        a, b = (gpu.DeviceArray(np.ascontiguousarray(x[:, :cols])) for x in (F, f))
        q = gpu.DeviceArray(np.ascontiguousarray(Q[:, :cols])) if with_source else None
        gpu.ops.energy_half(a, b, *tabs, h, dg, rho, Ng, cols, 1, Q1=q, straggling=straggling)
        return a.numpy()[:, :lanes], b.numpy()[:, :lanes]

    for narrow, full in zip(run(lanes), run(wide)):
        np.testing.assert_array_equal(narrow, full)


@pytest.mark.parametrize("Ng,over", [(17, dict(Ny=2, Nz=1, Nmu=2, Nom=3)),
                                     (33, dict(Ny=3, Nz=2, Nmu=3, Nom=3)),
                                     (500, dict(Ny=6, Nz=5, Nmu=5, Nom=5))])
@pytest.mark.parametrize("straggling", [0, 1])
def test_paired_sweeps_at_group_and_lane_edges(gpu, oracle_mod, Ng, over, straggling):
    """Whole steps with the secondary (paired sweeps with two sources) against
    the oracle, and in one call against one call per step, bit for bit."""
    c = small_case(Ng=Ng, Lg=259.0 * Ng / 500, energy=1.0 + 0.4 * 259.0 * Ng / 500,
                   flags=dict(eq15_straggling=straggling), **over)
    ref = oracle_mod.Solver(c)
    ref.advance(5)
    for precision, tol in ((gpu.FP64, 1e-10), (gpu.FP32, 2e-4)):
        with gpu.Solver(c, precision) as one, gpu.Solver(c, precision) as many:
            one.advance(5)
            for _ in range(5):
                many.advance(1)
            np.testing.assert_array_equal(one.history()[0], many.history()[0])
            for k in range(4):
                a, r = one.state(k), ref.state(k)
                np.testing.assert_array_equal(a, many.state(k))
                assert np.abs(a - r).max() <= tol * max(np.abs(r).max(), 1e-300)


@pytest.mark.parametrize("over", [dict(Ny=5, Nz=7, Nmu=7, Nom=6), dict(Ny=9, Nz=4, Nmu=11, Nom=11),
                                  dict(Ny=4, Nz=5, Nmu=18, Nom=17), dict(Ny=15, Nz=2, Nmu=3, Nom=9)])
@pytest.mark.parametrize("no_clip", [0, 1])
def test_both_arrays_in_one_launch(gpu, oracle_mod, over, no_clip):
    """Whole steps on grids whose transport and angular launches take both
    arrays of a species, the primary's psi^1 clipped or signed."""
    c = small_case(Ng=60, Lg=31.08, energy=20.0, flags=dict(no_spatial_clipping=no_clip), **over)
    ref = oracle_mod.Solver(c)
    ref.advance(4)
    for precision, tol in ((gpu.FP64, 1e-10), (gpu.FP32, 2e-4)):
        with gpu.Solver(c, precision) as s:
            s.advance(4)
            np.testing.assert_allclose(s.history()[0], ref.history()[0], rtol=tol)
            for k in range(4):
                a, r = s.state(k), ref.state(k)
                assert np.abs(a - r).max() <= tol * max(np.abs(r).max(), 1e-300)


@pytest.mark.parametrize("dtype,lanes", [(np.float32, 46999), (np.float32, 47001), (np.float32, 47008),
                                         (np.float32, 65520), (np.float32, 65536),
                                         (np.float64, 43499), (np.float64, 43500)])
def test_half_sweep_on_both_sides_of_its_limits(gpu, dtype, lanes):
    """The split sweep and the one of a thread per lane: the same bits as the
    first columns of a wide grid have."""
    rng = np.random.default_rng(lanes)
    Ng, wide = 19, (1 << 16) + 32
    S, sig, T = 5.0 + 100.0 * rng.random(Ng + 1), 0.02 * rng.random(Ng), 0.01 * rng.random(Ng)
    F, f, Q = (rng.standard_normal((Ng, wide)).astype(dtype) for _ in range(3))
    tabs = [gpu.DeviceArray(a) for a in (S, sig, T)]

    def run(cols):
        a, b, q = (gpu.DeviceArray(np.ascontiguousarray(x[:, :cols])) for x in (F, f, Q))
        gpu.ops.energy_half(a, b, *tabs, 0.01, 0.518, 1.1, Ng, cols, 1, Q1=q, straggling=True)
        return a.numpy()[:, :lanes], b.numpy()[:, :lanes]

    for narrow, full in zip(run(lanes), run(wide)):
        np.testing.assert_array_equal(narrow, full)


@pytest.mark.parametrize("precision,over", [("FP32", dict(Ny=12, Nz=15, Nmu=13, Nom=16)),   # 43,264
                                            ("FP32", dict(Ny=13, Nz=14, Nmu=14, Nom=15)),   # 44,100
                                            ("FP64", dict(Ny=8, Nz=16, Nmu=14, Nom=14)),    # 29,988
                                            ("FP64", dict(Ny=10, Nz=13, Nmu=14, Nom=14))])  # 30,184
def test_paired_sweep_on_both_sides_of_its_limits(gpu, oracle_mod, precision, over):
    c = small_case(Ng=17, Lg=0.518 * 17, energy=5.0, flags=dict(eq15_straggling=1), **over)
    ref = oracle_mod.Solver(c)
    ref.advance(3)
    tol = 1e-10 if precision == "FP64" else 2e-4
    with gpu.Solver(c, getattr(gpu, precision)) as one, gpu.Solver(c, getattr(gpu, precision)) as many:
        one.advance(3)
        for _ in range(3):
            many.advance(1)
        np.testing.assert_allclose(one.history()[0], ref.history()[0], rtol=tol)
        for k in range(4):
            a, r = one.state(k), ref.state(k)
            np.testing.assert_array_equal(a, many.state(k))
            assert np.abs(a - r).max() <= tol * max(np.abs(r).max(), 1e-300)


@pytest.mark.parametrize("Ng", [110, 90])  # 220 and 180 work-groups of 32 directions
@pytest.mark.parametrize("no_clip", [0, 1])
def test_both_arrays_of_wide_planes_in_one_launch(gpu, oracle_mod, Ng, no_clip):
    """65 columns, with the shape of whole cache lines and with the one for fewer
    work-groups."""
    c = small_case(Ng=Ng, Lg=0.518 * Ng, energy=0.3 * Ng, Ny=64, Nz=2, Nmu=6, Nom=6,
                   flags=dict(no_spatial_clipping=no_clip))
    ref = oracle_mod.Solver(c)
    ref.advance(3)
    for precision, tol in ((gpu.FP64, 1e-10), (gpu.FP32, 2e-4)):
        with gpu.Solver(c, precision) as s:
            s.advance(3)
            np.testing.assert_allclose(s.history()[0], ref.history()[0], rtol=tol)
            for k in range(4):
                a, r = s.state(k), ref.state(k)
                assert np.abs(a - r).max() <= tol * max(np.abs(r).max(), 1e-300)
