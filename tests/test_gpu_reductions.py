"""The dose sum and the dose plane at the edges of their group chunks and
lane blocks, against the oracle.

Both sum in FP64 whatever the state type, so the only difference is the order:
at most n 2^-53 of the sum of magnitudes, n below 1e6 terms here: 1.2e-10.
"""
import numpy as np
import pytest

from gpu_cases import small_case

pytestmark = pytest.mark.gpu

TOL = 1.2e-10


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("have", range(8))  # bit 0: f, 1: F1, 2: f1
@pytest.mark.parametrize("Ng,Ny,Nz,nang", [(1, 1, 1, 1), (7, 1, 2, 5), (8, 3, 1, 32), (17, 4, 6, 9),
                                           (50, 15, 15, 7)])
def test_dose_over_chunks(gpu, oracle_mod, dtype, have, Ng, Ny, Nz, nang):
    rng = np.random.default_rng(Ng)
    n = Ng * (Ny + 1) * (Nz + 1) * nang
    st = [rng.standard_normal(n).astype(dtype) for _ in range(4)]
    st = [a if k == 0 or (have >> (k - 1)) & 1 else None for k, a in enumerate(st)]
    S, sig = 1.0 + rng.random(Ng + 1), rng.uniform(-0.2, 0.5, Ng)
    en = np.cumsum(0.5 + rng.random(Ng + 1))
    args = (Ng, Ny, Nz, nang, 0.5, 0.1, 0.2, 0.3, 0.4, 1.3)
    dev = [None if a is None else gpu.DeviceArray(a) for a in st]
    got = gpu.ops.idd(*dev, *(gpu.DeviceArray(t) for t in (S, sig, en)), *args, trapezoidal=True)
    ref = [None if a is None else a.astype(np.float64) for a in st]
    want = oracle_mod.idd(*ref, S, sig, en, *args, trapezoidal=True, catastrophic=True)
    size = oracle_mod.idd(*(None if a is None else np.abs(a) for a in ref), S, np.abs(sig), en, *args,
                          trapezoidal=True, catastrophic=True)
    assert abs(got - want) <= TOL * size


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("have", [0, 5, 7])
@pytest.mark.parametrize("Ng,nang", [(5, 256), (6, 256), (7, 256), (7, 255)])
def test_dose_of_wide_arrays(gpu, oracle_mod, dtype, have, Ng, nang):
    """512 nodes: 2^17 lanes, and one direction fewer."""
    test_dose_over_chunks(gpu, oracle_mod, dtype, have, Ng, 15, 31, nang)


@pytest.mark.parametrize("Ng,over", [(2, dict(Ny=1, Nz=1, Nmu=1, Nom=1)),
                                     (17, dict(Ny=2, Nz=3, Nmu=7, Nom=9)),
                                     (65, dict(Ny=4, Nz=2, Nmu=8, Nom=9))])
def test_dose_plane_over_chunks(gpu, oracle_mod, Ng, over):
    c = small_case(Ng=Ng, Lg=259.0 * Ng / 500, energy=1.0 + 0.2 * Ng,
                   flags=dict(normalize_initial_mass=0, discrete_angle_delta=0), **over)
    d = oracle_mod.deltas(c)
    rng = np.random.default_rng(Ng)
    st = [rng.random(c.cells) for _ in range(4)]
    with gpu.Solver(c, gpu.FP64) as s:
        t = {k: s.table(k) for k in ("S", "sigma", "en")}
        for k, a in enumerate(st):
            s.set_state(k, a)
        got = s.spot_plane()
    want = oracle_mod.spot_plane(*st, t["S"], t["sigma"], t["en"], c.Ng, c.nyz, c.nang, d.dg, d.du,
                                 d.dv, 1.0)
    assert np.abs(got - want).max() <= TOL * np.abs(want).max()
