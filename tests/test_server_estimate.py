"""The memory that admission charges for a beam covers every array a context
makes (host only: nothing is allocated)."""
import pytest

import bfpn_gpu_amd as bg
from gpu_cases import small_case


@pytest.mark.parametrize("precision", [bg.FP32, bg.FP64])
@pytest.mark.parametrize("over,flags,per_partial", [
    (dict(Ny=8, Nz=8, Nmu=7, Nom=7), {}, 32),  # few lanes: a partial per 32
    (dict(Ny=4, Nz=2, Nmu=3, Nom=1), {}, 32),
    (dict(Ny=40, Nz=40, Nmu=20, Nom=19), {}, 256),
    (dict(Ny=8, Nz=8, Nmu=7, Nom=7), dict(legacy_energy=1), 256),
    (dict(Ny=8, Nz=8, Nmu=7, Nom=7), dict(lite_memory=1), 256)])
def test_dose_partials_are_counted(precision, over, flags, per_partial):
    """Five sets of dose partials, four of them with a proxy: nine doubles a partial."""
    c = small_case(flags=flags, **over)
    lanes = (c.Ny + 1) * (c.Nz + 1) * c.Nmu * c.Nom
    arrays = 1 if flags.get("lite_memory") else 10
    state = arrays * lanes * c.Ng * (8 if precision == bg.FP64 else 4)
    history = 2 * max(16, c.Nx) * 8
    beam, _ = bg.Server.estimate(c, precision)
    assert beam - state - history == 9 * 8 * (-(-lanes // per_partial))
