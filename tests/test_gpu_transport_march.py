"""The transport march at the edges of its parts and launch shapes.

Marches of 2 to 23 rows end in every place of the unrolled blocks; the column
counts give one column per thread or more (the last thread sharing columns with
its neighbour or not) and, in FP64, 8, 16 and 24 directions per work-group.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the bounds of one transport application against the oracle (test_gpu_ops.py)
TOL = {np.float64: 1e-12, np.float32: 5e-5}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("Ny,Nz,nang", [(13, n, 17) for n in range(1, 23)] +
                         [(1, 9, 5), (2, 5, 23), (10, 11, 49), (20, 12, 25), (21, 8, 24), (33, 6, 40),
                          (66, 4, 9), (81, 13, 33), (95, 3, 8), (96, 5, 3), (169, 2, 3)])
def test_against_the_oracle(gpu, oracle_mod, Ny, Nz, nang, dtype):
    rng = np.random.default_rng(1000 * Ny + Nz)
    Ng, n = 3, (Ny + 1) * (Nz + 1) * nang
    F = rng.standard_normal(Ng * n)
    F[::5] = np.round(F[::5])  # ties and flat runs
    F = F.astype(dtype).astype(np.float64)
    om = rng.uniform(-0.9, 0.9, 2 * nang)
    d_om = gpu.DeviceArray(om.astype(np.float64))
    for preserve in (True, False):
        ref = F.copy()
        dF = gpu.DeviceArray(F.astype(dtype))
        gpu.ops.transport_half(dF, d_om, Ny, Nz, Ng, nang, 0.2, 0.3, 0.05, preserve)
        oracle_mod.transport_half(ref, om, Ny, Nz, Ng, nang, 0.2, 0.3, 0.05, preserve)
        err = np.abs(dF.numpy().astype(np.float64) - ref).max() / np.abs(ref).max()
        assert err <= TOL[dtype]


def _check(gpu, oracle_mod, Ny, Nz, nang, Ng, dtype):
    rng = np.random.default_rng(1000 * Ny + Nz)
    F = rng.standard_normal(Ng * (Ny + 1) * (Nz + 1) * nang).astype(dtype)
    om = rng.uniform(-0.9, 0.9, 2 * nang)
    d_om = gpu.DeviceArray(om.astype(np.float64))
    for preserve in (True, False):
        ref = F.astype(np.float64)
        dF = gpu.DeviceArray(F)
        gpu.ops.transport_half(dF, d_om, Ny, Nz, Ng, nang, 0.2, 0.3, 0.05, preserve)
        oracle_mod.transport_half(ref, om, Ny, Nz, Ng, nang, 0.2, 0.3, 0.05, preserve)
        err = np.abs(dF.numpy().astype(np.float64) - ref).max() / np.abs(ref).max()
        assert err <= TOL[dtype]


@pytest.mark.parametrize("Ny,Nz", [(64, n) for n in range(1, 21)] + [(65, 6), (66, 7), (80, 8), (95, 9)])
@pytest.mark.parametrize("nang,Ng", [(1, 205), (33, 128), (1, 204)])
def test_planes_of_whole_cache_lines(gpu, oracle_mod, Ny, Nz, nang, Ng):
    """65 to 96 columns: 32 directions and three columns per thread where their
    work-groups fill at least four fifths of the CUs (the last case: one too
    few), every end of the march with four rows in flight."""
    _check(gpu, oracle_mod, Ny, Nz, nang, Ng, np.float32)


@pytest.mark.parametrize("Ny,nang", [(4, 24), (12, 25), (16, 24), (20, 9), (27, 8), (28, 8), (28, 65),
                                     (35, 7), (36, 7), (47, 16), (48, 16), (96, 9), (130, 5)])
def test_fp64_shapes(gpu, oracle_mod, Ny, nang):
    """Both sides of each line of the FP64 launch shapes."""
    for Nz in (1, 5, 10):
        _check(gpu, oracle_mod, Ny, Nz, nang, 2, np.float64)
