"""The FP32 source on grids of few lanes and on rows of any length.

A node's source depends on that node alone, so the same nodes give the same
bits on a grid of at most 32,768 lanes (tiles over output groups) and as the
first nodes of a larger one (the march over the source groups).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nang", [1, 7, 9, 49, 64, 121, 130])
def test_few_lanes_equal_the_march(gpu, oracle_mod, nang):
    rng = np.random.default_rng(nang)
    Ng, few, many = 70, 32768 // nang, 32768 // nang + 1 + 300 // nang
    ke1, ke2 = np.zeros((Ng, Ng)), np.zeros((Ng, Ng))
    beg, end = np.zeros(Ng, np.int32), np.zeros(Ng, np.int32)
    for g in range(Ng - 1):
        beg[g], end[g] = g + 1, min(Ng, g + 25)
        ke1[g, beg[g]:end[g]] = rng.random(end[g] - beg[g])
        ke2[g, beg[g]:end[g]] = rng.standard_normal(end[g] - beg[g])
    kv = rng.random((Ng, nang, nang)) * (rng.random((Ng, nang, nang)) < 0.4)
    F, f = (rng.standard_normal((Ng, many, nang)).astype(np.float32) for _ in range(2))
    tabs = [gpu.DeviceArray(a) for a in (ke1, ke2, kv, beg, end)]

    def run(nodes):
        a, b = (np.ascontiguousarray(x[:, :nodes]) for x in (F, f))
        q = gpu.DeviceArray(np.full(a.shape, np.nan, np.float32))
        gpu.ops.secondary_source(gpu.DeviceArray(a), gpu.DeviceArray(b), q, *tabs, Ng, nodes, nang, 0.5)
        return q.numpy().reshape(a.shape)

    narrow, wide = run(few), run(many)
    np.testing.assert_array_equal(narrow, wide[:, :few])
    n = min(few, 40)  # and the oracle (the bound of one source in test_gpu_ops.py)
    want = oracle_mod.secondary_source_factorized(
        np.ascontiguousarray(F[:, :n]).astype(np.float64).reshape(-1),
        np.ascontiguousarray(f[:, :n]).astype(np.float64).reshape(-1), ke1, ke2, kv, beg, end, Ng, n,
        nang, 0.5).reshape(Ng, n, nang)
    assert np.abs(narrow[:, :n] - want).max() <= 1e-4 * np.abs(want).max()
