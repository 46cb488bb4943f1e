"""Operators called from several host threads, each with its own workspace, at
sizes that take one kernel with very different amounts of LDS."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _angle(gpu, n, nyz=40, Ng=3):
    rng = np.random.default_rng(n)
    F, sig, ws = rng.standard_normal(Ng * nyz * n * n), rng.uniform(0.0, 4.0, Ng), gpu.Workspace()

    def call():
        d = gpu.DeviceArray(F)
        gpu.ops.angle_full(d, sig, nyz, Ng, n, n, 0.2, 0.13, 0.05, 1.2, ws=ws)
        return d.numpy()
    return call


def _transport(gpu, Ny, Nz=3, Ng=3, nang=9):
    rng = np.random.default_rng(Ny)
    F, om = rng.standard_normal(Ng * (Ny + 1) * (Nz + 1) * nang), rng.uniform(-0.9, 0.9, 2 * nang)
    ws, d_om = gpu.Workspace(), gpu.DeviceArray(om)

    def call():
        d = gpu.DeviceArray(F)
        gpu.ops.transport_half(d, d_om, Ny, Nz, Ng, nang, 0.2, 0.3, 0.05, True, ws=ws)
        return d.numpy()
    return call


@pytest.mark.parametrize("make,sizes", [(_angle, (1, 5, 8, 21, 32)), (_transport, (100, 130, 169))])
def test_sizes_that_share_a_kernel(gpu, make, sizes):
    calls = [make(gpu, n) for n in sizes]
    alone = [c() for c in calls]
    bad, start = [], threading.Barrier(len(calls))

    def work(call, want):
        start.wait(timeout=30)
        try:
            for _ in range(30):
                if not np.array_equal(call(), want):
                    bad.append("other result")
        except Exception as e:  # reported by the main thread
            bad.append(repr(e))

    threads = [threading.Thread(target=work, args=a) for a in zip(calls, alone)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not bad and not any(t.is_alive() for t in threads)
