"""sbp43 steps go by slopes from 64 MB of step data on, as sbp63's, whose halos are as wide; below, states are as fast or faster.

The sizes lie on either side of the line; on both a step equals the one composed of right-hand sides and vector
updates (rk4_mod.f90:28-40) bit for bit, as both forms take the same operations.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)


@pytest.mark.parametrize("bits,N,slopes", [(64, 256, False), (64, 329, False), (64, 330, True), (32, 463, False), (32, 471, True)])
def test_sbp43(bits, N, slopes):
    import bench
    import cubedsphere_sbp_swm_amd as swm
    print(f"[rk4 form 43 {bits} {N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names(43), scale=A, omega=OM, grav=G0, precision=bits)
    assert bench.by_slopes(op) is slopes
    rng = np.random.default_rng(N)
    shp = op.host_shape()
    x = swm.create_stvec_swm(op)
    x.upload(1.0e4 + 50.0 * rng.standard_normal(shp), *(20.0 * rng.standard_normal(shp) for _ in range(2)))
    k1, k2, k3, k4, y, v0 = (x.create_similar() for _ in range(6))
    v0.assign(1.0, x, 0.0, x)
    dt = 9000.0 / N
    op.apply(k1, v0)
    for k, nxt, c in ((k1, k2, 0.5), (k2, k3, 0.5), (k3, k4, 1.0)):
        y.assign(1.0, v0, c * dt, k)
        op.apply(nxt, y)
    v0.update(dt / 6.0, k1, dt / 3.0, k2)
    v0.update(dt / 3.0, k3, dt / 6.0, k4)
    swm.create_timescheme(op, "rk4").step(x, dt)
    for a, b in zip(x.download(), v0.download()):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
