"""RK4 steps on both sides of the grid size from which their first stages write slopes only.

A step equals the one composed of right-hand sides and vector updates (rk4_mod.f90:28-40) bit for bit:
both forms take the same operations, whichever values go through memory.  The sizes lie on either
side of the line of each family and precision.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)


@pytest.mark.parametrize("order,bits,N", [(21, 64, 240), (21, 64, 258), (42, 64, 241), (42, 64, 256), (42, 64, 263),
                                          (43, 64, 257), (63, 64, 325), (63, 64, 341), (21, 32, 481), (42, 32, 460),
                                          (42, 32, 479), (63, 32, 487)])
@pytest.mark.parametrize("mountain", [False, True])
def test_step_equals_composition(order, bits, N, mountain):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[rk4 slopes order={order} bits={bits} N={N} mountain={mountain}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names(order), scale=A, omega=OM, grav=G0, precision=bits)
    rng = np.random.default_rng(N)
    shp = op.host_shape()
    if mountain:
        op.set_orography(300.0 * rng.random(shp))
    x = swm.create_stvec_swm(op)
    x.upload(1.0e4 + 50.0 * rng.standard_normal(shp), *(20.0 * rng.standard_normal(shp) for _ in range(2)))
    v0 = x.create_similar()
    v0.assign(1.0, x, 0.0, x)
    k1, k2, k3, k4, y = (x.create_similar() for _ in range(5))
    dt = 9000.0 / N
    op.apply(k1, v0)
    y.assign(1.0, v0, 0.5 * dt, k1)
    op.apply(k2, y)
    y.assign(1.0, v0, 0.5 * dt, k2)
    op.apply(k3, y)
    y.assign(1.0, v0, dt, k3)
    op.apply(k4, y)
    v0.update(dt / 6.0, k1, dt / 3.0, k2)
    v0.update(dt / 3.0, k3, dt / 6.0, k4)
    swm.create_timescheme(op, "rk4").step(x, dt)
    for a, b in zip(x.download(), v0.download()):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
