"""Tile orders of the kernels at the sizes where the closure tiles are first dealt apart from the inner ones.

Below a number of tiles all go in one band order; above, the ring of tiles with closure rows goes first.  The
sizes lie on either side of that number for each kernel, with last tiles 1 to 16 points wide, and each
point is checked: against the oracle bit for bit, or for the adjoint against its two-launch form.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)


def _noise(rng, shp):
    return [1.0e4 + 50.0 * rng.standard_normal(shp)] + [20.0 * rng.standard_normal(shp) for _ in range(2)]


@pytest.mark.parametrize("N", [103, 104, 105, 111, 112, 113, 128, 137])
def test_c_grid(oracle_lib, N):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[tile order c N={N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names("c42"), scale=A, omega=OM, grav=G0)
    C = oracle_lib.CGrid(N, A, OM, G0)
    rng = np.random.default_rng(N)
    f = [C.embed(t, mean + amp * rng.standard_normal(C.interior(t, C.geometry(t, "r")[0]).shape))
         for t, (mean, amp) in zip("oxy", ((5.0e3, 50.0), (0.0, 20.0), (0.0, 20.0)))]
    x = swm.create_stvec_swm(op)
    x.upload(*f, C.hw)
    k = x.create_similar()
    op.apply(k, x)
    for t, a, b in zip("oxy", k.download(C.hw), C.rhs(*(a.copy() for a in f))):
        assert np.array_equal(C.interior(t, a), C.interior(t, b)), t


@pytest.mark.parametrize("order,N", [(21, 176), (21, 191), (42, 175), (42, 176), (42, 191), (42, 192), (63, 176), (63, 207)])
def test_laplace(oracle_lib, order, N):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[tile order laplace order={order} N={N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names(42), scale=A, omega=OM, grav=G0)
    G = oracle_lib.Grid(N, grad_order=42, div_kind=42, scale=A, omega=OM, grav=G0)
    x, out = swm.create_stvec_swm(op), swm.create_stvec_swm(op)
    f = _noise(np.random.default_rng(N), op.host_shape(G.hw))
    x.upload(*f, G.hw)
    op.laplace(out, x, f"laplace_ah_sbp{order}_narrow")
    a, b = G.interior(out.download(G.hw)[0]), G.interior(G.laplace(f[0], order))
    assert np.all(np.isfinite(a)) and np.array_equal(a, b)


@pytest.mark.parametrize("order,N", [(42, 207), (42, 208), (42, 223), (43, 209), (63, 208), (63, 225)])
def test_vjp(order, N):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[tile order vjp order={order} N={N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names(order), scale=A, omega=OM, grav=G0)
    rng = np.random.default_rng(N)
    y, mu, g = (swm.create_stvec_swm(op) for _ in range(3))
    y.upload(*_noise(rng, op.host_shape()))
    mu.upload(*(rng.standard_normal(op.host_shape()) for _ in range(3)))
    out = {}
    for tile in (32, 16, 0):
        op.set_adjoint_tiling(tile)
        op.rhs_vjp(g, y, mu)
        out[tile] = g.download()
    for tile in (32, 16):
        for a, b in zip(out[tile], out[0]):
            assert np.all(np.isfinite(a)) and np.array_equal(a, b)
