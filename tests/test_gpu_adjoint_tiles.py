"""Transposed right-hand side at panel sizes around multiples of its 16 x 16 tiles.

The fused kernel takes closure columns from a table, panel-edge points one wave per edge and, from three
tiles a side on, tiles of interior columns only; the two-launch form has every column written out.  Both
evaluate the same terms in the same order, so they agree bit for bit; the last tile of a line is 1 to 16
points wide over the sizes.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)


@pytest.mark.parametrize("order,N", [(42, 14), (42, 15), (42, 16), (42, 20), (42, 31), (42, 32), (42, 37), (42, 47),
                                     (42, 48), (42, 63), (43, 14), (43, 16), (43, 32), (43, 53), (63, 22), (63, 24),
                                     (63, 31), (63, 32), (63, 40), (63, 47), (63, 64)])
def test_vjp_fused_equals_two_launches(order, N):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[adjoint tiles order={order} N={N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names(order), scale=A, omega=OM, grav=G0)
    rng = np.random.default_rng(N)
    shp = op.host_shape()
    y, mu, g = (swm.create_stvec_swm(op) for _ in range(3))
    y.upload(1.0e4 + 50.0 * rng.standard_normal(shp), *(20.0 * rng.standard_normal(shp) for _ in range(2)))
    mu.upload(*(rng.standard_normal(shp) for _ in range(3)))
    out = {}
    for tile in (16, 0):
        op.set_adjoint_tiling(tile)
        op.rhs_vjp(g, y, mu)
        out[tile] = g.download()
    for a, b in zip(out[16], out[0]):
        assert np.all(np.isfinite(a)) and np.array_equal(a, b)
