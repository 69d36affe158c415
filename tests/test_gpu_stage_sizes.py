"""Stage kernel at the sizes where its tiles and edge segments change shape, against the oracle.

An edge segment holds 64 - 2 REACH points (58 for sbp42, 54 for sbp43 and sbp63); tiles whose rows are
all interior start at NE points from the panel edge and leave NE points beyond their end.  The sizes
sit on both sides of one and two segments and of the first and last size with such a tile, and at the
smallest panels.  Every value takes the reference's operations in the reference's order, so the bound is
equality.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)
QUAD = {42: 42, 43: 63, 63: 63}


@pytest.mark.parametrize("tile", [(64, 8), (32, 8), (16, 32)])
@pytest.mark.parametrize("order,N", [(42, 8), (42, 39), (42, 40), (42, 57), (42, 58), (42, 59), (42, 115), (42, 116),
                                     (43, 8), (43, 53), (43, 54), (43, 107), (43, 108),
                                     (63, 8), (63, 43), (63, 44), (63, 53), (63, 54), (63, 55), (63, 108)])
def test_rhs_at_segment_and_tile_edges(oracle_lib, order, N, tile):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[stage sizes order={order} N={N} tile={tile}]", flush=True)
    if N + 1 <= tile[1]:
        pytest.skip("tile taller than the panel")
    op = swm.create_swm_operator(N, **swm.operator_names(order), scale=A, omega=OM, grav=G0)
    op.set_tiling(tile_rows=tile[1], tile_cols=tile[0])
    G = oracle_lib.Grid(N, order, order, A, OM, G0)
    rng = np.random.default_rng(N)
    f = [G.zeros() for _ in range(3)]
    for a, (mean, amp) in zip(f, ((1.0e4, 50.0), (0.0, 20.0), (0.0, 20.0))):
        G.interior(a)[:] = mean + amp * rng.standard_normal(G.interior(a).shape)
    x = swm.create_stvec_swm(op)
    x.upload(*f, G.hw)
    k = x.create_similar()
    op.apply(k, x)
    got = k.download(G.hw)
    ref = G.rhs(*(a.copy() for a in f))
    for name, a, b in zip("huv", got, ref):
        assert np.array_equal(G.interior(a), G.interior(b)), name


@pytest.mark.parametrize("value", [0.0, float("inf"), float("nan")])
@pytest.mark.parametrize("field", [0, 1, 2])
def test_special_values_spread_as_in_division(oracle_lib, field, value):
    """A zero, an infinity or a NaN at an inner point and at an edge point gives the same finite values,
    infinities and NaN as the oracle's plain divisions (the kernel divides by shared reciprocals)."""
    import cubedsphere_sbp_swm_amd as swm
    N = 48
    op = swm.create_swm_operator(N, **swm.operator_names(42), scale=A, omega=OM, grav=G0)
    G = oracle_lib.Grid(N, 42, 42, A, OM, G0)
    rng = np.random.default_rng(7)
    f = [G.zeros() for _ in range(3)]
    for a, (mean, amp) in zip(f, ((1.0e4, 50.0), (0.0, 20.0), (0.0, 20.0))):
        G.interior(a)[:] = mean + amp * rng.standard_normal(G.interior(a).shape)
    G.interior(f[field])[2, 20, 21] = value
    G.interior(f[field])[4, 0, 17] = value
    x = swm.create_stvec_swm(op)
    x.upload(*f, G.hw)
    k = x.create_similar()
    op.apply(k, x)
    got = k.download(G.hw)
    with np.errstate(all="ignore"):
        ref = G.rhs(*(a.copy() for a in f))
    for name, a, b in zip("huv", got, ref):
        assert np.array_equal(G.interior(a), G.interior(b), equal_nan=True), name
