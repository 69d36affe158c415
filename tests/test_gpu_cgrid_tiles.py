"""C-grid right-hand side at panel sizes around multiples of the 16 x 8 tiles, against the oracle.

The last tile of a line holds 1 to 16 (8) cells and the face N+1; its closure rows reach back over a
narrow tile, and from N = 20 on a panel has tiles of interior rows only.  Random values at every point, so
that no interface penalty vanishes.  Same operations in the same order as the oracle: the bound is
equality.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)


@pytest.mark.parametrize("N", [8, 9, 10, 12, 15, 16, 17, 18, 20, 23, 24, 25, 27, 28, 31, 33, 36, 37, 44, 49, 63])
def test_c_rhs_around_tile_edges(oracle_lib, N):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[c tiles N={N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names("c42"), scale=A, omega=OM, grav=G0)
    C = oracle_lib.CGrid(N, A, OM, G0)
    rng = np.random.default_rng(N)
    f = []
    for t, (mean, amp) in zip("oxy", ((5.0e3, 50.0), (0.0, 20.0), (0.0, 20.0))):
        z = C.embed(t, mean + amp * rng.standard_normal(C.interior(t, C.geometry(t, "r")[0]).shape))
        f.append(z)
    hs = C.embed("o", 300.0 * rng.standard_normal(C.interior("o", f[0]).shape)) if N % 2 else None
    op.set_orography(hs, C.hw)
    x = swm.create_stvec_swm(op)
    x.upload(*f, C.hw)
    k = x.create_similar()
    op.apply(k, x)
    ref = C.rhs(*(a.copy() for a in f), hs)
    for t, a, b in zip("oxy", k.download(C.hw), ref):
        assert np.array_equal(C.interior(t, a), C.interior(t, b)), t
