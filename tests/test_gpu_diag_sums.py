"""Final sums of the diagnostics over few and many block partials, against the oracle.

The C grid's number of partials follows the size (6 at N = 8, 1014 at N = 207, 1176 at N = 208, on either side
of the 1024 that the final block takes in one round); the Ah grid always has 1024, most of them empty
at N = 8.  The oracle adds the same terms serially: with 3e5 terms of one sign its rounding error stays
near sqrt(3e5) 1.1e-16 = 6e-14, so 1e-12 relative bounds the difference; extrema are equal.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)


@pytest.mark.parametrize("N", [8, 15, 16, 47, 191, 207, 208])
def test_c_grid(oracle_lib, N):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[diagnostics c N={N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names("c42"), scale=A, omega=OM, grav=G0)
    C = oracle_lib.CGrid(N, A, OM, G0)
    rng = np.random.default_rng(N)
    f = [C.embed(t, mean + amp * rng.standard_normal(C.interior(t, C.geometry(t, "r")[0]).shape))
         for t, (mean, amp) in zip("oxy", ((5.0e3, 50.0), (0.0, 20.0), (0.0, 20.0)))]
    x = swm.create_stvec_swm(op)
    x.upload(*f, C.hw)
    got, ref = op.get_diagnostics(x), C.diagnostics(*f, None)
    assert got["hmin"] == ref["hmin"] and got["hmax"] == ref["hmax"]
    for k in ("mass", "TE", "KE", "PE"):
        assert abs(got[k] - ref[k]) <= 1e-12 * abs(ref[k]), (k, got[k], ref[k])


@pytest.mark.parametrize("N", [8, 23, 106, 209])
def test_ah_grid(oracle_lib, N):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[diagnostics ah N={N}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names(42), scale=A, omega=OM, grav=G0)
    G = oracle_lib.Grid(N, 42, 42, A, OM, G0)
    f = [a.copy() for a in op.initial_state(5, 4, halo_width=G.hw)]
    x = swm.create_stvec_swm(op)
    x.upload(*f, G.hw)
    d = op.get_diagnostics(x)
    got = [d[k] for k in ("hmin", "hmax", "mass", "TE", "KE", "PE", "Enstrophy")]
    ref = G.diagnostics(42, *f)
    assert got[0] == ref[0] and got[1] == ref[1]
    for a, b in zip(got, ref):
        assert abs(a - b) <= 1e-12 * abs(b)
