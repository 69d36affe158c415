"""Quotients at the ends of the number range: overflowing ones, subnormal denominators, tiny numerators.

A finite a / b beyond the range is an infinity, one with a subnormal a or b is rounded once, as IEEE
division gives it; a state that blows up then spreads infinities and NaN in the kernels as in the oracle.  The
unit sphere makes hx * scale small, so that gradients and divergences of values near the end of the range overflow
there.  FP64 values equal the oracle's bit for bit; the transposed tile kernel equals its two-launch form.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 40
# mean and amplitude of h, amplitude of u, v; and the points that get `h` instead (an inner one, one on a panel edge)
CASES = {"huge h": ((0.0, 1.0e307), 1.0e-3, None), "huge velocity": ((1.0, 0.1), 1.0e153, None),
         "subnormal h": ((1.0, 0.1), 1.0, 3.0e-310), "tiny velocity": ((1.0, 0.1), 1.0e-304, None),
         "tiny state": ((1.0e-303, 1.0e-304), 1.0e-5, None)}


def _values(case, rng, shapes):
    (mean, amp), vel, _ = CASES[case]
    return [m + a * rng.standard_normal(s) for (m, a), s in zip(((mean, amp), (0.0, vel), (0.0, vel)), shapes)]


def _put(case, inner):
    if CASES[case][2] is not None:
        inner[2, 20, 21] = CASES[case][2]
        inner[4, 0, 17] = CASES[case][2]


def _ah(oracle_lib, order, bits=64):
    import cubedsphere_sbp_swm_amd as swm
    return (swm, swm.create_swm_operator(N, **swm.operator_names(order), scale=1.0, omega=1.0, grav=1.0, precision=bits),
            oracle_lib.Grid(N, order, order if order != 21 else 2, 1.0, 1.0, 1.0))


def _same(got, want, name):
    assert np.array_equal(got, want, equal_nan=True), (name, int(np.sum(~((got == want) | (np.isnan(got) & np.isnan(want))))))


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("order", [42, 63])
def test_rhs(oracle_lib, order, case):
    print(f"[quotients rhs {order} {case}]", flush=True)
    swm, op, G = _ah(oracle_lib, order)
    f = _values(case, np.random.default_rng(order), [op.host_shape(G.hw)] * 3)
    _put(case, G.interior(f[0]))
    x = swm.create_stvec_swm(op)
    x.upload(*f, G.hw)
    k = x.create_similar()
    op.apply(k, x)
    with np.errstate(all="ignore"):
        ref = G.rhs(*(a.copy() for a in f))
    for name, a, b in zip("huv", k.download(G.hw), ref):
        _same(G.interior(a), G.interior(b), name)


@pytest.mark.parametrize("case", CASES)
def test_c_rhs(oracle_lib, case):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[quotients c {case}]", flush=True)
    op = swm.create_swm_operator(N, **swm.operator_names("c42"), scale=1.0, omega=1.0, grav=1.0)
    C = oracle_lib.CGrid(N, 1.0, 1.0, 1.0)
    shapes = [C.interior(t, C.geometry(t, "r")[0]).shape for t in "oxy"]
    f = _values(case, np.random.default_rng(3), shapes)
    _put(case, f[0])
    f = [C.embed(t, a) for t, a in zip("oxy", f)]
    x = swm.create_stvec_swm(op)
    x.upload(*f, C.hw)
    k = x.create_similar()
    op.apply(k, x)
    with np.errstate(all="ignore"):
        ref = C.rhs(*(a.copy() for a in f))
    for t, a, b in zip("oxy", k.download(C.hw), ref):
        _same(C.interior(t, a), C.interior(t, b), t)


@pytest.mark.parametrize("amp", [1.0e305, 1.0e-306])
@pytest.mark.parametrize("order", [21, 42, 63])
def test_laplace(oracle_lib, order, amp):
    print(f"[quotients laplace {order} {amp}]", flush=True)
    swm, op, G = _ah(oracle_lib, 42)
    f = [amp * np.random.default_rng(order).standard_normal(op.host_shape(G.hw)) for _ in range(3)]
    x, out = swm.create_stvec_swm(op), swm.create_stvec_swm(op)
    x.upload(*f, G.hw)
    op.laplace(out, x, f"laplace_ah_sbp{order}_narrow")
    with np.errstate(all="ignore"):
        ref = G.laplace(f[0], order)
    _same(G.interior(out.download(G.hw)[0]), G.interior(ref), "laplace")


@pytest.mark.parametrize("amp", [1.0e307, 1.0e-304])
@pytest.mark.parametrize("order", [42, 43, 63])
def test_vjp(oracle_lib, order, amp):
    print(f"[quotients vjp {order} {amp}]", flush=True)
    swm, op, _ = _ah(oracle_lib, order)
    rng = np.random.default_rng(order)
    y, mu, g = (swm.create_stvec_swm(op) for _ in range(3))
    y.upload(*(1.0 + 0.1 * rng.standard_normal(op.host_shape()) for _ in range(3)))
    # off the panel edges, where the fused kernel's gathers hold entries of weight zero
    seed = np.zeros((3,) + op.host_shape())
    seed[:, :, 12:-12, 12:-12] = amp * rng.standard_normal(seed[:, :, 12:-12, 12:-12].shape)
    mu.upload(*seed)
    out = {}
    for tile in (16, 32, 0):
        op.set_adjoint_tiling(tile)
        op.rhs_vjp(g, y, mu)
        out[tile] = g.download()
    for tile in (16, 32):
        for name, a, b in zip("huv", out[tile], out[0]):
            _same(a, b, name)


@pytest.mark.parametrize("order", [21, 42, 63])
def test_fp32_overflow(order):
    """h of about 2e37 on the unit sphere: off the panel edges, where a tendency of u, v is the quotient of a row's
    sum (at most a few 1e38, which FP32 holds), one beyond FP32 is an infinity of the FP64 value's sign.  The two sums
    differ by a few units in the last place of their terms, so values within 1 % of the range's end are left out."""
    import cubedsphere_sbp_swm_amd as swm
    print(f"[quotients fp32 {order}]", flush=True)
    big = float(np.finfo(np.float32).max)
    got = {}
    f = None
    for bits in (64, 32):
        op = swm.create_swm_operator(N, **swm.operator_names(order), scale=1.0, omega=1.0, grav=1.0, precision=bits)
        if f is None:
            rng = np.random.default_rng(order)
            f = [(a * rng.uniform(-1.0, 1.0, op.host_shape())).astype(np.float32).astype(np.float64)
                 for a in (2.0e37, 1e-3, 1e-3)]
        x = swm.create_stvec_swm(op)
        x.upload(*f)
        k = x.create_similar()
        op.apply(k, x)
        got[bits] = [a[:, 1:-1, 1:-1] for a in k.download()]
    some = 0
    for a, b in zip(got[32], got[64]):
        assert np.all(np.isfinite(b))
        over, under = np.abs(b) > 1.01 * big, np.abs(b) < 0.99 * big
        some += int(np.sum(over))
        assert np.array_equal(a[over], np.sign(b[over]) * np.inf) and np.all(np.isfinite(a[under]))
    assert some > 100


@pytest.mark.parametrize("order", [42, 63])
def test_fp32_subnormal_h(order):
    """A subnormal h: hv and its product with the Coriolis parameter hold a few bits, their quotient by h is of
    the size of the velocity.  h = 1e-39 is 7e5 and fz hv at least 1e4 units of the last subnormal bit (both at u, v = 1 and
    fz of order 1 and more), so three roundings leave 1e-3 of the terms."""
    import cubedsphere_sbp_swm_amd as swm
    print(f"[quotients fp32 subnormal h {order}]", flush=True)
    got = {}
    rng = np.random.default_rng(order)
    f = None
    for bits in (64, 32):
        op = swm.create_swm_operator(N, **swm.operator_names(order), scale=1.0, omega=1.0, grav=1.0, precision=bits)
        if f is None:
            f = [np.full(op.host_shape(), 1.0)] + [1.0 + 0.1 * rng.standard_normal(op.host_shape()) for _ in range(2)]
            f[0][2, 20, 21] = f[0][4, 0, 17] = 1.0e-39
            f = [a.astype(np.float32).astype(np.float64) for a in f]
        x = swm.create_stvec_swm(op)
        x.upload(*f)
        k = x.create_similar()
        op.apply(k, x)
        got[bits] = k.download()
    for a, b in zip(got[32], got[64]):
        assert np.all(np.isfinite(a)) and np.max(np.abs(a - b)) < 1e-3 * np.max(np.abs(b))
