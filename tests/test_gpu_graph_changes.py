"""Runs of RK4 steps whose graph was captured before something that it holds changed.

Two runs of 8 steps leave a graph of 8 steps behind (the first run of a state is launched step by step); a third
run replays it.  After a change of orography, time step, state, tile shape, launch grid or stream the next run must take
the new values and buffers, and so must the graph that the run after it captures.  Reference: another operator and
state taken through the same sequence by calls of one step, which never use a graph.  Same kernels in
the same order: the bound is equality.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)
RUNS = (8, 8, 8)


def _op(key, N, bits=64):
    import cubedsphere_sbp_swm_amd as swm
    return swm, swm.create_swm_operator(N, **swm.operator_names(key), scale=A, omega=OM, grav=G0,
                                        **({} if key == "c42" else {"precision": bits}))


def _state(swm, op, seed):
    x = swm.create_stvec_swm(op)
    rng = np.random.default_rng(seed)
    h, u, v = (a.shape for a in x.download())
    x.upload(1.0e4 + 5.0 * rng.standard_normal(h), 2.0 * rng.standard_normal(u), 2.0 * rng.standard_normal(v))
    return x


def _mountain(op, amp):
    f = np.zeros(op.host_shape())
    N = f.shape[1]
    f[2, N // 3: 2 * N // 3, N // 4: N // 2] = amp
    return f


def _equal(xs, ys, what):
    for x, y in zip(xs, ys):
        for name, a, b in zip("huv", x.download(), y.download()):
            assert np.all(np.isfinite(a)) and np.array_equal(a, b), (what, name)


# (change, argument): applied between groups of runs
ORO = [("oro", 900.0), ("oro", 300.0), ("oro", None), ("oro", 500.0)]
CHANGES = {"orography": ORO, "dt": [("dt", 500.0), ("dt", 900.0), ("dt", 250.0)], "state": [("state", 1), ("state", 0), ("state", 1)],
           "tile": [("tile", (16, 32)), ("tile", (8, 64)), ("oro", 400.0)], "stream": [("stream", True), ("oro", 700.0), ("stream", False)],
           "mixed": [("oro", 900.0), ("state", 1), ("dt", 450.0), ("oro", None), ("state", 0)]}


@pytest.mark.parametrize("key,N,bits", [(42, 20, 64), (63, 24, 64), (21, 16, 64), (42, 20, 32), ("c42", 12, 64)])
@pytest.mark.parametrize("change", CHANGES)
def test_one_grid(change, key, N, bits):
    import torch
    if key == "c42" and change in ("tile", "stream"):
        pytest.skip("no such setting on the C grid")
    print(f"[graph changes {change} {key} {bits}]", flush=True)
    side = torch.cuda.Stream()
    swm, op = _op(key, N, bits)
    _, ref = _op(key, N, bits)
    xs, ys = ([_state(swm, o, s) for s in (1, 2)] for o in (op, ref))
    ts, ts_ref = (swm.create_timescheme(o, "rk4") for o in (op, ref))
    dt, at = 900.0, 0
    for kind, arg in [("start", None)] + CHANGES[change]:
        if kind == "oro":
            for o in (op, ref):
                o.set_orography(None if arg is None else _mountain(o, arg))
        elif kind == "dt":
            dt = arg
        elif kind == "state":
            at = arg
        elif kind == "tile":
            op.set_tiling(tile_rows=arg[0], tile_cols=arg[1])
        elif kind == "stream":
            op.set_stream(side.cuda_stream if arg else None)
        for r in RUNS:
            ts.steps(xs[at], dt, r)
            for _ in range(r):
                ts_ref.steps(ys[at], dt, 1)
        op.synchronize()
        _equal(xs, ys, (kind, arg))

ENS = {"orography": ORO, "dt": CHANGES["dt"], "tile": [("tile", (8, 64)), ("oro", 400.0), ("tile", (16, 32))],
       "member": [("member", None), ("oro", 600.0), ("member", None)], "mixed": [("oro", 900.0), ("dt", 450.0), ("tile", (8, 32)), ("oro", None)]}


@pytest.mark.parametrize("order,bits", [(42, 64), (63, 64), (43, 32)])
@pytest.mark.parametrize("change", ENS)
def test_ensemble(change, order, bits):
    print(f"[graph changes ensemble {change} {order} {bits}]", flush=True)
    Ns = (18, 25, 33)
    swm = None
    ops, refs = [], []
    for N in Ns:
        for l in (ops, refs):
            swm, o = _op(order, N, bits)
            l.append(o)
    xs, ys = ([_state(swm, o, k) for k, o in enumerate(l)] for l in (ops, refs))
    ens = swm.Ensemble(ops, xs)
    one = [swm.create_timescheme(o, "rk4") for o in refs]
    own = [swm.create_timescheme(o, "rk4") for o in ops]
    dts = [600.0, 500.0, 400.0]
    for kind, arg in [("start", None)] + ENS[change]:
        if kind == "oro":     # of one member, or of all
            for l in (ops, refs):
                for o in l[1:2] if arg == 300.0 else l:
                    o.set_orography(None if arg is None else _mountain(o, arg))
        elif kind == "dt":
            dts = [arg / (k + 1) for k in range(len(Ns))]
        elif kind == "tile":
            ens.set_tiling(tile_rows=arg[0], tile_cols=arg[1], metric_on_the_fly=False, blocks_per_slot=0)
        elif kind == "member":   # a member steps by itself between the ensemble's runs, in its own work buffers
            for r in RUNS:
                own[1].steps(xs[1], 350.0, r)
                for _ in range(r):
                    one[1].steps(ys[1], 350.0, 1)
        for r in RUNS:
            ens.steps(dts, r)
            for ts, y, d in zip(one, ys, dts):
                for _ in range(r):
                    ts.steps(y, d, 1)
        ens.synchronize()
        _equal(xs, ys, (kind, arg))
