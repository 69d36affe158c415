"""Runs of RK4 steps by plain launches, by graphs and by both.

A state's first run is launched step by step (a long one from its second step on by graphs); later runs take graphs of
4, 8, ... 64 steps and launch the rest.  Single-step calls never use a graph.  The same kernels run in the
same order, so a state stepped in runs equals one stepped by single calls bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

A, G0 = 0.6371229e7, 9.80616
OM = 2.0 * np.pi / (23 * 60 * 60 + 56 * 60 + 4)


def _c_state(swm, op):
    rng = np.random.default_rng(4)
    h, u, v = (a.shape for a in swm.create_stvec_swm(op).download())
    return 1.0e4 + 5.0 * rng.standard_normal(h), 2.0 * rng.standard_normal(u), 2.0 * rng.standard_normal(v)


@pytest.mark.parametrize("runs", [(1, 3, 4), (5, 7, 8, 8), (127, 2), (128, 4), (129, 64, 5), (2, 131), (4, 0, 60, 63)])
@pytest.mark.parametrize("kind", ["42", "c42", "ensemble"])
def test_runs_equal_single_steps(kind, runs):
    import cubedsphere_sbp_swm_amd as swm
    print(f"[step runs {kind} {runs}]", flush=True)
    Ns = (16, 21) if kind == "ensemble" else (12,)
    key = "c42" if kind == "c42" else 42
    ops = [swm.create_swm_operator(N, **swm.operator_names(key), scale=A, omega=OM, grav=G0) for N in Ns]
    dts = [900.0 / (k + 1) for k in range(len(Ns))]
    ics = [op.initial_state(3, 4) if kind != "c42" else _c_state(swm, op) for op in ops]
    xs, ys = ([swm.create_stvec_swm(op) for op in ops] for _ in range(2))
    for x, y, ic in zip(xs, ys, ics):
        x.upload(*ic)
        y.upload(*ic)
    ones = [swm.create_timescheme(op, "rk4") for op in ops]
    for op, y, dt, ts in zip(ops, ys, dts, ones):
        for _ in range(sum(runs)):
            ts.steps(y, dt, 1)
    if kind == "ensemble":
        ens = swm.Ensemble(ops, xs)
        for r in runs:
            ens.steps(dts, r)
    else:
        for r in runs:
            ones[0].steps(xs[0], dts[0], r)
    for x, y in zip(xs, ys):
        for a, b in zip(x.download(), y.download()):
            assert np.all(np.isfinite(a)) and np.array_equal(a, b)


def test_capture_is_refused():
    import torch
    import cubedsphere_sbp_swm_amd as swm
    print("[step runs under capture]", flush=True)
    op = swm.create_swm_operator(12, **swm.operator_names(42), scale=A, omega=OM, grav=G0)
    x = swm.create_stvec_swm(op)
    x.upload(*op.initial_state(3, 4))
    before = x.download()
    ts = swm.create_timescheme(op, "rk4")
    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    buf = torch.zeros(8, device="cuda")
    op.set_stream(s.cuda_stream)
    with torch.cuda.graph(graph, stream=s):
        with pytest.raises(swm.SwmError):
            ts.steps(x, 900.0, 3)
        buf.add_(1.0)
    op.set_stream(None)
    torch.cuda.synchronize()
    assert all(np.array_equal(a, b) for a, b in zip(before, x.download()))
