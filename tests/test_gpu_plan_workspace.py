"""A prepared reduction of a small expression without a compiled kernel runs in
the block its caller gives: nothing outside the reported size is written, it
can be captured on a stream that never ran anything (an allocation would end
the capture), and captured launches stay valid when the stream's own workspace
is grown (and its old one freed) between replays."""

import ctypes as C

import numpy as np
import pytest

import xtensor_amd as xt
from xtensor_amd import _abi as A

pytestmark = pytest.mark.gpu

# float32 and float64 expressions, split and unsplit, by rows, columns and all
CASES = [((1029, 575), "float32", [1]), ((1029, 575), "float32", [0]), ((3, 20001), "float32", [1]),
         ((300, 41), "float64", None), ((7, 5), "float64", [0])]


def _make(shape, dtype, axes, seed=0):
    """(reducer, its output, the numpy operand, its sum of magnitudes and sum)."""
    h = np.random.default_rng(seed).normal(size=shape).astype(dtype)
    a = xt.from_numpy(h)
    r = xt.sum(a * a * 3 - a, axes)
    v = h * h * np.asarray(3, dtype) - h  # exact product order of the expression
    ax = None if axes is None else tuple(axes)
    return r, xt.empty(r.shape, r.dtype), v.astype(np.longdouble).sum(ax), np.abs(v).astype(np.longdouble).sum(ax)


def _check(out, want, mag, dtype):
    """Compensated sums: one rounding of the sum, relative to the magnitudes."""
    eps = np.finfo(dtype).eps
    assert np.all(np.abs(out.to_numpy().astype(np.longdouble) - want) <= eps * mag)


def _run(plan, block, stream):
    assert A.lib().xg_plan_execute(plan.handle, block, C.c_void_p(stream)) == A.OK


@pytest.mark.parametrize("shape,dtype,axes", CASES)
def test_in_the_callers_block(shape, dtype, axes):
    import torch
    r, out, want, mag = _make(shape, dtype, axes)
    p = xt.plan(out, r)
    need = A.lib().xg_plan_workspace_size(p.handle)
    assert need >= np.prod(shape) * np.dtype(dtype).itemsize
    guard = 4096
    block = torch.full((need + guard,), 0xA5, dtype=torch.uint8, device="cuda")
    _run(p, block.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert bool((block[need:] == 0xA5).all())
    _check(out, want, mag, dtype)
    got = out.to_numpy()
    assert xt.eval(r).to_numpy().tobytes() == got.tobytes()  # xg_reduce: the same kernels


@pytest.mark.parametrize("shape,dtype,axes", CASES)
@pytest.mark.parametrize("own_block", [True, False])
def test_captured(shape, dtype, axes, own_block):
    """Captured with and without a block; the stream's workspace grows between
    the replays, and the operand changes."""
    import torch
    r, out, want, mag = _make(shape, dtype, axes)
    p = xt.plan(out, r)
    need = A.lib().xg_plan_workspace_size(p.handle)
    block = torch.empty(need, dtype=torch.uint8, device="cuda") if own_block else None
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    if not own_block:
        p.run(stream=s.cuda_stream)  # one eager pass, as before any capture
    g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        _run(p, block.data_ptr() if own_block else None, s.cuda_stream)
    big = xt.from_numpy(np.random.default_rng(1).normal(size=(1 << 22,)).astype("float32"))
    for rep in range(3):
        xt.noalias(out).assign(out * 0)
        g.replay()
        torch.cuda.synchronize()
        _check(out, want, mag, dtype)
        with torch.cuda.stream(s):
            for k in (1, 2, 4):  # flattened scans of expressions: a temporary each, larger every time
                xt.cumsum(big[: (1 << 20) * k] * 2.0)
        torch.cuda.synchronize()


def test_plan_graph_and_many():
    import torch
    made = [_make(*c) for c in CASES]
    g = xt.PlanGraph([xt.plan(m[1], m[0]) for m in made])
    eager = [xt.empty(m[1].shape, m[1].dtype) for m in made]
    plans = [xt.plan(o, m[0]) for o, m in zip(eager, made)]
    for rep in range(3):
        for m, o in zip(made, eager):
            xt.noalias(m[1]).assign(m[1] * 0)
            xt.noalias(o).assign(o * 0)
        g.replay()
        xt.execute_many(plans)
        torch.cuda.synchronize()
        for m, o, c in zip(made, eager, CASES):
            _check(m[1], m[2], m[3], c[1])
            assert m[1].to_numpy().tobytes() == o.to_numpy().tobytes()
        with torch.cuda.stream(g._stream):
            xt.cumsum(xt.zeros(((1 << 21) + (1 << 20) * rep,), "float32") + 1.0)
        torch.cuda.synchronize()


@pytest.mark.parametrize("shape,dtype,axes", CASES)
def test_eager_call_captured(shape, dtype, axes):
    """A captured xg_reduce that is not split keeps no address of the stream's
    workspace: its replays are right after the workspace has grown.  (A split
    one keeps its partials there, so it is replayed without growing it.)"""
    import torch
    r, out, want, mag = _make(shape, dtype, axes)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        xt.noalias(out).assign(r)  # one eager pass
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        xt.noalias(out).assign(r)
    for rep in range(3):
        xt.noalias(out).assign(out * 0)
        g.replay()
        torch.cuda.synchronize()
        _check(out, want, mag, dtype)
        if shape == (1029, 575) and axes == [1]:  # 1029 outputs: no split
            with torch.cuda.stream(s):
                xt.cumsum(xt.zeros(((1 << 20) * (rep + 1),), "float32") + 1.0)
            torch.cuda.synchronize()


def test_captured_variance_matches_eager():
    """Its mean is in the stream's workspace anyway; captured after an eager
    pass it runs the same kernels."""
    import torch
    rng = np.random.default_rng(3)
    a = xt.from_numpy(rng.normal(size=(200, 300)).astype("float32"))
    r = xt.variance(a * a + a, [1])
    out = xt.empty(r.shape, r.dtype)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        want = xt.eval(r).to_numpy()
        g = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(g, stream=s):
        xt.noalias(out).assign(r)
    for _ in range(3):
        xt.noalias(out).assign(out * 0)
        g.replay()
        torch.cuda.synchronize()
        assert out.to_numpy().tobytes() == want.tobytes()


@pytest.mark.parametrize("n,first", [((1 << 21) - 3, True), ((1 << 21) + 1, False)])
def test_bound_without_the_compiler(n, first):
    """With the run-time compiler off the temporary's 8 MiB are the bound, not
    the compiler's threshold of 2^20 elements."""
    L = A.lib()
    L.xg_debug_jit(0)
    try:
        h = np.random.default_rng(4).normal(size=n).astype("float32")
        a = xt.from_numpy(h)
        r = xt.sum(a * a * 3 - a)
        out = xt.empty(r.shape, r.dtype)
        p = xt.plan(out, r)
        assert (L.xg_plan_workspace_size(p.handle) >= 4 * n) == first
        p.run()
        v = h * h * np.float32(3) - h
        _check(out, v.astype(np.longdouble).sum(), np.abs(v).astype(np.longdouble).sum(), "float32")
    finally:
        L.xg_debug_jit(1)
