"""Rows that do not start on a vector boundary: odd pitches, inner views and
offsets are read and written with wide accesses at element addresses
(compiled programs), and nothing outside the view changes."""

import numpy as np
import pytest

import xtensor_amd as xt
from xtensor_amd import _abi as A

from helpers import Dual, oracle_for, same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _compiled():
    """Run-time compile every program, however small the launch."""
    A.lib().xg_debug_jit(2)
    yield
    A.lib().xg_debug_jit(1)


# (rows, pitch, first column, columns): rows shorter than a vector, whole
# vectors off a boundary, remainders, an even pitch with an odd offset
VIEWS = [(3, 7, 1, 2), (5, 33, 1, 32), (4, 515, 3, 511), (6, 512, 1, 509), (2, 4099, 2, 4095)]


@pytest.mark.parametrize("dtype", ["int8", "int16", "float32", "float64"])
@pytest.mark.parametrize("rows,pitch,c0,cols", VIEWS)
def test_assign_inner_view(dtype, rows, pitch, c0, cols):
    rng = np.random.default_rng(rows * pitch + c0)
    draw = (lambda: rng.integers(-100, 100, (rows, pitch)).astype(dtype)) if dtype.startswith("int") else \
        (lambda: rng.normal(size=(rows, pitch)).astype(dtype))
    x, y, o = Dual.of(draw()), Dual.of(draw()), Dual.of(draw())
    cut = (slice(None), slice(c0, c0 + cols))
    xv, yv, ov = x.view(*cut), y.view(*cut), o.view(*cut)
    xt.noalias(ov.dev).assign(xv.dev + yv.dev)
    want = o.host.copy()
    want[cut] = xv.host + yv.host
    assert same_bits(o.dev.to_numpy(), want)


def test_shifted_views_of_one_array():
    """A stencil: overlapping leaves share cache lines and workgroups are
    numbered per XCD (more than 8 of them, no multiple of 8)."""
    u = np.random.default_rng(1).normal(size=(301, 2051))
    d, o = xt.from_numpy(u), xt.from_numpy(np.zeros_like(u))
    e = d[:-2, 1:-1] + d[2:, 1:-1] + d[1:-1, :-2] + d[1:-1, 2:] - d[1:-1, 1:-1]
    xt.noalias(o[1:-1, 1:-1]).assign(e)
    want = np.zeros_like(u)
    want[1:-1, 1:-1] = u[:-2, 1:-1] + u[2:, 1:-1] + u[1:-1, :-2] + u[1:-1, 2:] - u[1:-1, 1:-1]
    assert same_bits(o.to_numpy(), want)


@pytest.mark.parametrize("dtype,tol", [("bfloat16", 1e-7), ("float32", 1e-7), ("float64", 1e-15), ("int32", 0)])
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("rows,pitch,c0,cols", VIEWS)
def test_reduce_inner_view(dtype, tol, axis, rows, pitch, c0, cols):
    """Compensated float sums are within one rounding of the long-double sum
    relative to the sum of magnitudes; integer sums exact."""
    rng = np.random.default_rng(rows + pitch)
    h = rng.integers(-1000, 1000, (rows, pitch)).astype("int32") if dtype == "int32" else \
        rng.normal(size=(rows, pitch)).astype("float32" if dtype == "bfloat16" else dtype)
    v = Dual.of(h, dtype if dtype == "bfloat16" else None).view(slice(None), slice(c0, c0 + cols))
    r = xt.sum(v.dev, [axis])
    got = xt.eval(r).to_numpy()
    o = oracle_for(v)
    if not tol:
        assert same_bits(got, o.reduce(r))
        return
    ref = o.reduce(r, high_precision=True)
    mag = o.reduce(xt.sum(xt.abs(v.dev), [axis]), high_precision=True)
    assert np.all(np.abs(got.astype(np.float64) - ref) <= tol * mag)
    m = xt.amax(v.dev, [axis])
    assert same_bits(xt.eval(m).to_numpy(), o.reduce(m))


@pytest.mark.parametrize("dtype", ["bfloat16", "float32", "float64", "int32"])
@pytest.mark.parametrize("shape,axes", [((3, 5, 7, 7), [0, 2, 3]), ((9, 2, 1, 3), [0, 2, 3]), ((33, 1, 5, 13), [0, 2, 3]),
                                        ((130, 300, 2, 9), [0, 2, 3]), ((1, 700, 3, 3), [0, 2, 3]), ((5, 1001), [0]),
                                        ((2000, 131), [0]), ((1100, 520), [0]), ((70, 3), [0, 1])])
def test_channel_and_ragged_reductions(dtype, shape, axes):
    """Rows of [outputs | reduced | fast], columns whose last chunk is shifted,
    one output, rows shorter than a vector: sums within one rounding relative
    to the sum of magnitudes (as above), maxima and infinities exact."""
    rng = np.random.default_rng(sum(shape))
    h = rng.integers(-1000, 1000, shape).astype("int32") if dtype == "int32" else \
        rng.normal(size=shape).astype("float32" if dtype == "bfloat16" else dtype)
    d = Dual.of(h, dtype if dtype == "bfloat16" else None)
    o = oracle_for(d)
    r = xt.sum(d.dev, axes)
    got = xt.eval(r).to_numpy()
    if dtype == "int32":
        assert same_bits(got, o.reduce(r))
    else:
        mag = o.reduce(xt.sum(xt.abs(d.dev), axes), high_precision=True)
        tol = 1e-15 if dtype == "float64" else 1e-7
        assert np.all(np.abs(got.astype(np.float64) - o.reduce(r, high_precision=True)) <= tol * mag)
    for m in (xt.amax(d.dev, axes), xt.amin(d.dev, axes)):
        assert same_bits(xt.eval(m).to_numpy(), o.reduce(m))
    if dtype in ("float32", "float64"):
        h2 = np.full(shape, -np.inf, dtype)  # folds to lowest(), but where the infinity is
        h2.reshape(-1)[-1] = np.inf
        d2 = Dual.of(h2)
        m = xt.amax(d2.dev, axes)
        assert same_bits(xt.eval(m).to_numpy(), oracle_for(d2).reduce(m))
