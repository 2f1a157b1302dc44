"""The generic interpreter: programs of 32-bit types (four elements a lane)
and with 64-bit ones (two), made of light ops only or with called ones, over
row lengths around a lane's elements, strides, views, ranks and leaf counts,
against the oracle."""

import numpy as np
import pytest

import xtensor_amd as xt
from xtensor_amd import _abi as A

from helpers import Dual, oracle_for, same_bits

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _interpreter():
    A.lib().xg_debug_force_dynamic(1)
    yield
    A.lib().xg_debug_force_dynamic(0)


def draw(rng, shape, dtype):
    if dtype == "bool":
        return rng.integers(0, 2, shape).astype(bool)
    if dtype in ("float32", "float64", "bfloat16"):
        return rng.normal(size=shape).astype("float32" if dtype == "bfloat16" else dtype)
    return rng.integers(1, 100, shape).astype(dtype)


def check(e, duals, out_dtype=None):
    shape = e.shape
    o = xt.empty(shape, out_dtype or e.dtype)
    xt.noalias(o).assign(e)
    assert xt.last_kernel() == "dynamic"
    assert same_bits(o.to_numpy(), oracle_for(*duals).assign(e, dtype=out_dtype))


@pytest.mark.parametrize("cols", [1, 2, 3, 4, 5, 7, 8, 257, 1029])
@pytest.mark.parametrize("dtype", ["int8", "uint8", "int16", "bfloat16", "float32", "int32", "float64", "int64"])
def test_light_ops_row_lengths(dtype, cols):
    rng = np.random.default_rng(cols)
    x, r, c = (Dual.of(draw(rng, s, dtype), dtype if dtype == "bfloat16" else None) for s in ((5, cols), (5, 1), (cols,)))
    check(xt.where(x.dev > r.dev, x.dev * r.dev - c.dev, c.dev + x.dev), (x, r, c))


@pytest.mark.parametrize("dtype", ["uint32", "float32", "float64", "uint64", "uint16"])
def test_called_ops(dtype):
    rng = np.random.default_rng(3)
    x, y = Dual.of(draw(rng, (3, 131), dtype)), Dual.of(draw(rng, (3, 131), dtype))
    if dtype.startswith("float"):
        check(xt.fmod(x.dev, y.dev) + xt.maximum(x.dev, y.dev) * 2.0, (x, y))
    else:
        check((x.dev % y.dev) + x.dev / y.dev, (x, y))


def test_leaf_counts_ranks_and_strides():
    rng = np.random.default_rng(4)
    many = [Dual.of(rng.normal(size=(7, 37)).astype(np.float32)) for _ in range(11)]
    e = many[0].dev
    for d in many[1:]:
        e = e + d.dev
    check(e, many)  # more leaves than are read ahead
    big = Dual.of(rng.normal(size=(3, 2, 3, 2, 5, 4, 9)))
    v = big.view(slice(None, None, 2), slice(None), slice(None, None, -1), slice(None), slice(None, None, 2), slice(None),
                 slice(None, None, 3))
    check(v.dev * 2.0, (v,))  # rank beyond the compact form
    t = Dual.of(rng.integers(-9, 9, (33, 18)).astype(np.int16)).transpose()
    check(t.dev * 3 - 1, (t,))


def test_gather_and_mixed_conversions():
    rng = np.random.default_rng(5)
    x = Dual.of(rng.normal(size=(300,)).astype(np.float32))
    i = Dual.of(rng.integers(0, 300, 77))
    g = xt.index_view(x.dev, i.dev)
    assert same_bits(xt.eval(g * 2.0).to_numpy(), x.host[i.host].astype(np.float64) * 2.0)
    b = Dual.of(draw(rng, (300,), "bool"))
    check(xt.cast(b.dev, "int64") + xt.cast(x.dev, "int32") * 2, (b, x))
    check(x.dev * 1.5, (x,), "int8")


# either side of the lines between one element a lane and several, for programs
# that call functions: 2^18 elements, and 2^19 for 32-bit ones of mostly calls
@pytest.mark.parametrize("n", [1, 63, 1000, (1 << 18) - 1, 1 << 18, (1 << 19) - 1, (1 << 19) + 1])
@pytest.mark.parametrize("dtype", ["int8", "uint16", "int32", "int64"])
def test_called_ops_by_size(n, dtype):
    """Integer divisions and remainders (called), bit for bit; a contiguous
    output, one inside a larger array, and operands that are views."""
    rng = np.random.default_rng(n)
    a, b = (Dual.of(rng.integers(1, 100, n + 3).astype(dtype)) for _ in range(2))
    av, bv = a.view(slice(1, n + 1)), b.view(slice(2, n + 2))
    e = (av.dev / bv.dev) + (av.dev % bv.dev) * (bv.dev % av.dev)
    want = oracle_for(av, bv).assign(e)
    assert same_bits(xt.eval(e).to_numpy(), want)
    whole = xt.from_numpy(np.full(n + 2, 7, want.dtype))
    xt.noalias(whole[1:-1]).assign(e)
    got = whole.to_numpy()
    assert same_bits(got[1:-1], want) and got[0] == 7 and got[-1] == 7


@pytest.mark.parametrize("n", [1, 1000, (1 << 18) - 1, (1 << 19) - 1, (1 << 19) + 1])
def test_gather_and_many_leaves_by_size(n):
    rng = np.random.default_rng(n)
    x = Dual.of(rng.normal(size=500).astype(np.float32))
    i = Dual.of(rng.integers(0, 500, n).astype(np.int64))
    g = xt.index_view(x.dev, i.dev)
    assert same_bits(xt.eval(g * np.float32(2)).to_numpy(), x.host[i.host] * np.float32(2))
    ls = [Dual.of(rng.normal(size=n).astype(np.float32)) for _ in range(9)]
    e, want = ls[0].dev, ls[0].host
    for l in ls[1:]:
        e, want = e + l.dev, want + l.host
    assert same_bits(xt.eval(e).to_numpy(), want)
