"""The compiled tree walker lays out the same descriptor as core.serialize(),
and refuses what it refuses."""

import ctypes as C

import numpy as np
import pytest

import xtensor_amd as xt
from xtensor_amd import _abi as A
from xtensor_amd import core

from test_abi_frontend import random_expr


def raw(e):
    return core._pack(e, core._placeholder_for).raw()


def serialized(e):
    s = core.serialize(e, reducer_fn=core._placeholder_for)
    n = s.expr
    return tuple(bytes(C.string_at(p, k * C.sizeof(t))) for p, k, t in
                 ((n.nodes, n.n_nodes, A.Node), (n.leaves, n.n_leaves, A.Tensor), (n.consts, n.n_consts, A.Scalar)))


@pytest.mark.parametrize("seed", range(20))
def test_same_descriptor(seed):
    rng = np.random.default_rng(seed)
    for _ in range(20):
        e = random_expr(rng, 4, [])
        assert raw(e) == serialized(e)


def test_shared_nodes_views_gathers_reducers_and_constants():
    a = core._Placeholder(A.FLOAT64, (6, 5))
    v = core.view(a, slice(4, 0, -2), xt.newaxis(), 3)
    t = a * a
    e = xt.where(t > t, xt.scalar(2**64 - 1, "uint64"), xt.scalar(-7, "int64")) + v * -1.5 + xt.sum(a, [0]) + True
    assert raw(e) == serialized(e)
    i = core.IndexView.__new__(core.IndexView)
    i.source, i.offsets = a, core._Placeholder(A.INT64, (3,)) * xt.scalar(5, "int64")
    assert raw(i + 1) == serialized(i + 1)


def test_refusals():
    a = core._Placeholder(A.FLOAT32, (4,))
    e = a
    for _ in range(A.MAX_NODES):
        e = e + a
    with pytest.raises(NotImplementedError, match="too many nodes"):
        raw(e)
    for _ in range(100000):
        e = -e
    with pytest.raises(RecursionError):
        raw(e)
    with pytest.raises(TypeError, match="not an expression"):
        core._pack(3, None)
    with pytest.raises(RuntimeError, match="evaluation context"):
        core._pack(xt.sum(a) + 1, None)
    with pytest.raises(IndexError):
        raw(core._Placeholder(A.FLOAT32, (1,) * 9))
    with pytest.raises(RuntimeError, match="too many axes"):
        core._pack(a, None).reduce_info(xt.sum(a, list(range(9))))
    host = xt.empty((4,), "float32", device="cpu")
    with pytest.raises(RuntimeError, match="device"):
        core._pack(host + a, None).assign(host, 0)


def test_nodes_are_ordinary_objects():
    """Expression nodes take weak references, attributes, copies and every
    pickle protocol, as any instance does."""
    import copy
    import pickle
    import weakref
    a = core._Placeholder(A.FLOAT32, (4,))
    s = xt.scalar(3, "int64")
    for e in (a + s, -(a * a), s):
        assert weakref.ref(e)() is e
        e.note = "kept"
        assert vars(e)["note"] == "kept" and copy.copy(e).note == "kept"
    for protocol in range(pickle.HIGHEST_PROTOCOL + 1):
        e = pickle.loads(pickle.dumps(s + 2, protocol))
        assert raw(e) == raw(s + 2)


def test_host_arrays_are_refused_as_such():
    """With and without a GPU: before torch is asked for a stream."""
    a, s = (xt.empty(n, "float32", device="cpu") for n in ((4,), ()))
    for call in (lambda: xt.noalias(a).assign(a + a), lambda: xt.noalias(s).assign(xt.sum(a)),
                 lambda: xt.noalias(a).assign(a * 2)):
        with pytest.raises(RuntimeError, match="needs device"):
            call()
