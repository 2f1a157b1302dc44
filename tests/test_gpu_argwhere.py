"""argwhere around the edges of its workgroups (4096 positions, 16 a thread),
of one to four dimensions, in both orders, against numpy; rows past a given
output are dropped."""

import numpy as np
import pytest

import xtensor_amd as xt
from xtensor_amd import _abi as A
from xtensor_amd import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4095, 4096, 4097, 3 * 4096 + 5, 4096 * 4097 + 3])
@pytest.mark.parametrize("fill", ["none", "all", "some", "last"])
def test_lengths(n, fill):
    h = {"none": np.zeros(n, bool), "all": np.ones(n, bool), "some": np.random.default_rng(n).random(n) < 0.3,
         "last": np.arange(n) == n - 1}[fill]
    got = xt.argwhere(xt.from_numpy(h))
    assert np.array_equal(got.to_numpy(), np.argwhere(h))


@pytest.mark.parametrize("layout", ["row_major", "column_major"])
@pytest.mark.parametrize("shape", [(3, 5000), (5000, 3), (17, 31, 29), (1, 9, 1, 700)])
def test_dimensions(shape, layout):
    h = np.random.default_rng(7).normal(size=shape)
    want = np.argwhere(h > 0.5) if layout == "row_major" else np.argwhere((h > 0.5).T)[:, ::-1]
    x = xt.from_numpy(h)
    assert np.array_equal(xt.argwhere(x > 0.5, layout).to_numpy(), want)
    assert np.array_equal(xt.eval(xt.filter(x, x > 0.5, layout)).to_numpy(), h[tuple(want.T)])
    # one call into a given output with padded rows, fewer than there are
    rows = len(want) // 2
    out = xt.zeros((rows, 2 * len(shape)), "int64")
    s, t = core.serialize(x > 0.5), out[:, ::2].to_abi()
    core._check(A.lib().xg_argwhere(s.ptr(), int(layout == "column_major"), t, core._stream()))
    got = out.to_numpy()
    assert np.array_equal(got[:, ::2], want[:rows]) and not got[:, 1::2].any()
