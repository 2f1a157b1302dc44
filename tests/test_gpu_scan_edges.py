"""Scans whose rows are no whole vectors: narrow matrices (several row groups
to a wave), odd pitches, inner views and short axes, against long double."""

import numpy as np
import pytest

import xtensor_amd as xt

from test_gpu_scan import _check_scan, _scan_ref, _tiled_input

pytestmark = pytest.mark.gpu

# (shape, kernel along axis 0): short axes, one column, narrow rows of 1 .. 16
# row groups, an odd number of chunks, column tiles that end inside a vector
SHAPES = [((77, 5), "scan_short"), ((128, 333), "scan_short"), ((129, 5), "scan_tiles_1p"), ((1000, 1), None),
          ((4097, 3), "scan_tiles_1p"), ((16054, 25), "scan_tiles_1p"), ((300, 33), "scan_tiles_1p"),
          ((515, 257), "scan_tiles_1p"), ((700, 1023), "scan_tiles_1p")]


@pytest.mark.parametrize("dtype", ["float32", "float64", "int32", "int64"])
@pytest.mark.parametrize("shape,kernel", SHAPES)
def test_ragged_scans(dtype, shape, kernel):
    x = _tiled_input(np.random.default_rng(sum(shape)), shape, dtype, "cumsum")
    X = xt.from_numpy(x)
    got = xt.cumsum(X, 0).to_numpy()
    if kernel:
        assert xt.last_kernel() == kernel
    _check_scan(got, _scan_ref(x, 0, "cumsum"), dtype, shape)
    _check_scan(xt.cumsum(X, 1).to_numpy(), _scan_ref(x, 1, "cumsum"), dtype, shape)


@pytest.mark.parametrize("dtype", ["float32", "int64"])
@pytest.mark.parametrize("axis", [0, 1])
@pytest.mark.parametrize("shape", [(100, 40), (900, 37), (2, 70001)])
def test_scan_of_inner_view_into_inner_view(dtype, axis, shape):
    """Offset by one element on both sides; what lies around the output stays."""
    rng = np.random.default_rng(9)
    full = (shape[0], shape[1] + 3)
    x, y = _tiled_input(rng, full, dtype, "cumsum"), _tiled_input(rng, full, dtype, "cumsum")
    X, Y = xt.from_numpy(x), xt.from_numpy(y)
    xt.plan(Y[:, 1:-2], xt.Scan("cumsum", X[:, 1:-2], axis)).run()
    got = Y.to_numpy()
    _check_scan(got[:, 1:-2].copy(), _scan_ref(x[:, 1:-2], axis, "cumsum"), dtype, shape)
    assert np.array_equal(got[:, :1], y[:, :1]) and np.array_equal(got[:, -2:], y[:, -2:])
