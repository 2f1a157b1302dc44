"""Copies between layouts contiguous along different dimensions, by tiles of
64 x 64 through LDS: the copy itself against numpy, bit for bit."""

import ctypes as C

import numpy as np
import pytest

import xtensor_amd as xt
from xtensor_amd import _abi as A

pytestmark = pytest.mark.gpu

DTYPES = [np.int16, np.float32, np.int64]
EDGES = [(17, 64), (18, 64), (33, 34), (34, 34), (63, 65), (64, 64), (65, 127), (130, 40), (257, 191)]  # from either side of the line on


def distinct(shape, dtype):
    n = int(np.prod(shape))
    return (np.arange(n, dtype=np.int64) * 7919 % 30011).astype(dtype).reshape(shape)


def copied(view, dtype, tiles=True):
    """The copy; tiles: whether the tiles' kernel makes it (None: either)."""
    out = xt.zeros(view.shape, str(np.dtype(dtype)))
    xt.noalias(out).assign(view)
    if tiles is not None:
        assert (xt.last_kernel() == "transpose") == tiles
    return out.to_numpy()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("c,hw", EDGES)
def test_matrix_and_images(c, hw, dtype):
    """Edges of a tile either way, with none, one and two other dimensions; a
    tile of 17 x 64 is just below the line."""
    tiles = (c, hw) != (17, 64)
    x = distinct((c, hw), dtype)
    assert np.array_equal(copied(xt.transpose(xt.from_numpy(x), (1, 0)), dtype, tiles), x.T)
    x = distinct((3, c, hw), dtype)
    assert np.array_equal(copied(xt.transpose(xt.from_numpy(x), (0, 2, 1)), dtype, tiles), x.transpose(0, 2, 1))
    x = distinct((2, c, 3, hw), dtype)
    assert np.array_equal(copied(xt.transpose(xt.from_numpy(x), (2, 3, 0, 1)), dtype), x.transpose(2, 3, 0, 1))
    assert np.array_equal(copied(xt.transpose(xt.from_numpy(x), (0, 3, 2, 1)), dtype, tiles), x.transpose(0, 3, 2, 1))


@pytest.mark.parametrize("dtype", DTYPES)
def test_parts_of_arrays(dtype):
    """A leaf and an output that start inside a row and whose rows are apart:
    the elements around the output's part stay."""
    x = distinct((71, 203), dtype)
    part = xt.view(xt.from_numpy(x), xt.range_(1, 68), xt.range_(3, 200))
    whole = xt.from_numpy(np.full((230, 90), 7, dtype))
    xt.noalias(xt.view(whole, xt.range_(5, 202), xt.range_(1, 68))).assign(xt.transpose(part, (1, 0)))
    assert xt.last_kernel() == "transpose"
    want = np.full((230, 90), 7, dtype)
    want[5:202, 1:68] = x[1:68, 3:200].T
    assert np.array_equal(whole.to_numpy(), want)


def test_bfloat16_bits():
    """Every bfloat16 pattern: the tiles store what the element-wise program does."""
    import torch
    bits = np.arange(65536, dtype=np.uint16).reshape(128, 512)
    x, by_tiles, by_elements = (xt.zeros(s, "bfloat16") for s in ((128, 512), (512, 128), (512, 128)))
    x.storage.view(torch.int16)[:65536].copy_(torch.from_numpy(bits.view(np.int16).ravel()))
    xt.noalias(by_tiles).assign(xt.transpose(x, (1, 0)))
    assert xt.last_kernel() == "transpose"
    for r in range(0, 128, 16):   # 16 columns at a time are below the tiles' line
        part = xt.transpose(xt.view(x, xt.range_(r, r + 16), xt.all_()), (1, 0))
        xt.noalias(xt.view(by_elements, xt.all_(), xt.range_(r, r + 16))).assign(part)
        assert xt.last_kernel() != "transpose"
    got, ref = (o.storage.view(torch.int16)[:65536].cpu().numpy() for o in (by_tiles, by_elements))
    assert np.array_equal(got, ref)
    nan = (bits & 0x7FFF) > 0x7F80
    assert np.array_equal(got.view(np.uint16).reshape(512, 128).T, np.where(nan, bits | 0x40, bits))


def test_prepared_and_graph_replays():
    """A prepared plan and replays of its graph, with new values between them."""
    import torch
    x = distinct((2, 70, 33, 5), np.float32)
    dx = xt.from_numpy(x)
    direct, replayed = (xt.zeros((2, 33, 5, 70), "float32") for _ in range(2))
    plan = xt.plan(direct, xt.transpose(dx, (0, 2, 3, 1)))
    g = xt.PlanGraph([xt.plan(replayed, xt.transpose(dx, (0, 2, 3, 1)))])
    for k in range(4):
        dx.storage.view(torch.float32).add_(1.0)
        plan.run()
        g.replay()
        torch.cuda.synchronize()
        want = (x + np.float32(k + 1)).transpose(0, 2, 3, 1)
        assert np.array_equal(direct.to_numpy(), want) and np.array_equal(replayed.to_numpy(), want)


@pytest.mark.parametrize("dtype", ["int16", "float32", "float64"])
def test_large_copy_compiles_nothing(dtype):
    """Past the run-time compiler's threshold too: no kernel is compiled,
    loaded or looked up for a copy that goes by tiles."""
    x = distinct((1100, 1000), np.dtype(dtype))
    d = xt.from_numpy(x)
    before, after = ((C.c_int64 * 4)() for _ in range(2))
    L = A.lib()
    L.xg_debug_jit_stats(before)
    got = copied(xt.transpose(d, (1, 0)), np.dtype(dtype))
    plan_out = xt.zeros((1000, 1100), dtype)
    xt.plan(plan_out, xt.transpose(d, (1, 0))).run()
    L.xg_debug_jit_stats(after)
    assert list(before) == list(after)
    assert np.array_equal(got, x.T) and np.array_equal(plan_out.to_numpy(), x.T)
