"""Convolutions and data gradients on register-staged tiles (conv_tile_kernel.h): strides above
one as several products, channel counts off a slice, ragged tiles, split reductions, filters in
other layouts, against torch's f32 convolutions of whole numbers on the CPU (exact in f32, and so
equal after the one rounding)."""
import numpy as np
import pytest
import torch

from fusilli_amd import capi
from oracle import oracle
from helpers import HT, rand
from test_generic_ops_gpu import run_conv, run_conv_dgrad

pytestmark = pytest.mark.gpu

LAY = oracle.channels_last_strides


def _whole(seed, i, dims, lim, dtype, strides=None):
    flat = rand(seed, i, [4099], "int", lo=-lim, hi=lim + 1)
    return HT.from_logical(np.resize(flat, dims), dtype, strides or LAY(dims))


def _equal(got, want, dtype):
    t = {capi.BFLOAT16: torch.bfloat16, capi.HALF: torch.float16, capi.FLOAT: torch.float32}[dtype]
    assert float(want.abs().max()) < 2 ** 24
    assert np.array_equal(got, want.to(t).float().numpy())


@pytest.mark.parametrize("x,w,pad,st,dil,parts", [
    ([3, 24, 11, 9], [40, 24, 3, 3], 1, [2, 2], [1, 1], 4),       # odd sizes, K-taps inside a slice
    ([2, 64, 12, 14], [136, 64, 3, 2], 1, [2, 1], [1, 1], 2),     # a stride in one dim
    ([2, 72, 13, 10], [72, 72, 1, 1], 0, [2, 2], [1, 1], 4),      # remainders without a tap: zeros
    ([2, 8, 10, 11], [8, 8, 5, 5], 2, [3, 3], [1, 1], 9),
    ([2, 16, 17, 18], [24, 16, 3, 3], 2, [4, 4], [2, 2], 16),     # stride and dilation share a factor
    ([2, 16, 13, 13], [24, 16, 3, 3], 2, [2, 3], [2, 2], 6),
    ([1, 16, 30, 9], [24, 16, 3, 3], 1, [5, 4], [1, 1], 0),       # more products than a launch: spread
    ([16, 296, 62, 62], [64, 296, 5, 5], 2, [2, 2], [1, 1], 4),   # tiles of 128 x 128, the last ones ragged
    ([20, 64, 11, 11], [384, 64, 5, 5], 2, [1, 1], [1, 1], 1),    # a split reduction
    ([5, 200, 20, 20], [104, 200, 3, 3], 1, [1, 1], [1, 1], 1),
    ([3, 40, 50], [64, 40, 4], 1, [2], [1], 2),                   # one spatial dim
])
@pytest.mark.parametrize("dtype,flat", [(capi.BFLOAT16, False), (capi.HALF, True)])
def test_data_gradient(ctx, x, w, pad, st, dil, parts, dtype, flat):
    sp = len(x) - 2
    geom = ([pad] * sp, st, dil)
    yd = oracle.conv_output_dims(x, w, *geom)
    ws = None
    if flat:  # channels-first filter
        ws = [int(np.prod(w[i + 1:])) for i in range(len(w))]
    wt = _whole(81, 1, w, 2, dtype, ws)
    dy = _whole(81, 2, yd, 3, dtype)
    dx = run_conv_dgrad(ctx, dy, wt, x, *geom, dtype, tuned=None)
    name = ctx.last_kernel()
    if parts != 1:
        assert ("parts=" in name) == (parts > 1) and (parts == 0 or f"parts={parts}" in name), name
    elif not flat:  # (a filter that is copied first: whichever is faster)
        assert "parts=1" in name, name
    if x[0] == 20:
        assert "split=1" not in name, name
    grad = torch.nn.grad.conv2d_input if sp == 2 else torch.nn.grad.conv1d_input
    ref = grad(x, torch.from_numpy(wt.logical()), torch.from_numpy(dy.logical()), st, geom[0], dil)
    _equal(dx.logical(), ref, dtype)


@pytest.mark.parametrize("x,w,pad,st", [
    ([9, 128, 12, 12], [128, 128, 5, 5], 2, 1),    # few tiles, a long reduction
    ([31, 192, 11, 11], [180, 192, 5, 5], 2, 1),   # columns off a tile
    ([7, 456, 13, 14], [61, 456, 3, 3], 1, 2),     # odd columns, channels off a slice
    ([40, 264, 30, 30], [260, 264, 3, 3], 1, 1),   # wide tiles; with a chain conv_gather.hip
    ([2, 520, 6, 6], [64, 520, 5, 5], 2, 1),
])
@pytest.mark.parametrize("chain", [False, True])
def test_forward(ctx, x, w, pad, st, chain, dtype=capi.BFLOAT16, route=""):
    geom = ([pad, pad], [st, st], [1, 1])
    yd = oracle.conv_output_dims(x, w, *geom)
    xs, wt = _whole(82, 0, x, 3, dtype), _whole(82, 1, w, 2, dtype)
    bias = _whole(82, 2, [1, w[0], 1, 1], 9, dtype)
    res = _whole(82, 3, yd, 9, dtype)
    epi = [capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=bias.desc()),
           capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=res.desc(), operand_index=1),
           capi.epilogue_op(capi.PW["RELU_FWD"], dtype)] if chain else []
    y = run_conv(ctx, xs, wt, *geom, capi.FLOAT, out_dtype=dtype if chain else capi.FLOAT, epilogue=epi,
                 epi_tensors=[bias, res] if chain else [], channels_last_out=True)
    assert ctx.last_kernel().startswith(f"conv_igemm unpadded {route}"), ctx.last_kernel()
    ref = torch.nn.functional.conv2d(torch.from_numpy(xs.logical()), torch.from_numpy(wt.logical()), None, st, pad)
    if chain:
        ref = (ref + torch.from_numpy(bias.logical()) + torch.from_numpy(res.logical())).clamp(min=0)
    _equal(y.logical(), ref, dtype if chain else capi.FLOAT)


# every tile of the forward kernel, whole and in parts (teams=0: the kernel for short reductions)
@pytest.mark.parametrize("x,w,pad,st,chain,route", [
    ([33, 120, 22, 38], [200, 120, 3, 3], 1, 1, False, "128x128 split=1 teams=1"),
    ([13, 120, 36, 33], [196, 120, 3, 3], 1, 1, True, "128x128 split=1 teams=1"),
    ([27, 296, 36, 9], [76, 296, 3, 3], 1, 1, False, "128x128 split=3 teams=1"),
    ([10, 416, 24, 36], [68, 416, 3, 3], 1, 1, True, "128x128 split=3 teams=1"),
    ([33, 184, 17, 34], [144, 184, 3, 3], 1, 1, True, "128x64 split=1 teams=1"),
    ([31, 288, 27, 7], [140, 288, 5, 5], 2, 1, False, "128x64 split=3 teams=1"),
    ([30, 112, 39, 25], [104, 112, 3, 3], 1, 1, False, "64x128 split=1 teams=1"),
    ([13, 56, 25, 38], [216, 56, 5, 5], 2, 1, True, "64x128 split=1 teams=1"),
    ([11, 216, 19, 14], [72, 216, 5, 5], 2, 1, False, "64x128 split=5 teams=1"),
    ([8, 184, 24, 26], [72, 184, 5, 5], 2, 1, True, "64x128 split=3 teams=1"),
    ([9, 176, 25, 15], [264, 176, 3, 3], 1, 1, True, "64x64 split=1 teams=0"),
    ([2, 104, 5, 8], [92, 104, 3, 3], 1, 1, True, "64x64 split=5 teams=0"),
    ([12, 128, 10, 27], [200, 128, 3, 3], 1, 2, False, "64x64 split=1 teams=2"),
    ([1, 216, 28, 18], [37, 216, 5, 5], 2, 2, False, "64x64 split=11 teams=2"),
])
@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
def test_forward_tiles(ctx, x, w, pad, st, chain, route, dtype):
    test_forward(ctx, x, w, pad, st, chain, dtype, route)
