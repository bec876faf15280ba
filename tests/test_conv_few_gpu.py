"""Convolutions over few input channels, channels-first (conv_few.hip), through the C
ABI vs the oracle: forward with bias and ReLU, data gradient, weight gradient."""
import numpy as np
import pytest

from fusilli_amd import capi
from oracle import oracle
from helpers import HT, assert_close, rand
from test_generic_ops_gpu import run_conv, run_conv_dgrad, run_conv_wgrad

pytestmark = pytest.mark.gpu

CASES = [
    # the reference benchmark's shape (reduced batch): tiles of 256 pixels, the last short
    dict(x=[3, 3, 32, 32], w=[32, 3, 3, 3], pad=[0, 0], s=[1, 1], d=[1, 1]),
    dict(x=[2, 1, 57, 57], w=[64, 1, 5, 5], pad=[2, 2], s=[1, 1], d=[1, 1]),
    # 100 pairs; rows of 17 (no multiple of 4 or 16)
    dict(x=[2, 4, 16, 17], w=[16, 4, 5, 5], pad=[2, 2], s=[1, 1], d=[1, 1]),
    # fewest output channels, fewer pixels than one wavefront's
    dict(x=[1, 2, 5, 4], w=[8, 2, 3, 3], pad=[1, 1], s=[1, 1], d=[1, 1]),
    # two blocks of output channels, stride, dilation (data gradient: direct kernel)
    dict(x=[2, 3, 20, 33], w=[70, 3, 3, 5], pad=[1, 0], s=[2, 1], d=[1, 2]),
    # widest rows of the data gradient; single output rows per band
    dict(x=[1, 3, 5, 252], w=[24, 3, 3, 3], pad=[1, 1], s=[1, 1], d=[1, 1]),
    # padding beyond the filter, narrow image, many rows
    dict(x=[1, 1, 150, 3], w=[9, 1, 2, 3], pad=[0, 4], s=[1, 1], d=[1, 1]),
    # most pairs (112)
    dict(x=[1, 7, 9, 9], w=[20, 7, 4, 4], pad=[1, 2], s=[1, 1], d=[1, 1]),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16, capi.HALF])
def test_conv_few_channels_vs_oracle(ctx, case, dtype):
    geom = (case["pad"], case["s"], case["d"])
    yd = oracle.conv_output_dims(case["x"], case["w"], *geom)
    x = HT.from_logical(rand(51, 0, case["x"]), dtype)
    w = HT.from_logical(rand(51, 1, case["w"], std=0.2), dtype)
    dy = HT.from_logical(rand(51, 2, yd), dtype)
    bias = HT.from_logical(rand(51, 3, [1, case["w"][0], 1, 1]), dtype)
    epi = [capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=bias.desc()),
           capi.epilogue_op(capi.PW["RELU_FWD"], dtype)]
    y = run_conv(ctx, x, w, *geom, dtype, epilogue=epi, epi_tensors=[bias])
    assert ctx.last_kernel().startswith("conv_few fprop"), ctx.last_kernel()
    plain = oracle.conv_fprop(x.logical(), w.logical(), *geom)
    assert_close(y.logical(), np.maximum(plain + bias.logical(), 0), dtype, f"fprop {case}")
    # an operand of Y's own size is not one value per channel
    res = HT.from_logical(rand(51, 4, yd), dtype)
    y = run_conv(ctx, x, w, *geom, dtype, epi_tensors=[res],
                 epilogue=[capi.epilogue_op(capi.PW["ADD"], dtype, operand=res.desc())])
    assert ctx.last_kernel().startswith("conv_direct"), ctx.last_kernel()
    assert_close(y.logical(), plain + res.logical(), dtype, f"fprop + residual {case}")
    dx = run_conv_dgrad(ctx, dy, w, case["x"], *geom, dtype, False, tuned=None)
    few = case["x"][1] <= 4 and case["w"][3] in (3, 5) and case["s"] == case["d"] == [1, 1]
    assert ctx.last_kernel().startswith("conv_few dgrad" if few else "conv_direct"), ctx.last_kernel()
    assert_close(dx.logical(), oracle.conv_dgrad(dy.logical(), w.logical(), case["x"], *geom),
                 dtype, f"dgrad {case}")
    dw = run_conv_wgrad(ctx, dy, x, case["w"], *geom, dtype, False, tuned=None)
    assert ctx.last_kernel().startswith("conv_few wgrad"), ctx.last_kernel()
    assert_close(dw.logical(), oracle.conv_wgrad(dy.logical(), x.logical(), case["w"], *geom),
                 dtype, f"wgrad {case}")


@pytest.mark.parametrize("x,w,pad", [
    ([64, 3, 64, 64], [32, 3, 3, 3], [1, 1]),   # many bands per workgroup
    ([8, 1, 28, 28], [16, 1, 5, 5], [2, 2]),    # one
    ([4, 12, 16, 16], [64, 12, 3, 3], [1, 1]),  # the widest tiles
])
def test_weight_gradient_rounds_in_short_chains(ctx, x, w, pad):
    # Groups of 16 pixels, a wavefront's groups and the workgroups' sums are chains of
    # their own, at most 64 roundings each; a chain of n adds about sqrt(n) / 3 * 2^-24 of
    # a random sum's size (one chain of all a workgroup's pixels reached 4e-7)
    geom = (pad, [1, 1], [1, 1])
    xs = HT.from_logical(rand(52, 0, x), capi.FLOAT)
    dy = HT.from_logical(rand(52, 1, oracle.conv_output_dims(x, w, *geom)), capi.FLOAT)
    dw = run_conv_wgrad(ctx, dy, xs, w, *geom, capi.FLOAT, False, tuned=None).logical()
    assert ctx.last_kernel().startswith("conv_few wgrad"), ctx.last_kernel()
    xp = np.pad(xs.logical().astype(np.float64), [(0, 0), (0, 0), (pad[0],) * 2, (pad[1],) * 2])
    g = dy.logical().astype(np.float64)
    p, q = g.shape[2:]
    ref = np.empty(w)
    for r in range(w[2]):
        for s in range(w[3]):
            ref[:, :, r, s] = np.einsum("nkpq,ncpq->kc", g, xp[:, :, r:r + p, s:s + q], optimize=True)
    assert np.linalg.norm(dw - ref) <= 8 / 3 * 2.0 ** -24 * np.linalg.norm(ref)


@pytest.mark.parametrize("n,forward,gradient", [(2, 16, 1), (160, 32, 4), (400, 64, 4)])
def test_few_tiles_take_fewer_channels_each(ctx, n, forward, gradient):
    # blocks of channels by the number of tiles; operands per channel and per image
    x = HT.from_logical(np.resize(rand(53, 0, [2, 3, 20, 20]), [n, 3, 20, 20]), capi.FLOAT)
    w = HT.from_logical(rand(53, 1, [64, 3, 3, 3], std=0.2), capi.FLOAT)
    bias = HT.from_logical(rand(53, 2, [1, 64, 1, 1]), capi.BFLOAT16)
    full = np.zeros([n, 64, 1, 1])
    full[1] = rand(53, 3, [64, 1, 1])
    image = HT.from_logical(full, capi.FLOAT)  # a value per image and channel
    epi = [capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=bias.desc(), operand_index=0),
           capi.epilogue_op(capi.PW["MUL"], capi.FLOAT, scalar=0.5),
           capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=image.desc(), operand_index=1),
           capi.epilogue_op(capi.PW["GELU_FWD"], capi.FLOAT)]
    geom = ([0, 0], [1, 1], [1, 1])
    y = run_conv(ctx, x, w, *geom, capi.FLOAT, epilogue=epi, epi_tensors=[bias, image])
    assert ctx.last_kernel() == f"conv_few fprop channels={forward}", ctx.last_kernel()
    ref = oracle.conv_fprop(x.logical()[:2], w.logical(), *geom) + bias.logical()
    ref = oracle.pointwise(capi.PW["GELU_FWD"], [ref * 0.5 + full[:2]])
    assert_close(y.logical()[:2], ref, capi.FLOAT)
    dy = HT.from_logical(rand(53, 4, [n, 64, 18, 18]), capi.FLOAT)
    dw = run_conv_wgrad(ctx, dy, x, [64, 3, 3, 3], *geom, capi.FLOAT, False, tuned=None)
    assert ctx.last_kernel() == f"conv_few wgrad tiles={gradient}x2", ctx.last_kernel()
    assert_close(dw.logical(), oracle.conv_wgrad(dy.logical(), x.logical(), [64, 3, 3, 3], *geom), capi.FLOAT)


@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("x,w,pad,dense,kind", [
    ([3, 3, 32, 32], [32, 3, 3, 3], [0, 0], True, "products"),
    ([2, 2, 21, 30], [32, 2, 3, 3], [1, 1], True, "products"),    # rows of 30: the last quad reaches behind
    ([1, 1, 6, 4], [9, 1, 3, 3], [0, 0], True, "products"),       # rows of two, odd channels
    ([2, 4, 40, 9], [37, 4, 3, 3], [2, 2], True, "products"),     # three tiles of pairs, channels in two blocks
    ([2, 3, 20, 24], [65, 3, 5, 5], [2, 2], True, "products"),    # passes side by side, 65 channels
    ([300, 2, 12, 12], [40, 2, 5, 5], [2, 2], True, None),        # passes one after the other (16 bits)
    ([300, 3, 12, 12], [16, 3, 5, 5], [2, 2], True, "channels"),  # few output channels: vector instructions
    ([1, 1, 30, 200], [24, 1, 5, 5], [0, 1], True, "products"),   # bands cut in columns
    ([2, 1, 3, 250], [8, 1, 2, 3], [3, 3], True, "products"),     # DY beside the image
    ([2, 3, 20, 18], [16, 3, 3, 3], [1, 1], False, "products"),   # rows of DY with gaps
    # both sides of the line for much work per compute unit: vector instructions (f32)
    ([69, 1, 33, 33], [16, 1, 5, 5], [2, 2], True, None),
    ([67, 1, 48, 48], [32, 1, 5, 5], [0, 0], True, "products"),
    ([120, 1, 39, 39], [32, 1, 5, 5], [2, 2], True, None),
    ([50, 1, 63, 63], [16, 1, 3, 3], [1, 1], True, None),
    ([104, 4, 38, 38], [16, 4, 3, 3], [1, 1], True, "products"),
    ([106, 3, 61, 61], [16, 3, 3, 3], [1, 1], True, None),
    ([69, 1, 33, 33], [460, 1, 5, 5], [2, 2], True, "products"),  # a filter that LDS does not hold there
])
def test_data_gradient_products_first(ctx, x, w, pad, dense, kind, dtype):
    geom = (pad, [1, 1], [1, 1])
    yd = oracle.conv_output_dims(x, w, *geom)
    wt = HT.from_logical(rand(54, 0, w, std=0.2), dtype)
    if dense:
        dy = HT.from_logical(rand(54, 1, yd), dtype)
    else:
        pitch = yd[3] + 3
        st = [yd[1] * yd[2] * pitch, yd[2] * pitch, pitch, 1]
        dy = HT.from_logical(rand(54, 1, yd), dtype, strides=st)
    dx = run_conv_dgrad(ctx, dy, wt, x, *geom, dtype, False, tuned=None)
    if kind is None:
        kind = "channels" if dtype == capi.FLOAT else "products"
    assert ctx.last_kernel().startswith(f"conv_few dgrad {kind}"), ctx.last_kernel()
    assert_close(dx.logical(), oracle.conv_dgrad(dy.logical(), wt.logical(), x, *geom), dtype, f"{x} {w}")


def test_data_gradient_keeps_infinities_where_they_fall(ctx):
    # one infinite value of DY reaches the pixels under its filter and no others
    geom = ([1, 1], [1, 1], [1, 1])
    g = rand(55, 0, [2, 12, 10, 11])
    g[0, 11, 4, 10] = np.inf  # last column, last channel
    wt = HT.from_logical(np.abs(rand(55, 1, [12, 3, 3, 3])) + 0.1, capi.FLOAT)
    dx = run_conv_dgrad(ctx, HT.from_logical(g, capi.FLOAT), wt, [2, 3, 10, 11], *geom, capi.FLOAT, False,
                        tuned=None).logical()
    assert ctx.last_kernel().startswith("conv_few dgrad products"), ctx.last_kernel()
    hit = np.zeros(dx.shape, bool)
    hit[0, :, 3:6, 9:11] = True
    assert np.isposinf(dx[hit]).all() and np.isfinite(dx[~hit]).all()


@pytest.mark.parametrize("dtype,tiny", [(capi.HALF, 2.0 ** -22), (capi.BFLOAT16, 2.0 ** -130)])
def test_data_gradient_keeps_subnormal_values(ctx, dtype, tiny):
    # 16-bit DY below the normal range times whole numbers: exact sums of 12 * 9 values at most
    dy = HT.from_logical(np.full([1, 12, 8, 8], tiny), dtype)
    wt = HT.from_logical(np.full([12, 3, 3, 3], 64.0 if dtype == capi.HALF else 4.0), dtype)
    dx = run_conv_dgrad(ctx, dy, wt, [1, 3, 8, 8], [1, 1], [1, 1], [1, 1], dtype, False, tuned=None).logical()
    assert ctx.last_kernel().startswith("conv_few dgrad products"), ctx.last_kernel()
    scale = 12 * wt.logical().flat[0] * tiny
    assert np.array_equal(dx[0, 0, 1:-1, 1:-1], np.full([6, 6], 9 * scale)), dx[0, 0]
    assert np.array_equal(dx[0, :, 0, 0], np.full([3], 4 * scale))


# X staged by steps of 256 elements: rows longer than that, channels of fewer elements, several batches
# of loads, gaps between rows, channels and images; filters that do not lie pair behind pair; more
# bands than workgroups.  Whole numbers: every sum is exact.
@pytest.mark.parametrize("x,w,pad,s,d,gaps", [
    ([2, 3, 6, 300], [16, 3, 3, 3], [1, 1], [1, 1], [1, 1], False),
    ([3, 9, 2, 3], [20, 9, 3, 3], [1, 1], [1, 1], [1, 1], True),
    ([2, 12, 40, 31], [17, 12, 3, 3], [1, 1], [1, 1], [1, 1], True),
    ([2, 4, 25, 256], [30, 4, 5, 5], [2, 2], [2, 1], [1, 3], True),
    ([2, 1, 1, 700], [8, 1, 1, 5], [0, 7], [1, 3], [1, 2], False),
    ([2, 2, 700, 1], [8, 2, 5, 1], [3, 0], [2, 1], [1, 1], True),
    ([200, 3, 40, 40], [16, 3, 3, 3], [1, 1], [1, 1], [1, 1], False),
])
@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16])
def test_staged_rows(ctx, x, w, pad, s, d, gaps, dtype):
    rng = np.random.default_rng(x[0] + x[3])
    pitch, plane = x[3] + 5, x[2] * (x[3] + 5) + 11
    xt = HT.from_logical(rng.integers(-2, 3, size=x), dtype, [x[1] * plane + 3, plane, pitch, 1] if gaps else None)
    turned = [w[1] * w[2] * w[3], 1, w[1] * w[3], w[1]]  # channel beside channel
    wt = HT.from_logical(rng.integers(-1, 2, size=w), dtype, turned if gaps else None)
    y = run_conv(ctx, xt, wt, pad, s, d, dtype)
    assert ctx.last_kernel().startswith("conv_few fprop"), ctx.last_kernel()
    # (sums of at most 112 products of 2 x 1: whole in 16 bits too)
    np.testing.assert_array_equal(y.logical(), oracle.conv_fprop(xt.logical(), wt.logical(), pad, s, d))
    dy = HT.from_logical(rng.integers(-1, 2, size=y.dims), dtype)
    dw = run_conv_wgrad(ctx, dy, xt, w, pad, s, d, dtype, False, tuned=None)
    assert ctx.last_kernel().startswith("conv_few wgrad"), ctx.last_kernel()
    ref = oracle.conv_wgrad(dy.logical(), xt.logical(), w, pad, s, d)
    np.testing.assert_array_equal(dw.logical(), HT.from_logical(ref, dtype).logical())
