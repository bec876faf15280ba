"""Weight gradient on gathered MFMA tiles (conv_wgrad.hip), through the C ABI vs the
oracle: channel counts off the tiles, tap runs across column tiles, strides, dilation,
padding beyond the image, pixel counts off the steps, several chunks of pixels."""
import numpy as np
import pytest

from fusilli_amd import capi
from oracle import oracle
from helpers import HT, assert_close, rand
from test_generic_ops_gpu import run_conv_wgrad

pytestmark = pytest.mark.gpu

CASES = [
    # 48 channels: a tap's runs straddle the column tiles; rows and columns padded
    dict(x=[3, 48, 12, 9], w=[48, 48, 3, 3], pad=[2, 2], s=[1, 1], d=[1, 1]),
    # least channels, fewer than 32 pixels, one run
    dict(x=[1, 8, 5, 4], w=[8, 8, 3, 3], pad=[1, 1], s=[1, 1], d=[1, 1]),
    # unequal strides, dilation in both dims
    dict(x=[2, 40, 17, 19], w=[72, 40, 3, 2], pad=[1, 0], s=[2, 1], d=[2, 3]),
    # stride 2; K over one 128-row tile, J over one 128-column tile
    dict(x=[4, 136, 15, 15], w=[200, 136, 3, 3], pad=[1, 1], s=[2, 2], d=[1, 1]),
    # 1 x 1 with stride (256 rows x 64 columns), 5 x 5 with wide padding
    dict(x=[2, 56, 13, 11], w=[256, 56, 1, 1], pad=[0, 0], s=[2, 2], d=[1, 1]),
    dict(x=[2, 16, 6, 7], w=[32, 16, 5, 5], pad=[4, 4], s=[1, 1], d=[1, 1]),
    # a run of more than 2048 pixels (two chunks, images crossed inside both)
    dict(x=[40, 512, 17, 16], w=[512, 512, 3, 3], pad=[0, 1], s=[1, 1], d=[1, 1]),
    # whole image inside the padding on one side: many pixels per image, one column
    dict(x=[5, 24, 70, 1], w=[104, 24, 3, 3], pad=[0, 1], s=[1, 1], d=[1, 1]),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("f32_out", [False, True])
def test_conv_wgrad_gather_vs_oracle(ctx, case, dtype, f32_out):
    lay = oracle.channels_last_strides
    geom = (case["pad"], case["s"], case["d"])
    yd = oracle.conv_output_dims(case["x"], case["w"], *geom)
    x = HT.from_logical(rand(61, 0, case["x"]), dtype, lay(case["x"]))
    dy = HT.from_logical(rand(61, 1, yd), dtype, lay(yd))
    if case["x"][0] * case["x"][1] > 4096:
        # (large reduction: checked on a slice, the gradient of the first 8 of K and C)
        if f32_out:
            pytest.skip("covered by the 16-bit output")
        dw = run_conv_wgrad(ctx, dy, x, case["w"], *geom, dtype, tuned=None)
        ref = oracle.conv_wgrad(dy.logical()[:, :8], x.logical()[:, :8], [8, 8, 3, 3], *geom)
        assert_close(dw.logical()[:8, :8], ref, dtype, f"wgrad {case}")
    else:
        dw = run_conv_wgrad(ctx, dy, x, case["w"], *geom, dtype, tuned=None,
                            w_dtype=capi.FLOAT if f32_out else None)
        assert_close(dw.logical(), oracle.conv_wgrad(dy.logical(), x.logical(), case["w"], *geom),
                     dtype, f"wgrad {case}")
    assert ctx.last_kernel().startswith("conv_wgrad_gather"), ctx.last_kernel()


@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("x,w,stride,tile", [
    ([4, 256, 48, 60], [256, 256, 5, 5], 1, "128x128"),
    ([6, 512, 24, 24], [192, 512, 5, 5], 1, "64x256"),
    ([6, 512, 24, 24], [96, 512, 5, 5], 1, "32x256"),
    ([8, 320, 64, 60], [2560, 320, 1, 1], 2, "256x64"),
])
def test_f32_weight_gradient_rounds_in_short_chains(ctx, dtype, x, w, stride, tile):
    # Few runs of many pixels: 30 additions of 16 products each, at most seven such groups per
    # run, at most ten runs are chains of their own.  A chain of n adds about sqrt(n) / 3 *
    # 2^-24 of a random sum's size: 2.4 together (one chain of a run's 770 to 2900 pixels: 2.4
    # to 4.6).
    pad = w[2] // 2
    geom = ([pad, pad], [stride, stride], [1, 1])
    lay = oracle.channels_last_strides
    yd = oracle.conv_output_dims(x, w, *geom)
    xs = HT.from_logical(rand(62, 0, x), dtype, lay(x))
    dy = HT.from_logical(rand(62, 1, yd), dtype, lay(yd))
    dw = run_conv_wgrad(ctx, dy, xs, w, *geom, dtype, tuned=None, w_dtype=capi.FLOAT).logical()
    assert ctx.last_kernel().startswith(f"conv_wgrad_gather {tile} "), ctx.last_kernel()
    xp = np.pad(xs.logical().astype(np.float64), [(0, 0), (0, 0), (pad, pad), (pad, pad)])
    for r, s in ((0, 0), (w[2] - 1, w[3] // 2)):
        shifted = xp[:, :, r:r + stride * (yd[2] - 1) + 1:stride, s:s + stride * (yd[3] - 1) + 1:stride]
        ref = (dy.logical().astype(np.float64).transpose(1, 0, 2, 3).reshape(w[0], -1)
               @ shifted.transpose(0, 2, 3, 1).reshape(-1, w[1]))
        err = np.linalg.norm(dw[:, :, r, s] - ref) / np.linalg.norm(ref)
        assert err <= 2.6 * 2.0 ** -24, (ctx.last_kernel(), err * 2.0 ** 24)
