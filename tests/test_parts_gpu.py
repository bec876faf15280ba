"""Launches that add partial results, at part counts on both sides of their rounds of loads:
small whole numbers, so that every sum is exact in f32 whatever its order."""
import numpy as np
import pytest

from fusilli_amd import capi
from oracle import oracle
from helpers import HT
from test_generic_ops_gpu import conv_bwd_desc, run_batchnorm, run_conv_dgrad, run_conv_wgrad

pytestmark = pytest.mark.gpu


def whole(seed, dims, dtype, span):
    v = np.random.default_rng(seed).integers(-span, span + 1, size=dims).astype(np.float64)
    return HT.from_logical(v, dtype, oracle.channels_last_strides(dims))


# 64 rows of 32 channels are a round of the row lanes, eight of them a block: blocks on both sides of
# the rounds of loads that add them, channels in one and several groups, the last one part of a group
@pytest.mark.parametrize("n,c,parts", [
    (1, 32, 1), (8, 32, 1), (9, 32, 2), (129, 32, 17), (1032, 32, 129), (2048, 32, 256), (2200, 32, 256),
    (5, 8, 1), (7, 136, 2), (130, 72, 21), (9, 1032, 3), (13, 2048, 4),
])
@pytest.mark.parametrize("dtype,affine", [(capi.BFLOAT16, capi.FLOAT), (capi.FLOAT, capi.HALF)])
def test_batchnorm_parts(ctx, n, c, parts, dtype, affine):
    if dtype == capi.FLOAT and c > 1024:
        pytest.skip("more channels than the kernel takes")
    x = whole(n, [n, c, 8, 8], dtype, 3)
    one = HT.from_logical(np.ones(c), affine)
    y, m, v = run_batchnorm(ctx, x, training=True, eps=1e-3, scale=one, bias=one)
    if dtype == capi.BFLOAT16:
        assert ctx.last_kernel().endswith(f"workgroups={parts}"), ctx.last_kernel()
    # (one division and one addition to the pivot, each rounded once)
    mean = x.logical().mean(axis=(0, 2, 3))
    np.testing.assert_allclose(m, mean, rtol=0, atol=3 * 2.0 ** -23)
    # (exact sums: a few roundings of values near one, the last one to Y's type)
    inv = 1 / np.sqrt(x.logical().astype(np.float64).var(axis=(0, 2, 3)) + 1e-3)
    np.testing.assert_allclose(v, inv, rtol=2.0 ** -20)
    ref = (x.logical() - mean[:, None, None]) * inv[:, None, None] + 1
    step = 2.0 ** -8 if dtype == capi.BFLOAT16 else 2.0 ** -19
    np.testing.assert_allclose(y.logical() if hasattr(y, "logical") else y, ref, rtol=step, atol=step)


# (the pivot is a value of X)
def test_batchnorm_writes_over_its_input(ctx):
    x = whole(3, [9, 72, 17, 16], capi.BFLOAT16, 3)
    y, m, _ = run_batchnorm(ctx, x, training=True, eps=1e-3)
    d = capi.BatchNormDesc()
    d.x, d.y, d.training, d.epsilon = x.desc(), x.desc(), 1, 1e-3
    d.scale_dtype = d.bias_dtype = d.running_dtype = d.stats_dtype = capi.FLOAT
    mean, inv = HT.empty([72], capi.FLOAT), HT.empty([72], capi.FLOAT)
    bx, bm, bi = x.upload(ctx), mean.upload(ctx), inv.upload(ctx)
    ctx.batchnorm_fwd(d, bx, bx, None, None, None, None, bm, bi)
    np.testing.assert_array_equal(mean.fetch(ctx, bm).logical(), m)
    np.testing.assert_array_equal(x.fetch(ctx, bx).logical(), y)


# gathered tiles: runs of 32-pixel steps, added one by one, four and sixteen at a time
@pytest.mark.parametrize("n", [2, 3, 5, 8, 9, 17, 33, 36, 39, 65, 130])
@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.FLOAT])
def test_weight_gradient_parts(ctx, n, dtype):
    x, dy = whole(n, [n, 8, 16, 16], capi.BFLOAT16, 2), whole(n + 1, [n, 24, 16, 16], capi.BFLOAT16, 1)
    dw = run_conv_wgrad(ctx, dy, x, [24, 8, 1, 3], [0, 1], [1, 1], [1, 1], capi.BFLOAT16, tuned=None,
                        w_dtype=capi.FLOAT if dtype == capi.FLOAT else None)
    assert ctx.last_kernel().startswith("conv_wgrad_gather"), ctx.last_kernel()
    ref = oracle.conv_wgrad(dy.logical(), x.logical(), [24, 8, 1, 3], [0, 1], [1, 1], [1, 1])
    np.testing.assert_array_equal(dw.logical(), HT.from_logical(ref, dtype).logical())


# 3 x 3 filters at unit stride: rows of one to four 16-pixel steps, shares of the batch's rows that
# start and end inside images, cross several, or are empty
@pytest.mark.parametrize("x,k,steps", [
    ([1, 32, 3, 1], 32, 1), ([21, 32, 5, 15], 64, 1), ([300, 32, 1, 16], 32, 1), ([40, 96, 14, 16], 64, 1),
    ([9, 64, 13, 17], 32, 2), ([14, 320, 24, 24], 480, 2), ([3, 32, 50, 32], 160, 2),
    ([5, 32, 19, 33], 96, 3), ([4, 64, 48, 48], 192, 3), ([2, 96, 7, 49], 32, 4), ([11, 32, 56, 56], 64, 4),
])
def test_direct_weight_gradient_shares(ctx, x, k, steps):
    xt, dy = whole(k, x, capi.BFLOAT16, 2), whole(k + 1, [x[0], k] + x[2:], capi.BFLOAT16, 1)
    w = [k, x[1], 3, 3]
    dw = run_conv_wgrad(ctx, dy, xt, w, [1, 1], [1, 1], [1, 1], capi.BFLOAT16, tuned=True, w_dtype=capi.FLOAT)
    assert ctx.last_kernel().startswith(f"conv_wgrad_direct steps={steps}"), ctx.last_kernel()
    got = dw.logical()
    if k > 300:  # (some blocks of a large one)
        xt, dy = xt.logical()[:, 256:], dy.logical()[:, 416:]
        np.testing.assert_array_equal(got[416:, 256:], oracle.conv_wgrad(dy, xt, [64, 64, 3, 3], [1, 1], [1, 1], [1, 1]))
    else:
        np.testing.assert_array_equal(got, oracle.conv_wgrad(dy.logical(), xt.logical(), w, [1, 1], [1, 1], [1, 1]))


# paddings of 0 to 2, channels off the blocks of 32: the same kernel in place of the
# gathered tiles, whose workspace it is given
@pytest.mark.parametrize("x,k,pad,steps", [
    ([16, 48, 48, 32], 48, 2, 3), ([9, 64, 31, 19], 72, 0, 2), ([40, 200, 9, 18], 40, 0, 1),
    ([60, 32, 20, 58], 32, 0, 4), ([30, 40, 17, 14], 64, 2, 1), ([25, 96, 4, 31], 200, 2, 3),
    ([12, 136, 16, 54], 24, 2, 4), ([11, 8, 60, 40], 72, 1, 3), ([60, 88, 1, 16], 200, 2, 2),
])
@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
def test_direct_weight_gradient_of_other_paddings_and_channels(ctx, x, k, pad, steps, dtype):
    yd = [x[0], k, x[2] + 2 * pad - 2, x[3] + 2 * pad - 2]
    xt, dy = whole(k, x, dtype, 2), whole(k + 1, yd, dtype, 1)
    w = [k, x[1], 3, 3]
    geom = ([pad, pad], [1, 1], [1, 1])
    ref = oracle.conv_wgrad(dy.logical(), xt.logical(), w, *geom)
    dw = run_conv_wgrad(ctx, dy, xt, w, *geom, dtype, tuned=None)
    name = ctx.last_kernel()
    big = np.prod(yd) * x[1] >= 1.4e7
    assert name.startswith(f"conv_wgrad_direct steps={steps}" if big else "conv_wgrad_gather"), name
    np.testing.assert_array_equal(dw.logical(), HT.from_logical(ref, dtype).logical())
    # stored in f32: the gathered tiles' shorter chains
    dw = run_conv_wgrad(ctx, dy, xt, w, *geom, dtype, tuned=None, w_dtype=capi.FLOAT)
    assert ctx.last_kernel().startswith("conv_wgrad_gather"), ctx.last_kernel()
    np.testing.assert_array_equal(dw.logical(), ref)


def test_direct_weight_gradient_meets_no_channels_outside(ctx):
    # infinite values in the channel next to a gradient's own, in the same blocks
    x, dy = whole(5, [8, 40, 40, 30], capi.BFLOAT16, 2), whole(6, [8, 72, 40, 30], capi.BFLOAT16, 1)
    xv, w = x.logical().copy(), [72, 40, 3, 3]
    xv[:, 39] = np.inf
    dw = run_conv_wgrad(ctx, dy, HT.from_logical(xv, capi.BFLOAT16, oracle.channels_last_strides([8, 40, 40, 30])), w,
                        [1, 1], [1, 1], [1, 1], capi.BFLOAT16, tuned=None).logical()
    assert ctx.last_kernel().startswith("conv_wgrad_direct"), ctx.last_kernel()
    ref = oracle.conv_wgrad(dy.logical(), x.logical(), w, [1, 1], [1, 1], [1, 1])
    np.testing.assert_array_equal(dw[:, :39], HT.from_logical(ref, capi.BFLOAT16).logical()[:, :39])
    assert not np.isfinite(dw[:, 39]).any()


# Infinite values of X in border rows and columns, a channel for each: the taps that meet them show it and no
# other (DY rows and columns that do not exist are zeros in registers).  Steps of 16 pixels full and not,
# channels in whole blocks of 32 and off them, every padding.
@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("n,p,q,steps", [(60, 17, 14, 1), (16, 40, 30, 2), (20, 27, 32, 2), (12, 36, 45, 3),
                                         (20, 16, 50, 4), (12, 29, 56, 4), (400, 1, 20, 2), (260, 2, 17, 2)])
@pytest.mark.parametrize("c,k", [(40, 72), (64, 32)])
def test_direct_weight_gradient_meets_no_rows_or_columns_outside(ctx, pad, n, p, q, steps, c, k):
    h, w = p + 2 - 2 * pad, q + 2 - 2 * pad
    if h < 1:
        pytest.skip("no rows of X")
    x, dy = whole(n, [n, c, h, w], capi.BFLOAT16, 2), whole(n + 1, [n, k, p, q], capi.BFLOAT16, 1)
    xv = x.logical().copy()
    for i, (axis, at) in enumerate((a, b) for a in (2, 3) for b in (0, 1, 2, -3, -2, -1)):
        if -xv.shape[axis] <= at < xv.shape[axis]:
            np.moveaxis(xv[:, 3 * i], axis - 1, 0)[at] = np.inf
    xt = HT.from_logical(xv, capi.BFLOAT16, oracle.channels_last_strides(xv.shape))
    geom = ([k, c, 3, 3], [pad, pad], [1, 1], [1, 1])
    got = run_conv_wgrad(ctx, dy, xt, *geom, capi.BFLOAT16, tuned=None).logical()
    assert ctx.last_kernel().startswith(f"conv_wgrad_direct steps={steps}"), ctx.last_kernel()
    ref = HT.from_logical(oracle.conv_wgrad(dy.logical(), xt.logical(), *geom), capi.BFLOAT16).logical()
    np.testing.assert_array_equal(np.isfinite(got), np.isfinite(ref))
    assert np.isfinite(ref).any(axis=(0, 2, 3)).sum() > 20  # (and most channels meet none)
    np.testing.assert_array_equal(got[np.isfinite(ref)], ref[np.isfinite(ref)])


# Layers for which more parts would be faster than the descriptor's workspace holds, its own and the gathered
# tiles': all parts lie there all the same (graphs with a workspace each share nothing else).
@pytest.mark.parametrize("x,k,parts", [([45, 448, 21, 1], 320, 1), ([1, 264, 45, 22], 128, 2)])
def test_direct_weight_gradient_stays_in_the_workspace(ctx, x, k, parts):
    xt, dy = whole(k, x, capi.BFLOAT16, 2), whole(k + 1, [x[0], k] + x[2:], capi.BFLOAT16, 1)
    w, geom = [k, x[1], 3, 3], ([1, 1], [1, 1], [1, 1])
    dw = HT.empty(w, capi.BFLOAT16, oracle.channels_last_strides(w))
    d = conv_bwd_desc(xt, dw, dy, *geom)
    need, used = ctx.conv_wgrad_workspace(d), parts * -(-k // 32) * -(-x[1] // 32) * 9 * 1024
    assert need >= used * 4
    space = ctx.to_device(np.full(need // 4, np.nan, np.float32))
    bdy, bx, bdw = dy.upload(ctx), xt.upload(ctx), dw.upload(ctx)
    ctx.conv_wgrad(d, bdy, bx, bdw, space)
    name = ctx.last_kernel()
    assert name.startswith("conv_wgrad_direct") and name.endswith(f"parts={parts}"), name
    assert np.isfinite(space.download(np.float32)[:used]).all()
    ref = HT.from_logical(oracle.conv_wgrad(dy.logical(), xt.logical(), w, *geom), capi.BFLOAT16)
    np.testing.assert_array_equal(dw.fetch(ctx, bdw).logical(), ref.logical())


# Gradients stored in f32 keep the parts that their workspace has room for, however few are faster: fewer parts
# are longer chains of f32 additions.  16-bit gradients take the planner's count.
@pytest.mark.parametrize("x,k,parts,few", [([14, 320, 24, 24], 480, 2, 1), ([14, 64, 14, 14], 192, 28, 5)])
@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16])
def test_direct_weight_gradient_parts_by_type(ctx, x, k, parts, few, dtype):
    xt, dy = whole(k, x, capi.BFLOAT16, 2), whole(k + 1, [x[0], k] + x[2:], capi.BFLOAT16, 1)
    w, geom = [k, x[1], 3, 3], ([1, 1], [1, 1], [1, 1])
    dw = HT.empty(w, dtype, oracle.channels_last_strides(w))
    assert ctx.conv_wgrad_workspace(conv_bwd_desc(xt, dw, dy, *geom)) == parts * (k // 32) * (x[1] // 32) * 36864
    got = run_conv_wgrad(ctx, dy, xt, w, *geom, capi.BFLOAT16, tuned=True, w_dtype=dtype).logical()
    assert ctx.last_kernel().endswith(f" parts={parts if dtype == capi.FLOAT else few}"), ctx.last_kernel()
    # (some blocks of a large one)
    ref = oracle.conv_wgrad(dy.logical()[:, -64:], xt.logical()[:, -64:], [64, 64, 3, 3], *geom)
    np.testing.assert_array_equal(got[-64:, -64:], HT.from_logical(ref, dtype).logical())


# the mirrored filter of a data gradient, copied in blocks of 64 x 64: edges of the blocks, groups, and a
# channel count that the copy takes element by element
@pytest.mark.parametrize("x,k,w", [
    ([4, 64, 13, 12], 8, [3, 3]), ([4, 72, 13, 12], 136, [3, 3]), ([2, 192, 9, 30], 64, [5, 1]),
    ([3, 256, 12, 12], 128, [3, 3]), ([2, 64, 20, 21], 200, [1, 3]), ([2, 64, 20, 21], 100, [3, 3]),
])
@pytest.mark.parametrize("groups", [1, 2])
def test_mirrored_filter(ctx, x, k, w, groups):
    if groups == 2 and (x[1] % 128 or k % 128):
        pytest.skip("groups of whole slices")
    wd = [k, x[1] // groups] + w
    dy = whole(k, [x[0], k] + x[2:], capi.BFLOAT16, 1)
    wt = whole(k + 1, wd, capi.BFLOAT16, 2)
    pad = [(w[0] - 1) // 2, (w[1] - 1) // 2]
    dx = run_conv_dgrad(ctx, dy, wt, x, pad, [1, 1], [1, 1], capi.BFLOAT16, tuned=None)
    ref = oracle.conv_dgrad(dy.logical(), wt.logical(), x, pad, [1, 1], [1, 1])
    np.testing.assert_array_equal(dx.logical(), HT.from_logical(ref, capi.BFLOAT16).logical())
