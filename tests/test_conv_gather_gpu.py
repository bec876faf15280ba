"""Forward convolution and data gradient on unpadded gathered tiles (conv_gather.hip),
through the C ABI vs the oracle: channel counts off 64, output
channels off 8 and off the tiles, strides, dilation, a split reduction, fused chains."""
import numpy as np
import pytest

from fusilli_amd import capi
from oracle import oracle
from helpers import HT, assert_close, rand
from test_generic_ops_gpu import run_conv, run_conv_dgrad

pytestmark = pytest.mark.gpu

CASES = [
    # 48 channels: taps straddle the steps of 64; output channels under one tile
    dict(x=[2, 48, 11, 9], w=[48, 48, 3, 3], pad=[2, 2], s=[1, 1], d=[1, 1]),
    # 8 channels: eight taps a step; output channels no multiple of 8 or 4
    dict(x=[3, 8, 7, 13], w=[37, 8, 3, 3], pad=[1, 1], s=[1, 1], d=[1, 1]),
    # stride and dilation, more than one tile of channels, N a multiple of 4 only
    dict(x=[2, 72, 17, 15], w=[140, 72, 3, 2], pad=[1, 1], s=[2, 1], d=[1, 2]),
    # several tiles of pixels (the last short), channels past one slice
    dict(x=[5, 136, 14, 14], w=[96, 136, 1, 1], pad=[0, 0], s=[1, 1], d=[1, 1]),
    # few pixels, a long reduction (split)
    dict(x=[1, 200, 6, 6], w=[64, 200, 5, 5], pad=[2, 2], s=[1, 1], d=[1, 1]),
    # whole slices too, where forced
    dict(x=[2, 128, 9, 8], w=[72, 128, 3, 3], pad=[1, 1], s=[1, 1], d=[1, 1]),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("forced", [True, False])
def test_conv_gather_vs_oracle(ctx, case, dtype, forced, knobs):
    if forced:
        knobs(CONV_GATHER="1")
    elif case["x"][1] % 64 == 0:
        pytest.skip("covered with the switch")
    lay = oracle.channels_last_strides
    geom = (case["pad"], case["s"], case["d"])
    yd = oracle.conv_output_dims(case["x"], case["w"], *geom)
    x = HT.from_logical(rand(71, 0, case["x"]), dtype, lay(case["x"]))
    w = HT.from_logical(rand(71, 1, case["w"], std=0.1), dtype, lay(case["w"]))
    bias = HT.from_logical(rand(71, 2, [1, case["w"][0], 1, 1]), dtype)
    res = HT.from_logical(rand(71, 3, yd), dtype, lay(yd))
    epi = [capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=bias.desc()),
           capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=res.desc(), operand_index=1),
           capi.epilogue_op(capi.PW["RELU_FWD"], dtype)]
    y = run_conv(ctx, x, w, *geom, capi.FLOAT, out_dtype=dtype, epilogue=epi,
                 epi_tensors=[bias, res], channels_last_out=True)
    name = ctx.last_kernel()
    assert name.startswith("conv_igemm unpadded"), name
    plain = oracle.conv_fprop(x.logical(), w.logical(), *geom)
    assert_close(y.logical(), np.maximum(plain + bias.logical() + res.logical(), 0), dtype,
                 f"fprop {case} {name}")
    y = run_conv(ctx, x, w, *geom, capi.FLOAT, out_dtype=capi.FLOAT, channels_last_out=True)
    assert_close(y.logical(), plain, dtype, f"fprop f32 out {case} {name}")
    if case["w"][0] % 8 == 0:
        dy = HT.from_logical(rand(71, 4, yd), dtype, lay(yd))
        dx = run_conv_dgrad(ctx, dy, w, case["x"], *geom, dtype, tuned=None)
        assert_close(dx.logical(), oracle.conv_dgrad(dy.logical(), w.logical(), case["x"], *geom),
                     dtype, f"dgrad {case} {ctx.last_kernel()}")


@pytest.mark.parametrize("x,w,pad,stride,plain,fused", [  # whether gathered
    ([8, 200, 60, 60], [256, 200, 3, 3], 1, 1, False, False),  # tiles of 256 rows, a long reduction
    ([44, 80, 58, 58], [256, 80, 1, 1], 0, 1, True, False),    # 1 x 1 over very many results
    ([12, 328, 56, 56], [256, 328, 1, 1], 0, 2, True, True),   # strided
    ([18, 224, 46, 46], [144, 224, 3, 3], 1, 1, True, True),   # tiles half empty
    ([11, 16, 64, 64], [560, 16, 3, 3], 1, 2, True, True),     # a short reduction
    ([39, 216, 30, 18], [352, 216, 3, 3], 1, 1, False, False),  # halo tiles, full rounds
    ([32, 136, 28, 28], [256, 136, 3, 3], 1, 1, True, True),
    ([22, 56, 48, 48], [256, 56, 3, 3], 1, 1, False, False),   # halo tiles of 256 rows
    ([27, 40, 36, 36], [384, 40, 3, 3], 1, 1, True, False),    # much padding
    ([11, 472, 48, 48], [128, 472, 3, 3], 1, 1, False, False),  # a split reduction
    ([11, 248, 48, 48], [128, 248, 3, 3], 1, 1, True, True),
])
@pytest.mark.parametrize("relu", [False, True])
def test_padded_copies_where_they_pay(ctx, knobs, x, w, pad, stride, plain, fused, relu):
    # both sides of the rule, and the same sums (of whole numbers: exact in f32) on either route
    gathered = fused if relu else plain
    lay = oracle.channels_last_strides
    xs = HT.from_logical(np.resize(rand(72, 0, [4099], "int", lo=-3, hi=4), x), capi.BFLOAT16, lay(x))
    ws = HT.from_logical(np.resize(rand(72, 1, [4093], "int", lo=-3, hi=4), w), capi.BFLOAT16, lay(w))
    geom = ([pad, pad], [stride, stride], [1, 1])
    epi = [capi.epilogue_op(capi.PW["RELU_FWD"], capi.FLOAT)] if relu else []
    y = run_conv(ctx, xs, ws, *geom, capi.FLOAT, epilogue=epi, channels_last_out=True).logical()
    assert ("unpadded" in ctx.last_kernel()) == gathered, ctx.last_kernel()
    knobs(CONV_GATHER=0 if gathered else 1)
    z = run_conv(ctx, xs, ws, *geom, capi.FLOAT, epilogue=epi, channels_last_out=True).logical()
    assert ("unpadded" in ctx.last_kernel()) != gathered, ctx.last_kernel()
    assert np.array_equal(y, z)


@pytest.mark.parametrize("relu", [False, True])
def test_narrow_layers_by_tiles_and_fused_operations(ctx, relu):
    # 64 output channels at most: gathered below 128 tiles of 128 rows, without fused
    # operations below 192
    for n, gathered in ((12, True), (16, not relu), (25, False)):  # 96, 128, 200 tiles
        x = HT.from_logical(np.resize(rand(73, 0, [4099]), [n, 64, 32, 32]), capi.BFLOAT16,
                            oracle.channels_last_strides([n, 64, 32, 32]))
        w = HT.from_logical(rand(73, 1, [32, 64, 3, 3], std=0.05), capi.BFLOAT16,
                            oracle.channels_last_strides([32, 64, 3, 3]))
        epi = [capi.epilogue_op(capi.PW["RELU_FWD"], capi.BFLOAT16)] if relu else []
        y = run_conv(ctx, x, w, [1, 1], [1, 1], [1, 1], capi.BFLOAT16, epilogue=epi, channels_last_out=True).logical()
        assert ("unpadded" in ctx.last_kernel()) == gathered, (n, ctx.last_kernel())
        ref = oracle.conv_fprop(x.logical()[:1], w.logical(), [1, 1], [1, 1], [1, 1])
        assert_close(y[:1], np.maximum(ref, 0) if relu else ref, capi.BFLOAT16)
