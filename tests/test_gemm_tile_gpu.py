"""Products whose K ends inside a 128-byte slice, whose rows start on any element or whose tiles
are few: the register-staged LDS tiles (gemm_tile_kernel.h) and the tiled GEMM's cut slices,
against the oracle."""
import numpy as np
import pytest

from fusilli_amd import capi
from helpers import HT, assert_close, rand
from oracle import oracle
from test_gemm_mfma_gpu import make_operand, ref_matmul

pytestmark = pytest.mark.gpu
BYTES = [capi.INT8, capi.FP8E4M3, capi.FP8E5M2]
DTYPES = [capi.BFLOAT16, capi.HALF] + BYTES


def run(ctx, a, b, epilogue=(), epi_tensors=()):
    i8 = a.dtype == capi.INT8
    cdt, odt = (capi.INT32, capi.INT32) if i8 else (capi.FLOAT, capi.HALF if a.dtype == capi.HALF else capi.BFLOAT16)
    dims = a.dims[:-2] + [a.dims[-2], b.dims[-1]]
    out = HT.empty(dims, odt)
    d = capi.MatmulDesc()
    d.a, d.b, d.out, d.out_dtype = a.desc(), b.desc(), out.desc(), odt
    d.c = capi.TensorDesc.make(dims, out.strides, cdt)
    d.epilogue = capi.make_epilogue(list(epilogue))
    bufs = [t.upload(ctx) for t in epi_tensors]
    da, db, do = a.upload(ctx), b.upload(ctx), out.upload(ctx)
    ctx.matmul(d, da, db, do, epilogue_operands=bufs)
    return out.fetch(ctx, do).logical(), ctx.last_kernel(), odt


def check(got, ref, odt, what):
    if odt == capi.INT32:
        assert np.array_equal(got, ref), what
    else:
        # one rounding to the result's type over f32 sums: half a unit in the last place, and as
        # much again where the sum's own error crosses a rounding boundary
        ulp = 2.0 ** -8 if odt == capi.BFLOAT16 else 2.0 ** -11
        rms = np.sqrt(np.mean(np.square(ref)))
        assert np.all(np.abs(got - ref) <= 1.01 * ulp * np.abs(ref) + 1e-4 * rms), what


# tile rows and columns, remainders on either side, one slice and a cut one, K odd
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(640, 1089, 2051), (705, 705, 3001), (1153, 641, 1999), (1025, 1027, 1033)])
def test_tiles_of_64(ctx, dtype, ta, tb, m, n, k):
    a, b = make_operand(81, 0, m, k, dtype, ta), make_operand(81, 1, k, n, dtype, tb)
    got, name, odt = run(ctx, a, b)
    check(got, ref_matmul(a, b), odt, name)
    assert name.startswith("gemm_mfma") and "x64 " in name, name


@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.FP8E4M3, capi.INT8])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(1299, 1930, 777), (2049, 1282, 1001)])
def test_wide_tiles(ctx, dtype, ta, tb, m, n, k):
    a, b = make_operand(82, 0, m, k, dtype, ta), make_operand(82, 1, k, n, dtype, tb)
    got, name, odt = run(ctx, a, b)
    check(got, ref_matmul(a, b), odt, name)
    assert name.startswith("gemm_mfma") and "128x128 waves=4" in name, name


# 64 x 128 and 128 x 64 tiles, whole and in parts
HALF_WIDE = [
    (capi.BFLOAT16, 1059, 1928, 623, False, False, "64x128 waves=4 split=1"),
    (capi.HALF, 1944, 1098, 692, False, True, "64x128 waves=4 split=1"),
    (capi.BFLOAT16, 1581, 1217, 258, True, False, "64x128 waves=4 split=1"),
    (capi.HALF, 1311, 1705, 264, True, True, "64x128 waves=4 split=1"),
    (capi.BFLOAT16, 910, 352, 4928, False, False, "64x128 waves=4 split=5"),
    (capi.BFLOAT16, 225, 2051, 4303, True, False, "64x128 waves=4 split=3"),
    (capi.HALF, 193, 2252, 4521, True, True, "64x128 waves=4 split=3"),
    (capi.FP8E4M3, 816, 2320, 1248, True, True, "64x128 waves=4 split=1"),
    (capi.FP8E5M2, 1155, 1623, 426, False, True, "64x128 waves=4 split=1"),
    (capi.INT8, 824, 2329, 285, True, False, "64x128 waves=4 split=1"),
    (capi.BFLOAT16, 1399, 1572, 273, True, True, "128x64 waves=4 split=1"),
    (capi.HALF, 1626, 300, 4271, True, False, "128x64 waves=4 split=3"),
    (capi.BFLOAT16, 464, 1072, 4368, False, True, "128x64 waves=4 split=3"),
    (capi.FP8E4M3, 847, 1534, 350, False, False, "128x64 waves=4 split=1"),
    (capi.INT8, 466, 2978, 208, True, True, "128x64 waves=4 split=1"),
]


@pytest.mark.parametrize("dtype,m,n,k,ta,tb,route", HALF_WIDE)
def test_half_wide_tiles(ctx, dtype, m, n, k, ta, tb, route):
    a, b = make_operand(86, 0, m, k, dtype, ta), make_operand(86, 1, k, n, dtype, tb)
    got, name, odt = run(ctx, a, b)
    assert name.endswith(route), name
    check(got, ref_matmul(a, b), odt, name)


# whole 16-byte chunks of K, and any K where neither operand lies along it: the tiled GEMM (its
# other tiles and split reductions: test_cut_slice_after_garbage), but for the last row, whose few
# tiles are staged
@pytest.mark.parametrize("dtype,k16", [(capi.BFLOAT16, 8), (capi.HALF, 8), (capi.INT8, 16), (capi.FP8E5M2, 16)])
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,slices,rest", [(3072, 2064, 8, 1), (2064, 2064, 7, 7), (2576, 2592, 3, 3), (256, 4096, 33, 5)])
def test_cut_slices(ctx, dtype, k16, ta, tb, m, n, slices, rest):
    k = slices * 8 * k16 + rest * k16 + (3 if ta and not tb else 0)
    a, b = make_operand(83, 0, m, k, dtype, ta), make_operand(83, 1, k, n, dtype, tb)
    got, name, odt = run(ctx, a, b)
    assert name.endswith("256x128 waves=8 split=1" if m > 256 else "64x64 waves=8 split=1"), name
    check(got, ref_matmul(a, b), odt, name)


# one whole slice of K: the tiled GEMM, also in batches (the direct kernels take up to seven times as long)
@pytest.mark.parametrize("dtype,m,n,k,batch", [
    (capi.BFLOAT16, 1536, 448, 64, 4), (capi.HALF, 2048, 1160, 64, 1), (capi.FP8E4M3, 640, 2240, 128, 1),
    (capi.INT8, 256, 400, 128, 3)])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
def test_one_whole_slice(ctx, dtype, m, n, k, batch, ta, tb):
    of = batch if batch > 1 else None
    a, b = make_operand(90, 0, m, k, dtype, ta, batch=of), make_operand(90, 1, k, n, dtype, tb, batch=of)
    got, name, odt = run(ctx, a, b)
    assert name.startswith("gemm_mfma") and name.endswith("waves=8 split=1"), name
    check(got, ref_matmul(a, b), odt, name)


# every tile of the tiled GEMM, operands along M / N (whole K-rows are masked) and along K, split
# reductions whose last part is the shorter one, a slice of a few values
CUT = [
    (capi.HALF, 601, 4736, 808, False, False, "128x128 waves=8 split=1"),
    (capi.BFLOAT16, 4104, 4104, 75, True, False, "128x128 waves=8 split=1"),
    (capi.FP8E4M3, 2576, 2592, 4000, True, True, "256x128 waves=8 split=1"),
    (capi.BFLOAT16, 4096, 4096, 72, True, False, "256x256 waves=8 split=1"),
    (capi.HALF, 6936, 2240, 592, True, True, "256x256 waves=8 split=1"),
    (capi.FP8E4M3, 4096, 4096, 131, True, False, "256x256 waves=8 split=1"),
    (capi.FP8E4M3, 6936, 2240, 1168, False, False, "256x256 waves=8 split=1"),
    (capi.INT8, 6936, 2240, 1168, False, True, "256x256 waves=8 split=1"),
    (capi.BFLOAT16, 232, 2232, 5664, True, True, "128x128 waves=8 split=6"),
    (capi.BFLOAT16, 1059, 1152, 5744, False, False, "128x128 waves=8 split=3"),
    (capi.INT8, 1248, 800, 8752, True, True, "128x128 waves=8 split=3"),
]


@pytest.mark.parametrize("dtype,m,n,k,ta,tb,route", CUT)
def test_cut_slice_after_garbage(ctx, dtype, m, n, k, ta, tb, route):
    # What a masked part of the last slice holds in LDS must not reach the sums: the same product
    # of NaNs (127 in int8) has just left its operands there.
    a, b = make_operand(87, 0, m, k, dtype, ta), make_operand(87, 1, k, n, dtype, tb)
    full = 127 if dtype == capi.INT8 else np.nan
    fill = [HT.from_logical(np.full(t.dims, full), dtype, t.strides) for t in (a, b)]
    run(ctx, *fill)
    got, name, odt = run(ctx, a, b)
    assert name.endswith(route), name
    check(got, ref_matmul(a, b), odt, name)


@pytest.mark.parametrize("dtype,m,n,k", [
    (capi.FP8E5M2, 1024, 512, 13), (capi.FP8E4M3, 256, 272, 15), (capi.BFLOAT16, 512, 512, 7), (capi.HALF, 264, 1040, 3)])
def test_few_values_of_k_into_f32(ctx, dtype, m, n, k):
    # exact products and an f32 sum: each addition may be off by half a unit of its partial sum
    a, b = make_operand(89, 0, m, k, dtype, True), make_operand(89, 1, k, n, dtype, False)
    out = HT.empty([m, n], capi.FLOAT)
    d = capi.MatmulDesc()
    d.a, d.b, d.out, d.out_dtype = a.desc(), b.desc(), out.desc(), capi.FLOAT
    d.c = capi.TensorDesc.make([m, n], out.strides, capi.FLOAT)
    d.epilogue = capi.make_epilogue([])
    da, db, do = a.upload(ctx), b.upload(ctx), out.upload(ctx)
    ctx.matmul(d, da, db, do)
    got, size = out.fetch(ctx, do).logical(), np.abs(a.logical()) @ np.abs(b.logical())
    assert np.all(np.abs(got - ref_matmul(a, b)) <= k * 2.0 ** -24 * size), ctx.last_kernel()


@pytest.mark.parametrize("m,n,k,ta,tb", [(4096, 4096, 72, True, False), (601, 4736, 808, False, False)])
def test_infinities_in_front_of_a_cut(ctx, m, n, k, ta, tb):
    # the last row of K is fetched again in place of those behind it: neither operand's may count
    a, b = make_operand(88, 0, m, k, capi.BFLOAT16, ta), make_operand(88, 1, k, n, capi.BFLOAT16, tb)
    av, bv = a.logical(), b.logical()
    av[5, k - 1], bv[k - 1, 7] = np.inf, -np.inf
    a = HT.from_logical(av, capi.BFLOAT16, a.strides)
    b = HT.from_logical(bv, capi.BFLOAT16, b.strides)
    got, name, _ = run(ctx, a, b)
    ref = ref_matmul(a, b)
    assert "waves=8 split=1" in name, name
    assert np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref)), name
    finite = np.isfinite(ref)
    assert_close(got[finite], ref[finite], capi.BFLOAT16, name)


@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("m,n,k,batch,route", [
    # the direct kernels
    (130, 250, 1003, 1, "gemm_direct 16x16"), (140, 140, 6001, 1, "split=4"), (90, 200, 700, 5, "gemm_direct"),
    # staged tiles of every size, whole, in parts, of a batch
    (700, 1300, 1500, 1, "64x64 waves=8 split=1"), (576, 2402, 263, 1, "64x64 waves=4 split=1"),
    (205, 216, 3456, 1, "64x64 waves=4 split=11"), (1368, 69, 4977, 1, "64x64 waves=8 split=5"),
    (354, 589, 273, 3, "64x64 waves=8 split=1"), (77, 400, 5771, 3, "64x64 waves=8 split=6"),
    (778, 2381, 446, 1, "64x128 waves=4 split=1"), (267, 610, 4957, 3, "64x128 waves=4 split=3"),
    (330, 1138, 339, 5, "128x64 waves=4 split=1"), (207, 1430, 5666, 1, "128x64 waves=4 split=5"),
    (1212, 883, 241, 3, "128x128 waves=4 split=1"), (866, 1248, 2483, 1, "128x128 waves=4 split=3")])
def test_fused_chains(ctx, dtype, m, n, k, batch, route):
    # a column operand alone (requested early), and with a full one
    lead = [batch] if batch > 1 else []
    a = make_operand(84, 0, m, k, dtype, False, batch=batch if batch > 1 else None)
    b = make_operand(84, 1, k, n, dtype, True, batch=batch if batch > 1 else None)
    bias = HT.from_logical(rand(84, 2, [1] * (len(lead) + 1) + [n]), dtype)
    full = HT.from_logical(rand(84, 3, lead + [m, n]), capi.FLOAT)
    product = ref_matmul(a, b)
    add = capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=bias.desc(), operand_index=0)
    mul = capi.epilogue_op(capi.PW["MUL"], dtype, operand=full.desc(), operand_index=1)
    scale = capi.epilogue_op(capi.PW["MUL"], capi.FLOAT, scalar=0.25)
    gelu = capi.epilogue_op(capi.PW["GELU_FWD"], dtype)
    for ops, tensors, ref in (
            ([add, gelu], [bias], oracle.pointwise(capi.PW["GELU_FWD"], [product + bias.logical()])),
            ([scale, add, mul], [bias, full], (0.25 * product + bias.logical()) * full.logical())):
        got, name, odt = run(ctx, a, b, ops, tensors)
        assert route in name, name
        assert_close(got, ref, dtype, name)


@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("m,n,k", [
    (777, 1400, 1000),  # sixteen columns a thread, the last run of eight
    (700, 1301, 1500),  # ... of five
    (520, 520, 4001),   # split: four columns
    (1299, 1930, 777),  # wide tiles
])
def test_chains_of_four(ctx, dtype, m, n, k):
    # 2 - (swish_0.7(0.25 x) - bias): a scalar in front, a unary with a parameter, the accumulator
    # as the second operand of a scalar and the first of a column's, roundings between
    a, b = make_operand(85, 0, m, k, dtype, False), make_operand(85, 1, k, n, dtype, True)
    bias = HT.from_logical(rand(85, 2, [1, n]), capi.FLOAT)
    swish = capi.PointwiseParams.default()
    swish.swish_beta = 0.7
    ops = [capi.epilogue_op(capi.PW["MUL"], capi.FLOAT, scalar=0.25),
           capi.epilogue_op(capi.PW["SWISH_FWD"], dtype, params=swish),
           capi.epilogue_op(capi.PW["SUB"], capi.FLOAT, operand=bias.desc()),
           capi.epilogue_op(capi.PW["SUB"], dtype, scalar=2.0, acc_is_in1=True)]
    got, name, odt = run(ctx, a, b, ops, [bias])
    assert name.startswith("gemm_mfma") and "waves=" in name, name
    x = 0.25 * ref_matmul(a, b)
    act = oracle.pointwise(capi.PW["SWISH_FWD"], [x], swish_beta=0.7)
    assert_close(got, 2.0 - (act - bias.logical()), dtype, name)


# 257 to 512 tiles of 128 x 128 in place of 256 x 128 ones; flat results, cut slices and row-major bytes
# stay on those
@pytest.mark.parametrize("dtype,m,n,k,tb,tile", [
    (capi.BFLOAT16, 2176, 1984, 1216, False, "128x128"), (capi.HALF, 3177, 1920, 896, True, "128x128"),
    (capi.FP8E4M3, 3328, 1792, 2432, True, "128x128"), (capi.INT8, 1728, 2656, 2560, True, "128x128"),
    (capi.INT8, 569, 7296, 2304, True, "256x128"), (capi.BFLOAT16, 1264, 4928, 2608, True, "256x128"),
    (capi.FP8E4M3, 832, 5520, 1792, False, "256x128"),
])
def test_tiles_in_pairs(ctx, dtype, m, n, k, tb, tile):
    a, b = make_operand(87, 0, m, k, dtype, False), make_operand(87, 1, k, n, dtype, tb)
    got, name, odt = run(ctx, a, b)
    assert name.endswith(f"{tile} waves=8 split=1"), name
    check(got, ref_matmul(a, b), odt, name)
