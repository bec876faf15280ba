"""Direct matrix-product kernels (fragments straight from global memory) vs the
oracle, at the sizes where they can go wrong: one row, tile edges, K tails of
every length class, rows that start on odd elements, batches, split K."""
import math

import numpy as np
import pytest

from fusilli_amd import capi
from oracle import oracle
from helpers import HT, assert_close, rand
from test_gemm_mfma_gpu import make_operand, ref_matmul

pytestmark = pytest.mark.gpu

DTYPES = [capi.FLOAT, capi.BFLOAT16, capi.HALF, capi.INT8, capi.FP8E4M3, capi.FP8E5M2]


def run(ctx, a, b, c_dtype, out_dtype=None, epilogue=(), epi_tensors=()):
    out_dtype = c_dtype if out_dtype is None else out_dtype
    cdims = list(np.broadcast_shapes(tuple(a.dims[:-2]), tuple(b.dims[:-2]))) + [a.dims[-2], b.dims[-1]]
    out = HT.empty(cdims, out_dtype)
    d = capi.MatmulDesc()
    d.a, d.b = a.desc(), b.desc()
    d.c = capi.TensorDesc.make(cdims, out.strides, c_dtype)
    d.out, d.out_dtype = out.desc(), out_dtype
    d.epilogue = capi.make_epilogue(list(epilogue))
    assert ctx.lib.fhip_matmul_supported(d) == 1
    bufs = [t.upload(ctx) for t in epi_tensors]
    da, db, do = a.upload(ctx), b.upload(ctx), out.upload(ctx)
    ctx.matmul(d, da, db, do, epilogue_operands=bufs)
    name = ctx.last_kernel()
    assert name.startswith("gemm_direct"), name
    return out.fetch(ctx, do), name


def check(got, ref, dtype):
    if dtype == capi.INT8:
        assert np.array_equal(got, ref)
    else:
        assert_close(got, ref, capi.FLOAT, rtol=1e-4)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [
    (1, 40, 16),      # one row, the shortest K of 8-bit types
    (16, 16, 128),    # exactly one tile, whole steps
    (7, 37, 131),     # tails of K and N, odd row pitches
    (17, 65, 77),     # two row tiles
    (33, 66, 300),    # four row tiles, a second tile with one row
    (130, 70, 1029),  # several tiles, K split over four wavefronts
])
def test_direct_orientations_and_edges(ctx, dtype, ta, tb, m, n, k):
    a = make_operand(90, 0, m, k, dtype, ta)
    b = make_operand(90, 1, k, n, dtype, tb)
    out, _ = run(ctx, a, b, capi.INT32 if dtype == capi.INT8 else capi.FLOAT)
    check(out.logical(), ref_matmul(a, b), dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tb", [False, True])
@pytest.mark.parametrize("m", [3, 20, 50])
def test_direct_split_k(ctx, dtype, tb, m):
    # few tiles over a long K: parts on workgroups of their own, added in order
    k = (24704 if capi.DTYPE_SIZE[dtype] > 1 else 49408) + 8
    a = make_operand(91, 0, m, k, dtype, False)
    b = make_operand(91, 1, k, 34, dtype, tb)
    out, name = run(ctx, a, b, capi.INT32 if dtype == capi.INT8 else capi.FLOAT)
    assert "split=" in name and not name.endswith("split=1"), name
    check(out.logical(), ref_matmul(a, b), dtype)


@pytest.mark.parametrize("dtype,ta,tb,m,n,batch,tiled,direct", [
    (capi.FLOAT, False, False, 600, 1100, 1, [9, 128, 149], [150]),   # 180 tiles
    (capi.FLOAT, True, False, 33, 65, 100, [9, 64, 129], [130, 160]),  # 200, a second one for a row and a column
    (capi.FLOAT, False, True, 1500, 1450, 1, [9, 64, 112, 152], [96, 113, 153]),  # 552, both K-contiguous
    (capi.FLOAT, True, False, 1500, 1450, 1, [64, 84], [85, 96, 129]),
    (capi.FLOAT, False, True, 700, 900, 1, [9, 16], [17]),
    (capi.HALF, False, False, 1100, 1200, 1, [9, 23], [24]),
    (capi.BFLOAT16, True, True, 1100, 1200, 1, [9, 49], [50]),
    (capi.HALF, False, True, 600, 1100, 1, [9, 33], [34]),
])
def test_short_k_takes_the_f32_tiles(ctx, dtype, ta, tb, m, n, batch, tiled, direct):
    # both sides of the rule's lines, whole slices of 32 and cut ones
    for k in tiled + direct:
        a = make_operand(96, 0, m, k, dtype, ta, batch=batch if batch > 1 else None)
        b = make_operand(96, 1, k, n, dtype, tb, batch=1 if batch > 1 else None)
        out = HT.empty(([batch] if batch > 1 else []) + [m, n], dtype)
        d = capi.MatmulDesc()
        d.a, d.b, d.c, d.out, d.out_dtype = a.desc(), b.desc(), out.desc(), out.desc(), dtype
        d.c.dtype = capi.FLOAT
        d.epilogue = capi.make_epilogue([])
        da, db, do = a.upload(ctx), b.upload(ctx), out.upload(ctx)
        ctx.matmul(d, da, db, do)
        name = ctx.last_kernel()
        assert name.startswith("gemm_direct" if k in direct else "matmul_f32_tiled"), (k, name)
        got, ref = out.fetch(ctx, do).logical(), ref_matmul(a, b)
        check(got, ref, dtype) if dtype == capi.FLOAT else assert_close(got, ref, dtype)
        if dtype == capi.FLOAT:
            # Steps of 16 products and their sums are chains of their own: n additions round n
            # times sums of half the result's size on average by 2^-24 / sqrt(12) of it, 0.41
            # sqrt(n) 2^-24 together; 16 + 10 here (one chain of 152: 3.7 measured)
            exact = a.logical().astype(np.float64) @ b.logical().astype(np.float64)
            assert np.linalg.norm(got - exact) <= 0.41 * 26 ** 0.5 * 2.0 ** -24 * np.linalg.norm(exact), k


@pytest.mark.parametrize("dtype", [capi.HALF, capi.BFLOAT16])
def test_16_bit_operands_into_f32_keep_the_direct_kernel(ctx, dtype):
    # (the f32 tiles' chains would show in the result)
    a, b = make_operand(97, 0, 1100, 17, dtype, True), make_operand(97, 1, 17, 1200, dtype, True)
    out, _ = run(ctx, a, b, capi.FLOAT)
    exact = a.logical().astype(np.float64) @ b.logical().astype(np.float64)
    assert np.linalg.norm(out.logical() - exact) <= 2.0 ** -24 * np.linalg.norm(exact)


@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.HALF, capi.INT8])
def test_direct_batched(ctx, dtype):
    a = make_operand(92, 0, 19, 45, dtype, False, batch=3)
    cdt = capi.INT32 if dtype == capi.INT8 else capi.FLOAT
    for batch in (3, 1):
        b = make_operand(92, 1, 45, 33, dtype, False, batch=batch)
        out, _ = run(ctx, a, b, cdt)
        check(out.logical(), ref_matmul(a, b), dtype)


@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16, capi.FP8E4M3])
@pytest.mark.parametrize("m,k", [(5, 90), (60, 90), (5, 49000)])
def test_direct_epilogue(ctx, dtype, m, k):
    # a row vector, a full operand and a unary step, also behind a split K
    a = make_operand(93, 0, m, k, dtype, False)
    b = make_operand(93, 1, k, 41, dtype, True)
    bias = HT.from_logical(rand(93, 2, [1, 41]), capi.BFLOAT16)
    full = HT.from_logical(rand(93, 3, [m, 41]), capi.FLOAT)
    epi = [capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=bias.desc(), operand_index=0),
           capi.epilogue_op(capi.PW["MUL"], capi.FLOAT, operand=full.desc(), operand_index=1),
           capi.epilogue_op(capi.PW["GELU_FWD"], capi.BFLOAT16)]
    out, _ = run(ctx, a, b, capi.FLOAT, out_dtype=capi.BFLOAT16, epilogue=epi, epi_tensors=[bias, full])
    ref = (ref_matmul(a, b) + bias.logical()) * full.logical()
    assert_close(out.logical(), oracle.pointwise(capi.PW["GELU_FWD"], [ref]), capi.BFLOAT16)


@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
def test_direct_gelu_of_infinities(ctx, dtype):
    a = make_operand(94, 0, 20, 64, dtype, False)
    b = make_operand(94, 1, 64, 40, dtype, True)
    v = np.zeros([1, 40], np.float32)
    v[0, 3], v[0, 9] = np.inf, np.nan
    bias = HT.from_logical(v, dtype)
    epi = [capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=bias.desc(), operand_index=0),
           capi.epilogue_op(capi.PW["GELU_FWD"], dtype)]
    out, _ = run(ctx, a, b, capi.FLOAT, out_dtype=dtype, epilogue=epi, epi_tensors=[bias])
    got = out.logical()
    assert (got[:, 3] == np.inf).all() and np.isnan(got[:, 9]).all()
    assert np.isfinite(np.delete(got, [3, 9], axis=1)).all()


@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("fused", [True, False])
def test_gelu_rounds_once(ctx, dtype, fused):
    # every value of the type from -13 to 13, as the bias of an empty product or as the input
    # of the pointwise operation: half a unit in the last place is the result's own rounding,
    # 0.01 what the function and the hardware's exp2 and reciprocal add (measured 0.003)
    bits = np.arange(1 << 16, dtype=np.uint16)
    v = oracle.dequantize(bits.view(oracle.storage_dtype(dtype)), dtype)
    x = v[np.isfinite(v) & (np.abs(v) <= 13)]
    x = x[:len(x) // 8 * 8].astype(np.float64).reshape(1, -1)
    t = HT.from_logical(x, dtype)
    if fused:
        a = make_operand(95, 0, 1, 16, dtype, False)
        b = HT.from_logical(np.zeros([16, x.size]), dtype)
        epi = [capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=t.desc(), operand_index=0),
               capi.epilogue_op(capi.PW["GELU_FWD"], dtype)]
        got = run(ctx, a, b, capi.FLOAT, out_dtype=dtype, epilogue=epi, epi_tensors=[t])[0].logical()
    else:
        out = HT.empty([1, x.size], dtype)
        d = capi.PointwiseDesc()
        d.mode, d.num_inputs, d.params = capi.PW["GELU_FWD"], 1, capi.PointwiseParams.default()
        d.in_[0], d.out = t.desc(), out.desc()
        bi, bo = t.upload(ctx), out.upload(ctx)
        ctx.pointwise(d, bi, None, None, bo)
        assert ctx.last_kernel().startswith("pointwise_fast"), ctx.last_kernel()
        got = out.fetch(ctx, bo).logical()
    exact = np.array([0.5 * e * math.erfc(-e / math.sqrt(2)) for e in x.ravel()]).reshape(x.shape)
    digits, least = (10, -14) if dtype == capi.HALF else (7, -126)
    size = np.where(exact == 0, 1e-300, np.abs(exact))
    ulp = np.exp2(np.maximum(np.floor(np.log2(size)), least) - digits)
    worst = np.abs(got - exact) / ulp
    assert worst.max() <= 0.51, (float(worst.max()), float(x.ravel()[worst.argmax()]))
