"""Row-reduction kernel (trailing dims of a dense tensor) through the C ABI vs
the oracle; every case asserts that the tuned kernel is the one chosen."""
import numpy as np
import pytest

from fusilli_amd import capi
from oracle import oracle
from helpers import HT, assert_close, rand

pytestmark = pytest.mark.gpu

MODES = ["ADD", "SUM", "MUL", "MIN", "MAX", "AMAX", "AVG", "NORM1", "NORM2",
         "MUL_NO_ZEROS"]


def run(ctx, x, odims, mode, y_dtype=None, expect_tuned=True):
    y = HT.empty(odims, x.dtype if y_dtype is None else y_dtype)
    d = capi.ReduceDesc()
    d.x, d.y, d.mode = x.desc(), y.desc(), capi.RED[mode]
    assert ctx.lib.fhip_reduce_supported(d) == (2 if expect_tuned else 1)
    dx, dy = x.upload(ctx), y.upload(ctx)
    ctx.reduce(d, dx, dy)
    return y.fetch(ctx, dy)


def make_x(seed, dims, dtype, mode):
    if mode in ("MUL", "MUL_NO_ZEROS"):
        v = 1.0 + 0.02 * rand(seed, 0, dims)  # products stay in range
        if mode == "MUL_NO_ZEROS":
            v.reshape(-1)[::7] = 0.0
    else:
        v = rand(seed, 0, dims)
    return HT.from_logical(v, dtype)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("dims,odims", [
    ([2, 16, 8, 8], [2, 16, 1, 1]),      # the reference sample's shape: 64-element rows
    ([37, 1000], [37, 1]),               # one wavefront per row, ragged chunk count
    ([5, 3, 4096], [5, 3, 1]),           # one workgroup per row
    ([3, 1, 6000, 8], [3, 1, 1, 1]),     # long rows, odd number of chunk pairs
])
def test_reduce_rows_vs_oracle(ctx, mode, dtype, dims, odims):
    x = make_x(61, dims, dtype, mode)
    out = run(ctx, x, odims, mode, y_dtype=capi.FLOAT)
    ref = oracle.reduction(x.logical(), odims, capi.RED[mode])
    rtol = 1e-4 if dtype == capi.FLOAT else 2e-2
    assert_close(out.logical(), ref, capi.FLOAT, f"{mode} {dims}", rtol=rtol)


def test_reduce_reference_table_known_answers(ctx):
    # samples/reduction/reduction_ops.cpp: inputs i % 100 - 50 on [2,16,8,8]
    dims, odims = [2, 16, 8, 8], [2, 16, 1, 1]
    vals = (np.arange(int(np.prod(dims))) % 100 - 50).astype(np.float64).reshape(dims)
    x = HT.from_logical(vals, capi.FLOAT)
    g = vals.reshape(2, 16, 64)
    assert np.array_equal(run(ctx, x, odims, "SUM").logical().reshape(2, 16), g.sum(2))
    assert np.array_equal(run(ctx, x, odims, "MIN").logical().reshape(2, 16), g.min(2))
    assert np.array_equal(run(ctx, x, odims, "AMAX").logical().reshape(2, 16), np.abs(g).max(2))
    assert np.array_equal(run(ctx, x, odims, "NORM1").logical().reshape(2, 16), np.abs(g).sum(2))


def test_reduce_output_rounding_and_bf16_store(ctx):
    x = make_x(62, [64, 512], capi.BFLOAT16, "SUM")
    out = run(ctx, x, [64, 1], "SUM")  # bf16 result
    ref = oracle.reduction(x.logical(), [64, 1], capi.RED["SUM"])
    assert_close(out.logical(), ref, capi.BFLOAT16)


def test_reduce_not_chosen_outside_contract(ctx):
    # leading-dim reduction and int32 input keep the generic kernel
    x = make_x(63, [16, 64], capi.FLOAT, "SUM")
    out = run(ctx, x, [1, 64], "SUM", expect_tuned=False)
    assert_close(out.logical(), oracle.reduction(x.logical(), [1, 64], capi.RED["SUM"]),
                 capi.FLOAT)
    xi = HT.from_logical(np.arange(128).reshape(2, 64) - 60, capi.INT32)
    out = run(ctx, xi, [2, 1], "MAX", expect_tuned=False)
    assert np.array_equal(out.logical().reshape(-1), [3, 67])


def test_reduce_headline_size(ctx):
    # [8192, 4096] bf16 row sums and row maxima of |x| at full size
    x = make_x(64, [8192, 4096], capi.BFLOAT16, "SUM")
    xl = x.logical()
    out = run(ctx, x, [8192, 1], "SUM", y_dtype=capi.FLOAT).logical()
    assert_close(out, xl.sum(1, keepdims=True), capi.FLOAT, rtol=1e-4)
    out = run(ctx, x, [8192, 1], "AMAX", y_dtype=capi.FLOAT).logical()
    assert np.array_equal(out, np.abs(xl).max(1, keepdims=True))


@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("mode", ["MIN", "MAX", "AMAX"])
def test_reduce_min_max_propagate_nan_and_inf(ctx, mode, dtype):
    # aten.amin / amax semantics: a NaN anywhere in the row gives NaN; an
    # infinity is an ordinary extreme value
    v = rand(65, 0, [6, 640])
    v[1, 17] = np.nan
    v[2, 600] = -np.inf
    v[3, 5] = np.inf
    out = run(ctx, HT.from_logical(v, dtype), [6, 1], mode, y_dtype=capi.FLOAT).logical().reshape(-1)
    assert np.isnan(out[1]) and not np.isnan(out[[0, 2, 3, 4, 5]]).any()
    assert out[2] == (-np.inf if mode == "MIN" else np.inf if mode == "AMAX" else out[2])
    assert out[3] == (np.inf if mode in ("MAX", "AMAX") else out[3])


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("dims,odims,channels_last", [
    ([4, 40, 9, 7], [1, 40, 1, 1], True),    # columns in 16-byte vectors, one slice
    ([16, 128, 20, 20], [1, 128, 1, 1], True),  # several slices
    ([3, 13, 11, 5], [1, 13, 1, 1], True),   # odd channel count: element loads
    ([6000, 70], [1, 70], False),            # column sums of a matrix
    ([5, 3, 8, 8], [1, 3, 1, 1], False),     # channels first, whole vectors per run
    ([50, 4, 30, 31], [1, 4, 1, 1], False),  # runs of odd length, several slices
    ([7, 600, 2], [1, 600, 1], False),       # short runs
    ([3, 5], [1, 1], False),                 # everything, no whole vector
])
def test_reduce_in_front_of_kept_dims_vs_oracle(ctx, mode, dtype, dims, odims, channels_last):
    x = make_x(66, dims, dtype, mode)
    y = HT.empty(odims, capi.FLOAT)
    if channels_last:
        x = HT.from_logical(x.logical(), dtype, oracle.channels_last_strides(dims))
        y = HT.empty(odims, capi.FLOAT, oracle.channels_last_strides(odims))
    d = capi.ReduceDesc()
    d.x, d.y, d.mode = x.desc(), y.desc(), capi.RED[mode]
    dx, dy = x.upload(ctx), y.upload(ctx)
    ctx.reduce(d, dx, dy)
    assert ctx.last_kernel().startswith(("reduce_cols", "reduce_mid")), ctx.last_kernel()
    got = y.fetch(ctx, dy).logical()
    ref = oracle.reduction(x.logical(), odims, capi.RED[mode])
    rtol = 1e-4 if dtype == capi.FLOAT else 2e-2
    assert_close(got, ref, capi.FLOAT, f"{mode} {dims}", rtol=rtol)


@pytest.mark.parametrize("mode", ["MIN", "MAX", "AMAX"])
def test_reduce_columns_propagate_nan(ctx, mode):
    v = rand(67, 0, [700, 24])
    v[33, 5], v[650, 11], v[2, 17] = np.nan, -np.inf, np.inf
    out = run(ctx, HT.from_logical(v, capi.BFLOAT16), [1, 24], mode, y_dtype=capi.FLOAT,
              expect_tuned=False).logical().reshape(-1)
    assert np.isnan(out[5]) and np.isnan(out).sum() == 1
    assert out[11] == (-np.inf if mode == "MIN" else np.inf if mode == "AMAX" else out[11])
    assert out[17] == (np.inf if mode in ("MAX", "AMAX") else out[17])


@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16])
@pytest.mark.parametrize("dims,odims", [([40000, 64], [1, 64]), ([200, 24, 20, 20], [1, 24, 1, 1])])
def test_column_sums_round_about_once(ctx, dtype, dims, odims):
    # Running sums in f64 over f32 sums of four: what is left is the rounding of the
    # slices' sums and of the result, 2^-24 of a value each at most.  As a 2-norm both
    # stay below one such step (the strided kernel this replaced: 4.5e-8 to 6.9e-8).
    x = HT.from_logical(rand(68, 0, dims), dtype)
    got = run(ctx, x, odims, "SUM", y_dtype=capi.FLOAT, expect_tuned=False).logical().astype(np.float64)
    axes = tuple(i for i, n in enumerate(odims) if n == 1)
    ref = x.logical().astype(np.float64).sum(axis=axes, keepdims=True)
    assert np.linalg.norm(got - ref) <= 2.0 ** -24 * np.linalg.norm(ref)


@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.HALF])
@pytest.mark.parametrize("kernel", ["reduce_cols", "reduce_mid", "reduce_rows"])
@pytest.mark.parametrize("n", [41, 47, 55, 82, 83, 94, 97])
def test_mean_of_equal_values_is_that_value(ctx, dtype, kernel, n):
    # (n times the f32 nearest to 1 / n is not 1 for these n)
    assert np.float32(n) * (np.float32(1) / np.float32(n)) != 1
    dims, odims = {"reduce_cols": ([n, 5], [1, 5]), "reduce_mid": ([2, 3, n, 2], [1, 3, 1, 1]),
                   "reduce_rows": ([3, 8 * n], [3, 1])}[kernel]
    x = HT.from_logical(np.ones(dims), dtype)
    out = run(ctx, x, odims, "AVG", y_dtype=capi.FLOAT, expect_tuned=kernel == "reduce_rows").logical()
    assert ctx.last_kernel().startswith(kernel), ctx.last_kernel()
    assert (out == 1).all()


@pytest.mark.parametrize("mode", ["SUM", "AVG", "MAX", "AMAX", "MUL"])
@pytest.mark.parametrize("dtype", [capi.FLOAT, capi.BFLOAT16])
@pytest.mark.parametrize("dims,odims,least", [
    ([2, 3, 256, 256], [1, 3, 1, 1], 60),  # two long runs per result: slices end inside them
    ([1, 3, 129, 131], [1, 3, 1, 1], 8),   # one run of odd length per result
    ([1, 100003], [1, 1], 48),             # everything, one run
    ([3, 5, 4099], [1, 5, 1], 6),          # slices that start at odd elements of a run
    ([4, 20, 2050], [1, 20, 1], 4),
])
def test_reduce_slices_of_few_long_runs(ctx, mode, dtype, dims, odims, least):
    x = make_x(69, dims, dtype, mode)
    if mode == "MUL":  # ((1 + 0.02 r)^100000 is out of range)
        x = HT.from_logical(1 + 2e-3 * rand(69, 0, dims), dtype)
    out = run(ctx, x, odims, mode, y_dtype=capi.FLOAT, expect_tuned=False)
    kernel, slices = ctx.last_kernel().split(" slices=")
    assert kernel == "reduce_mid" and int(slices) >= least, ctx.last_kernel()
    ref = oracle.reduction(x.logical(), odims, capi.RED[mode])
    assert_close(out.logical(), ref, capi.FLOAT, f"{mode} {dims}", rtol=1e-4 if dtype == capi.FLOAT else 2e-2)


@pytest.mark.parametrize("mode", ["SUM", "MAX"])
@pytest.mark.parametrize("dims", [[2, 8], [512, 40], [513, 40], [64, 2048], [300, 16392], [33, 4101]])
def test_reduce_few_rows_in_one_launch(ctx, mode, dims):
    x = make_x(70, dims, capi.BFLOAT16, mode)
    out = run(ctx, x, [1, dims[1]], mode, y_dtype=capi.FLOAT, expect_tuned=False)
    assert (ctx.last_kernel() == "reduce_cols slices=1") == (dims[0] <= 512), ctx.last_kernel()
    assert_close(out.logical(), oracle.reduction(x.logical(), [1, dims[1]], capi.RED[mode]), capi.FLOAT, rtol=2e-2)
