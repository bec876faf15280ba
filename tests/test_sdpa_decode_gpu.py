"""Attention with the keys split over workgroups (few query rows per key / value
head), and the tiled kernel on the same problems, vs the oracle."""
import numpy as np
import pytest

from fusilli_amd import capi
from oracle import oracle
from helpers import HT, assert_close, rand
from test_sdpa_flash_gpu import CASES, bshd_strides, run

pytestmark = pytest.mark.gpu

DECODE = [
    dict(B=1, Hq=1, Hkv=1, Sq=1, Skv=1, causal=False),       # one key
    dict(B=2, Hq=4, Hkv=2, Sq=1, Skv=33, causal=False),      # one key past a chunk
    dict(B=3, Hq=8, Hkv=1, Sq=1, Skv=1000, causal=False),    # grouped heads, splits
    dict(B=1, Hq=8, Hkv=2, Sq=5, Skv=777, causal=False),     # 20 rows: a second tile
    dict(B=1, Hq=2, Hkv=1, Sq=8, Skv=515, causal=True),      # exactly one tile, masked
    dict(B=1, Hq=3, Hkv=3, Sq=90, Skv=300, causal=True),     # wavefronts without a live key
    dict(B=1, Hq=1, Hkv=1, Sq=40, Skv=7, causal=True),       # fewer keys than queries
]


@pytest.mark.parametrize("case", DECODE + CASES)
@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("hd", [128, 64])
@pytest.mark.parametrize("decode", [1, 0])
def test_both_kernels_vs_oracle(ctx, knobs, case, dtype, hd, decode):
    knobs(SDPA_DECODE=decode)
    c = case
    q = HT.from_logical(rand(56, 0, [c["B"], c["Hq"], c["Sq"], hd], std=2.0), dtype)
    k = HT.from_logical(rand(56, 1, [c["B"], c["Hkv"], c["Skv"], hd], std=2.0), dtype)
    v = HT.from_logical(rand(56, 2, [c["B"], c["Hkv"], c["Skv"], hd]), dtype)
    out = run(ctx, q, k, v, causal=c["causal"])
    assert ctx.last_kernel().startswith("sdpa_decode" if decode else "sdpa_fwd"), ctx.last_kernel()
    ref = oracle.sdpa(q.logical(), k.logical(), v.logical(), is_causal=c["causal"])
    assert_close(out.logical(), ref, dtype, str(case))


@pytest.mark.parametrize("hd", [128, 64])
def test_decode_layout_and_scale(ctx, knobs, hd):
    # heads interleaved per position, custom scale, several splits
    knobs(SDPA_DECODE=1)
    dims_q, dims_k = [2, 6, 3, hd], [2, 2, 900, hd]
    q = HT.from_logical(rand(57, 0, dims_q), capi.BFLOAT16, bshd_strides(dims_q))
    k = HT.from_logical(rand(57, 1, dims_k), capi.BFLOAT16, bshd_strides(dims_k))
    v = HT.from_logical(rand(57, 2, dims_k), capi.BFLOAT16, bshd_strides(dims_k))
    out = run(ctx, q, k, v, scale=0.31, o_strides=bshd_strides(dims_q))
    assert "splits=" in ctx.last_kernel() and not ctx.last_kernel().endswith("splits=1"), ctx.last_kernel()
    assert_close(out.logical(), oracle.sdpa(q.logical(), k.logical(), v.logical(), scale=0.31),
                 capi.BFLOAT16)


@pytest.mark.parametrize("hd", [128, 64])
@pytest.mark.parametrize("decode", [1, 0])
@pytest.mark.parametrize("sq,group,first", [
    (100, 4, 64),   # a tile of 16 packed rows holds the end of one head and the start of the next
    (100, 1, 64),
    (20, 3, None),  # one tile of 64 keys: the tiled kernel multiplies masked values there as well
])
def test_causal_rows_do_not_meet_late_values(ctx, knobs, hd, decode, sq, group, first):
    # the last key's value is infinite: only the rows whose 64 keys hold it may show that
    knobs(SDPA_DECODE=decode)
    q = HT.from_logical(rand(58, 0, [1, 2 * group, sq, hd]), capi.BFLOAT16)
    k = HT.from_logical(rand(58, 1, [1, 2, sq, hd]), capi.BFLOAT16)
    v = rand(58, 2, [1, 2, sq, hd])
    ref = oracle.sdpa(q.logical(), k.logical(), HT.from_logical(v, capi.BFLOAT16).logical(), is_causal=True)
    v[:, :, -1, :] = np.inf
    out = run(ctx, q, k, HT.from_logical(v, capi.BFLOAT16), causal=True).logical()
    assert ctx.last_kernel().startswith("sdpa_decode" if decode else "sdpa_fwd"), ctx.last_kernel()
    assert not np.isfinite(out[:, :, -1]).any()
    if first is not None:
        assert_close(out[:, :, :first], ref[:, :, :first], capi.BFLOAT16)


@pytest.mark.parametrize("case", [
    dict(B=8, Hq=32, Hkv=8, Sq=1, Skv=4000, hd=128, causal=False),
    dict(B=2, Hq=16, Hkv=4, Sq=128, Skv=128, hd=64, causal=True),
    dict(B=2, Hq=8, Hkv=2, Sq=16, Skv=2000, hd=64, causal=False),
])
@pytest.mark.parametrize("dtype", [capi.BFLOAT16, capi.HALF])
@pytest.mark.parametrize("std", [1.0, 3.0])
def test_split_keys_lose_no_precision(ctx, knobs, case, dtype, std):
    # Both kernels round the probabilities to 16 bits, against different reference points;
    # the error against 64 bits may not grow by it.  (The two errors are sums over at least
    # 32 000 independent roundings: their ratio moves by a percent or so.)
    c = case
    q = HT.from_logical(rand(59, 0, [c["B"], c["Hq"], c["Sq"], c["hd"]], std=std), dtype)
    k = HT.from_logical(rand(59, 1, [c["B"], c["Hkv"], c["Skv"], c["hd"]]), dtype)
    v = HT.from_logical(rand(59, 2, [c["B"], c["Hkv"], c["Skv"], c["hd"]]), dtype)
    group = c["Hq"] // c["Hkv"]
    ql, kl, vl = (t.logical().astype(np.float64) for t in (q, k, v))
    ref = np.empty(q.dims, np.float64)
    for b in range(c["B"]):
        for h in range(c["Hq"]):
            s = ql[b, h] @ kl[b, h // group].T / np.sqrt(c["hd"])
            if c["causal"]:
                s[np.triu_indices(c["Sq"], 1)] = -np.inf
            p = np.exp(s - s.max(1, keepdims=True))
            ref[b, h] = p @ vl[b, h // group] / p.sum(1, keepdims=True)
    err = []
    for decode in (0, 1):
        knobs(SDPA_DECODE=decode)
        out = run(ctx, q, k, v, causal=c["causal"])
        assert ctx.last_kernel().startswith("sdpa_decode" if decode else "sdpa_fwd"), ctx.last_kernel()
        err.append(np.linalg.norm(out.logical() - ref) / np.linalg.norm(ref))
    assert err[1] <= 1.02 * err[0], err


def test_route_of_short_products_and_many_tiles(ctx):
    # the kernel that measured faster on each side of the rule
    def name(b, hq, hkv, sq, skv, hd, causal):
        q = HT.from_logical(rand(60, 0, [b, hq, sq, hd]), capi.BFLOAT16)
        k = HT.from_logical(rand(60, 1, [b, hkv, skv, hd]), capi.BFLOAT16)
        run(ctx, q, k, k, causal=causal)
        return ctx.last_kernel().split()[0]
    assert name(1, 8, 2, 1, 2000, 128, False) == "sdpa_decode"
    assert name(2, 16, 4, 128, 128, 64, True) == "sdpa_decode"
    assert name(4, 64, 8, 68, 68, 128, True) == "sdpa_fwd"
    assert name(5, 32, 32, 266, 266, 64, True) == "sdpa_fwd"
    assert name(2, 32, 32, 65, 65, 128, True) == "sdpa_decode"
    assert name(7, 32, 32, 1, 175, 128, False) == "sdpa_decode"
    assert name(5, 32, 32, 1, 64, 128, False) == "sdpa_decode"
