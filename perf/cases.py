"""Performance cases of the operator library: what a program calls it for.

Every case goes through ``fusilli_amd.capi.Context`` with descriptors, output
buffers and workspaces made once, as a program that runs a plan many times
keeps them.  The context lives on one torch stream, on which the inputs are
made as well.

Kinds of case
  matmul  [batch x] M x K times K x N, operands stored either way round, with
          the fused operations of a linear layer (bias, bias + GELU) or of a
          quantised one (a scale on fp8 products; int8 sums stay int32)
  sdpa    attention forward: prefill (causal or not), cross attention, a mask
          tensor, grouped heads, and decode over a key / value cache
  conv    one training step of a convolution layer: forward, activation,
          bias gradient, data gradient, weight gradient
  norm    RMSNorm (inference, with the multiplication that follows it) and
          LayerNorm (training, with its statistics)
"""
import math

import torch

from fusilli_amd import capi

_DT = {"f32": (torch.float32, capi.FLOAT), "bf16": (torch.bfloat16, capi.BFLOAT16),
       "f16": (torch.float16, capi.HALF), "i8": (torch.int8, capi.INT8),
       "fp8": (torch.float8_e4m3fn, capi.FP8E4M3)}
_SIZE = {"f32": 4, "bf16": 2, "f16": 2, "i8": 1, "fp8": 1}
_FP8_SCALE = 1.0 / (448.0 * 448.0)
_held = {}


def _program():
    """The context and the stream that the whole program works on."""
    if not _held:
        stream = torch.cuda.Stream()
        _held["stream"] = stream
        _held["ctx"] = capi.Context(torch.cuda.current_device(), stream.cuda_stream)
    return _held["ctx"], _held["stream"]


# ---- cases -------------------------------------------------------------------
def _matmul(dtype, m, n, k, batch=1, ta=False, tb=False, epi="none"):
    return {"kind": "matmul", "dtype": dtype, "m": m, "n": n, "k": k, "batch": batch,
            "ta": ta, "tb": tb, "epi": epi}


def _sdpa(dtype, b, hq, hkv, sq, skv, d, causal=False, mask=False):
    return {"kind": "sdpa", "dtype": dtype, "b": b, "hq": hq, "hkv": hkv, "sq": sq,
            "skv": skv, "d": d, "causal": causal, "mask": mask}


def _conv(dtype, layout, n, c, h, w, k, r, pad, stride, act):
    return {"kind": "conv", "dtype": dtype, "layout": layout, "n": n, "c": c, "h": h,
            "w": w, "k": k, "r": r, "pad": pad, "stride": stride, "act": act}


def _norm(dtype, op, rows, cols):
    return {"kind": "norm", "dtype": dtype, "op": op, "rows": rows, "cols": cols}


def listed():
    return [dict(c, name=name) for name, c in (
        # the benchmark list's smallest product: one call's latency
        ("matmul_f32_small", _matmul("f32", 16, 32, 64, ta=True, tb=True, epi="bias")),
        # one token each of 16 sequences through a linear layer (weights N x K)
        ("matmul_bf16_decode", _matmul("bf16", 16, 4096, 4096, tb=True, epi="bias")),
        # sizes that fit no tile: a batch of short sequences through an MLP layer
        ("matmul_f16_ragged", _matmul("f16", 777, 1400, 1000, epi="bias_gelu")),
        # the quantised product of the benchmark (scaled fp8, bf16 result)
        ("matmul_fp8_large", _matmul("fp8", 4096, 4096, 8192, epi="scale")),
        # benchmark attention shapes: grouped heads over a short sequence ...
        ("sdpa_f16_gqa_short", _sdpa("f16", 2, 16, 4, 128, 128, 64, causal=True)),
        # ... and prefill of 2048 tokens
        ("sdpa_bf16_prefill", _sdpa("bf16", 4, 32, 32, 2048, 2048, 128, causal=True)),
        # decode: one new query per sequence over a cache of some thousand keys
        ("sdpa_bf16_decode", _sdpa("bf16", 8, 32, 8, 1, 4000, 128)),
        # training steps of convolution layers: a ResNet-sized one with bias and ReLU,
        ("conv_bf16_c64_train", _conv("bf16", "nhwc", 32, 64, 56, 56, 128, 3, 1, 1, "bias_relu")),
        # one whose channel count fits no tile, with batch norm,
        ("conv_f16_c48_train", _conv("f16", "nhwc", 16, 48, 48, 32, 48, 3, 2, 1, "batchnorm")),
        # and the first layer of a network on f32 images
        ("conv_f32_nchw_train", _conv("f32", "nchw", 100, 3, 32, 32, 32, 3, 0, 1, "bias_relu")),
        # the headline norm of the benchmark, and its normalisation over whole images
        ("rmsnorm_bf16_mul", _norm("bf16", "rmsnorm", 8192, 4096)),
        ("layernorm_bf16_long_rows", _norm("bf16", "layernorm", 16, 262144)),
    )]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(rng, size, steps):
    """`size` as a multiple of one of `steps` (a list of (step, weight))."""
    step = rng.choices([s for s, _ in steps], [w for _, w in steps])[0]
    return max(step, size // step * step)


def _draw_matmul(rng):
    dtype = rng.choice(["f32", "bf16", "bf16", "f16", "fp8", "i8"])
    ta, tb = rng.choice([(False, False), (False, True), (False, True), (True, False), (True, True)])
    if dtype == "f32":  # the benchmark's f32 products are small, some of them batched
        any_ = [(16, 2), (1, 1)]
        m, n, k = (_near(rng, _log(rng, 16, 512), any_) for _ in range(3))
        return _matmul(dtype, m, n, k, rng.choice([1, 1, 10]), ta, tb, rng.choice(["none", "bias"]))
    m = _near(rng, _log(rng, 1, 4096), [(64, 1), (1, 2)])
    if dtype in ("bf16", "f16"):
        some = [(64, 10), (8, 7), (1, 3)]
        n, k = (_near(rng, _log(rng, 256, 8192), some) for _ in range(2))
        return _matmul(dtype, m, n, k, 1, False if m % 8 else ta, tb,
                       rng.choice(["none", "bias", "bias_gelu"]))
    n, k = (_near(rng, _log(rng, 512, 8192), [(128, 2), (16, 1)]) for _ in range(2))
    return _matmul(dtype, m, n, k, 1, False, tb, "scale" if dtype == "fp8" else "none")


def _draw_sdpa(rng):
    dtype, d = rng.choice(["bf16", "f16"]), rng.choice([64, 128])
    hkv = rng.choice([1, 4, 8, 16, 32])
    hq = hkv * rng.choice([1, 1, 4, 8]) if hkv < 32 else 32
    mode = rng.choice(["prefill", "prefill", "cross", "mask", "decode", "decode"])
    b = _log(rng, 1, 8)
    skv = _near(rng, _log(rng, 64, 4096), [(64, 1), (1, 1)])
    sq = skv
    if mode == "decode":
        b, sq = _log(rng, 1, 32), 1
    elif mode == "cross":
        sq = _near(rng, _log(rng, 16, 2048), [(64, 1), (1, 1)])
    elif mode == "mask":
        sq = skv = _near(rng, skv, [(8, 1)])
    causal = mode == "prefill" and rng.random() < 0.7
    while 4 * b * hq * sq * skv * d > 2.7e11:
        b, hq, hkv = (b // 2, hq, hkv) if b > 1 else (b, hq // 2, max(1, hkv // 2))
    return _sdpa(dtype, b, hq, hkv, sq, skv, d, causal, mode == "mask")


def _draw_conv(rng):
    if rng.random() < 0.25:  # first layers: few input channels, channels first
        r = rng.choice([3, 3, 5])
        hw = _log(rng, 16, 64)
        return _conv(rng.choice(["f32", "bf16"]), "nchw", _log(rng, 16, 128), rng.choice([1, 3, 3, 4]),
                     hw, hw, rng.choice([16, 32, 64]), r, rng.choice([0, r // 2]), 1, "bias_relu")
    r = rng.choice([1, 3, 3, 3, 5])
    h = _log(rng, 7, 64)
    w = h if rng.random() < 0.7 else _log(rng, 7, 64)
    c, k = (_near(rng, _log(rng, 32, 512), [(64, 3), (16, 2), (8, 1)]) for _ in range(2))
    n = _log(rng, 8, 64)
    stride = rng.choice([1, 1, 1, 2])
    while n > 1 and n * h * w * c * k * r * r // stride ** 2 > 1.5e10:
        n //= 2
    return _conv(rng.choice(["bf16", "f16"]), "nhwc", n, c, h, w, k, r, r // 2, stride,
                 rng.choice(["bias_relu", "batchnorm"]))


def _draw_norm(rng):
    op, dtype = rng.choice(["rmsnorm", "layernorm"]), rng.choice(["bf16", "bf16", "f16", "f32"])
    if rng.random() < 0.25:  # whole images: few rows, long ones
        return _norm(dtype, op, _log(rng, 1, 32), _near(rng, _log(rng, 32768, 524288), [(1024, 1)]))
    rows = _log(rng, 1, 16384)
    return _norm(dtype, op, rows, _near(rng, _log(rng, 128, 16384), [(64, 3), (8, 2), (1, 1)]))


def draw(rng):
    return rng.choice([_draw_matmul, _draw_sdpa, _draw_conv, _draw_norm])(rng)


# ---- inputs ------------------------------------------------------------------
class _Inputs:
    """Seeded tensors on the device (activations N(0, 1), weights scaled by
    their fan-in, 8-bit operands over their whole range)."""

    def __init__(self, seed):
        self.gen = torch.Generator(device="cuda")
        self.gen.manual_seed(seed)

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        t = torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32)
        return t.mul_(std).add_(mean).to(_DT[dtype][0])

    def operand(self, shape, dtype, std=1.0):
        if dtype == "i8":
            return torch.randint(-127, 128, shape, generator=self.gen, device="cuda", dtype=torch.int8)
        if dtype == "fp8":
            t = torch.rand(shape, generator=self.gen, device="cuda", dtype=torch.float32)
            return t.mul_(896.0).sub_(448.0).to(torch.float8_e4m3fn)
        return self.normal(shape, dtype, std)


def _empty(shape, dtype):
    t = torch.int32 if dtype == "i32" else _DT[dtype][0]
    return torch.empty(shape, device="cuda", dtype=t)


def _desc(dims, strides, dtype):
    return capi.TensorDesc.make(dims, strides, capi.INT32 if dtype == "i32" else _DT[dtype][1])


def _contiguous(dims):
    out, step = [], 1
    for d in reversed(dims):
        out.insert(0, step)
        step *= d
    return out


def _buffer(bytes_):
    return torch.empty(max(bytes_, 1), device="cuda", dtype=torch.uint8)


def _prepare_matmul(c, put):
    m, n, k, batch, dt = c["m"], c["n"], c["k"], c["batch"], c["dtype"]
    lead = [batch] if batch > 1 else []
    a = put.operand(lead + ([k, m] if c["ta"] else [m, k]), dt)
    b = put.operand(lead + ([n, k] if c["tb"] else [k, n]), dt, 1.0 / math.sqrt(k))
    out_dt = {"f32": "f32", "i8": "i32", "fp8": "bf16"}.get(dt, dt)
    out = _empty(lead + [m, n], out_dt)

    def strides(rows, cols, flip):
        return ([rows * cols] if lead else []) + ([1, rows] if flip else [cols, 1])

    d = capi.MatmulDesc()
    d.a = _desc(lead + [m, k], strides(m, k, c["ta"]), dt)
    d.b = _desc(lead + [k, n], strides(k, n, c["tb"]), dt)
    acc = "i32" if dt == "i8" else "f32"
    d.c = _desc(lead + [m, n], strides(m, n, False), acc)
    d.out = _desc(lead + [m, n], strides(m, n, False), out_dt)
    d.out_dtype = d.out.dtype
    s, ops = {"d": d, "a": a, "b": b, "out": out}, []
    if c["epi"] == "scale":
        ops = [capi.epilogue_op(capi.PW["MUL"], d.out_dtype, scalar=_FP8_SCALE)]
    elif c["epi"] != "none":
        s["bias"] = put.normal([n], dt)
        row = _desc(([1] if lead else []) + [1, n], ([n] if lead else []) + [n, 1], dt)
        last = c["epi"] == "bias"
        ops = [capi.epilogue_op(capi.PW["ADD"], d.out_dtype if last else capi.FLOAT, operand=row)]
        if not last:
            ops.append(capi.epilogue_op(capi.PW["GELU_FWD"], d.out_dtype))
    d.epilogue = capi.make_epilogue(ops)
    return s


def _run_matmul(ctx, s):
    p = s["p"]
    ctx.matmul(s["d"], p["a"], p["b"], p["out"], [p["bias"]] if "bias" in p else ())
    return s["out"]


def _prepare_sdpa(c, put):
    b, hq, hkv, sq, skv, hd, dt = (c[x] for x in ("b", "hq", "hkv", "sq", "skv", "d", "dtype"))
    # decode reads the first skv keys of a cache with room for more
    room = (skv + 255) // 256 * 256 if sq == 1 else skv
    q = put.normal([b, hq, sq, hd], dt)
    k, v = (put.normal([b, hkv, room, hd], dt) for _ in range(2))
    o = _empty([b, hq, sq, hd], dt)
    d = capi.SdpaDesc()
    d.q = _desc([b, hq, sq, hd], _contiguous([b, hq, sq, hd]), dt)
    d.k = _desc([b, hkv, skv, hd], _contiguous([b, hkv, room, hd]), dt)
    d.v = _desc([b, hkv, skv, hd], _contiguous([b, hkv, room, hd]), dt)
    d.o = _desc([b, hq, sq, hd], _contiguous([b, hq, sq, hd]), dt)
    d.is_causal = 1 if c["causal"] else 0
    s = {"d": d, "q": q, "k": k, "v": v, "o": o}
    if c["mask"]:
        s["mask"] = put.normal([b, 1, sq, skv], dt)
        d.mask = _desc([b, 1, sq, skv], _contiguous([b, 1, sq, skv]), dt)
    return s


def _run_sdpa(ctx, s):
    p = s["p"]
    ctx.sdpa_fwd(s["d"], p["q"], p["k"], p["v"], p["o"], p.get("mask"))
    return s["o"]


def _out_size(c):
    return tuple((c[x] + 2 * c["pad"] - c["r"]) // c["stride"] + 1 for x in ("h", "w"))


def _prepare_conv(c, put):
    dt, n, ch, k, r = c["dtype"], c["n"], c["c"], c["k"], c["r"]
    p, q = _out_size(c)
    nhwc = c["layout"] == "nhwc"

    def stored(dims):  # the shape in memory of logical [d0, d1, h, w]
        return [dims[0], dims[2], dims[3], dims[1]] if nhwc else dims

    def desc(dims, dtype=dt):
        st = [dims[1] * dims[2] * dims[3], 1, dims[3] * dims[1], dims[1]] if nhwc else _contiguous(dims)
        return _desc(dims, st, dtype)

    xd, wd, yd = [n, ch, c["h"], c["w"]], [k, ch, r, r], [n, k, p, q]
    s = {"x": put.normal(stored(xd), dt), "w": put.normal(stored(wd), dt, 1.0 / math.sqrt(ch * r * r)),
         "dy": put.normal(stored(yd), dt), "y": _empty(stored(yd), dt), "z": _empty(stored(yd), dt),
         "dx": _empty(stored(xd), dt), "dw": _empty(stored(wd), dt)}
    per_channel = lambda dtype: desc([1, k, 1, 1], dtype)  # noqa: E731

    def conv_desc(y_dtype):
        d = capi.ConvDesc()
        d.x, d.w, d.y = desc(xd), desc(wd), desc(yd, y_dtype)
        d.spatial_rank = 2
        for i in range(2):
            d.padding[i], d.stride[i], d.dilation[i] = c["pad"], c["stride"], 1
        return d

    fwd, bwd = conv_desc("f32"), conv_desc(dt)
    fwd.out, fwd.out_dtype = desc(yd), _DT[dt][1]
    bwd.epilogue = capi.make_epilogue([])
    act = capi.PointwiseDesc()
    act.params = capi.PointwiseParams.default()
    act.in_[0], act.out = desc(yd), desc(yd)
    if c["act"] == "bias_relu":
        s["bias"] = put.normal([k], dt)
        s["db"] = _empty([k], "f32")
        fwd.epilogue = capi.make_epilogue([
            capi.epilogue_op(capi.PW["ADD"], capi.FLOAT, operand=per_channel(dt)),
            capi.epilogue_op(capi.PW["RELU_FWD"], _DT[dt][1])])
        act.mode, act.num_inputs = capi.PW["RELU_BWD"], 2
        act.in_[1] = desc(yd)
        red = capi.ReduceDesc()
        red.x, red.y, red.mode = desc(yd), per_channel("f32"), capi.RED["SUM"]
        s["reduce"] = red
    else:
        s["scale"], s["shift"] = put.normal([k], "f32", 0.1, 1.0), put.normal([k], "f32")
        s["mean"], s["inv"], s["b"] = _empty([k], "f32"), _empty([k], "f32"), _empty(stored(yd), dt)
        fwd.epilogue = capi.make_epilogue([])
        bn = capi.BatchNormDesc()
        bn.x, bn.y = desc(yd), desc(yd)
        bn.training = bn.has_scale = bn.has_bias = 1
        bn.scale_dtype = bn.bias_dtype = bn.stats_dtype = capi.FLOAT
        bn.epsilon = 1e-5
        act.mode, act.num_inputs = capi.PW["RELU_FWD"], 1
        s["bn"] = bn
    ctx, _ = _program()
    need = max(ctx.conv_dgrad_workspace(bwd), ctx.conv_wgrad_workspace(bwd))
    s.update(fwd=fwd, bwd=bwd, act=act, ws=_buffer(need))
    return s


def _run_conv(ctx, s):
    p = s["p"]
    if "bias" in p:
        # y = relu(conv(x, w) + bias);  z = dL/d(conv) = dy where y > 0;  db = sum z
        ctx.conv_fprop(s["fwd"], p["x"], p["w"], p["y"], [p["bias"]])
        ctx.pointwise(s["act"], p["dy"], p["y"], None, p["z"])
        ctx.reduce(s["reduce"], p["z"], p["db"])
        dz, more = p["z"], {"db": s["db"]}
    else:
        # y = relu(batchnorm(conv(x, w))); dy is the gradient at the convolution
        ctx.conv_fprop(s["fwd"], p["x"], p["w"], p["z"])
        ctx.batchnorm_fwd(s["bn"], p["z"], p["b"], p["scale"], p["shift"],
                          saved_mean=p["mean"], saved_inv_variance=p["inv"])
        ctx.pointwise(s["act"], p["b"], None, None, p["y"])
        dz, more = p["dy"], {"mean": s["mean"], "inv": s["inv"]}
    ctx.conv_dgrad(s["bwd"], dz, p["w"], p["dx"], workspace=p["ws"])
    ctx.conv_wgrad(s["bwd"], dz, p["x"], p["dw"], workspace=p["ws"])
    return {"y": s["y"], "dx": s["dx"], "dw": s["dw"], **more}


def _prepare_norm(c, put):
    rows, cols, dt = c["rows"], c["cols"], c["dtype"]
    layer = c["op"] == "layernorm"
    full = _desc([rows, cols], [cols, 1], dt)
    row = _desc([1, cols], [cols, 1], dt)
    d = capi.NormDesc()
    d.x, d.scale, d.out = full, row, full
    d.out_dtype = _DT[dt][1]
    d.y = full if layer else _desc([rows, cols], [cols, 1], "f32")
    d.epsilon = 1e-5 if layer else 1e-6
    s = {"d": d, "x": put.normal([rows, cols], dt), "scale": put.normal([cols], dt, 0.02, 1.0),
         "out": _empty([rows, cols], dt)}
    if layer:
        d.is_layernorm = d.emit_stats = 1
        d.stats_dtype = capi.FLOAT
        d.bias = row
        d.epilogue = capi.make_epilogue([])
        s.update(bias=put.normal([cols], dt, 0.02), mean=_empty([rows], "f32"), inv=_empty([rows], "f32"))
    else:
        d.epilogue = capi.make_epilogue([capi.epilogue_op(capi.PW["MUL"], d.out_dtype, scalar=0.5)])
    return s


def _run_norm(ctx, s):
    p = s["p"]
    ctx.norm_fwd(s["d"], p["x"], p["scale"], p.get("bias"), p["out"], p.get("mean"), p.get("inv"))
    return s["out"] if "mean" not in s else {"y": s["out"], "mean": s["mean"], "inv": s["inv"]}


_PREPARE = {"matmul": _prepare_matmul, "sdpa": _prepare_sdpa, "conv": _prepare_conv, "norm": _prepare_norm}
_RUN = {"matmul": _run_matmul, "sdpa": _run_sdpa, "conv": _run_conv, "norm": _run_norm}


def prepare(case, seed):
    ctx, stream = _program()
    with torch.cuda.stream(stream):
        s = _PREPARE[case["kind"]](case, _Inputs(seed))
    s["p"] = {key: t.data_ptr() for key, t in s.items() if isinstance(t, torch.Tensor)}
    s["run"] = _RUN[case["kind"]]
    s["ctx"] = ctx
    return s


def run(state):
    return state["run"](state["ctx"], state)


# ---- what a pass cannot do without -------------------------------------------
def work(case):
    e = _SIZE[case["dtype"]]
    if case["kind"] == "matmul":
        m, n, k, batch = case["m"], case["n"], case["k"], case["batch"]
        out = {"i8": 4, "fp8": 2}.get(case["dtype"], e)
        bias = n * e if "bias" in case["epi"] else 0
        return {"bytes": batch * (e * (m * k + k * n) + out * m * n) + bias, "flops": 2 * batch * m * n * k}
    if case["kind"] == "sdpa":
        b, hq, hkv, sq, skv, d = (case[x] for x in ("b", "hq", "hkv", "sq", "skv", "d"))
        # a causal query sees the keys up to its own position
        pairs = sum(min(i + 1, skv) for i in range(sq)) if case["causal"] else sq * skv
        mask = b * sq * skv * e if case["mask"] else 0
        return {"bytes": e * b * d * (2 * hq * sq + 2 * hkv * skv) + mask, "flops": 4 * b * hq * d * pairs}
    if case["kind"] == "conv":
        p, q = _out_size(case)
        x = case["n"] * case["c"] * case["h"] * case["w"]
        y = case["n"] * case["k"] * p * q
        w = case["k"] * case["c"] * case["r"] ** 2
        # x, w, dy in; y, dx, dw out; vectors per channel; three products
        vectors = case["k"] * (e + 4 if case["act"] == "bias_relu" else 16)
        return {"bytes": e * (2 * x + 2 * y + 2 * w) + vectors,
                "flops": 3 * 2 * y * case["c"] * case["r"] ** 2}
    rows, cols = case["rows"], case["cols"]
    layer = case["op"] == "layernorm"
    return {"bytes": e * (2 * rows * cols + (2 if layer else 1) * cols) + (8 * rows if layer else 0),
            "flops": (8 if layer else 5) * rows * cols}


def tolerance(case):
    # About four times what the path differs by from the same arithmetic in 64
    # bits rounded to the result's type.  Sums in another order move a 16-bit
    # result by a unit in its last place here and there (bf16 up to 1.5e-4 over
    # 8192 terms, f16 up to 4e-5); attention also rounds its probabilities
    # (bf16 2.6e-3, f16 3.2e-4); the mean of centred data cancels (3e-5).
    half = case["dtype"] == "f16"
    if case["dtype"] == "i8":
        return "exact"
    if case["dtype"] == "f32":
        return {"rel": 1e-4 if case.get("op") == "layernorm" else 1e-5, "max": 1e-3}
    if case["kind"] == "sdpa":
        return {"rel": 1.3e-3, "max": 1e-2} if half else {"rel": 1e-2, "max": 0.13}
    return {"rel": 2e-4, "max": 1e-2} if half else {"rel": 6e-4, "max": 6e-2}
