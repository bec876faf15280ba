"""Calls recorded into a graph: on a context that has never run one, paths that would
have to grow the context's scratch do without it; on one that has, the scratch that the
graph names outlives later growth.  Every replay is compared with the eager result of a
second context."""
import ctypes

import pytest

from fusilli_amd import capi

pytestmark = pytest.mark.gpu


def _norm(torch):
    x = torch.randn(2, 70001, device="cuda")
    out = torch.empty_like(x)
    d = capi.NormDesc()
    d.x = d.y = d.out = capi.TensorDesc.make([2, 70001], [70001, 1], capi.FLOAT)
    d.out_dtype, d.epsilon = capi.FLOAT, 1e-6
    d.epilogue = capi.make_epilogue([capi.epilogue_op(capi.PW["MUL"], capi.FLOAT, scalar=0.5)])
    return x, out, lambda c: c.norm_fwd(d, x.data_ptr(), None, None, out.data_ptr()), 1e-5


def _sdpa(torch):
    q, k, v = (torch.randn(1, 2, s, 64, device="cuda", dtype=torch.bfloat16) for s in (1, 2000, 2000))
    out = torch.empty_like(q)
    d = capi.SdpaDesc()
    for f, t in (("q", q), ("k", k), ("v", v), ("o", out)):
        setattr(d, f, capi.TensorDesc.make(list(t.shape), list(t.stride()), capi.BFLOAT16))
    return q, out, lambda c: c.sdpa_fwd(d, q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()), 2e-2


def _matmul(torch):
    a = torch.randn(16, 4096, device="cuda", dtype=torch.bfloat16)
    b = torch.randn(4096, 128, device="cuda", dtype=torch.bfloat16)
    out = torch.empty(16, 128, device="cuda", dtype=torch.bfloat16)
    d = capi.MatmulDesc()
    d.a = capi.TensorDesc.make([16, 4096], [4096, 1], capi.BFLOAT16)
    d.b = capi.TensorDesc.make([4096, 128], [128, 1], capi.BFLOAT16)
    d.c = capi.TensorDesc.make([16, 128], [128, 1], capi.FLOAT)
    d.out = capi.TensorDesc.make([16, 128], [128, 1], capi.BFLOAT16)
    d.out_dtype = capi.BFLOAT16
    d.epilogue = capi.make_epilogue([])
    return a, out, lambda c: c.matmul(d, a.data_ptr(), b.data_ptr(), out.data_ptr()), 2e-2


def _matmul_tiled(torch):
    a = torch.randn(512, 8192, device="cuda", dtype=torch.bfloat16)
    b = torch.randn(256, 8192, device="cuda", dtype=torch.bfloat16)
    out = torch.empty(512, 256, device="cuda", dtype=torch.bfloat16)
    d = capi.MatmulDesc()
    d.a = capi.TensorDesc.make([512, 8192], [8192, 1], capi.BFLOAT16)
    d.b = capi.TensorDesc.make([8192, 256], [1, 8192], capi.BFLOAT16)
    d.c = capi.TensorDesc.make([512, 256], [256, 1], capi.FLOAT)
    d.out = capi.TensorDesc.make([512, 256], [256, 1], capi.BFLOAT16)
    d.out_dtype = capi.BFLOAT16
    d.epilogue = capi.make_epilogue([])
    return a, out, lambda c: c.matmul(d, a.data_ptr(), b.data_ptr(), out.data_ptr()), 2.0 ** -8


def _conv(torch, n, c, k, hw, pad=1):
    cl = lambda n, c, h, w: capi.TensorDesc.make([n, c, h, w], [c * h * w, 1, c * w, c], capi.BFLOAT16)  # noqa: E731
    x = torch.randn(n, hw, hw, c, device="cuda", dtype=torch.bfloat16)
    w = torch.randn(k, 1 + 2 * pad, 1 + 2 * pad, c, device="cuda", dtype=torch.bfloat16)
    out = torch.empty(n, hw, hw, k, device="cuda", dtype=torch.bfloat16)
    d = capi.ConvDesc()
    d.x, d.w = cl(n, c, hw, hw), cl(k, c, 1 + 2 * pad, 1 + 2 * pad)
    d.y = d.out = cl(n, k, hw, hw)
    d.out_dtype, d.spatial_rank = capi.BFLOAT16, 2
    for i in range(2):
        d.stride[i] = d.dilation[i] = 1
        d.padding[i] = pad
    d.epilogue = capi.make_epilogue([])
    return x, out, lambda c: c.conv_fprop(d, x.data_ptr(), w.data_ptr(), out.data_ptr()), 2.0 ** -8  # two roundings to bf16


def _conv_padded(torch):
    return _conv(torch, 8, 200, 256, 60)


def _conv_split(torch):
    return _conv(torch, 4, 512, 128, 7)


def _reduce(torch, channels_last):
    dims = [8, 24, 50, 50]
    x = torch.randn(dims, device="cuda")
    if channels_last:
        x = x.contiguous(memory_format=torch.channels_last)
    out = torch.empty(24, device="cuda")
    d = capi.ReduceDesc()
    d.x = capi.TensorDesc.make(dims, list(x.stride()), capi.FLOAT)
    d.y = capi.TensorDesc.make([1, 24, 1, 1], [24, 1, 1, 1], capi.FLOAT)
    d.mode = capi.RED["AVG"]
    return x, out, lambda c: c.reduce(d, x.data_ptr(), out.data_ptr()), 1e-5


def _bias_gradient(torch):
    return _reduce(torch, True)


def _channel_means(torch):
    return _reduce(torch, False)


# (more parts than the workspace holds would be faster: recorded or not, it bounds them, so the bits agree)
def _weight_gradient(torch, n, c, h, w, k):
    cl = lambda n, c, h, w: capi.TensorDesc.make([n, c, h, w], [c * h * w, 1, c * w, c], capi.BFLOAT16)  # noqa: E731
    x = torch.randn(n, h, w, c, device="cuda", dtype=torch.bfloat16)
    dy = torch.randn(n, h, w, k, device="cuda", dtype=torch.bfloat16)
    out = torch.empty(k, 3, 3, c, device="cuda", dtype=torch.bfloat16)
    d = capi.ConvDesc()
    d.x, d.w, d.y = cl(n, c, h, w), cl(k, c, 3, 3), cl(n, k, h, w)
    d.spatial_rank = 2
    for i in range(2):
        d.stride[i] = d.dilation[i] = d.padding[i] = 1
    d.epilogue = capi.make_epilogue([])
    need = ctypes.c_size_t(0)
    assert capi.load().fhip_conv_wgrad_workspace_size(ctypes.byref(d), ctypes.byref(need)) == 0
    space = torch.empty(need.value, device="cuda", dtype=torch.uint8)
    return x, out, lambda c: c.conv_wgrad(d, dy.data_ptr(), x.data_ptr(), out.data_ptr(), space.data_ptr()), 0.0


def _weight_gradient_own(torch):
    return _weight_gradient(torch, 45, 448, 21, 1, 320)


def _weight_gradient_gathered(torch):
    return _weight_gradient(torch, 1, 264, 45, 22, 128)


# what runs where there is scratch
ROUTES = {_matmul_tiled: "gemm_mfma bf16 128x128 waves=8 split=16",
          _conv_padded: "conv_igemm gather 256x128 split=1 padded=1 groups=1",
          _conv_split: "conv_igemm gather 128x128 split=8 padded=0 groups=1",
          _weight_gradient_own: "conv_wgrad_direct steps=1 parts=1",
          _weight_gradient_gathered: "conv_wgrad_direct steps=2 parts=2"}


@pytest.mark.parametrize("make", [_norm, _sdpa, _matmul])
def test_replay_after_scratch_has_grown(make):
    import torch
    torch.manual_seed(2)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        x, out, call, tol = make(torch)
        big = capi.ConvDesc()  # 4 MB of partial sums
        xs = torch.randn(8, 32, 32, 64, device="cuda", dtype=torch.bfloat16)
        dy = torch.randn(8, 32, 32, 256, device="cuda", dtype=torch.bfloat16)
        dw = torch.empty(256, 1, 1, 64, device="cuda")
        cl = lambda n, c, h, w: capi.TensorDesc.make([n, c, h, w], [c * h * w, 1, c * w, c], capi.BFLOAT16)  # noqa: E731
        big.x, big.y = cl(8, 64, 32, 32), cl(8, 256, 32, 32)
        big.w = capi.TensorDesc.make([256, 64, 1, 1], [64, 1, 64, 64], capi.FLOAT)
        big.spatial_rank = 2
        for i in range(2):
            big.stride[i] = big.dilation[i] = 1
        big.epilogue = capi.make_epilogue([])
        warm = capi.Context(torch.cuda.current_device(), stream.cuda_stream)
        other = capi.Context(torch.cuda.current_device(), stream.cuda_stream)
        call(warm)
        graph = torch.cuda.CUDAGraph()
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            call(warm)
        for i in range(4):
            if i == 1:
                warm.conv_wgrad(big, dy.data_ptr(), xs.data_ptr(), dw.data_ptr())
                assert warm.last_kernel() == "conv_wgrad_gather 256x64 runs=64"
            x.copy_(torch.randn_like(x))
            call(other)
            want = out.clone()
            out.zero_()
            # memory that went back to the device would be handed out again here
            fill = [torch.full((1 << 18,), 7.0, device="cuda") for _ in range(8)]
            graph.replay()
            stream.synchronize()
            assert torch.equal(out, want), i
            assert all(bool((f == 7.0).all()) for f in fill), i
            del fill
        del graph
        warm.close()
        other.close()


@pytest.mark.parametrize("make", [_norm, _sdpa, _matmul, _matmul_tiled, _conv_padded, _conv_split, _bias_gradient,
                                  _channel_means, _weight_gradient_own, _weight_gradient_gathered])
def test_first_call_under_capture(make):
    import torch
    torch.manual_seed(1)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        x, out, call, tol = make(torch)
        cold = capi.Context(torch.cuda.current_device(), stream.cuda_stream)
        warm = capi.Context(torch.cuda.current_device(), stream.cuda_stream)
        graph = torch.cuda.CUDAGraph()
        stream.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            call(cold)
        assert "split=1" in cold.last_kernel() or "split=" not in cold.last_kernel()
        for i in range(3):
            x.copy_(torch.randn_like(x))
            call(warm)
            assert warm.last_kernel() == ROUTES.get(make, warm.last_kernel())
            want = out.float().clone()
            out.zero_()
            graph.replay()
            stream.synchronize()
            got = out.float()
            err = (got - want).norm() / want.norm()
            assert err <= tol, (i, float(err))
        del graph
        cold.close()
        warm.close()
