"""The natively registered operators (csrc/host_args.cpp) against the Python implementations of the same operators: outputs,
their layouts, what else the tuples hold, and the calls that are handed on."""

import threading

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu
aten = torch.ops.aten


@pytest.fixture(scope="module")
def impl(gpu_device):
    import torch_neuronx_amd  # noqa: F401
    from torch_neuronx_amd.python_ops import scaled_dot_product_fused_attention as impl

    return impl


def _make(dev, dtype, B, Hq, Hkv, L, S, D, layout, Dv=None):
    g = torch.Generator(device=dev).manual_seed(L * 7 + S + D)

    def one(H, n, d):
        if layout == "seq_major":
            return torch.randn(B, n, H, d, generator=g, device=dev).to(dtype).transpose(1, 2)
        if layout == "strided":  # no unit stride on the head dim
            return torch.randn(B, H, d, n, generator=g, device=dev).to(dtype).transpose(2, 3)
        if layout == "broadcast":
            return torch.randn(1, H, n, d, generator=g, device=dev).to(dtype).expand(B, H, n, d)
        return torch.randn(B, H, n, d, generator=g, device=dev).to(dtype)

    return one(Hq, L, D), one(Hkv, S, D), one(Hkv, S, Dv or D)


def _same(got, want):
    assert len(got) == len(want)
    for a, b in zip(got, want):
        if isinstance(b, torch.Tensor):
            assert (a.shape, a.dtype, a.device, a.stride()) == (b.shape, b.dtype, b.device, b.stride())
            assert torch.equal(a, b)  # (the same kernels on the same inputs)
        else:
            assert a == b


@pytest.mark.parametrize("layout", ["plain", "seq_major", "strided", "broadcast"])
@pytest.mark.parametrize("dtype,B,Hq,Hkv,L,S,D,causal,scale", [
    (torch.bfloat16, 2, 4, 2, 130, 130, 64, True, None),
    (torch.float16, 1, 4, 4, 1, 700, 128, False, 0.3),     # the library asks for a workspace
    (torch.float32, 2, 3, 3, 33, 65, 64, False, None),
    (torch.bfloat16, 2, 2, 2, 65, 40, 80, False, 0.0),     # an explicit scale of zero
    (torch.float64, 1, 2, 2, 20, 20, 32, True, None),      # handed on
])
def test_operators_match_the_python_implementations(impl, gpu_device, layout, dtype, B, Hq, Hkv, L, S, D, causal, scale):
    q, k, v = _make(gpu_device, dtype, B, Hq, Hkv, L, S, D, layout)
    kw = {} if scale is None else {"scale": scale}
    r = aten._scaled_dot_product_flash_attention(q, k, v, 0.0, causal, False, **kw)
    w = impl.scaled_dot_product_flash_attention(q, k, v, 0.0, causal, False, scale)
    _same(r, w)
    do = torch.randn_like(w[0])
    args = (do, q, k, v, w[0], w[1], w[2], w[3], w[4], w[5], 0.0, causal, w[6], w[7])
    _same(aten._scaled_dot_product_flash_attention_backward(*args, **kw), impl.scaled_dot_product_flash_attention_backward(*args, scale))
    for lse in (True, False):
        e = impl.scaled_dot_product_efficient_attention(q, k, v, None, lse, 0.0, causal, scale)
        _same(aten._scaled_dot_product_efficient_attention(q, k, v, None, lse, 0.0, causal, **kw), e)
    e = impl.scaled_dot_product_efficient_attention(q, k, v, None, True, 0.0, causal, scale)
    args = (do, q, k, v, None, e[0], e[1], e[2], e[3], 0.0, [True, True, True, False], causal)
    _same(aten._scaled_dot_product_efficient_attention_backward(*args, **kw), impl.scaled_dot_product_efficient_attention_backward(*args, scale))


def test_calls_that_are_handed_on(impl, gpu_device, monkeypatch):
    q, k, v = _make(gpu_device, torch.bfloat16, 2, 4, 4, 64, 64, 64, "plain")
    bias = torch.randn(2, 1, 64, 64, device=gpu_device).to(torch.bfloat16)
    _same(aten._scaled_dot_product_efficient_attention(q, k, v, bias, True), impl.scaled_dot_product_efficient_attention(q, k, v, bias, True))
    with pytest.raises(NotImplementedError):
        aten._scaled_dot_product_flash_attention(q, k, v, 0.0, False, True)
    with pytest.raises(RuntimeError, match="batch sizes must match"):
        aten._scaled_dot_product_flash_attention(q, k[:1], v[:1], 0.0, False)
    out = aten._scaled_dot_product_flash_attention(q, k, v, 0.5, False)
    assert out[6].dim() == 0 and not torch.equal(out[0], aten._scaled_dot_product_flash_attention(q, k, v, 0.0, False)[0])
    # a program that binds the kernel, or wraps the functions behind the operators
    monkeypatch.setenv("TORCH_NEURONX_AMD_ENABLE_MFMA_SDPA", "0")
    generic = aten._scaled_dot_product_flash_attention(q, k, v)[0]
    _same([generic], [impl.scaled_dot_product_flash_attention(q, k, v)[0]])
    monkeypatch.delenv("TORCH_NEURONX_AMD_ENABLE_MFMA_SDPA")
    seen = []
    real = impl.ops.sdpa_forward
    monkeypatch.setattr(impl.ops, "sdpa_forward", lambda *a, **kw: (seen.append(1), real(*a, **kw))[1])
    aten._scaled_dot_product_flash_attention(q, k, v)
    assert seen == [1]
    monkeypatch.setattr(impl, "_force_kernel", lambda: 1 / 0)
    with pytest.raises(ZeroDivisionError):
        aten._scaled_dot_product_flash_attention(q, k, v)


def test_streams_threads_and_training(impl, gpu_device):
    """Forward + backward from several threads, each on a stream of its own, and under a capture."""
    q, k, v = _make(gpu_device, torch.bfloat16, 2, 8, 2, 200, 200, 128, "plain")
    do = torch.randn_like(q)

    def step():
        a = [t.detach().requires_grad_(True) for t in (q, k, v)]
        out = F.scaled_dot_product_attention(*a, is_causal=True, enable_gqa=True)
        return (out.detach(), *torch.autograd.grad(out, a, do))

    want = step()
    got = [None] * 4

    def work(i):
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.default_stream())
        with torch.cuda.stream(stream):
            for _ in range(10):
                got[i] = step()
            stream.synchronize()

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    for r in got:
        _same(r, want)
    with torch.inference_mode():
        assert torch.equal(F.scaled_dot_product_attention(q, k, v, is_causal=True, enable_gqa=True), want[0])
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        r = step()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        _same(r, want)
