"""The native argument marshalling: what it refuses, and the block it writes against the tensors it was given."""

import ctypes as C
import sys
import threading
import time

import pytest
import torch


@pytest.fixture(scope="module")
def amd():
    import torch_neuronx_amd as amd

    return amd


def test_refuses_what_is_no_gpu_tensor(amd):
    p = amd._lib.FwdParams()
    t = torch.zeros(1, 1, 2, 8)
    with pytest.raises(ValueError, match="query"):
        amd._lib.host().forward(C.addressof(p), t, t, t, None, True, False, 1.0, 0, False)
    with pytest.raises(TypeError):
        amd._lib.host().forward(C.addressof(p), None, t, t, None, True, False, 1.0, 0, False)
    with pytest.raises(TypeError, match="arguments"):
        amd._lib.host().backward(C.addressof(p), t)
    with pytest.raises(ValueError):
        amd.decode_fp8kv(t, t.to(torch.float8_e4m3fn), t.to(torch.float8_e4m3fn), t, t)


@pytest.mark.parametrize("block,error", [(0, ValueError), (None, TypeError), ("0", TypeError), (-1 << 80, OverflowError)])
def test_refuses_what_is_no_block(amd, block, error):
    t, host = torch.zeros(1, 1, 2, 8), amd._lib.host()
    with pytest.raises(error):
        host.forward(block, t, t, t, None, True, False, 1.0, 0, False)
    with pytest.raises(error):
        host.backward(block, t, t, t, t, t, t, None, None, False, 1.0, 0, False)
    with pytest.raises(error):
        host.decode(block, t, t, t, t, t, None, None, None, True, 1.0, 0)


def test_refuses_a_scale_that_is_no_number(amd):
    p, t = amd._lib.FwdParams(), torch.zeros(1, 1, 2, 8)
    with pytest.raises(TypeError, match="real number"):
        amd._lib.host().forward(C.addressof(p), t, t, t, None, True, False, "1", 0, False)
    with pytest.raises(TypeError, match="real number"):
        amd._lib.host().validate(t, t, t, False, "0", False)


def test_takes_whole_numbers_of_any_type(amd):
    p, t = amd._lib.FwdParams(), torch.zeros(1, 1, 2, 8)
    for n in (2, 2.0, True, torch.tensor(2)):
        with pytest.raises(ValueError, match="GPU tensor"):  # (past the conversions)
            amd._lib.host().forward(C.addressof(p), t, t, t, None, True, False, torch.tensor(1.0), n, False)


def test_placeholders_made_under_inference_mode_serve_training(amd, monkeypatch):
    from torch_neuronx_amd.python_ops import scaled_dot_product_fused_attention as ops

    monkeypatch.setattr(ops, "_rng_placeholders", {})
    monkeypatch.setattr(ops, "_scalar_rng_pair", None)
    with torch.inference_mode():
        pairs = ops._empty_rng(torch.device("cpu")) + ops._scalar_rng()
    assert not any(t.is_inference() for t in pairs)


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["plain", "seq_major_view", "expanded_kv", "strided_head_dim", "one_row"])
def test_block_and_outputs_of_a_call(amd, gpu_device, layout):
    B, Hq, Hkv, L, S, E, Dv = 2, 4, 2, 5, 7, 16, 8
    if layout == "one_row":
        L = 1
    q, k, v = (torch.randn(s, device=gpu_device) for s in ((B, Hq, L, E), (B, Hkv, S, E), (B, Hkv, S, Dv)))
    if layout == "seq_major_view":
        q, k, v = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (q, k, v))
    elif layout == "expanded_kv":
        k, v = k[:, :1].expand(B, Hkv, S, E), v[:, :1].expand(B, Hkv, S, Dv)
    elif layout == "strided_head_dim":
        q = q.transpose(2, 3).contiguous().transpose(2, 3)
    p = amd._lib.FwdParams()
    out, lse, hold = amd._lib.host().forward(C.addressof(p), q, k, v, None, True, True, 0.25, 2, False)
    assert tuple(out.shape) == (B, Hq, L, Dv) and out.dtype == q.dtype and tuple(lse.shape) == (B, Hq, L)
    want = amd.ops.empty_like_layout(q, (B, Hq, L, Dv))
    assert out.stride() == (want.stride() if want.stride(3) == 1 else torch.empty(out.shape).stride())
    assert len(hold) == (layout == "strided_head_dim" and L > 1)
    for t, f in ((hold[0] if hold else q, p.q), (k, p.k), (v, p.v), (out, p.out)):
        assert f.data == t.data_ptr() and tuple(f.size) == tuple(t.shape) and tuple(f.stride) == t.stride()
    assert (p.lse, p.bias.data, p.dtype, p.is_causal, p.scale, p.force_kernel) == (lse.data_ptr(), None, amd._lib.F32, 1, 0.25, 2)
    b = amd._lib.BwdParams()
    go = torch.randn(out.shape, device=gpu_device)
    dq, dk, dv, hold = amd._lib.host().backward(C.addressof(b), go, q, k, v, out, lse.double(), None, None, False, 0.5, 0, True)
    for g, x, f in ((dq, q, b.grad_q), (dk, k, b.grad_k), (dv, v, b.grad_v)):
        assert g.shape == x.shape and g.transpose(1, 2).is_contiguous() and f.data == g.data_ptr() and tuple(f.stride) == g.stride()
    assert hold[-1].dtype == torch.float32 and b.lse == hold[-1].data_ptr()  # (a float64 log-sum-exp is converted)


@pytest.mark.gpu
def test_the_debug_mask_of_a_call_is_its_own(amd, gpu_device):
    """The flash operator's (empty) debug mask: changed by one caller, or made under inference mode, it is no other
    call's."""
    q = torch.randn(1, 2, 8, 64, device=gpu_device, dtype=torch.bfloat16)
    call = lambda: torch.ops.aten._scaled_dot_product_flash_attention(q, q, q)[8]
    with torch.inference_mode():
        first = call()
    second = call()
    assert first.is_inference() and not second.is_inference()
    second.resize_(3)
    assert call().shape == (0,)


@pytest.mark.gpu
def test_a_lazily_cloned_output_is_written_alone(amd, gpu_device):
    """torch._lazy_clone shares memory until one side is written: a call's output is written."""
    q = torch.randn(2, 4, 1, 64, device=gpu_device, dtype=torch.bfloat16)
    kv = torch.randn(2, 2, 40, 64, device=gpu_device).to(torch.float8_e4m3fn)
    one = torch.ones(2, device=gpu_device)
    want, _ = amd.decode_fp8kv(q, kv, kv, one, one)
    base = torch.zeros_like(want)
    got, _ = amd.decode_fp8kv(q, kv, kv, one, one, out=torch._lazy_clone(base))
    same, untouched = torch.equal(got, want), not bool(base.any())
    assert same and untouched


@pytest.mark.gpu
def test_other_threads_run_while_a_call_allocates(amd, gpu_device):
    """A thread that waits for the interpreter gets it while a call's outputs are allocated (which waits for the
    GPU where memory is short).  No thread is made to give it up by time here, and the outputs are kept (freeing a
    tensor lets others in), so only the allocation can."""
    q = torch.randn(1, 2, 64, 64, device=gpu_device, dtype=torch.bfloat16)
    p, host, go, ran, kept = amd._lib.FwdParams(), amd._lib.host(), threading.Event(), [], []
    thread = threading.Thread(target=lambda: (go.wait(), ran.append(True)))
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1000.0)
    try:
        thread.start()
        go.set()
        end = time.monotonic() + 3.0
        while not ran and time.monotonic() < end and len(kept) < 20000:
            kept.append(host.forward(C.addressof(p), q, q, q, None, True, False, 1.0, 0, False))
        in_time = bool(ran)
    finally:
        sys.setswitchinterval(interval)
        thread.join()
    assert in_time
