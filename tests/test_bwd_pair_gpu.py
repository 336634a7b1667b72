"""Backward at head dims above 128, full width, without a bias or dropout (the dK/dV kernel that puts two wavefronts on
32 keys): sizes around its 32-row items and 128-key blocks, one to a few items, narrow rows, grouped
heads, key counts that leave blocks and wavefronts without a key, windows with and without sink keys, each score functor,
query tiles shared out over workgroups.

Bound, against the same attention in float64 on the kernel's inputs: P, dS, O (through delta) and the gradient are
each rounded once to the input dtype, 2^-9 relative in bf16, 2^-12 in f16, and P once more times the derivative of a
functor, which adds up to at most four times that in the 2-norm of a gradient: 8e-3 and 1e-3."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd(gpu_device):
    import torch_neuronx_amd as amd

    return amd


def _functors(dev, names, Hq, S, B, L):
    g = torch.Generator(device=dev).manual_seed(5)
    kw = {}
    if "alibi" in names:
        kw["alibi_slopes"] = torch.linspace(0.02, 0.4, Hq, device=dev)
    if "bias" in names:
        kw["key_bias"] = torch.randn(Hq, S, generator=g, device=dev)
    if "weight" in names:
        kw["key_weight"] = torch.rand(Hq, S, generator=g, device=dev) + 0.5
    if "docs" in names:
        kw["doc_ids_q"] = (torch.arange(L, device=dev) // 50).to(torch.int32).expand(B, L).contiguous()
        kw["doc_ids_k"] = (torch.arange(S, device=dev) // 50).to(torch.int32).expand(B, S).contiguous()
    return kw


CASES = [
    # B, Hq, Hkv, L, S, D, Dv, causal, window, sinks, lens, cap, functors
    (1, 1, 1, 1, 1, 256, 256, False, 0, 0, None, 0.0, ""),
    (1, 2, 2, 31, 33, 256, 256, False, 0, 0, None, 0.0, ""),
    (1, 2, 1, 33, 129, 136, 136, False, 0, 0, None, 0.0, ""),
    (2, 4, 2, 129, 129, 256, 160, True, 0, 0, None, 0.0, ""),
    (3, 2, 2, 100, 193, 160, 160, False, 0, 0, [193, 0, 65], 0.0, ""),
    (2, 2, 2, 300, 300, 256, 256, True, 0, 0, [300, 129], 0.0, ""),
    (1, 4, 2, 300, 300, 256, 256, True, 40, 0, None, 0.0, ""),
    (1, 2, 2, 261, 261, 256, 256, True, 70, 5, None, 5.0, ""),
    (2, 4, 4, 200, 200, 256, 256, True, 64, 0, [200, 77], 50.0, ""),
    (1, 2, 1, 97, 225, 200, 200, False, 0, 0, None, 2.0, ""),
    (1, 16, 2, 640, 160, 256, 256, False, 0, 0, None, 30.0, ""),   # a key block's query tiles go to several workgroups
    (1, 8, 8, 700, 700, 256, 256, True, 0, 0, None, 0.0, ""),      # ... under a causal mask
    (1, 2, 2, 130, 130, 256, 256, True, 0, 0, None, 0.0, "alibi"),
    (1, 4, 2, 100, 150, 256, 256, False, 0, 0, None, 20.0, "bias weight"),
    (2, 2, 2, 190, 190, 256, 256, True, 0, 0, None, 10.0, "alibi docs"),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "H%d_%d_L%d_S%d_D%d_%d_c%d_w%d_cap%g_%s" % (c[1:9] + (c[11], c[12].replace(" ", "+"))))
def test_against_float64(amd, gpu_device, case, dtype):
    B, Hq, Hkv, L, S, D, Dv, causal, window, sinks, lens, cap, names = case
    dev, rep = gpu_device, Hq // Hkv
    g = torch.Generator(device=dev).manual_seed(L * 7 + S)
    q, k, v, do = (torch.randn(s, generator=g, device=dev).to(dtype) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, Dv), (B, Hq, L, Dv)))
    kw = dict(is_causal=causal, **_functors(dev, names, Hq, S, B, L))
    if cap:
        kw["softcap"] = cap
    if window:
        kw.update(window=window, sink_keys=sinks)
    lens_t = torch.tensor([S] * B if lens is None else lens, device=dev)
    if lens is not None:
        kw["kv_lens"] = lens_t.to(torch.int32)
        for b, n in enumerate(lens):  # (what lies behind a batch's keys takes no part, whatever it is)
            k[b, :, n:], v[b, :, n:] = math.nan, math.nan
    out, lse = amd.sdpa_forward(q, k, v, **kw)
    dq, dk, dv, _ = amd.sdpa_backward(do, q, k, v, out, lse, **kw)[:4]
    Q, DO = q.double().requires_grad_(), do.double()
    K, V = (t.double().nan_to_num(0.0).requires_grad_() for t in (k, v))
    i, j = torch.arange(L, device=dev)[:, None], torch.arange(S, device=dev)[None]
    s = Q @ K.repeat_interleave(rep, 1).transpose(-1, -2).contiguous() / math.sqrt(D)
    if "key_weight" in kw:
        s = s * kw["key_weight"].double()[None, :, None]
    if "key_bias" in kw:
        s = s + kw["key_bias"].double()[None, :, None]
    if "alibi_slopes" in kw:
        s = s + kw["alibi_slopes"].double()[None, :, None, None] * (j - i)
    if cap:
        s = cap * torch.tanh(s / cap)
    dead = (j[None] >= lens_t[:, None, None])[:, None].expand(B, 1, L, S).clone()
    if causal:
        dead |= j > i
    if window:
        dead |= (j < i - window + 1) & (j >= sinks)
    if "doc_ids_q" in kw:
        dead |= (kw["doc_ids_q"][:, :, None] != kw["doc_ids_k"][:, None, :])[:, None]
    P = torch.softmax(s.masked_fill(dead, -1e300), -1).masked_fill(dead, 0.0)
    want = torch.autograd.grad(P @ V.repeat_interleave(rep, 1), (Q, K, V), DO)
    for name, a, r in zip(("dq", "dk", "dv"), (dq, dk, dv), want):
        assert torch.isfinite(a).all(), name
        far = float((a.double() - r).norm() / r.norm().clamp_min(1e-30)) if float(r.norm()) else float(a.double().norm())
        assert far <= (8e-3 if dtype is torch.bfloat16 else 1e-3), (name, far)
    if lens is not None:
        for b, n in enumerate(lens):
            assert not dk[b, :, n:].any() and not dv[b, :, n:].any()
