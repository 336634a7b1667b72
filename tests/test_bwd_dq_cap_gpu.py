"""dQ above head dim 128 under a soft cap and no other functor (the cap's three stages ride on the dP products, the
masks of an edge tile follow in one block): query rows and keys around the 32-wide tiles and 128-row workgroups, both
widths the kernel is built for, windows with and without sink keys, key counts, a cap that saturates.

Bound, against dS = P (dP - delta) (1 - tanh^2) in float64 on the kernel's inputs, the forward's rounded output (whose
rounding delta takes up, many times over where a row has a probability near one) among them: dS and the gradient
are each rounded once to the input dtype, 2^-9 relative in bf16, 2^-12 in f16; twice their sum, 8e-3 and 1e-3."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [
    # B, Hq, Hkv, L, S, D, Dv, causal, window, sinks, lens, cap, size of the scores
    (1, 1, 1, 1, 2, 256, 256, False, 0, 0, None, 50.0, 1.0),
    (1, 2, 1, 33, 31, 192, 128, False, 0, 0, None, 20.0, 1.0),
    (2, 2, 2, 129, 129, 192, 128, True, 0, 0, [129, 65], 30.0, 1.0),
    (1, 4, 2, 300, 300, 160, 96, True, 40, 3, None, 5.0, 1.0),
    (2, 2, 2, 128, 128, 256, 256, True, 0, 0, None, 50.0, 1.0),
    (3, 2, 1, 65, 161, 256, 200, False, 0, 0, [161, 0, 32], 50.0, 1.0),
    (1, 2, 2, 257, 257, 256, 256, True, 32, 33, None, 50.0, 1.0),
    (1, 2, 2, 160, 160, 256, 256, True, 2, 0, None, 50.0, 1.0),
    (1, 2, 2, 200, 200, 256, 256, True, 64, 0, None, 2.0, 8.0),   # most scores at the cap
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "L%d_S%d_D%d_%d_c%d_w%d_sink%d_cap%g" % (*c[3:10], c[11]))
def test_against_float64(gpu_device, case, dtype):
    import torch_neuronx_amd as amd

    B, Hq, Hkv, L, S, D, Dv, causal, window, sinks, lens, cap, size = case
    dev, rep = gpu_device, Hq // Hkv
    g = torch.Generator(device=dev).manual_seed(L * 11 + S)
    q, k, v, do = (torch.randn(s, generator=g, device=dev).to(dtype) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, Dv), (B, Hq, L, Dv)))
    q = q * size
    kw = dict(is_causal=causal, softcap=cap)
    if window:
        kw.update(window=window, sink_keys=sinks)
    lens_t = torch.tensor([S] * B if lens is None else lens, device=dev)
    if lens is not None:
        kw["kv_lens"] = lens_t.to(torch.int32)
        for b, n in enumerate(lens):  # (what lies behind a batch's keys takes no part, whatever it is)
            k[b, :, n:], v[b, :, n:] = math.nan, math.nan
    out, lse = amd.sdpa_forward(q, k, v, **kw)
    dq = amd.sdpa_backward(do, q, k, v, out, lse, **kw)[0]
    Q, DO = q.double(), do.double()
    K, V = (x.double().nan_to_num(0.0).repeat_interleave(rep, 1) for x in (k, v))
    i, j = torch.arange(L, device=dev)[:, None], torch.arange(S, device=dev)[None]
    th = torch.tanh(Q @ K.transpose(-1, -2).contiguous() / (math.sqrt(D) * cap))
    dead = (j[None] >= lens_t[:, None, None])[:, None].expand(B, 1, L, S).clone()
    if causal:
        dead |= j > i
    if window:
        dead |= (j < i - window + 1) & (j >= sinks)
    P = torch.softmax((cap * th).masked_fill(dead, -1e300), -1).masked_fill(dead, 0.0)
    delta = (DO * out.double()).sum(-1, keepdim=True)
    want = P * (DO @ V.transpose(-1, -2).contiguous() - delta) * (1 - th * th) @ K / math.sqrt(D)
    assert torch.isfinite(dq).all()
    far = float((dq.double() - want).norm() / want.norm())
    assert far <= (8e-3 if dtype is torch.bfloat16 else 1e-3), far
