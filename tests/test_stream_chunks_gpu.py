"""Calls whose streams (a (batch, kv head)'s keys and values) an XCD takes in chunks, forward, backward and with dropout: every
(batch, head, row) is computed, once, also where the last chunk is a smaller one or some XCDs serve a stream less than others.

Bound, against the same attention in float64 on the kernel's inputs: P and the output are each rounded once to bf16,
2^-9 relative, which adds up to at most twice that in the 2-norm: 4e-3; the log-sum-exp is a float32 sum, 1e-5."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,D,causal", [
    (24, 12, 12, 577, 64, False),   # 36 streams an XCD in chunks of 7
    (11, 32, 16, 333, 104, False),  # 22 in chunks of 7, two heads a kv head
    (12, 8, 8, 900, 128, False),    # 12 (5.5 MB) at a time, 12 of 1030 keys (6.3 MB) in chunks of four
    (12, 8, 8, 1030, 128, False),
    (11, 16, 8, 1100, 72, False),   # 11 in chunks of four, the last one of three
    (10, 32, 8, 1100, 128, False),  # four heads a kv head: one by one
    (43, 24, 24, 1024, 64, True),   # 129 in chunks of 16: eight and a last one of a single stream
    (19, 16, 8, 2048, 128, True),   # 19 in chunks of 4 are fewer than eight chunks: one after the other
    (9, 8, 8, 4096, 256, True),     # 9 of 4 MB each: at a time
    (17, 8, 8, 2830, 128, True),    # 17, two of which fill the L2: in five chunks of four, the last one of a single stream
    (35, 8, 8, 1500, 128, True),    # 35, chunks of five
    (35, 16, 8, 2048, 128, True),   # 35: nine
    (31, 12, 12, 512, 64, False),   # 372 streams: the last four XCDs serve one less, in chunks of 8
    (21, 28, 4, 512, 128, True),    # 84, seven heads a kv head, no chunks
    (9, 12, 12, 785, 64, False),    # 108 would need a turn of workgroups more: not pinned
])
def test_every_stream_is_computed(gpu_device, B, Hq, Hkv, S, D, causal):
    import torch_neuronx_amd as amd

    g = torch.Generator(device=gpu_device).manual_seed(S)
    q, k, v = (torch.randn(B, h, S, D, generator=g, device=gpu_device).to(torch.bfloat16) for h in (Hq, Hkv, Hkv))
    out, lse = amd.sdpa_forward(q, k, v, is_causal=causal)
    dead = ~torch.ones(S, S, dtype=torch.bool, device=gpu_device).tril() if causal else None
    for b in range(B):
        K, V = (t[b].double().repeat_interleave(Hq // Hkv, 0) for t in (k, v))
        s = q[b].double() @ K.transpose(-1, -2).contiguous() / math.sqrt(D)
        if causal:
            s.masked_fill_(dead, -math.inf)
        far = (lse[b] - torch.logsumexp(s, -1)).abs().amax(-1)
        assert float(far.max()) <= 1e-5, b
        ref = torch.softmax(s, -1) @ V
        far = (out[b].double() - ref).norm(dim=(-2, -1)) / ref.norm(dim=(-2, -1))
        assert float(far.max()) <= 4e-3, (b, far)


@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,causal,lens", [
    (57, 8, 8, 1100, 1100, 128, True, None),    # 57 streams an XCD in chunks of 7, in both kernels
    (9, 16, 8, 3000, 300, 104, False, None),    # 9 one by one in dK/dV, which walks Q and dO of two heads
    (18, 4, 4, 5000, 400, 128, True, None),     # 9, one of which fills the L2: in three chunks of three in dK/dV
    (20, 8, 4, 400, 5000, 128, True, None),     # 10: four, four and two in dQ
    (13, 48, 48, 1000, 1000, 128, False, 1000), # 78 in chunks of 8, key counts
    (11, 16, 16, 1024, 1024, 64, True, None),   # 22 at a time at head dim 64
    (25, 8, 8, 900, 900, 64, False, None),      # 25 in chunks of 4
    (31, 12, 12, 512, 512, 64, False, None),    # 372 streams: the last four XCDs serve one less
    (15, 12, 12, 500, 500, 64, True, None),     # 180
    (5, 12, 4, 300, 300, 64, True, None),       # 20: not pinned
    (29, 12, 4, 300, 300, 64, True, None),      # 116, three heads a kv head
    (70, 8, 8, 200, 200, 64, True, None),       # causal, up to three key blocks: 70 (3.6 MB) in five chunks of 14, 64 at a time
    (64, 8, 8, 200, 200, 64, True, None),
    (32, 8, 8, 300, 288, 64, True, None),       # three, 32 at a time, 33 of 288 keys and rows in three chunks, of 287 at a time
    (33, 8, 8, 288, 288, 64, True, None),
    (33, 8, 8, 287, 290, 64, True, None),
    (33, 16, 8, 300, 300, 64, True, None),      # two heads a kv head: 33 of 5 MB for dK/dV
    (56, 8, 8, 270, 270, 64, True, None),       # 56 of 3.9 MB at a time, 62 of 4.3 in four chunks
    (62, 8, 8, 270, 270, 64, True, None),
    (24, 8, 8, 500, 500, 64, True, None),       # four: 24 at a time, 25 and 31 in two chunks, 25 of 2.3 MB at a time
    (25, 8, 8, 400, 390, 64, True, None),
    (31, 8, 8, 385, 512, 64, True, None),
    (25, 8, 8, 385, 360, 56, True, None),       # (three key blocks)
    (32, 8, 8, 500, 500, 64, True, None),       # 32 of 4.1 MB in two of 16, of 3.9 at a time
    (32, 8, 8, 480, 480, 64, True, None),
    (33, 8, 8, 490, 490, 64, True, None),       # 33 and 42 in three, 43 in six
    (42, 8, 8, 400, 400, 64, True, None),
    (43, 8, 8, 400, 400, 64, True, None),
    (28, 16, 8, 400, 400, 64, True, None),      # two heads a kv head: 28 of 5.7 MB for dK/dV in four
    (19, 12, 12, 1100, 900, 64, True, None),    # 228: the last four XCDs serve one less than 29, at a time
    (12, 16, 16, 700, 4100, 64, True, None),    # 24 of 4100 keys, more than 24 MB: in two chunks of 12 for dQ
    (12, 16, 16, 4100, 700, 48, True, None),    # ... of 4100 rows for dK/dV
])
def test_every_gradient_is_computed(gpu_device, B, Hq, Hkv, L, S, D, causal, lens):
    """The same in the backward.  P, dS, O and the gradients are rounded once each: 8e-3, as in test_bwd_d64_gpu.py."""
    import torch_neuronx_amd as amd

    g = torch.Generator(device=gpu_device).manual_seed(S)
    q, k, v, do = (torch.randn(B, h, n, D, generator=g, device=gpu_device).to(torch.bfloat16) for h, n in ((Hq, L), (Hkv, S), (Hkv, S), (Hq, L)))
    kw = dict(is_causal=causal)
    if lens:
        kw["kv_lens"] = torch.tensor([lens - 37 * i for i in range(B)], dtype=torch.int32, device=gpu_device)
    out, lse = amd.sdpa_forward(q, k, v, **kw)
    grads = amd.sdpa_backward(do, q, k, v, out, lse, **kw)[:3]
    rep = Hq // Hkv
    for b in range(B):
        n = lens - 37 * b if lens else S
        Q, DO = q[b].double(), do[b].double()
        K, V = (t[b, :, :n].double().repeat_interleave(rep, 0) for t in (k, v))
        s = Q @ K.transpose(-1, -2).contiguous() / math.sqrt(D)
        if causal:
            s.masked_fill_(~torch.ones(L, n, dtype=torch.bool, device=gpu_device).tril(), -math.inf)
        P = torch.softmax(s, -1)
        dS = P * (DO @ V.transpose(-1, -2).contiguous() - (DO * (P @ V)).sum(-1, keepdim=True)) / math.sqrt(D)
        want = (dS @ K, (dS.transpose(-1, -2).contiguous() @ Q).view(Hkv, rep, n, D).sum(1), (P.transpose(-1, -2).contiguous() @ DO).view(Hkv, rep, n, D).sum(1))
        for name, a, r in zip(("dq", "dk", "dv"), grads, want):
            got = a[b] if name == "dq" else a[b, :, :n]
            far = (got.double() - r).norm(dim=(-2, -1)) / r.norm(dim=(-2, -1))
            assert float(far.max()) <= 8e-3, (name, b, far)


@pytest.mark.parametrize("lens", [False, True])
@pytest.mark.parametrize("B,H,L,S,causal", [
    (26, 8, 900, 700, False),   # 26 streams an XCD, in chunks of 5 and a last one of a single stream (dQ, by the keys) and of 4 and 2 (dK/dV, by the rows)
    (31, 12, 512, 512, False),  # 372: the last four XCDs serve one less than 47, in chunks of 8
    (13, 12, 300, 400, False),  # 156: 20 at a time, the last four 19
    (45, 8, 500, 470, True),    # causal, four key blocks: 45 in chunks of 8 and 5
    (61, 8, 1000, 1000, True),  # more than 15 MB: 61 in chunks of 16 and 13
    (37, 8, 300, 384, True),    # three: 37 in chunks of 13 and 11
    (29, 8, 450, 512, True),    # 29 in chunks of 15 and 14
    (35, 8, 500, 460, True),    # 35 in chunks of 12 and 11
    (23, 12, 300, 300, True),   # three: 276 of which the last four XCDs serve one less than 35
])
def test_keep_bits_reach_every_stream(gpu_device, B, H, L, S, causal, lens):
    """With dropout: the dQ kernel leaves the keep bits that the dK/dV kernel reads, each in the order of its own chunks."""
    import torch_neuronx_amd as amd

    g = torch.Generator(device=gpu_device).manual_seed(S)
    D, p = 64, 0.25
    q, k, v, do = (torch.randn(B, H, n, D, generator=g, device=gpu_device).to(torch.bfloat16) for n in (L, S, S, L))
    keep = amd.ops.padded_keep_mask(B, H, L, S, gpu_device).bernoulli_(1 - p, generator=g)
    kw = dict(is_causal=causal, dropout_p=p, dropout_keep=keep)
    if lens:
        kw["kv_lens"] = torch.tensor([S - 9 * i for i in range(B)], dtype=torch.int32, device=gpu_device)
    out, lse = amd.sdpa_forward(q, k, v, **kw)
    grads = amd.sdpa_backward(do, q, k, v, out, lse, **kw)[:3]
    for b in range(B):
        n = S - 9 * b if lens else S
        Q, DO, K, V, kp = q[b].double(), do[b].double(), k[b, :, :n].double(), v[b, :, :n].double(), keep[b, :, :, :n].double() / (1 - p)
        s = Q @ K.transpose(-1, -2).contiguous() / math.sqrt(D)
        if causal:
            s.masked_fill_(~torch.ones(L, n, dtype=torch.bool, device=gpu_device).tril(), -math.inf)
        P = torch.softmax(s, -1)
        dS = P * ((DO @ V.transpose(-1, -2).contiguous()) * kp - (DO * ((P * kp) @ V)).sum(-1, keepdim=True)) / math.sqrt(D)
        want = (dS @ K, dS.transpose(-1, -2).contiguous() @ Q, (P * kp).transpose(-1, -2).contiguous() @ DO)
        for name, a, r in zip(("dq", "dk", "dv"), grads, want):
            got = a[b] if name == "dq" else a[b, :, :n]
            far = (got.double() - r).norm(dim=(-2, -1)) / r.norm(dim=(-2, -1))
            assert float(far.max()) <= 8e-3, (name, b, far)
