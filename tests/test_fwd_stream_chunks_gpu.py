"""Forward calls whose streams (a (batch, kv head)'s keys and values) an XCD takes in chunks: every (batch, head, row) is
computed, once, also where the last chunk is a smaller one.

Bound, against the same attention in float64 on the kernel's inputs: P and the output are each rounded once to bf16,
2^-9 relative, which adds up to at most twice that in the 2-norm: 4e-3; the log-sum-exp is a float32 sum, 1e-5."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,Hq,Hkv,S,D,causal", [
    (24, 12, 12, 577, 64, False),   # 36 streams an XCD in chunks of 7
    (11, 32, 16, 333, 104, False),  # 22 in chunks of 7, two heads a kv head
    (43, 24, 24, 1024, 64, True),   # 129 in chunks of 16: eight and a last one of a single stream
    (19, 16, 8, 2048, 128, True),   # 19 in chunks of 4 are fewer than eight chunks: one after the other
    (35, 16, 8, 2048, 128, True),   # 35: nine
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
