"""The backward at head dims up to 64 with few workgroups (dQ and dK/dV in one launch): tile edges, both sides of the rule's
lines, grouped heads with and without a split of the items, key counts, narrow rows, rows without a key.

Bounds: P, dS and a gradient are each rounded to the input dtype once (2^-9 relative for bfloat16, 2^-12 for float16): in
the 2-norm below 3 * 2^-9 = 6e-3 and 3 * 2^-12 = 8e-4."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,bound", [(torch.bfloat16, 6e-3), (torch.float16, 8e-4)])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,causal,lens", [
    (1, 1, 1, 1, 1, 64, False, None),
    (1, 3, 3, 65, 63, 64, True, None),          # workgroups that are no multiple of eight
    (2, 6, 6, 129, 300, 48, False, [300, 17]),
    (3, 4, 2, 33, 200, 64, True, [0, 200, 64]),  # a batch without a key
    (1, 16, 4, 1021, 1021, 64, True, None),     # parts
    (2, 12, 4, 192, 192, 64, True, None),       # three heads a kv head
    (1, 28, 4, 150, 150, 64, True, None),
    (1, 16, 2, 193, 193, 56, True, [150]),      # ... parts, past three query tiles: one
    (4, 32, 32, 129, 130, 64, False, None),     # 256 query and 256 key blocks: 512 in all, the last size here
    (2, 32, 32, 256, 256, 64, False, None),     # 256 in all are 2 * 32 * 2 * 2
    (8, 12, 12, 511, 511, 64, True, None),      # 768 in all
    (2, 16, 16, 1100, 700, 40, True, [700, 699]),
    (4, 16, 16, 1024, 1024, 64, True, None),    # 1024 in all
    # ... and past each: up to six query tiles 512, from seven 768, from fifteen 1024, with grouped heads 768
    (32, 8, 8, 128, 128, 64, True, None), (33, 8, 8, 128, 100, 64, True, [100 - i for i in range(33)]),
    (16, 8, 8, 256, 200, 56, True, None), (17, 8, 8, 256, 256, 64, True, None), (11, 8, 8, 384, 384, 64, True, None),
    (13, 8, 8, 500, 500, 64, True, None), (8, 16, 8, 512, 512, 64, True, None), (9, 16, 8, 449, 449, 64, True, None),
    (8, 8, 8, 896, 896, 64, True, None), (7, 8, 8, 896, 640, 64, True, None), (7, 8, 8, 1025, 1025, 64, True, None), (8, 8, 8, 1025, 1000, 48, True, None),
    # not causal, up to five query tiles 512 in all, from six and with three heads a kv head 768, 704 with two, and past each
    (32, 8, 8, 128, 100, 64, False, None), (33, 8, 8, 127, 128, 64, False, [128 - i for i in range(33)]),
    (16, 8, 8, 321, 321, 64, False, None), (17, 8, 8, 384, 300, 48, False, None), (16, 8, 8, 320, 320, 64, False, None),
    (7, 16, 8, 400, 400, 64, False, None), (8, 16, 8, 400, 500, 64, False, None),
    (6, 8, 4, 934, 934, 64, False, None), (2, 8, 4, 1498, 1498, 48, False, [1498, 1000]),  # ... 768 with split items
    (38, 16, 4, 65, 65, 64, False, None), (39, 16, 4, 65, 65, 64, False, None), (48, 12, 4, 65, 65, 64, False, None),
    # causal: three workgroups a compute unit above 640 and up to 768, up to eight query tiles
    (10, 8, 8, 448, 448, 64, True, None), (11, 8, 8, 448, 448, 64, True, None), (12, 8, 8, 500, 512, 40, True, [512 - 40 * i for i in range(12)]),
    (12, 8, 8, 512, 513, 64, True, None), (12, 8, 8, 513, 512, 64, True, None), (9, 8, 8, 640, 630, 64, True, None), (9, 8, 8, 641, 630, 64, True, None),
    # ... and long chains a block ahead
    (25, 2, 2, 1024, 1024, 64, True, None), (26, 2, 2, 1000, 1024, 48, True, [1024 - 30 * i for i in range(26)]), (24, 2, 2, 1217, 1280, 64, True, None), (11, 2, 2, 2561, 2500, 64, True, None),
])
def test_gradients(gpu_device, dtype, bound, B, Hq, Hkv, L, S, D, causal, lens):
    import torch_neuronx_amd as amd

    g = torch.Generator(device=gpu_device).manual_seed(L + S)
    make = lambda H, n: torch.randn(B, n, H, D, generator=g, device=gpu_device).to(dtype).transpose(1, 2)
    q, do, k, v = make(Hq, L), make(Hq, L), make(Hkv, S), make(Hkv, S)
    n = None if lens is None else torch.tensor(lens, dtype=torch.int32, device=gpu_device)
    out, lse = amd.sdpa_forward(q, k, v, is_causal=causal, kv_lens=n)
    got = amd.sdpa_backward(do, q, k, v, out, lse, is_causal=causal, kv_lens=n)[:3]
    rep = Hq // Hkv
    kd, vd = (t.double().repeat_interleave(rep, 1) for t in (k, v))
    s = q.double() @ kd.transpose(-1, -2).contiguous() / math.sqrt(D)
    i, j = torch.arange(L, device=gpu_device)[:, None], torch.arange(S, device=gpu_device)[None]
    live = (j <= i if causal else j >= 0).expand(B, 1, L, S)
    if n is not None:
        live = live & (j < n[:, None, None, None])
    p = torch.softmax(s.masked_fill(~live, -math.inf), -1).nan_to_num(0.0)
    dp = do.double() @ vd.transpose(-1, -2).contiguous()
    ds = p * (dp - (dp * p).sum(-1, keepdim=True)) / math.sqrt(D)
    fold = lambda t: t.view(B, Hkv, rep, S, D).sum(2)
    want = (ds @ kd, fold(ds.transpose(-1, -2).contiguous() @ q.double()), fold(p.transpose(-1, -2).contiguous() @ do.double()))
    for a, b in zip(got, want):
        # (one key: dS is 0 but for the rounding of the output that delta is formed from)
        assert float((a.double() - b).norm()) <= bound * max(float(b.norm()), 0.2 * math.sqrt(b.numel()))
