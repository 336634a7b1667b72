"""Backward at head dims up to 64 (the pair of kernels that keeps three workgroups on a compute unit): sizes around
its 32-row blocks and 64-row tiles, narrow rows, grouped heads, key counts, dropout over numbers of keys that
are no multiple of four or of a word of keep bits, items shared out over workgroups, many streams per XCD.

Bound, against the same attention in float64 on the kernel's inputs: P, dS, O (through delta) and the gradient are
each rounded once to the input dtype, 2^-9 relative in bf16, 2^-12 in f16, which adds up to at most four
times that in the 2-norm of a gradient: 8e-3 and 1e-3."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd(gpu_device):
    import torch_neuronx_amd as amd

    return amd


def _check(amd, dev, B, Hq, Hkv, L, S, D, causal, dtype, lens, p):
    g = torch.Generator(device=dev).manual_seed(L * 7 + S)
    q, k, v, do = (torch.randn(s, generator=g, device=dev).to(dtype) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, D), (B, Hq, L, D)))
    kw = dict(is_causal=causal)
    if lens is not None:
        kw["kv_lens"] = torch.tensor(lens, dtype=torch.int32, device=dev)
    keep = None
    if p:
        keep = amd.ops.padded_keep_mask(B, Hq, L, S, dev).bernoulli_(1 - p, generator=g)
        kw.update(dropout_p=p, dropout_keep=keep)
    out, lse = amd.sdpa_forward(q, k, v, **kw)
    dq, dk, dv, _ = amd.sdpa_backward(do, q, k, v, out, lse, **kw)
    rep = Hq // Hkv
    Q, DO = q.double(), do.double()
    K, V = (t.double().repeat_interleave(rep, 1) for t in (k, v))
    s = Q @ K.transpose(-1, -2).contiguous() / math.sqrt(D)
    dead = torch.zeros(B, 1, L, S, dtype=torch.bool, device=dev)
    if causal:
        dead |= ~torch.ones(L, S, dtype=torch.bool, device=dev).tril()
    if lens is not None:
        dead |= torch.arange(S, device=dev)[None, None, None] >= kw["kv_lens"][:, None, None, None]
    P = torch.softmax(s.masked_fill(dead, -math.inf), -1).nan_to_num(0.0)
    kp = 1.0 if keep is None else keep.double() / (1 - p)
    O = (P * kp) @ V
    dP = (DO @ V.transpose(-1, -2).contiguous()) * kp
    dS = P * (dP - (DO * O).sum(-1, keepdim=True)) / math.sqrt(D)
    want = (dS @ K, (dS.transpose(-1, -2).contiguous() @ Q).view(B, Hkv, rep, S, D).sum(2),
            ((P * kp).transpose(-1, -2).contiguous() @ DO).view(B, Hkv, rep, S, D).sum(2))
    for name, a, r in zip(("dq", "dk", "dv"), (dq, dk, dv), want):
        assert torch.isfinite(a).all(), name
        far = float((a.double() - r).norm() / r.norm().clamp_min(1e-30))
        assert far <= (8e-3 if dtype is torch.bfloat16 else 1e-3), (name, far)


CASES = [
    # B, Hq, Hkv, L, S, D, causal, lens, p
    (1, 1, 1, 31, 33, 64, False, None, 0.0),
    (2, 2, 2, 65, 127, 64, False, None, 0.0),
    (1, 4, 2, 129, 129, 64, True, None, 0.0),
    (1, 2, 1, 200, 90, 64, True, None, 0.0),
    (1, 2, 1, 90, 200, 64, True, None, 0.0),
    (3, 2, 2, 100, 193, 64, False, [193, 0, 64], 0.0),
    (2, 2, 2, 96, 160, 40, True, [97, 160], 0.0),
    (1, 2, 2, 70, 70, 8, False, None, 0.0),
    (2, 2, 2, 64, 197, 64, False, None, 0.25),
    (1, 4, 2, 131, 131, 64, True, None, 0.25),
    (3, 2, 2, 130, 261, 48, False, [261, 33, 0], 0.25),
    (2, 8, 1, 500, 140, 64, False, None, 0.1),   # the items of a key block go to several workgroups
    (1, 8, 1, 700, 300, 64, True, None, 0.0),
    (8, 20, 20, 130, 520, 64, False, None, 0.1),  # 20 streams per XCD, chunks of 15
    (4, 10, 10, 600, 600, 64, True, None, 0.0),  # 5 streams per XCD; key blocks of 384 to 512 workgroups
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_H%d_%d_L%d_S%d_D%d_c%d_p%s" % (c[:7] + (c[8],)))
def test_against_float64(amd, gpu_device, case, dtype):
    B, Hq, Hkv, L, S, D, causal, lens, p = case
    _check(amd, gpu_device, B, Hq, Hkv, L, S, D, causal, dtype, lens, p)
