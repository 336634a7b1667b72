"""Row counts whose last workgroup has wavefronts without a row (they feed LDS and compute nothing): every kernel that
cuts 128 or 256 rows into wavefronts of 32, one to three and seven of them idle, with each kind of mask.

Bound, in the 2-norm against the float32 oracle on the kernel's inputs: P and the output are each rounded once to the input
dtype, 2^-9 relative in bf16, at most twice that together, 4e-3; a gradient adds dS and O, 8e-3.  float32: sums of up to a
thousand products, 1e-5 (about 80 ulp)."""

import pytest
import torch

from helpers import oracle_bwd, oracle_fwd, qkv, rel_err

pytestmark = pytest.mark.gpu


def _keep(kind, B, L, S):
    """The mask of a kind as the oracle takes it: a boolean (B,1,L,S) tensor."""
    i, j = torch.arange(L)[:, None], torch.arange(S)[None]
    keep = torch.ones(B, 1, L, S, dtype=torch.bool)
    if kind == "window":
        keep &= (j <= i) & (j > i - 70)
    if kind == "lens":
        keep &= j < torch.tensor([S - 31 * b for b in range(B)])[:, None, None, None]
    if kind == "mask":
        keep &= (i * 7 + j * 3) % 5 != 0
    return keep


@pytest.mark.parametrize("kind", ["plain", "causal", "window", "lens", "mask"])
@pytest.mark.parametrize("B,Hq,Hkv,L,D,dtype", [
    (12, 8, 8, 129, 64, torch.bfloat16),   # 128 rows: three idle
    (12, 12, 12, 197, 64, torch.bfloat16),  # one
    (6, 12, 6, 325, 64, torch.bfloat16),   # two
    (8, 16, 16, 270, 128, torch.bfloat16), # 256 in the backward: seven
    (3, 8, 4, 530, 104, torch.bfloat16),
    (2, 16, 16, 289, 256, torch.bfloat16),
    (8, 12, 12, 261, 64, torch.float32),
])
def test_against_the_oracle(gpu_device, B, Hq, Hkv, L, D, dtype, kind):
    import torch_neuronx_amd as amd

    q, k, v, do = qkv(B, Hq, Hkv, L, L, D, dtype=dtype, seed=L, with_do=True)
    keep, causal = _keep(kind, B, L, L), kind == "causal"
    kw = dict(is_causal=causal)
    if kind == "window":
        kw.update(is_causal=True, window=70)
    if kind == "lens":
        kw.update(kv_lens=torch.tensor([L - 31 * b for b in range(B)], dtype=torch.int32).clamp_min(0).to(gpu_device))
    if kind == "mask":
        kw.update(attn_bias=keep.to(gpu_device))
    dev = [t.to(gpu_device) for t in (q, k, v, do)]
    out, lse = amd.sdpa_forward(*dev[:3], **kw)
    grads = amd.sdpa_backward(dev[3], *dev[:3], out, lse, **kw)[:3]
    mask = None if kind in ("plain", "causal") else keep
    ro, rl = oracle_fwd(q, k, v, attn_mask=mask, is_causal=causal)
    want = oracle_bwd(do, q, k, v, ro, rl, attn_mask=mask, is_causal=causal)[:3]
    f32 = dtype is torch.float32
    assert rel_err(out, ro) <= (1e-5 if f32 else 4e-3)
    assert rel_err(lse, rl) <= 1e-5
    for name, a, r in zip(("dq", "dk", "dv"), grads, want):
        assert rel_err(a, r) <= (1e-5 if f32 else 8e-3), name
