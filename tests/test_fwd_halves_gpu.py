"""The forward whose two halves of a workgroup share out its key tiles: tiles that do not divide by two, a half or a row
without a live key, ragged and narrow rows, and both sides of the line where it is taken.

Bounds: a probability and an output element are each rounded to the input dtype once (2^-9 relative for bfloat16,
2^-12 for float16), in the 2-norm below 2 * 2^-9 = 4e-3 with room for the sums; lse is float32, its exponents read
scores of at most 50 in units of 2^-23, 2e-5."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd(gpu_device):
    import torch_neuronx_amd as amd

    return amd


def _want(q, k, v, causal, lens, window, sink):
    rep = q.shape[1] // k.shape[1]
    q, k, v = q.double(), k.double().repeat_interleave(rep, 1), v.double().repeat_interleave(rep, 1)
    s = (q @ k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    i, j = torch.arange(q.shape[2], device=q.device)[:, None], torch.arange(k.shape[2], device=q.device)[None]
    dead = torch.zeros(q.shape[0], 1, q.shape[2], k.shape[2], dtype=torch.bool, device=q.device)
    if causal:
        dead = dead | (j > i)
    if window:
        dead = dead | ((j <= i - window) & (j >= 3))
    if lens is not None:
        dead = dead | (j >= lens[:, None, None, None])
    s = s.masked_fill(dead, -math.inf)
    if sink is not None:
        s = torch.cat([s, sink.double()[None, :, None, None].expand(*s.shape[:3], 1)], -1)
    lse = torch.logsumexp(s, -1)
    p = torch.exp(s - lse.masked_fill(lse == -math.inf, 0.0)[..., None])
    return p[..., : k.shape[2]] @ v, lse


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,Dv,causal,lens,window,sink", [
    (1, 8, 2, 97, 97, 128, 128, True, None, 0, False),      # four tiles, one key in the last
    (2, 4, 4, 160, 160, 64, 64, True, None, 0, False),      # five: three and two
    (1, 8, 8, 300, 300, 128, 128, True, None, 0, False),
    (1, 2, 1, 65, 1025, 128, 128, False, None, 0, False),   # more keys than rows
    (1, 4, 4, 500, 129, 64, 64, True, None, 0, False),      # rows past the last key
    (4, 4, 4, 256, 256, 64, 64, False, [256, 33, 32, 0], 0, False),  # a half, or both, without a key
    (3, 8, 4, 200, 200, 80, 72, True, [200, 1, 64], 0, False),
    (1, 4, 1, 513, 513, 120, 64, True, None, 0, True),
    (1, 8, 8, 700, 700, 128, 128, True, None, 100, False),  # window and leading keys
    (1, 6, 6, 1000, 1000, 64, 64, True, None, 70, True),
    (1, 16, 4, 769, 769, 128, 128, True, None, 0, False),   # 25 tiles, 112 workgroups of 128 rows: 64 rows
    (1, 24, 8, 769, 769, 128, 128, True, None, 0, False),   # 168: 128 rows
    (1, 28, 4, 1055, 1055, 128, 128, True, None, 0, False),
    (2, 28, 4, 800, 800, 128, 128, True, None, 0, False),   # 392 > 8 x 25: whole keys
    (1, 24, 24, 1055, 1055, 104, 104, True, [777], 0, True),
    (1, 32, 8, 801, 801, 128, 128, True, None, 0, False),   # 32 heads, whose last 128 rows are a quarter and three quarters full
    (2, 16, 4, 993, 993, 128, 128, True, [990, 400], 0, False),
    (1, 33, 11, 801, 801, 128, 128, True, None, 0, False),  # 231 > 8 x 28
])
def test_halves_of_a_workgroup(amd, gpu_device, dtype, B, Hq, Hkv, L, S, D, Dv, causal, lens, window, sink):
    g = torch.Generator(device=gpu_device).manual_seed(L + S + D)
    q, k, v = (torch.randn(s, generator=g, device=gpu_device).to(dtype) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, Dv)))
    k[:, :, S // 2] *= 4  # (a row's largest score in either half)
    n = None if lens is None else torch.tensor(lens, device=gpu_device, dtype=torch.int32)
    z = torch.linspace(-2, 6, Hq, device=gpu_device) if sink else None
    kw = dict(window=window, sink_keys=3) if window else {}
    out, lse = amd.sdpa_forward(q, k, v, is_causal=causal, kv_lens=n, sink_logit=z, **kw)
    want, want_lse = _want(q, k, v, causal, n, window, z)
    assert out.isfinite().all()
    assert float((out.double() - want).norm() / want.norm()) <= 4e-3
    live = want_lse != -math.inf
    assert bool((lse[~live] == -math.inf).all()) and bool((out[~live] == 0).all())
    assert float((lse.double() - want_lse)[live].abs().max()) <= 2e-5


def test_halves_under_a_verdict(amd, gpu_device):
    """A boolean mask that is causal with right padding: the kernel that reads the verdict, beside the masked one."""
    B, H, S = 2, 8, 333
    g = torch.Generator(device=gpu_device).manual_seed(3)
    q, k, v = (torch.randn(B, H, S, 128, generator=g, device=gpu_device).to(torch.bfloat16) for _ in range(3))
    lens = torch.tensor([S, 70], device=gpu_device)
    i = torch.arange(S, device=gpu_device)
    causal = (i[:, None] >= i[None])[None, None] & (i[None] < lens[:, None])[:, None, None]
    for mask in (causal, causal & ((i[:, None] == i[None]) | (i[None] % 7 != 3))[None, None]):
        out = torch.nn.functional.scaled_dot_product_attention(q, k, v, attn_mask=mask)
        s = (q.double() @ k.double().transpose(-1, -2).contiguous() / math.sqrt(128)).masked_fill(~mask, -math.inf)
        want = torch.softmax(s, -1) @ v.double()
        assert float((out.double() - want).norm() / want.norm()) <= 4e-3


def test_an_infinite_or_nan_row_stays_its_own(amd, gpu_device):
    q, k, v = (torch.randn(1, 2, 400, 64, device=gpu_device).to(torch.bfloat16) for _ in range(3))
    q[0, 0, 5] = float("nan")
    out, _ = amd.sdpa_forward(q, k, v)
    bad = out.isnan().any(-1)
    assert bool(bad[0, 0, 5]) and int(bad.sum()) == 1


def test_a_long_causal_call_and_its_prefix(amd, gpu_device):
    """The first rows depend on the first keys only.  A call that names its kernel sums them in the same order whatever
    follows; one that does not may share them out differently, which moves a result by its rounding (the bounds above)."""
    g = torch.Generator(device=gpu_device).manual_seed(8)
    q, k, v = (torch.randn(1, h, 16384, 128, generator=g, device=gpu_device).to(torch.bfloat16) for h in (4, 1, 1))
    n = 2048
    for force, bits in ((amd._lib.KERNEL_MFMA, True), (0, False)):
        out, lse = amd.sdpa_forward(q, k, v, is_causal=True, force_kernel=force)
        pre, pre_lse = amd.sdpa_forward(q[:, :, :n], k[:, :, :n], v[:, :, :n], is_causal=True, force_kernel=force)
        a, b = out[:, :, :n].double(), pre.double()
        if bits:
            assert torch.equal(a, b) and torch.equal(lse[:, :, :n], pre_lse)
        assert float((a - b).norm() / b.norm()) <= 4e-3
        assert float((lse[:, :, :n] - pre_lse).abs().max()) <= 4e-5  # (2e-5 of each)
