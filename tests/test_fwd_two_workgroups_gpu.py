"""The forward of 129 to 256 rows in two workgroups a head instead of one: both sides of each line of the rule, rows that leave
the second workgroup one wavefront or all four, narrow heads, key counts and a window, against float64.

Bounds: a probability and an output element are each rounded to float16 once (2^-12 relative), in the 2-norm below
2 * 2^-12 = 5e-4 with room for the sums; lse is float32, its exponents read scores of at most 50 in units of 2^-23, 2e-5."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,L,S,D,causal,lens,window", [
    (22, 4, 129, 129, 64, False, None, 0),    # 264 workgroups of 64 rows; the second workgroup has one row
    (43, 4, 160, 161, 64, True, None, 0),     # 516
    (128, 4, 225, 225, 64, False, None, 0),   # 512 heads past 224 rows: two
    (129, 4, 225, 225, 64, False, None, 0),   # ... 516: one
    (129, 4, 256, 256, 64, True, None, 0),
    (43, 6, 197, 700, 64, False, None, 0),    # 258 heads, more keys than rows: two
    (40, 6, 197, 700, 64, False, None, 0),    # 240 heads over more than 480 keys: one workgroup
    (48, 8, 200, 200, 56, False, list(range(0, 48 * 4, 4)), 0),
    (65, 4, 255, 255, 64, True, None, 33),
    (32, 4, 193, 193, 128, True, None, 0),    # 128 heads
    (43, 3, 193, 193, 128, False, None, 0),   # 129: one workgroup
    (20, 6, 256, 130, 80, False, None, 0),
])
def test_two_workgroups_a_head(gpu_device, B, H, L, S, D, causal, lens, window):
    import torch_neuronx_amd as amd

    g = torch.Generator(device=gpu_device).manual_seed(L + S + D)
    q, k, v = (torch.randn(B, H, n, D, generator=g, device=gpu_device).half() for n in (L, S, S))
    n = None if lens is None else torch.tensor(lens, device=gpu_device, dtype=torch.int32)
    out, lse = amd.sdpa_forward(q, k, v, is_causal=causal, kv_lens=n, **(dict(window=window) if window else {}))
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) / math.sqrt(D)
    i, j = torch.arange(L, device=gpu_device)[:, None], torch.arange(S, device=gpu_device)[None]
    dead = (j > i if causal else j < 0)[None, None]
    if window:
        dead = dead | (j <= i - window)
    if lens is not None:
        dead = dead | (j >= n[:, None, None, None])
    s = s.masked_fill(dead, -math.inf)
    want_lse = torch.logsumexp(s, -1)
    live = want_lse != -math.inf
    want = torch.exp(s - want_lse.masked_fill(~live, 0.0)[..., None]) @ v.double()
    assert float((out.double() - want).norm() / want.norm()) <= 5e-4
    assert bool((out[~live] == 0).all()) and bool((lse[~live] == -math.inf).all())
    assert float((lse.double() - want_lse)[live].abs().max()) <= 2e-5
