"""The forward with a soft cap and no other score functor (its variant of the 32-row kernels):
sizes around its 32-key tiles, windows, key counts that leave tiles and rows without a key, scores far beyond the
cap, a cap far beyond the scores, infinite scores of either sign.

Bounds, against the same attention in float64 on the kernel's inputs: the capped score is cap (1 - 2 r) with r
to 2^-22 relative, so a score is off by at most 2^-21 cap and what the float32 sum of its products loses
(2^-21 scale sum |q||k|), in lse as well (plus 2^-20 |lse| of its own sum); the output carries that, the rounding of P
(2^-9 in bf16, 2^-12 in f16) and its own: 2.5 roundings and twice the score's error times the largest |v|."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd(gpu_device):
    import torch_neuronx_amd as amd

    return amd


CASES = [
    # B, Hq, Hkv, L, S, D, causal, window, lens, cap, strength of the scores
    (1, 2, 2, 31, 33, 128, False, None, None, 5.0, 1.0),
    (1, 4, 2, 65, 127, 256, True, None, None, 50.0, 4.0),
    (2, 2, 1, 130, 130, 256, True, 40, None, 2.0, 1.0),
    (3, 2, 2, 100, 193, 160, False, None, [193, 0, 65], 5.0, 30.0),
    (2, 4, 4, 300, 300, 128, True, 64, [300, 129], 50.0, 1.0),
    (1, 2, 2, 40, 600, 256, True, 100, None, 30.0, 1.0),   # rows whose first tiles lie outside the window
    (1, 8, 2, 513, 513, 128, True, None, None, 1e4, 1.0),
    (2, 2, 1, 97, 225, 64, True, 50, [225, 96], 5.0, 2.0),
    (1, 3, 3, 200, 64, 40, False, None, None, 50.0, 8.0),
    (1, 1, 1, 2, 700, 256, False, None, None, 5.0, 1.0),
    # short windows at width 64 from 512 workgroups on run in the general functor variant, longer ones do not
    (64, 8, 8, 97, 97, 64, True, 40, None, 5.0, 1.0),
    (64, 16, 8, 300, 300, 64, True, 257, [300 - i for i in range(64)], 50.0, 1.0),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "L%d_S%d_D%d_c%d_w%s_cap%g_x%g" % (c[3:8] + c[9:]))
def test_against_float64(amd, gpu_device, case, dtype):
    B, Hq, Hkv, L, S, D, causal, window, lens, cap, strong = case
    dev = gpu_device
    g = torch.Generator(device=dev).manual_seed(L * 7 + S)
    q, k, v = (torch.randn(s, generator=g, device=dev) for s in ((B, Hq, L, D), (B, Hkv, S, D), (B, Hkv, S, D)))
    q, k, v = (q * strong).to(dtype), k.to(dtype), v.to(dtype)
    q[0, 0, 0], k[0, 0, 0] = math.inf, k[0, 0, 0].abs() + 0.5  # that row's scores: +inf at key 0, NaN at the others
    kw = dict(is_causal=causal, softcap=cap)
    if window:
        kw["window"] = window
    lens_t = torch.full((B,), S, device=dev) if lens is None else torch.tensor(lens, device=dev)
    if lens is not None:
        kw["kv_lens"] = lens_t.to(torch.int32)
    out, lse = amd.sdpa_forward(q, k, v, **kw)
    Q, (K, V) = q.double(), (t.double().repeat_interleave(Hq // Hkv, 1) for t in (k, v))
    s = cap * torch.tanh(Q @ K.transpose(-1, -2).contiguous() / math.sqrt(D) / cap)
    i, j = torch.arange(L, device=dev)[:, None], torch.arange(S, device=dev)[None]
    dead = (j[None] >= lens_t[:, None, None])[:, None].expand(B, 1, L, S).clone()
    if causal:
        dead |= j > i
    if window:
        dead |= j < i - window + 1
    s = s.masked_fill(dead, -math.inf)
    want, want_lse = torch.softmax(s, -1).nan_to_num(0.0) @ V, torch.logsumexp(s, -1)
    poisoned = torch.zeros(B, Hq, L, dtype=torch.bool, device=dev)
    poisoned[0, 0, 0] = bool(torch.isnan(s[0, 0, 0]).any())  # (a causal row 0 sees key 0 alone: its score is the cap)
    empty = dead.all(-1).expand(B, Hq, L)
    assert (out[empty & ~poisoned] == 0).all() and (lse[empty & ~poisoned] == -math.inf).all()
    ok = ~empty & ~poisoned
    products = (Q.abs() @ K.abs().transpose(-1, -2).contiguous() / math.sqrt(D)).masked_fill(torch.isinf(Q).any(-1, keepdim=True), 0.0)
    score_err = 2.0**-21 * (cap + float(products.max()))
    assert ((lse.double() - want_lse)[ok].abs() <= score_err + 2.0**-20 * want_lse[ok].abs() + 2.0**-20).all()
    eps = 2.0**-9 if dtype is torch.bfloat16 else 2.0**-12
    assert float((out.double() - want)[ok].abs().max()) <= (2.5 * eps + 2 * score_err) * float(V.abs().max())


def test_lse_of_a_large_cap_keeps_the_reference(amd, gpu_device):
    # A row's reference must not be rounded to the precision of the cap (cap log2(e) = 1443: 2^-14 of rounding step, 2.4e-5
    # of the lse by root mean square, from row to row).  What the scores carry themselves is at most 2^-22 cap each:
    # a common part (the reciprocal's rounding has a side it prefers), and one that averages out over the
    # keys, S / e of which carry the weight.
    g = torch.Generator(device=gpu_device).manual_seed(11)
    S, cap = 4096, 1000.0
    q, k, v = (torch.randn(1, 4, n, 128, generator=g, device=gpu_device).to(torch.bfloat16) for n in (300, S, S))
    lse = amd.sdpa_forward(q, k, v, softcap=cap)[1]
    s = cap * torch.tanh(q.double() @ k.double().transpose(-1, -2).contiguous() / math.sqrt(128) / cap)
    off = lse.double() - torch.logsumexp(s, -1)
    assert abs(float(off.mean())) <= 2.0**-22 * cap
    assert float(off.std()) <= 2.0**-22 * cap / math.sqrt(S / math.e) + 2.0**-22 * float(lse.abs().max())


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("L,S,causal,window,lens", [(70, 160, False, None, None), (97, 97, True, None, None), (130, 130, True, 40, None), (40, 193, False, None, [100, 65])])
def test_scores_of_minus_infinity_are_minus_the_cap(amd, gpu_device, D, L, S, causal, window, lens):
    """-cap like any score far below it, in tiles with a mask and without one: a row all of whose scores are -inf
    (or finite beyond -1e30) is the mean of the values it sees, a single such key keeps its share."""
    B, H, cap, dev = 2, 2, 5.0, gpu_device
    g = torch.Generator(device=dev).manual_seed(D + S)
    q, k, v = (torch.randn(B, H, n, D, generator=g, device=dev).to(torch.bfloat16) for n in (L, S, S))
    k[..., 0] = k[..., 0].abs() + 0.5
    q[0, :, ::3, 0] = -math.inf
    q[0, :, 1::3, 0] = -3e38                         # (scores of about -1e37 and below)
    q[1, :, :, 1], k[1, :, :, 1] = -1.0, 0.0
    k[1, :, 5::40, 1] = math.inf                     # keys whose score is -inf for every row
    kw = dict(is_causal=causal, softcap=cap)
    if window:
        kw["window"] = window
    lens_t = torch.tensor(lens or [S] * B, device=dev)
    if lens:
        kw["kv_lens"] = lens_t.to(torch.int32)
    out, lse = amd.sdpa_forward(q, k, v, **kw)
    i, j = torch.arange(L, device=dev)[:, None], torch.arange(S, device=dev)[None]
    dead = (j[None] >= lens_t[:, None, None])[:, None].expand(B, 1, L, S).clone()
    if causal:
        dead |= j > i
    if window:
        dead |= j < i - window + 1
    raw = q.double() @ k.double().transpose(-1, -2).contiguous() / math.sqrt(D)
    assert not torch.isnan(raw).any()
    s = (cap * torch.tanh(raw / cap)).masked_fill(dead, -math.inf)
    score_err = 2.0**-21 * (cap + 4 * math.sqrt(D))
    assert float((lse.double() - torch.logsumexp(s, -1)).abs().max()) <= score_err + 2.0**-19
    assert float((out.double() - torch.softmax(s, -1) @ v.double()).abs().max()) <= (2.5 * 2.0**-9 + 2 * score_err) * float(v.double().abs().max())
