"""Masks over an odd number of keys, in rows that start on dwords: taken as they are by the forward for 16-bit inputs, and
summed up row by row from any address on.

Bound of the forward: probabilities and outputs rounded once each to the input dtype, 2-norm below 4e-3 (bfloat16) and
5e-4 (float16).  Row summaries are whole numbers."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd(gpu_device):
    import torch_neuronx_amd as amd

    return amd


@pytest.mark.parametrize("dtype,bound", [(torch.bfloat16, 4e-3), (torch.float16, 5e-4)])
@pytest.mark.parametrize("L,S,pitch,D,kind", [
    (1, 1, 2, 64, "full"), (33, 31, 32, 64, "full"), (130, 33, 34, 128, "full"), (64, 255, 1000, 128, "heads"),
    (5, 97, 97, 64, "row"),      # one row for all queries, which ends with its storage
    (200, 129, 130, 256, "full"), (7, 1001, 1002, 128, "full"),  # few rows: the keys may be split
])
def test_forward_takes_an_odd_number_of_keys(amd, gpu_device, dtype, bound, L, S, pitch, D, kind):
    g = torch.Generator(device=gpu_device).manual_seed(S)
    B, Hq, Hkv = 2, 4, 2
    q, k, v = (torch.randn(B, h, n, D, generator=g, device=gpu_device).to(dtype) for h, n in ((Hq, L), (Hkv, S), (Hkv, S)))
    shape = {"full": (B, 1, L), "heads": (1, Hq, L), "row": (1, 1, 1)}[kind]
    rows = torch.full((*shape, pitch), math.nan, dtype=dtype, device=gpu_device)  # (what lies between the rows is nobody's)
    bias = rows[..., :S]
    bias.copy_(torch.randn(*shape, S, generator=g, device=gpu_device))
    bias[..., 1::3] = -math.inf
    out, lse = amd.sdpa_forward(q, k, v, attn_bias=bias, force_kernel=amd._lib.KERNEL_MFMA)
    kd, vd = (t.double().repeat_interleave(2, 1) for t in (k, v))
    s = q.double() @ kd.transpose(-1, -2).contiguous() / math.sqrt(D) + bias.double()
    assert float((out.double() - torch.softmax(s, -1) @ vd).norm() / (torch.softmax(s, -1) @ vd).norm()) <= bound
    assert float((lse.double() - torch.logsumexp(s, -1)).abs().max()) <= 2e-5


@pytest.mark.parametrize("dtype,bound", [(torch.bfloat16, 4e-3), (torch.float16, 5e-4)])
@pytest.mark.parametrize("L,S,pitch,D", [(33, 31, 32, 64), (130, 33, 34, 128), (65, 999, 1008, 128), (5, 97, 98, 64), (40, 129, 130, 256)])
def test_forward_with_dropout_over_an_odd_number_of_keys(amd, gpu_device, dtype, bound, L, S, pitch, D):
    """... together with a keep-mask, whose rows are padded to dwords as well."""
    g = torch.Generator(device=gpu_device).manual_seed(S + 1)
    B, Hq, Hkv, p = 2, 4, 2, 0.25
    q, k, v = (torch.randn(B, h, n, D, generator=g, device=gpu_device).to(dtype) for h, n in ((Hq, L), (Hkv, S), (Hkv, S)))
    rows = torch.full((B, Hq, L, pitch), math.nan, dtype=dtype, device=gpu_device)
    bias = rows[..., :S]
    bias.copy_(torch.randn(B, Hq, L, S, generator=g, device=gpu_device))
    bias[..., 2::3] = -math.inf
    keep = amd.ops.padded_keep_mask(B, Hq, L, S, q.device).bernoulli_(1 - p, generator=g)
    out, lse = amd.sdpa_forward(q, k, v, attn_bias=bias, dropout_p=p, dropout_keep=keep, force_kernel=amd._lib.KERNEL_MFMA)
    kd, vd = (t.double().repeat_interleave(2, 1) for t in (k, v))
    s = q.double() @ kd.transpose(-1, -2).contiguous() / math.sqrt(D) + bias.double()
    want = (torch.softmax(s, -1) * keep.double() / (1 - p)) @ vd
    assert float((out.double() - want).norm() / want.norm()) <= bound
    assert float((lse.double() - torch.logsumexp(s, -1)).abs().max()) <= 2e-5


@pytest.mark.parametrize("dtype", [torch.bool, torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("S,pitch,offset", [(1, 1, 0), (7, 9, 1), (16, 16, 3), (65, 67, 5), (999, 1008, 0), (1030, 1031, 15)])
def test_row_summaries_from_any_address(amd, gpu_device, dtype, S, pitch, offset):
    B, L = 3, 6
    g = torch.Generator().manual_seed(S)
    kept = torch.rand(B, L, S, generator=g) < torch.tensor([0.0, 1.0, 0.5, 0.95, 0.05, 0.5])[:, None]
    kept[0, 2] = torch.arange(S) < S // 2
    kept[1, 2] = torch.arange(S) >= S // 3
    flat = torch.zeros(offset + B * L * pitch, dtype=dtype, device=gpu_device)
    mask = flat.as_strided((B, 1, L, S), (L * pitch, L * pitch, pitch, 1), offset)
    mask.copy_(kept[:, None] if dtype == torch.bool else torch.zeros(B, 1, L, S).masked_fill(~kept[:, None], -math.inf))
    got = amd.ops.mask_verdict(mask, B, 2, L, S)[8 + B:8 + B + B * L * 4].view(B, L, 4).cpu()
    for b in range(B):
        for i in range(L):
            on = kept[b, i].nonzero().flatten().tolist()
            off = [j for j in range(S) if not kept[b, i, j]]
            hi = on[-1] if on else -1
            assert got[b, i].tolist() == [hi, len(on), off[0] if off else S, max([j for j in off if j < hi], default=-1) + 1]
