"""The forward of a decode step (at most 16 query rows per kv head): one step of 32 keys and its edges, wavefronts and parts
without a key, every count of rows, key counts, and layouts other than the contiguous one.

Bounds: a probability and an output element are each rounded to the input dtype once (2^-9 relative for bfloat16,
2^-12 for float16), in the 2-norm below 2 * 2^-9 = 4e-3, 2 * 2^-12 = 5e-4, with room for the sums; lse is float32, its
exponents read scores of at most 50 in units of 2^-23, 2e-5."""

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd(gpu_device):
    import torch_neuronx_amd as amd

    return amd


def _want(q, k, v, lens):
    rep = q.shape[1] // k.shape[1]
    q, k, v = q.double(), k.double().repeat_interleave(rep, 1), v.double().repeat_interleave(rep, 1)
    s = (q @ k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    if lens is not None:
        s = s.masked_fill(torch.arange(k.shape[2], device=q.device)[None, None, None] >= lens[:, None, None, None], -math.inf)
    lse = torch.logsumexp(s, -1)
    return torch.exp(s - lse.masked_fill(lse == -math.inf, 0.0)[..., None]) @ v, lse


@pytest.mark.parametrize("dtype,bound", [(torch.bfloat16, 4e-3), (torch.float16, 5e-4)])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,lens,seq_major", [
    (1, 1, 1, 1, 1, 64, None, False),
    (2, 4, 2, 1, 31, 128, None, False),
    (1, 16, 1, 1, 33, 64, None, True),      # 16 rows, one key in the second step
    (3, 7, 1, 1, 129, 128, None, False),    # a second step for one wavefront
    (2, 3, 1, 5, 257, 64, None, True),      # 15 rows: 3 heads, 5 rows each
    (1, 8, 8, 16, 383, 128, None, False),   # 12 steps: parts
    (2, 28, 4, 1, 1000, 128, None, True),
    (300, 2, 2, 1, 97, 64, None, False),    # more workgroups than compute units
    (5, 8, 4, 1, 700, 128, [700, 1, 0, 33, 352], False),  # parts without a key, a batch without one
    (4, 8, 2, 2, 90, 64, [0, 90, 32, 64], True),
    (1, 32, 8, 1, 20000, 128, None, False),
])
def test_few_query_rows(amd, gpu_device, dtype, bound, B, Hq, Hkv, L, S, D, lens, seq_major):
    g = torch.Generator(device=gpu_device).manual_seed(S + D + Hq)

    def make(H, n):
        t = torch.randn((B, n, H, D) if seq_major else (B, H, n, D), generator=g, device=gpu_device).to(dtype)
        return t.transpose(1, 2) if seq_major else t

    q, k, v = make(Hq, L), make(Hkv, S), make(Hkv, S)
    n = None if lens is None else torch.tensor(lens, device=gpu_device, dtype=torch.int32)
    out, lse = amd.sdpa_forward(q, k, v, kv_lens=n)
    want, want_lse = _want(q, k, v, n)
    live = want_lse != -math.inf
    assert float((out.double() - want).norm() / want.norm()) <= bound
    assert bool((out[~live] == 0).all()) and bool((lse[~live] == -math.inf).all())
    assert float((lse.double() - want_lse)[live].abs().max()) <= 2e-5


@pytest.mark.parametrize("S", [70, 1000])
def test_values_that_are_not_finite(amd, gpu_device, S):
    """An infinite last value row (the step it ends in is not whole) and a NaN query row, with and without parts."""
    q, k, v = (torch.randn(2, 4, n, 128, device=gpu_device).to(torch.bfloat16) for n in (1, S, S))
    v[0, 1, S - 1, 5] = math.inf
    q[1, 2] = math.nan
    out, _ = amd.sdpa_forward(q, k, v)
    assert float(out[0, 1, 0, 5]) == math.inf and int((~out[0].isfinite()).sum()) == 1
    assert bool(out[1, 2].isnan().all()) and int(out[1].isnan().any(-1).sum()) == 1
