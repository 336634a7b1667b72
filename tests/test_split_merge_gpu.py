"""The merge of split keys at the edges of its two forms (up to 16 parts a row, and more), with columns that
do not fill its last group of threads and with parts that hold no live key.

Bounds: a probability and an output element are each rounded to the input dtype once (2^-9 relative for
bfloat16), which in the 2-norm of a row stays below 2 * 2^-9 = 4e-3 with room for the sums; float32 rows carry
the exponent's rounding, 2e-7 per unit of a log-sum-exp of about 10, and 1e-5 covers it."""

import ctypes
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
    return torch.softmax(s, -1) @ v, torch.logsumexp(s, -1)


def _rel(a, b):
    return float((a.double() - b).norm() / b.norm())


# (parts of the call on 256 compute units: bf16 2, 16, 17, 64, 33; float32 2, 16, 17, 512, 64)
@pytest.mark.parametrize("dtype,B,Hq,Hkv,S,D,Dv,ragged", [
    (torch.bfloat16, 32, 8, 8, 513, 64, 64, False),
    (torch.bfloat16, 4, 8, 8, 4096, 128, 128, False),
    (torch.float16, 1, 32, 8, 17 * 256, 128, 72, False),
    (torch.bfloat16, 1, 32, 8, 32768, 128, 128, False),
    (torch.bfloat16, 2, 8, 8, 33 * 256, 256, 200, True),
    (torch.float32, 32, 16, 16, 512, 64, 40, True),
    (torch.float32, 8, 8, 8, 2048, 128, 128, False),
    (torch.float32, 3, 8, 4, 17 * 128, 128, 104, True),
    (torch.float32, 1, 2, 1, 65536, 64, 64, False),
    (torch.float32, 2, 8, 8, 8192, 256, 136, True),
])
def test_split_keys_of_the_forward(amd, gpu_device, dtype, B, Hq, Hkv, S, D, Dv, ragged):
    g = torch.Generator(device=gpu_device).manual_seed(S + D)
    q, k, v = (torch.randn(s, generator=g, device=gpu_device).to(dtype) for s in ((B, Hq, 1, D), (B, Hkv, S, D), (B, Hkv, S, Dv)))
    # (the last batch keeps 100 keys: most of its parts have none)
    lens = torch.tensor([S - 1] * (B - 1) + [100], device=gpu_device, dtype=torch.int32) if ragged else None
    out, lse = amd.sdpa_forward(q, k, v, kv_lens=lens)
    want, want_lse = _want(q, k, v, lens)
    assert _rel(out, want) <= (1e-5 if dtype is torch.float32 else 4e-3)
    assert float((lse.double() - want_lse).abs().max()) <= (1e-5 if dtype is torch.float32 else 2e-3)


@pytest.mark.parametrize("B,Hkv,S,D", [(1, 8, 128, 128), (1, 8, 16 * 128, 64), (1, 4, 20000, 128), (2, 1, 131072, 256), (70, 4, 4096, 128)])
def test_partials_of_the_fp8_decode(amd, gpu_device, B, Hkv, S, D):
    g = torch.Generator(device=gpu_device).manual_seed(S)
    q = torch.randn(B, 2 * Hkv, 1, D, generator=g, device=gpu_device, dtype=torch.bfloat16)
    k, v = ((torch.randn(B, Hkv, S, D, generator=g, device=gpu_device) * 32).to(torch.float8_e4m3fn) for _ in range(2))
    sc = torch.full((B, Hkv), 1.0 / 32, device=gpu_device)
    lens = torch.randint(1, S + 1, (B,), generator=g, device=gpu_device, dtype=torch.int32)
    out, lse = amd.decode_fp8kv(q, k, v, sc, sc, lens)
    want, want_lse = _want(q, k.float() / 32, v.float() / 32, lens)
    assert _rel(out, want) <= 4e-3
    assert float((lse.double() - want_lse).abs().max()) <= 2e-3


@pytest.mark.parametrize("H,S", [(64, 4096), (8, 65536)])
def test_a_large_lse_is_rounded_twice_and_no_more(amd, gpu_device, H, S):
    """Every score of a row is the same float32 value c between 512 and 1000, exactly: a part's lse is c + ln(keys),
    the row's that plus ln(parts), each sum rounded once to half a unit of 2^-14 (2^-20 for the two logarithms)."""
    c = 512.0 + 488.0 * torch.rand(H, generator=torch.Generator(device=gpu_device).manual_seed(H), device=gpu_device)
    q, k = torch.zeros(1, H, 1, 64, device=gpu_device), torch.zeros(1, H, S, 64, device=gpu_device)
    q[0, :, 0, 5], k[..., 5] = c, 1.0
    out, lse = amd.sdpa_forward(q, k, torch.ones_like(k), scale=1.0)
    assert float((lse[0, :, 0].double() - c.double() - math.log(S)).abs().max()) <= 2 * 2.0**-15 + 2.0**-20
    assert float((out - 1).abs().max()) <= 1e-5


@pytest.mark.parametrize("B,S,part,every", [(1, 8192, 8192, 1), (1, 8192, 100, 3), (1, 1024, 128, 4), (1, 1024, 128, 8), (16, 1024, 128, 4), (1, 32768, 256, 16)])
def test_nan_keys_of_the_fp8_decode_are_not_dropped(amd, gpu_device, B, S, part, every):
    """A cache with NaN keys gives rows without a sum (zeros, lse = -inf), whether the NaNs share their parts with
    ordinary keys or fill whole parts (of 128 keys, in the last case 256), those that one group of the merge's
    threads takes among them: never what the other keys alone would give."""
    g = torch.Generator(device=gpu_device).manual_seed(S)
    q = torch.randn(B, 16, 1, 128, generator=g, device=gpu_device, dtype=torch.bfloat16)
    k, v = (torch.randn(B, 8, S, 128, generator=g, device=gpu_device) for _ in range(2))
    k[:, :, torch.arange(S, device=gpu_device) // part % every == every - 1] = math.nan
    k, v = k.to(torch.float8_e4m3fn), v.to(torch.float8_e4m3fn)
    one = torch.ones(B, 8, device=gpu_device)
    out, lse = amd.decode_fp8kv(q, k, v, one, one)
    assert not out.any() and torch.isneginf(lse).all()


@pytest.mark.parametrize("dtype,Hq,Hkv,L,D,biased", [
    (torch.bfloat16, 8, 4, 1, 128, False),   # at most 16 rows a kv head
    (torch.float16, 8, 8, 2, 64, False),
    (torch.bfloat16, 8, 4, 1, 128, True),
    (torch.float16, 8, 4, 1, 96, False),
    (torch.bfloat16, 4, 4, 40, 128, False),  # 32 query rows a wavefront
    (torch.bfloat16, 8, 8, 1, 256, False),
    (torch.float32, 8, 4, 1, 64, False),
])
@pytest.mark.parametrize("where", ["a query row", "a key", "every key"])
def test_a_nan_stays_in_its_row_with_and_without_parts(amd, gpu_device, dtype, Hq, Hkv, L, D, biased, where):
    """Rows that a NaN reaches are NaN with lse = -inf, whether the keys are split (the NaN in one part of them) or not; the
    other rows are those of the call without it, bit for bit."""
    S = 2048
    g = torch.Generator(device=gpu_device).manual_seed(D)
    q, k, v = (torch.randn(1, h, n, D, generator=g, device=gpu_device).to(dtype) for h, n in ((Hq, L), (Hkv, S), (Hkv, S)))
    bias = torch.randn(1, 1, 1, S, generator=g, device=gpu_device).expand(1, Hq, L, S) if biased else None

    def call(workspace):
        p = amd._lib.FwdParams()
        out, lse, _ = amd._lib.host().forward(ctypes.addressof(p), q, k, v, bias, True, False, D**-0.5, 0, False)
        lib = amd._lib.load()
        need = lib.mi355_sdpa_fwd_workspace_bytes(ctypes.byref(p))
        assert need > 0  # (the keys are split)
        ws = torch.empty(need if workspace else 0, dtype=torch.uint8, device=gpu_device)
        if workspace:
            p.workspace, p.workspace_bytes = ws.data_ptr(), need
        amd._lib.check(lib.mi355_sdpa_fwd(ctypes.byref(p), amd._lib.current_stream(q.device)))
        return out, lse

    clean = [call(w) for w in (True, False)]
    reached = torch.zeros(1, Hq, L, dtype=torch.bool, device=gpu_device)
    if where == "a query row":
        q[0, 1, L - 1] = math.nan
        reached[0, 1, L - 1] = True
    else:
        k[0, 0, 1500 if where == "a key" else slice(None)] = math.nan
        reached[0, : Hq // Hkv] = True
    for (want, want_lse), (out, lse) in zip(clean, [call(w) for w in (True, False)]):
        assert bool(out[reached].isnan().all()) and bool((lse[reached] == -math.inf).all())
        assert torch.equal(out[~reached], want[~reached]) and torch.equal(lse[~reached], want_lse[~reached])
