"""Float32 forward with few query tiles: 32-row workgroups whose four wavefronts share out the key tiles, and with fewer
still 16-row workgroups whose eight wavefronts share out blocks of 16 keys.  Sizes around a tile, around a round of all
wavefronts and on both sides of the lines between the two and the 128-row kernel, and for each of the two ragged key
counts (none at all included), head dims below the width a kernel is built for, narrow V, grouped heads, L != S.

Bound: the tolerance of the float32 gate, 1e-5 on values of order 1 (float32 sums of at most 128 products and
1000 keys: about 3e-7 relative measured, and the rows are compared absolutely)."""

import pytest
import torch

from tests.helpers import max_abs, oracle_fwd, qkv

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def amd(gpu_device):
    import torch_neuronx_amd as amd

    return amd


@pytest.mark.parametrize("B,Hq,Hkv,L,S,E,Dv,causal", [
    (1, 2, 2, 33, 33, 64, 64, False),
    (1, 2, 2, 31, 33, 64, 64, True),
    (2, 4, 4, 128, 128, 64, 64, False),
    (2, 4, 2, 127, 129, 64, 64, True),
    (1, 4, 1, 65, 97, 128, 128, True),
    (1, 2, 2, 200, 161, 128, 72, True),
    (1, 3, 3, 1, 257, 40, 40, False),
    (2, 2, 2, 150, 500, 104, 8, False),
    (1, 4, 4, 1000, 1000, 64, 64, True),
    (20, 4, 4, 130, 130, 64, 64, False),   # 160 workgroups of 128 rows: the last size here
    (128, 1, 1, 128, 128, 64, 64, False),  # 512 workgroups of 32 rows: the last size here
    (103, 1, 1, 129, 129, 64, 64, False),  # ... and past it
    (23, 4, 4, 129, 129, 64, 64, False),   # ... and past it
    (15, 8, 8, 150, 150, 64, 64, True),    # 240, causal
])
def test_against_the_oracle(amd, gpu_device, B, Hq, Hkv, L, S, E, Dv, causal):
    q, k, v = qkv(B, Hq, Hkv, L, S, E, Dv, seed=L + S)
    out, lse = amd.sdpa_forward(*(t.to(gpu_device) for t in (q, k, v)), is_causal=causal)
    ro, rl = oracle_fwd(q, k, v, is_causal=causal)
    assert max_abs(out, ro) <= 1e-5 and max_abs(lse, rl) <= 1e-5


@pytest.mark.parametrize("causal", [False, True])
def test_key_counts(amd, gpu_device, causal):
    B, H, S, D = 4, 2, 140, 64
    q, k, v = qkv(B, H, H, S, S, D, seed=5)
    lens = torch.tensor([140, 0, 1, 97], dtype=torch.int32)
    k[2, :, 1:], v[2, :, 1:] = float("nan"), float("nan")  # (keys past a batch's count are never used)
    out, lse = amd.sdpa_forward(*(t.to(gpu_device) for t in (q, k, v)), is_causal=causal, kv_lens=lens.to(gpu_device))
    for b, n in enumerate(lens.tolist()):
        if n == 0:
            assert not out[b].any() and torch.isneginf(lse[b]).all()
            continue
        ro, rl = oracle_fwd(q[b:b + 1], k[b:b + 1, :, :n], v[b:b + 1, :, :n], is_causal=causal)
        assert max_abs(out[b:b + 1], ro) <= 1e-5 and max_abs(lse[b:b + 1], rl) <= 1e-5


@pytest.mark.parametrize("B,Hq,Hkv,L,S,E,Dv,causal", [
    (1, 2, 2, 1, 1, 64, 64, False),
    (1, 2, 1, 15, 16, 64, 64, True),
    (1, 2, 2, 17, 15, 8, 8, False),
    (2, 2, 1, 16, 129, 72, 24, True),     # a ninth block of 16 keys
    (1, 3, 1, 47, 128, 128, 128, False),
    (1, 2, 2, 250, 250, 128, 128, True),
    (32, 4, 4, 32, 40, 64, 64, False),    # 256 workgroups of 16 rows: the last size without the causal mask, and past it
    (32, 4, 4, 33, 40, 64, 64, False),
    (8, 8, 8, 128, 128, 128, 128, True),  # 512 with it
    (8, 8, 8, 129, 129, 128, 128, True),
    (8, 8, 8, 208, 208, 64, 64, True),    # 832 of short chains
    (2, 16, 16, 401, 401, 64, 64, True),  # ... and of longer ones
])
def test_sixteen_rows_against_the_oracle(amd, gpu_device, B, Hq, Hkv, L, S, E, Dv, causal):
    """The same in workgroups of 16 rows whose eight wavefronts take every eighth block of 16 keys."""
    test_against_the_oracle(amd, gpu_device, B, Hq, Hkv, L, S, E, Dv, causal)


@pytest.mark.parametrize("B,Hq,Hkv,L,S,E,Dv", [
    (10, 4, 2, 128, 128, 128, 128), (41, 1, 1, 128, 170, 128, 128),  # under the mask, head dims above 64: 320 of them of 33 to 128 rows, and past it
    (14, 4, 4, 129, 129, 104, 104), (19, 3, 3, 129, 140, 104, 104),  # 512 from 129 rows on
    (32, 4, 4, 32, 32, 128, 72), (43, 3, 1, 32, 90, 128, 128),       # 256 up to 32 rows
    (128, 4, 4, 16, 16, 128, 128), (171, 3, 3, 16, 16, 128, 128),    # 512 up to 16
    (64, 4, 4, 32, 32, 64, 64), (257, 1, 1, 20, 32, 64, 64),         # head dims up to 64: 512 of 17 to 32 rows
    (11, 3, 3, 400, 400, 64, 64), (17, 2, 2, 400, 400, 48, 48),      # 832 up to 400 rows
    (22, 1, 1, 210, 105, 128, 128), (23, 1, 1, 210, 105, 128, 128),  # half as many keys as rows: 320 at head dims above 64,
    (36, 1, 1, 210, 150, 128, 128), (18, 1, 1, 311, 264, 128, 64),   # not with more keys
    (32, 1, 1, 400, 47, 64, 64), (128, 2, 2, 64, 32, 64, 64),        # and not at head dims up to 64
    (24, 6, 2, 38, 38, 128, 128), (32, 4, 4, 38, 38, 128, 128),      # 288 of 32 rows, and 256
])
def test_on_both_sides_of_the_lines_of_sixteen_rows(amd, gpu_device, B, Hq, Hkv, L, S, E, Dv):
    test_against_the_oracle(amd, gpu_device, B, Hq, Hkv, L, S, E, Dv, True)


@pytest.mark.parametrize("B,Hq,Hkv,L,S,E,Dv,causal", [
    (15, 4, 2, 97, 161, 64, 64, False),     # 420 of 16 rows, 240 of 32, 60 of 128
    (17, 3, 1, 150, 129, 40, 8, False),
    (20, 4, 4, 100, 40, 72, 24, False),
    (10, 6, 2, 200, 700, 104, 104, False),
    (16, 12, 4, 70, 97, 64, 40, True),      # causal, D <= 64: 960 of 16, 192 of 128
    (50, 2, 1, 150, 333, 48, 48, True),
    (12, 6, 2, 128, 257, 128, 72, True),    # 576 of 16, 72 of 128
    (30, 4, 1, 130, 129, 80, 80, True),
])
def test_thirty_two_rows_against_the_oracle(amd, gpu_device, B, Hq, Hkv, L, S, E, Dv, causal):
    """32-row workgroups where there are too many of 16 rows: grouped heads, narrow rows, L != S."""
    test_against_the_oracle(amd, gpu_device, B, Hq, Hkv, L, S, E, Dv, causal)


@pytest.mark.parametrize("B,H,S,D,causal", [(20, 2, 140, 64, False), (20, 5, 140, 64, True), (20, 3, 140, 104, True)])
def test_key_counts_in_thirty_two_rows(amd, gpu_device, B, H, S, D, causal):
    q, k, v = qkv(B, H, H, S, S, D, seed=6)
    lens = torch.tensor([140, 0, 1, 97, 33] * 4, dtype=torch.int32)
    for b in range(B):
        k[b, :, lens[b]:], v[b, :, lens[b]:] = float("nan"), float("nan")
    out, lse = amd.sdpa_forward(*(t.to(gpu_device) for t in (q, k, v)), is_causal=causal, kv_lens=lens.to(gpu_device))
    for b, n in enumerate(lens.tolist()):
        if n == 0:
            assert not out[b].any() and torch.isneginf(lse[b]).all()
            continue
        ro, rl = oracle_fwd(q[b:b + 1], k[b:b + 1, :, :n], v[b:b + 1, :, :n], is_causal=causal)
        assert max_abs(out[b:b + 1], ro) <= 1e-5 and max_abs(lse[b:b + 1], rl) <= 1e-5


@pytest.mark.parametrize("B,H,S,D", [(2, 4, 128, 64), (2, 4, 500, 64), (2, 4, 300, 128), (1, 2, 97, 40)])
def test_log_sum_exp_of_sixteen_rows_is_rounded_once(amd, gpu_device, B, H, S, D):
    """The backward's probabilities take every error of the saved log-sum-exp.  Bound: its values lie between 4 and 8, where
    rounding leaves 0.29 ulp = 1.38e-7 (2-norm mean); scores, exponentials and sums of S keys average out to 1e-7 at
    most: together 1.7e-7.  (2.5e-7 with the log, the product and the sum rounded one by one.)"""
    q, k, v = qkv(B, H, H, S, S, D, seed=9)
    _, lse = amd.sdpa_forward(*(t.to(gpu_device) for t in (q, k, v)))
    want = torch.logsumexp(q.double() @ k.double().transpose(-1, -2) * D ** -0.5, -1)
    assert 4 < want.min() and want.max() < 8
    assert (lse.cpu().double() - want).pow(2).mean().sqrt() <= 1.7e-7
