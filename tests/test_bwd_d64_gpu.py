"""Backward at head dims up to 64 (the kernels of 128-row and 128-key workgroups): sizes around
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
    (19, 28, 4, 19, 1071, 64, True, None, 0.0),  # 684 key blocks, 76 of which have an item
    (2, 8, 1, 500, 140, 64, False, None, 0.1),   # the items of a key block go to several workgroups
    (1, 8, 1, 700, 300, 64, True, None, 0.0),
    (8, 20, 20, 130, 520, 64, False, None, 0.1),  # 20 streams per XCD
    (4, 10, 10, 600, 600, 64, True, None, 0.0),  # 5 streams per XCD; key blocks of 384 to 512 workgroups
    # causal calls of 380 to 1032 key blocks: two heads a kv head, short; one, 525 to 760 query tiles of 14 to 16 items
    (95, 8, 4, 65, 65, 64, True, None, 0.0),
    (96, 8, 4, 65, 65, 64, True, None, 0.0),
    (96, 8, 4, 65, 130, 40, True, [65 + i % 66 for i in range(96)], 0.0),
    (128, 16, 8, 65, 65, 64, True, None, 0.0),
    (129, 16, 8, 65, 65, 64, True, None, 0.0),
    (96, 8, 4, 65, 65, 64, True, None, 0.25),
    (25, 3, 3, 896, 896, 64, True, None, 0.0),
    (24, 3, 3, 897, 897, 64, True, None, 0.0),
    (24, 3, 3, 897, 897, 64, True, [897 - 30 * i for i in range(24)], 0.0),
    (19, 5, 5, 1020, 1020, 64, True, None, 0.0),
]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "B%d_H%d_%d_L%d_S%d_D%d_c%d_p%s" % (c[:7] + (c[8],)))
def test_against_float64(amd, gpu_device, case, dtype):
    B, Hq, Hkv, L, S, D, causal, lens, p = case
    _check(amd, gpu_device, B, Hq, Hkv, L, S, D, causal, dtype, lens, p)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("which", ["q", "do"])
def test_a_batch_beyond_32_bit_offsets(amd, gpu_device, which, causal):
    """Q or dO of one batch spans 2 GiB (two heads that far apart in one allocation), K and V do not: not
    these kernels' case, the 64-bit ones have it.  L: 256 workgroups of 256 rows."""
    B, H, L, S, D = 1, 2, 32768, 96, 64
    g = torch.Generator(device=gpu_device).manual_seed(3)
    q, k, v, do = (torch.randn(B, H, n, D, generator=g, device=gpu_device).to(torch.bfloat16) for n in (L, S, S, L))
    far = torch.empty((1 << 30) + L * D, dtype=torch.bfloat16, device=gpu_device).as_strided((B, H, L, D), ((1 << 30) + L * D, 1 << 30, D, 1))
    far.copy_(q if which == "q" else do)
    q, do = (far, do) if which == "q" else (q, far)
    out, lse = amd.sdpa_forward(q, k, v, is_causal=causal)
    dq, dk, dv, _ = amd.sdpa_backward(do, q, k, v, out, lse, is_causal=causal)
    for h in range(H):
        Q, K, V, DO = (t[0, h].double() for t in (q, k, v, do))
        s = Q @ K.t() / math.sqrt(D)
        if causal:
            s = s.masked_fill(~torch.ones(L, S, dtype=torch.bool, device=gpu_device).tril(), -math.inf)
        P = torch.softmax(s, -1)
        dS = P * (DO @ V.t() - (DO * (P @ V)).sum(-1, keepdim=True)) / math.sqrt(D)
        for name, a, r in (("dq", dq, dS @ K), ("dk", dk, dS.t() @ Q), ("dv", dv, P.t() @ DO)):
            off = float((a[0, h].double() - r).norm() / r.norm())
            assert off <= 8e-3, (name, h, off)


def _check_heads(amd, q, k, v, do, keep, p, heads):
    L, S, D = q.shape[2], k.shape[2], q.shape[3]
    kw = dict(dropout_p=p, dropout_keep=keep)
    out, lse = amd.sdpa_forward(q, k, v, **kw)
    dq, dk, dv, _ = amd.sdpa_backward(do, q, k, v, out, lse, **kw)
    for h in heads:
        Q, K, V, DO, kp = *(t[0, h].double() for t in (q, k, v, do)), keep[0, h].double() / (1 - p)
        P = torch.softmax(Q @ K.t() / math.sqrt(D), -1)
        dP = (DO @ V.t()) * kp
        dS = P * (dP - (DO * ((P * kp) @ V)).sum(-1, keepdim=True)) / math.sqrt(D)
        for name, a, r in (("dq", dq, dS @ K), ("dk", dk, dS.t() @ Q), ("dv", dv, (P * kp).t() @ DO)):
            off = float((a[0, h].double() - r).norm() / r.norm())
            assert off <= 8e-3, (name, h, off)


def test_keep_bits_of_a_batch_beyond_2_gib(amd, gpu_device):
    """Hq * L * ceil(S / 128) * 16 bytes of keep bits reach 2 GiB (every head reads the same Q, K, V and dO)."""
    H, L, S, D = 512, 1 << 18, 4, 8
    g = torch.Generator(device=gpu_device).manual_seed(4)
    q, k, v, do = (torch.randn(1, 1, n, D, generator=g, device=gpu_device).to(torch.bfloat16).expand(1, H, n, D) for n in (L, S, S, L))
    keep = torch.empty(1, H, L, S, dtype=torch.uint8, device=gpu_device).bernoulli_(0.75, generator=g)
    _check_heads(amd, q, k, v, do, keep, 0.25, (0, 300, 511))


def test_keep_mask_rows_far_apart(amd, gpu_device):
    """The rows of a keep-mask lie 1 MiB apart: 2.5 GiB from the first to the last."""
    L, S, D, ld = 2560, 100, 64, 1 << 20
    g = torch.Generator(device=gpu_device).manual_seed(5)
    q, k, v, do = (torch.randn(1, 1, n, D, generator=g, device=gpu_device).to(torch.bfloat16) for n in (L, S, S, L))
    keep = torch.empty(L * ld, dtype=torch.uint8, device=gpu_device).as_strided((1, 1, L, S), (L * ld, L * ld, ld, 1)).bernoulli_(0.75, generator=g)
    _check_heads(amd, q, k, v, do, keep, 0.25, (0,))


@pytest.mark.parametrize("p", [0.0, 0.25])
@pytest.mark.parametrize("L,causal", [(100, False), (97, True), (33, False)])
def test_nan_of_one_head_stays_in_it(amd, gpu_device, L, causal, p):
    """The rows past L of a head's last tile are the next head's in memory: a NaN there must not meet this head's
    zero probabilities.  (Heads are independent, so the others' gradients are the same bits.)"""
    B, H, S, D = 2, 3, 130, 64
    g = torch.Generator(device=gpu_device).manual_seed(L)
    q, k, v, do = (torch.randn(B, H, n, D, generator=g, device=gpu_device).to(torch.bfloat16) for n in (L, S, S, L))
    kw = dict(is_causal=causal)
    if p:
        kw.update(dropout_p=p, dropout_keep=amd.ops.padded_keep_mask(B, H, L, S, gpu_device).bernoulli_(1 - p, generator=g))

    def grads():
        out, lse = amd.sdpa_forward(q, k, v, **kw)
        return amd.sdpa_backward(do, q, k, v, out, lse, **kw)[:3]

    want = grads()
    q[:, 1], do[:, 1] = math.nan, math.inf
    for name, a, w in zip(("dq", "dk", "dv"), grads(), want):
        assert torch.isfinite(a[:, ::2]).all() and torch.equal(a[:, ::2], w[:, ::2]), name
        assert torch.isnan(a[:, 1]).any(), name


@pytest.mark.parametrize("L", [64, 100])
def test_every_row_of_the_gradient_in_one_place(amd, gpu_device, L):
    """dO with row stride 0 (a mean over the rows leaves such a gradient): rows past L are live data there."""
    B, H, S, D = 2, 2, 130, 64
    g = torch.Generator(device=gpu_device).manual_seed(L)
    q, k, v = (torch.randn(B, H, n, D, generator=g, device=gpu_device).to(torch.bfloat16) for n in (L, S, S))
    do = torch.randn(B, H, 1, D, generator=g, device=gpu_device).to(torch.bfloat16).expand(B, H, L, D)
    out, lse = amd.sdpa_forward(q, k, v)
    for a, w in zip(amd.sdpa_backward(do, q, k, v, out, lse)[:3], amd.sdpa_backward(do.contiguous(), q, k, v, out, lse)[:3]):
        assert torch.equal(a, w)


@pytest.mark.parametrize("p", [0.0, 0.25])
@pytest.mark.parametrize("Hq,Hkv,L,S,lens", [
    (1, 1, 3, 2, None), (3, 1, 32, 32, None), (2, 2, 33, 64, None), (2, 1, 64, 96, None), (3, 1, 96, 65, None), (2, 2, 160, 128, [128, 97]),
    (6, 2, 193, 193, [193, 33]), (8, 1, 640, 129, None),  # (the last: the items of a key block go to several workgroups)
])
def test_causal_blocks_in_two_phases_and_one_by_one(amd, gpu_device, Hq, Hkv, L, S, lens, p):
    """dK/dV takes items whose blocks are all live for a wavefront one block ahead, the others (the diagonal) block by block:
    none of the first kind, none of the second, both; a first item of fewer than 64 rows."""
    _check(amd, gpu_device, 2, Hq, Hkv, L, S, 64, True, torch.bfloat16, lens, p)


def test_rows_that_a_key_does_not_see_do_not_reach_it(amd, gpu_device):
    """Under a causal mask a NaN in rows of Q and dO stays with the blocks of 32 keys that have a key which sees them."""
    B, Hq, Hkv, L, D = 1, 4, 2, 320, 64
    g = torch.Generator(device=gpu_device).manual_seed(9)
    q, k, v, do = (torch.randn(B, h, L, D, generator=g, device=gpu_device).to(torch.bfloat16) for h in (Hq, Hkv, Hkv, Hq))
    out, lse = amd.sdpa_forward(q, k, v, is_causal=True)
    want = amd.sdpa_backward(do, q, k, v, out, lse, is_causal=True)[:3]
    for row in (5, 70, 130, 200):
        qn, dn = q.clone(), do.clone()
        qn[:, :, row], dn[:, :, row] = math.nan, math.inf
        got = amd.sdpa_backward(dn, qn, k, v, out, lse, is_causal=True)[:3]
        clean = (row // 32 + 1) * 32
        for name, a, w in zip(("dk", "dv"), got[1:], want[1:]):
            assert torch.equal(a[:, :, clean:], w[:, :, clean:]), (name, row)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,causal,lens", [
    (64, 8, 8, 64, 64, 64, False, None), (65, 8, 8, 64, 64, 64, False, None),    # 512 key blocks, and 520 block by block
    (96, 8, 8, 33, 31, 64, True, None), (97, 8, 8, 33, 31, 64, True, None),      # 768, and past them
    (48, 8, 8, 17, 200, 48, False, None),                                        # one item, two key blocks
    (96, 32, 8, 40, 40, 64, False, None),                                        # four heads' items of one query tile
    (80, 8, 8, 128, 128, 64, False, None), (80, 8, 8, 129, 128, 64, False, None),  # two items, three
    (42, 16, 8, 65, 140, 64, True, [140 - 3 * i for i in range(42)]),            # causal: eight items at the most, above 640
    (41, 8, 8, 190, 200, 64, True, [0, 33] * 20 + [200]),
    (20, 8, 8, 460, 460, 64, True, None), (21, 8, 8, 512, 512, 64, True, None), (21, 8, 8, 513, 512, 64, True, None),
])
def test_a_third_workgroup_on_a_compute_unit(amd, gpu_device, B, Hq, Hkv, L, S, D, causal, lens, dtype):
    """More key blocks than two per compute unit and at most three, of few items: dK/dV block by block, on both sides of the
    lines of that."""
    _check(amd, gpu_device, B, Hq, Hkv, L, S, D, causal, dtype, lens, 0.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,Hq,Hkv,L,S,D,lens", [
    (63, 6, 2, 321, 321, 64, None), (64, 6, 2, 321, 321, 64, None), (64, 6, 2, 320, 320, 64, None),  # 378 key blocks, 384, of five query tiles
    (43, 6, 2, 321, 700, 40, [700 - 15 * i for i in range(43)]),                                      # 516
    (64, 12, 4, 330, 200, 64, [200 - 3 * i for i in range(64)]),                                      # 512
    (65, 12, 4, 330, 200, 64, None), (64, 4, 2, 321, 321, 64, None),                                  # 520; two heads a kv head
])
def test_on_both_sides_of_the_lines_of_grouped_heads(amd, gpu_device, B, Hq, Hkv, L, S, D, lens, dtype):
    """Causal calls whose dK/dV is that of bwd_dkdv_w32.hip: three heads a kv head, 384 to 512 key blocks, six query tiles."""
    _check(amd, gpu_device, B, Hq, Hkv, L, S, D, True, dtype, lens, 0.0)
