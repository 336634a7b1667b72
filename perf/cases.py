"""The attention calls whose speed is tracked: what they are, their inputs, one pass, and the work it cannot avoid.

Every case goes through the public entry points the way a model or a serving loop does:
``F.scaled_dot_product_attention`` served by the registered operators (forward under ``no_grad``, training
through autograd), ``sdpa_forward`` / ``sdpa_backward`` for what the functional API cannot say (key counts with
a caller's dropout mask, a window with a soft cap), and ``decode_fp8kv`` for a quantised cache.  Inputs are
drawn on the GPU from N(0, 1), the distribution of the repository's tests and benchmark.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

# (the working folder is the root of the tree that is measured)
sys.path.insert(0, os.path.join(os.getcwd(), "torch-neuronx_amd"))

import torch_neuronx_amd as amd  # noqa: E402  (registers the attention operators)

_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_BYTES = {"bf16": 2, "f16": 2, "f32": 4}


def listed():
    return [
        # The smallest call: float32, no mask, a model nobody cast (latency: launches and host time).
        {"name": "f32_small", "kind": "forward", "dtype": "f32", "B": 2, "Hq": 4, "Hkv": 4, "S": 128, "D": 64, "causal": False},
        # A GPT-2-small layer in training: many small heads, head dim 64.
        {"name": "gpt2_train", "kind": "train", "dtype": "bf16", "B": 4, "Hq": 12, "Hkv": 12, "S": 1024, "D": 64, "causal": True},
        # One user's prompt of ordinary, odd length in front of a grouped-head model.
        {"name": "prompt_1021", "kind": "forward", "dtype": "bf16", "B": 1, "Hq": 32, "Hkv": 8, "S": 1021, "D": 128, "causal": True},
        # A long prompt: the Llama-3-8B layer shape of the headline metric.
        {"name": "prefill_8192", "kind": "forward", "dtype": "bf16", "B": 1, "Hq": 32, "Hkv": 8, "S": 8192, "D": 128, "causal": True},
        # The same layer in training, forward and backward.
        {"name": "llama_train", "kind": "train", "dtype": "bf16", "B": 2, "Hq": 32, "Hkv": 8, "S": 4096, "D": 128, "causal": True},
        # A batch of right-padded prompts with the boolean (B,1,L,S) mask that model code builds from them (which
        # repeats grouped key / value heads itself before such a call).
        {"name": "padded_batch", "kind": "padded", "dtype": "bf16", "B": 4, "Hq": 32, "Hkv": 32, "S": 999, "D": 128},
        # A vision encoder's layer over 196 patches and a class token, half precision, no mask.
        {"name": "vit_encode", "kind": "forward", "dtype": "f16", "B": 64, "Hq": 12, "Hkv": 12, "S": 197, "D": 64, "causal": False},
        # A BERT-base layer in training: attention dropout 0.1 and right padding.
        {"name": "bert_train", "kind": "dropout_train", "dtype": "bf16", "B": 32, "Hq": 12, "Hkv": 12, "S": 512, "D": 64, "p": 0.1},
        # A Gemma-2 layer in training: head dim 256, sliding window, soft cap on the scores.
        {"name": "gemma2_train", "kind": "window_train", "dtype": "bf16", "B": 2, "Hq": 16, "Hkv": 16, "S": 4096, "D": 256,
         "window": 1024, "softcap": 50.0},
        # A generation step of a small batch over a 16-bit cache, through the functional API.
        {"name": "decode_bf16", "kind": "decode", "dtype": "bf16", "B": 8, "Hq": 32, "Hkv": 8, "S": 2049, "D": 128},
        # Interactive serving: one long sequence over an fp8 cache.
        {"name": "decode_fp8_one", "kind": "decode_fp8", "dtype": "bf16", "B": 1, "Hq": 32, "Hkv": 8, "S": 32768, "D": 128, "low": 32768},
        # Batched serving over a padded fp8 cache, key counts between 512 and 8192.
        {"name": "decode_fp8_batch", "kind": "decode_fp8", "dtype": "bf16", "B": 64, "Hq": 32, "Hkv": 8, "S": 8192, "D": 128, "low": 512},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["f32", "train64", "prompt", "train128", "padded", "vit", "dropout", "window", "decode", "fp8_one", "fp8_batch"])
    grouped = rng.choice([(32, 8), (32, 8), (64, 8), (16, 4), (28, 4), (16, 16)])
    half = rng.choice(["bf16", "bf16", "f16"])
    if kind == "f32":
        S = _log(rng, 16, 1024)
        return {"kind": "forward", "dtype": "f32", "B": _log(rng, 1, 8), "Hq": 8, "Hkv": 8, "S": S, "D": rng.choice([64, 128]), "causal": rng.random() < 0.5}
    if kind == "train64":
        S = _log(rng, 64, 2048)
        H = rng.choice([6, 12, 16])
        return {"kind": "train", "dtype": half, "B": _log(rng, 1, min(16, 16384 // S)), "Hq": H, "Hkv": H, "S": S, "D": 64, "causal": True}
    if kind == "prompt":
        S = _log(rng, 16, 8192)
        return {"kind": "forward", "dtype": half, "B": 1, "Hq": grouped[0], "Hkv": grouped[1], "S": S, "D": 128, "causal": True}
    if kind == "train128":
        S = _log(rng, 256, 4096)
        Hq, Hkv = rng.choice([(32, 8), (28, 4), (16, 4), (16, 16)])
        return {"kind": "train", "dtype": half, "B": _log(rng, 1, min(8, 8192 // S)), "Hq": Hq, "Hkv": Hkv, "S": S, "D": 128, "causal": True}
    if kind == "padded":
        S = _log(rng, 64, 2048)
        H, D = rng.choice([(32, 128), (16, 128), (12, 64), (16, 64)])
        return {"kind": "padded", "dtype": half, "B": rng.randint(2, min(8, max(2, 8192 // S))), "Hq": H, "Hkv": H, "S": S, "D": D}
    if kind == "vit":
        S = _log(rng, 49, 785)
        H, D = rng.choice([(6, 64), (12, 64), (16, 64), (16, 80)])
        return {"kind": "forward", "dtype": half, "B": _log(rng, 1, max(2, 16384 // S)), "Hq": H, "Hkv": H, "S": S, "D": D, "causal": False}
    if kind == "dropout":
        S = _log(rng, 48, 512)
        H = rng.choice([12, 16])
        return {"kind": "dropout_train", "dtype": half, "B": _log(rng, 2, min(64, 16384 // S)), "Hq": H, "Hkv": H, "S": S, "D": 64, "p": 0.1}
    if kind == "window":
        S = _log(rng, 512, 4096)
        Hq, Hkv = rng.choice([(16, 16), (16, 8), (8, 4)])
        return {"kind": "window_train", "dtype": half, "B": rng.randint(1, max(1, min(4, 8192 // S))), "Hq": Hq, "Hkv": Hkv, "S": S, "D": 256,
                "window": rng.choice([256, 512, 1024]), "softcap": 50.0}
    if kind == "decode":
        S = _log(rng, 64, 16384)
        return {"kind": "decode", "dtype": half, "B": _log(rng, 1, min(64, 262144 // S)), "Hq": grouped[0], "Hkv": grouped[1], "S": S, "D": 128}
    D = rng.choice([128, 128, 128, 64])
    if kind == "fp8_one":
        S = _log(rng, 1000, 131072)
        return {"kind": "decode_fp8", "dtype": half, "B": 1, "Hq": grouped[0], "Hkv": grouped[1], "S": S, "D": D, "low": S}
    S = _log(rng, 512, 8192)
    return {"kind": "decode_fp8", "dtype": half, "B": _log(rng, 2, 64), "Hq": grouped[0], "Hkv": grouped[1], "S": S, "D": D, "low": max(1, S // 16)}


def _randn(g, dtype, *shape):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)


def _lens(case, lo):
    """Key counts of a batch, a fixed function of the case (so that `work` knows them): spread over [lo, S] in no order."""
    return [case["S"] - int((case["S"] - lo) * (i * 0.6180339887 % 1.0)) for i in range(case["B"])]


def _fp8_cache(g, B, Hkv, S, D):
    x = torch.randn((B, Hkv, S, D), generator=g, device="cuda", dtype=torch.float32)
    scale = (x.abs().amax((-2, -1)) / 448.0).contiguous()
    return (x / scale[:, :, None, None]).to(torch.float8_e4m3fn), scale


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, dt = case["kind"], _DTYPES[case["dtype"]]
    B, Hq, Hkv, S, D = (case[n] for n in ("B", "Hq", "Hkv", "S", "D"))
    s = {"case": case}
    if kind == "decode_fp8":
        s["q"] = _randn(g, dt, B, Hq, 1, D)
        s["k"], s["k_scale"] = _fp8_cache(g, B, Hkv, S, D)
        s["v"], s["v_scale"] = _fp8_cache(g, B, Hkv, S, D)
        s["lens"] = torch.tensor(_lens(case, case["low"]), dtype=torch.int32).cuda()
        return s
    s["q"] = _randn(g, dt, B, Hq, 1 if kind == "decode" else S, D)
    s["k"], s["v"] = _randn(g, dt, B, Hkv, S, D), _randn(g, dt, B, Hkv, S, D)
    if kind.endswith("train"):
        s["do"] = _randn(g, dt, B, Hq, S, D)
    if kind == "train":
        for n in "qkv":
            s[n].requires_grad_(True)
    if kind == "padded":
        i = torch.arange(S, device="cuda")
        live = i[None, :] < torch.tensor(_lens(case, max(1, S // 2)), device="cuda")[:, None]
        s["mask"] = (i[:, None] >= i[None, :])[None, None] & live[:, None, None, :]
    if kind == "dropout_train":
        s["lens"] = torch.tensor(_lens(case, max(1, S // 2)), dtype=torch.int32).cuda()
        s["keep"] = amd.ops.padded_keep_mask(B, Hq, S, S, s["q"].device).bernoulli_(1.0 - case["p"], generator=g)
    return s


def run(s):
    case = s["case"]
    kind, gqa = case["kind"], case["Hq"] != case["Hkv"]
    if kind == "decode_fp8":
        return amd.decode_fp8kv(s["q"], s["k"], s["v"], s["k_scale"], s["v_scale"], s["lens"])
    if kind == "train":
        out = F.scaled_dot_product_attention(s["q"], s["k"], s["v"], is_causal=case["causal"], enable_gqa=gqa)
        return (out, *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["do"]))
    if kind in ("dropout_train", "window_train"):
        if kind == "dropout_train":
            kw = dict(kv_lens=s["lens"], dropout_p=case["p"], dropout_keep=s["keep"])
        else:
            kw = dict(is_causal=True, window=case["window"], softcap=case["softcap"])
        out, lse = amd.sdpa_forward(s["q"], s["k"], s["v"], **kw)
        dq, dk, dv, _ = amd.sdpa_backward(s["do"], s["q"], s["k"], s["v"], out, lse, **kw)
        return out, lse, dq, dk, dv
    with torch.no_grad():
        if kind == "padded":
            return F.scaled_dot_product_attention(s["q"], s["k"], s["v"], attn_mask=s["mask"], enable_gqa=gqa)
        return F.scaled_dot_product_attention(s["q"], s["k"], s["v"], is_causal=case.get("causal", False), enable_gqa=gqa)


def _pairs(case):
    """(query, key) pairs that take part, over the batch, for one head."""
    kind, B, S = case["kind"], case["B"], case["S"]
    if kind == "decode":
        return B * S
    if kind == "decode_fp8":
        return sum(_lens(case, case["low"]))
    if kind == "padded":  # causal, keys below the batch's count
        return sum(n * (n + 1) // 2 + (S - n) * n for n in _lens(case, max(1, S // 2)))
    if kind == "dropout_train":
        return S * sum(_lens(case, max(1, S // 2)))
    if kind == "window_train":
        w = min(case["window"], S)
        return B * (w * (w + 1) // 2 + (S - w) * w)
    return B * (S * (S + 1) // 2 if case["causal"] else S * S)


def work(case):
    kind, B, Hq, Hkv, S, D = (case[n] for n in ("kind", "B", "Hq", "Hkv", "S", "D"))
    e, pairs = _BYTES[case["dtype"]], _pairs(case)
    if kind == "decode_fp8":
        return {"bytes": 2 * Hkv * D * pairs + 2 * B * Hq * D * e + 4 * B * Hq + 8 * B * Hkv + 4 * B, "flops": 4 * Hq * D * pairs}
    L = 1 if kind == "decode" else S
    q, kv = B * Hq * L * D * e, B * Hkv * S * D * e
    train = kind.endswith("train")  # (q, k, v, dO in; O, dQ, dK, dV out; two products forward, five backward)
    nbytes = (4 * q + 4 * kv) if train else (2 * q + 2 * kv)
    if kind == "padded":
        nbytes += B * S * S
    if kind in ("dropout_train", "window_train"):
        nbytes += 4 * B * Hq * S
    if kind == "dropout_train":
        nbytes += Hq * pairs
    return {"bytes": nbytes, "flops": (14 if train else 4) * Hq * D * pairs}


def tolerance(case):
    """About four times the distance of the path from the same attention in 64 bits on the same inputs, the largest
    over the outputs: rel 3.0e-3 / 3.7e-4 / 4e-7 (bf16 / f16 / f32), and per value 0.17 in a bf16 gradient, 0.05 in a
    bf16 output, an eighth of that in f16, 4e-6 in f32."""
    if case["dtype"] == "f32":
        return {"rel": 2e-6, "max": 2e-5}
    most = 0.6 if case["kind"].endswith("train") else 0.2
    return {"rel": 1.2e-2, "max": most} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": most / 8}
