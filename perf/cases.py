"""Performance cases of this package: what a program that uses it calls, at the sizes such programs have.

Six kinds of call, each through the public functions and as a user's program makes it:

  prefill   flash_attn_func on a dense batch, forward only (prompt processing, evaluation)
  varlen    flash_attn_varlen_func on packed sequences, forward only
  train     flash_attn_func or flash_attn_qkvpacked_func, forward and backward through autograd
  bert      flash_attn_varlen_qkvpacked_func with dropout, forward and backward (encoder training on unpadded batches)
  cache     flash_attn_with_kvcache: append new rows, rotate q and k, attend to the cache.  One new position is a
            decoding step, a few a speculative step, hundreds a chunk of a prompt
  rotary    apply_rotary_emb_qkv_ in place on a packed projection

All inputs are i.i.d. N(0, 1), which is what layer-normalised activations after a projection look like.
"""
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "flash-attention_amd"))

from flash_attn import (  # noqa: E402
    flash_attn_func,
    flash_attn_qkvpacked_func,
    flash_attn_varlen_func,
    flash_attn_varlen_qkvpacked_func,
    flash_attn_with_kvcache,
)
from flash_attn.layers.rotary import apply_rotary_emb_qkv_  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # the smallest ordinary call: a short non-causal batch of an encoder, bound by launches and host time
        dict(name="prefill_short", kind="prefill", dtype="fp16", b=2, sq=512, sk=512, h=8, hk=8, d=64, causal=False, left=-1),
        # the headline shape: causal prompts of 8k tokens
        dict(name="prefill_8k", kind="prefill", dtype="bf16", b=4, sq=8192, sk=8192, h=32, hk=32, d=128, causal=True, left=-1),
        # long context with grouped heads and a sliding window
        dict(name="prefill_window_16k", kind="prefill", dtype="bf16", b=2, sq=16384, sk=16384, h=32, hk=8, d=128, causal=True, left=4096),
        # a serving batch of prompts of all lengths, packed without padding
        dict(name="varlen_mixed", kind="varlen", dtype="bf16", n=64, lo=128, hi=4096, h=16, hk=16, d=128, causal=True),
        # language model training, long sequences
        dict(name="train_8k", kind="train", dtype="bf16", b=2, s=8192, h=16, hk=16, d=128, causal=True, packed=False),
        # the same with short sequences and small heads, from one packed projection
        dict(name="train_512", kind="train", dtype="fp16", b=32, s=512, h=32, hk=32, d=64, causal=True, packed=True),
        # wide heads, grouped, a length that fits no tile
        dict(name="train_wide_odd", kind="train", dtype="bf16", b=4, s=2039, h=16, hk=4, d=256, causal=True, packed=False),
        # encoder training: padding removed, dropout on the probabilities, no mask
        dict(name="train_bert_dropout", kind="bert", dtype="fp16", n=64, lo=64, hi=512, h=16, d=64, p=0.1),
        # one user's decoding step, bound by launches and latency
        dict(name="decode_single", kind="cache", dtype="bf16", b=1, sq=1, cap=4096, lo=2048, hi=4000, h=32, hk=8, d=128, rotary=128, interleaved=False),
        # a full server's decoding step over long caches, bound by memory
        dict(name="decode_64x32k", kind="cache", dtype="bf16", b=64, sq=1, cap=32768, lo=1024, hi=32767, h=64, hk=8, d=128, rotary=128, interleaved=True),
        # a prompt that arrives in chunks: 512 new tokens per sequence on caches of up to 16k
        dict(name="chunk_512_on_16k", kind="cache", dtype="bf16", b=8, sq=512, cap=16384, lo=1000, hi=15000, h=32, hk=8, d=128, rotary=128, interleaved=False),
        # rotary embedding of a training batch's projection, all of q and k
        dict(name="rotary_qkv", kind="rotary", dtype="bf16", b=4, s=4096, h=32, d=128, rotary=128, interleaved=False),
    ]


# no drawn case does more than these; the largest listed cases do (flops / bytes of one pass)
FORWARD_FLOPS, TRAIN_FLOPS, CACHE_BYTES, TOKENS = 1.5e12, 9e11, 3e9, 1 << 16


def _log(rng, lo, hi):
    """an integer spread evenly over the logarithm of [lo, hi]"""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def _heads(rng):
    h = rng.choice([8, 12, 16, 32])
    return h, h // rng.choice([g for g in (1, 1, 2, 4, 8) if h % g == 0])


def draw(rng):
    kind = rng.choice(["prefill", "prefill", "varlen", "train", "train", "bert", "cache", "cache", "cache", "rotary"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    d = rng.choice([64, 64, 80, 96, 128, 128, 128, 192, 256])
    h, hk = _heads(rng)
    while True:
        if kind == "prefill":
            sq = _log(rng, 64, 16384)
            sk = sq if rng.random() < 0.7 else _log(rng, sq, 16384)
            left = rng.choice([-1, -1, -1, 256, 1024, 4096])
            c = dict(kind=kind, dtype=dtype, b=_log(rng, 1, max(1, min(64, TOKENS // sk))), sq=sq, sk=sk, h=h, hk=hk, d=d,
                     causal=left >= 0 or rng.random() < 0.6, left=left)
        elif kind == "varlen":
            hi = _log(rng, 128, 8192)
            c = dict(kind=kind, dtype=dtype, n=_log(rng, 2, max(2, min(256, 2 * TOKENS // hi))), lo=_log(rng, 16, hi // 2), hi=hi, h=h, hk=hk,
                     d=d, causal=rng.random() < 0.8)
        elif kind == "train":
            s = _log(rng, 128, 8192)
            packed = rng.random() < 0.4
            c = dict(kind=kind, dtype=dtype, b=_log(rng, 1, max(1, min(64, TOKENS // 2 // s))), s=s, h=h, hk=h if packed else hk, d=d,
                     causal=rng.random() < 0.75, packed=packed)
        elif kind == "bert":
            hi = _log(rng, 64, 1024)
            c = dict(kind=kind, dtype=dtype, n=_log(rng, 4, max(4, min(256, TOKENS // hi))), lo=_log(rng, 8, hi // 2), hi=hi, h=rng.choice([8, 12, 16]),
                     d=rng.choice([64, 64, 128]), p=rng.choice([0.05, 0.1, 0.2]))
        elif kind == "cache":
            sq = rng.choice([1, 1, 1, 4, 4, _log(rng, 2, 16), _log(rng, 64, 1024)])
            cap = _log(rng, max(512, 2 * sq), 32768)
            hi = _log(rng, 256, cap) - sq
            h, hk = rng.choice([(32, 8), (32, 32), (64, 8), (16, 2), (8, 1)])
            c = dict(kind=kind, dtype=dtype, b=_log(rng, 1, 128), sq=sq, cap=cap, lo=_log(rng, 1, max(1, hi)), hi=hi, h=h, hk=hk,
                     d=rng.choice([64, 128, 128, 128]), interleaved=rng.random() < 0.5)
            c["rotary"] = c["d"]
            if hi < c["lo"] or 4 * c["b"] * cap * hk * c["d"] > 9e9:
                continue
        else:
            s = _log(rng, 64, 8192)
            c = dict(kind=kind, dtype=dtype, b=_log(rng, 1, max(1, min(64, TOKENS // 2 // s))), s=s, h=h, d=rng.choice([64, 128]),
                     interleaved=rng.random() < 0.3)
            c["rotary"] = c["d"] if rng.random() < 0.7 else c["d"] // 2
        w = work(c)
        if w["flops"] <= (TRAIN_FLOPS if kind in ("train", "bert") else FORWARD_FLOPS) and w["bytes"] <= CACHE_BYTES:
            return c


def _lengths(n, lo, hi):
    """n lengths spread evenly over [lo, hi]; the seed gives their order"""
    return [int(lo + (hi - lo) * (i + 0.5) / n) for i in range(n)]


def _pairs(sq, sk, causal, left):
    """(query, key) pairs the mask leaves, masks aligned to the bottom right"""
    last = np.arange(sq, dtype=np.int64) + (sk - sq) if causal else np.full(sq, sk - 1, dtype=np.int64)
    first = np.maximum(np.arange(sq, dtype=np.int64) + (sk - sq) - left, 0) if left >= 0 else np.zeros(sq, dtype=np.int64)
    return int(np.maximum(np.minimum(last, sk - 1) - first + 1, 0).sum())


def work(case):
    """Inputs read once, outputs written once; 2 operations per multiply-add of the products over the visible pairs:
    two products forward, five more backward.  Elements are 16-bit, the log-sum-exp a float per row and head."""
    c, kind, d = case, case["kind"], case["d"]
    if kind == "prefill":
        flops = 4 * d * c["h"] * c["b"] * _pairs(c["sq"], c["sk"], c["causal"], c["left"])
        return {"bytes": 2 * d * c["b"] * (2 * c["sq"] * c["h"] + 2 * c["sk"] * c["hk"]) + 4 * c["b"] * c["h"] * c["sq"], "flops": flops}
    if kind == "varlen":
        lens = _lengths(c["n"], c["lo"], c["hi"])
        flops = 4 * d * c["h"] * sum(_pairs(n, n, c["causal"], -1) for n in lens)
        return {"bytes": sum(lens) * (2 * d * (2 * c["h"] + 2 * c["hk"]) + 4 * c["h"]), "flops": flops}
    if kind in ("train", "bert"):
        lens = [c["s"]] * c["b"] if kind == "train" else _lengths(c["n"], c["lo"], c["hi"])
        causal, h, hk = (c["causal"], c["h"], c["hk"]) if kind == "train" else (False, c["h"], c["h"])
        flops = 14 * d * h * sum(_pairs(n, n, causal, -1) for n in lens)
        # forward: q, k, v in, out; backward: those and dout in, dq, dk, dv out
        return {"bytes": sum(lens) * (2 * d * (2 * h + 2 * hk) + 2 * d * (4 * h + 4 * hk) + 8 * h), "flops": flops}
    if kind == "cache":
        lens = [n + c["sq"] for n in _lengths(c["b"], c["lo"], c["hi"])]
        rows = c["b"] * c["sq"]
        flops = 4 * d * c["h"] * sum(_pairs(c["sq"], n, True, -1) for n in lens)
        return {"bytes": 4 * d * c["hk"] * sum(lens) + rows * (4 * d * c["h"] + 4 * d * c["hk"]), "flops": flops}
    assert kind == "rotary"
    turned = c["b"] * c["s"] * 2 * c["h"] * c["rotary"]       # elements of q and k, read and written
    return {"bytes": 4 * turned + 2 * c["s"] * c["rotary"], "flops": 3 * turned}


def tolerance(case):
    """About four times what the path shows against itself in float64 (largest over outputs and gradients, sequences of
    512 to 4096): bf16 rel 2.8e-3, max 6.3e-2; fp16 rel 3.2e-4, max 3.9e-3."""
    return {"rel": 1e-2, "max": 0.25} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 2e-2}


def prepare(case, seed):
    c, kind, dtype, d = case, case["kind"], DTYPES[case["dtype"]], case["d"]
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = random.Random(seed)

    def mk(*shape, grad=False):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=dtype).requires_grad_(grad)

    def lengths(n, lo, hi):
        lens = _lengths(n, lo, hi)
        rng.shuffle(lens)
        return lens

    def prefix(lens):
        return torch.tensor(np.concatenate([[0], np.cumsum(lens)]), dtype=torch.int32, device="cuda")

    def tables(rows, rotary):
        inv = 1.0 / (10000.0 ** (torch.arange(0, rotary, 2, device="cuda", dtype=torch.float32) / rotary))
        t = torch.outer(torch.arange(rows, device="cuda", dtype=torch.float32), inv)
        return torch.cos(t).to(dtype), torch.sin(t).to(dtype)

    s = dict(case=c)
    if kind == "prefill":
        s.update(q=mk(c["b"], c["sq"], c["h"], d), k=mk(c["b"], c["sk"], c["hk"], d), v=mk(c["b"], c["sk"], c["hk"], d))
    elif kind == "varlen":
        lens = lengths(c["n"], c["lo"], c["hi"])
        total = sum(lens)
        s.update(q=mk(total, c["h"], d), k=mk(total, c["hk"], d), v=mk(total, c["hk"], d), cu=prefix(lens), longest=max(lens))
    elif kind == "train":
        if c["packed"]:
            s.update(qkv=mk(c["b"], c["s"], 3, c["h"], d, grad=True))
        else:
            s.update(q=mk(c["b"], c["s"], c["h"], d, grad=True), k=mk(c["b"], c["s"], c["hk"], d, grad=True),
                     v=mk(c["b"], c["s"], c["hk"], d, grad=True))
        s.update(dout=mk(c["b"], c["s"], c["h"], d))
    elif kind == "bert":
        lens = lengths(c["n"], c["lo"], c["hi"])
        total = sum(lens)
        s.update(qkv=mk(total, 3, c["h"], d, grad=True), dout=mk(total, c["h"], d), cu=prefix(lens), longest=max(lens), seed=seed)
    elif kind == "cache":
        cos, sin = tables(c["cap"], c["rotary"])
        s.update(q=mk(c["b"], c["sq"], c["h"], d), k_new=mk(c["b"], c["sq"], c["hk"], d), v_new=mk(c["b"], c["sq"], c["hk"], d),
                 k_cache=mk(c["b"], c["cap"], c["hk"], d), v_cache=mk(c["b"], c["cap"], c["hk"], d), cos=cos, sin=sin,
                 lens=torch.tensor(lengths(c["b"], c["lo"], c["hi"]), dtype=torch.int32, device="cuda"))
    else:
        cos, sin = tables(c["s"], c["rotary"])
        s.update(qkv=mk(c["b"], c["s"], 3, c["h"], d), cos=cos, sin=sin)
    return s


def run(state):
    s, c = state, state["case"]
    kind = c["kind"]
    if kind == "prefill":
        return flash_attn_func(s["q"], s["k"], s["v"], causal=c["causal"], window_size=(c["left"], 0 if c["left"] >= 0 else -1))
    if kind == "varlen":
        return flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["longest"], s["longest"], causal=c["causal"])
    if kind == "train":
        if c["packed"]:
            out = flash_attn_qkvpacked_func(s["qkv"], causal=c["causal"])
            return (out, *torch.autograd.grad(out, s["qkv"], s["dout"]))
        out = flash_attn_func(s["q"], s["k"], s["v"], causal=c["causal"])
        return (out, *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"]))
    if kind == "bert":
        # (a training program seeds its steps so that a run can be repeated)
        torch.cuda.manual_seed(s["seed"])
        out = flash_attn_varlen_qkvpacked_func(s["qkv"], s["cu"], s["longest"], dropout_p=c["p"])
        return (out, *torch.autograd.grad(out, s["qkv"], s["dout"]))
    if kind == "cache":
        out = flash_attn_with_kvcache(s["q"], s["k_cache"], s["v_cache"], s["k_new"], s["v_new"], s["cos"], s["sin"], s["lens"],
                                      causal=True, rotary_interleaved=c["interleaved"])
        return out, s["k_cache"], s["v_cache"]
    return apply_rotary_emb_qkv_(s["qkv"], s["cos"], s["sin"], interleaved=c["interleaved"])
