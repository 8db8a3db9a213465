"""Attention workloads through the public entry points, for timing and for comparing results.

Nine kinds of call, which between them are what a model, a serving engine and a training loop ask of this package:

  prefill        F.scaled_dot_product_attention over a whole prompt, without gradients
  prefill_mask   the same with an additive attn_mask [B, 1, S, S] (document masks, relative position biases)
  varlen         packed sequences of different lengths, torch_mlu_amd.flash_attention_forward with cu_seqlens
  decode         one new token per sequence against a contiguous KV cache, F.scaled_dot_product_attention
  paged          one or a few new tokens per sequence against a paged KV cache of ragged fill, torch_mlu_amd.paged_attention
  chunk          a chunk of a long prompt against the cache of what came before, torch_mlu_amd.flash_attention_forward
  train          forward and backward of causal attention, F.scaled_dot_product_attention and autograd
  train_mask     forward and backward of an encoder: padding mask and dropout
  train_varlen   forward and backward over packed sequences

A case is a dict of plain values; lengths that vary inside a batch follow from its `lens` number alone, every tensor's
values from the seed given to prepare().
"""
import math
import random

import torch
import torch.nn.functional as F

import torch_mlu_amd

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(kind, *, batch, heads, kv_heads=None, seq, keys=None, head_dim=128, causal=False, dtype="bf16", **more):
    return dict(kind=kind, batch=batch, heads=heads, kv_heads=kv_heads or heads, seq=seq, keys=keys or seq,
                head_dim=head_dim, causal=causal, dtype=dtype, **more)


def listed():
    return [
        # the smallest call: a short prompt or a text encoder at inference; launches and host work are what it costs
        dict(name="prefill_short", **_case("prefill", batch=1, heads=8, seq=100, head_dim=64, dtype="fp16")),
        # an ordinary prompt batch with grouped kv heads, length not a multiple of anything
        dict(name="prefill_gqa_1000", **_case("prefill", batch=2, heads=32, kv_heads=8, seq=1000, causal=True)),
        # the large prefill: causal, S = 4096
        dict(name="prefill_4096", **_case("prefill", batch=4, heads=32, seq=4096, causal=True)),
        # an additive mask over the whole score matrix
        dict(name="prefill_mask_2048", **_case("prefill_mask", batch=1, heads=32, seq=2048)),
        # a server's prefill batch: 16 prompts of 256 ... 2048 tokens, packed
        dict(name="varlen_16", **_case("varlen", batch=16, heads=16, seq=2048, causal=True, dtype="fp16", lens=3)),
        # one conversation, one token: latency
        dict(name="decode_single", **_case("decode", batch=1, heads=32, kv_heads=8, seq=1, keys=4097)),
        # a full decode batch, bound by reading the cache
        dict(name="decode_64x8192", **_case("decode", batch=64, heads=32, kv_heads=8, seq=1, keys=8192)),
        # continuous batching: a paged cache, every sequence filled to another length
        dict(name="paged_32", **_case("paged", batch=32, heads=32, kv_heads=8, seq=1, keys=4096, page=64, lens=5)),
        # chunked prefill deep in a long prompt
        dict(name="chunk_256x32768", **_case("chunk", batch=1, heads=32, kv_heads=8, seq=256, keys=32768, causal=True)),
        # a training step's attention, the largest case
        dict(name="train_4096", **_case("train", batch=4, heads=32, seq=4096, causal=True)),
        # a small encoder in training: short sequences, head_dim 64, padding mask, dropout
        dict(name="train_encoder", **_case("train_mask", batch=16, heads=12, seq=384, head_dim=64, dropout=0.1, lens=7)),
        # fine-tuning on packed samples
        dict(name="train_varlen", **_case("train_varlen", batch=8, heads=16, kv_heads=4, seq=1500, causal=True, lens=9)),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_HEADS = ((8, 8), (12, 12), (16, 16), (16, 4), (32, 32), (32, 8), (28, 4))


def draw(rng):
    kind = rng.choice(("prefill", "prefill_mask", "varlen", "decode", "paged", "chunk", "train", "train_mask", "train_varlen"))
    heads, kv_heads = rng.choice(_HEADS)
    dtype = rng.choice(("bf16", "bf16", "fp16"))
    head_dim = rng.choice((64, 128, 128, 128))
    lens = rng.randrange(1 << 20)
    if kind in ("prefill", "train"):
        # up to 16k tokens a call; head_dim 96 and 256 are rarer
        head_dim = rng.choice((64, 64, 96, 128, 128, 128, 128, 256))
        seq = _log(rng, 64, 4096)
        batch = _log(rng, 1, max(1, min(32, (16384 if head_dim < 256 else 8192) // seq)))
        if head_dim == 256:
            heads, kv_heads = rng.choice(((8, 8), (16, 16), (16, 8)))
        causal = True if kind == "train" else rng.random() < 0.75
        return _case(kind, batch=batch, heads=heads, kv_heads=kv_heads, seq=seq, head_dim=head_dim, causal=causal, dtype=dtype)
    if kind == "prefill_mask":
        seq = _log(rng, 128, 4096)
        batch = _log(rng, 1, max(1, min(16, 8192 // seq)))
        return _case(kind, batch=batch, heads=heads, kv_heads=heads, seq=seq, head_dim=head_dim, dtype=dtype)
    if kind in ("varlen", "train_varlen"):
        seq = _log(rng, 200, 4096)
        batch = _log(rng, 2, max(2, min(32, 24576 // seq)))
        return _case(kind, batch=batch, heads=heads, kv_heads=kv_heads, seq=seq, head_dim=head_dim, causal=True, dtype=dtype, lens=lens)
    if kind == "decode":
        keys = _log(rng, 300, 65536)
        batch = _log(rng, 1, max(1, min(64, (1 << 19) // keys)))
        heads, kv_heads = rng.choice(((16, 16), (16, 4), (32, 8), (28, 4)))
        return _case(kind, batch=batch, heads=heads, kv_heads=kv_heads, seq=1, keys=keys, head_dim=head_dim, dtype=dtype)
    if kind == "paged":
        page = rng.choice((32, 64, 128, 256))
        keys = (_log(rng, 512, 32768) + page - 1) // page * page
        batch = _log(rng, 1, max(1, min(64, (1 << 18) // keys)))
        heads, kv_heads = rng.choice(((16, 4), (32, 8), (28, 4)))
        seq = rng.choice((1, 1, 1, 2, 4) if heads // kv_heads == 4 else (1, 1, 2))
        return _case(kind, batch=batch, heads=heads, kv_heads=kv_heads, seq=seq, keys=keys, dtype=dtype, page=page, lens=lens)
    if kind == "chunk":
        seq = _log(rng, 32, 1024)
        keys = _log(rng, max(1024, 2 * seq), 65536)
        return _case(kind, batch=1, heads=heads, kv_heads=kv_heads, seq=seq, keys=keys, head_dim=head_dim, causal=True, dtype=dtype)
    # an encoder in training
    seq = _log(rng, 64, 1024)
    batch = _log(rng, 2, max(2, min(64, 16384 // seq)))
    heads = rng.choice((8, 12, 16))
    return _case("train_mask", batch=batch, heads=heads, seq=seq, head_dim=64, dtype=dtype, dropout=0.1, lens=lens)


def _lengths(case):
    """Lengths of a batch's sequences: packed prompts spread from an eighth of the longest up to it, a paged cache's and
    an encoder's from a quarter and from half."""
    r = random.Random(case["lens"])
    longest = case["keys"]
    low = {"varlen": longest // 8, "train_varlen": longest // 8, "paged": longest // 4, "train_mask": longest // 2}[case["kind"]]
    got = [r.randint(max(low, case["seq"] if case["kind"] == "paged" else 1), longest) for _ in range(case["batch"])]
    if case["kind"] != "paged":
        got[r.randrange(len(got))] = longest
    return got


def prepare(case, seed):
    dev = torch.device("cuda")
    dt = _DTYPES[case["dtype"]]
    g = torch.Generator(device=dev).manual_seed(seed)
    kind, B, Hq, Hk, D = case["kind"], case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
    Sq, Sk = case["seq"], case["keys"]

    def normal(*shape):
        return torch.randn(shape, generator=g, device=dev, dtype=dt)

    s = {"case": case}
    if kind in ("varlen", "train_varlen"):
        lens = _lengths(case)
        total = sum(lens)
        cu = [0]
        for n in lens:
            cu.append(cu[-1] + n)
        s["cu"] = torch.tensor(cu, dtype=torch.int32, device=dev)
        s["q"], s["k"], s["v"] = normal(total, Hq, D), normal(total, Hk, D), normal(total, Hk, D)
    elif kind == "chunk":
        s["q"], s["k"], s["v"] = normal(B, Sq, Hq, D), normal(B, Sk, Hk, D), normal(B, Sk, Hk, D)
    elif kind == "paged":
        page, lens = case["page"], _lengths(case)
        per = Sk // page
        s["q"] = normal(B, Hq, Sq, D)
        s["k"], s["v"] = normal(B * per, page, Hk, D), normal(B * per, page, Hk, D)
        s["table"] = torch.randperm(B * per, generator=g, device=dev).to(torch.int32).reshape(B, per)
        s["used"] = torch.tensor(lens, dtype=torch.int32, device=dev)
    else:
        s["q"], s["k"], s["v"] = normal(B, Hq, Sq, D), normal(B, Hk, Sk, D), normal(B, Hk, Sk, D)
    if kind == "prefill_mask":
        s["mask"] = normal(B, 1, Sq, Sk)  # a relative position bias ...
        s["mask"][..., Sk - Sk // 16:] = float("-inf")  # ... and padding
    if kind == "train_mask":
        lens = torch.tensor(_lengths(case), device=dev)
        pad = torch.arange(Sk, device=dev)[None, :] >= lens[:, None]
        s["mask"] = torch.zeros(B, 1, 1, Sk, dtype=dt, device=dev).masked_fill_(pad[:, None, None, :], float("-inf"))
        torch.cuda.manual_seed(seed)  # the dropout mask is drawn from the device's generator
    if kind.startswith("train"):
        s["dout"] = normal(*s["q"].shape)
        for n in ("q", "k", "v"):
            s[n].requires_grad_()
    return s


def run(s):
    case = s["case"]
    kind, q, k, v = case["kind"], s["q"], s["k"], s["v"]
    gqa = case["heads"] != case["kv_heads"]
    if kind in ("prefill", "decode"):
        return F.scaled_dot_product_attention(q, k, v, is_causal=case["causal"], enable_gqa=gqa)
    if kind == "prefill_mask":
        return F.scaled_dot_product_attention(q, k, v, attn_mask=s["mask"])
    if kind == "varlen":
        return torch_mlu_amd.flash_attention_forward(q, k, v, s["cu"], s["cu"], case["seq"], case["keys"], is_causal=True)[:2]
    if kind == "chunk":
        return torch_mlu_amd.flash_attention_forward(q, k, v, None, None, case["seq"], case["keys"], is_causal=True)[:2]
    if kind == "paged":
        return torch_mlu_amd.paged_attention(q, k, v, s["table"], s["used"], is_causal=True)
    if kind == "train":
        out = F.scaled_dot_product_attention(q, k, v, is_causal=case["causal"], enable_gqa=gqa)
    elif kind == "train_mask":
        out = F.scaled_dot_product_attention(q, k, v, attn_mask=s["mask"], dropout_p=case["dropout"])
    else:
        out = torch_mlu_amd.flash_attention_forward(q, k, v, s["cu"], s["cu"], case["seq"], case["keys"], is_causal=True)[0]
    return (out.detach(),) + torch.autograd.grad(out, (q, k, v), s["dout"])


def work(case):
    kind, B, Hq, Hk, D = case["kind"], case["batch"], case["heads"], case["kv_heads"], case["head_dim"]
    Sq, Sk = case["seq"], case["keys"]
    if kind in ("varlen", "train_varlen"):
        lens = _lengths(case)
        pairs, rows, keys = sum(n * (n + 1) // 2 for n in lens), sum(lens), sum(lens)
    elif kind == "paged":
        lens = _lengths(case)
        pairs = sum(Sq * (n - Sq) + Sq * (Sq + 1) // 2 for n in lens)
        rows, keys = B * Sq, sum(lens)
    elif kind == "train_mask":
        # padded keys contribute nothing, and need neither be read nor multiplied
        lens = _lengths(case)
        pairs, rows, keys = Sq * sum(lens), B * Sq, sum(lens)
    else:
        rows, keys = B * Sq, B * Sk
        pairs = B * (Sq * (Sk - Sq) + Sq * (Sq + 1) // 2 if case["causal"] else Sq * Sk)
        if kind == "prefill_mask":
            pairs -= B * Sq * (Sk // 16)
    flops = 4.0 * Hq * D * pairs
    size = 2.0 * D * (2 * rows * Hq + 2 * keys * Hk)  # q, k, v and out
    if kind.startswith("train"):
        flops *= 3.5
        # dout in, three gradients out, and q, k, v, out once more for the backward
        size += 2.0 * D * (4 * rows * Hq + 4 * keys * Hk)
    if kind in ("varlen", "chunk", "paged"):
        size += 4.0 * rows * Hq  # logsumexp
    if kind == "prefill_mask":
        size += 2.0 * B * Sq * Sk
    return {"bytes": size, "flops": flops}


def tolerance(case):
    # probabilities (and, backward, their gradients) are rounded to the inputs' type before the second product
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 2e-3}
