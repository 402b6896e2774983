"""What a program that uses this package has it compute: the calls whose speed is measured.

Every case is one call of the package as a user's program makes it, over the range of sizes,
masks, data types and directions that the package is used for:

* ``forward``   inference over a whole sequence: the output only;
* ``train``     a training step's attention: the output and the gradients of q, k and v;
* ``continue``  a few new tokens against a long context that is already there (the end of a
                chunked prefill, a speculative or a plain decoding step): output and logsumexp;
* ``step``      what one device of a real ring does for one query shard: the carry starts empty,
                meets the device's own key/value shard and one that has travelled, is finalised,
                and the gradients of both (query shard, key/value shard) pairs follow.

A case is a dict of plain values; ``ring`` is the number of shards that the sequences are cut into.
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.abspath("ring-attention-jax-pallas_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

import ring_attention as ra  # noqa: E402
from ring_attention import ring as ring_steps  # noqa: E402

_DTYPES = {"bfloat16": torch.bfloat16, "float16": torch.float16, "float32": torch.float32}


def _case(path, mask, dtype, batch, heads, dim, q_len, kv_len, ring, *, window=0, mean_document=0, std=1.0, name=None):
    c = dict(path=path, mask=mask, dtype=dtype, batch=batch, heads=heads, dim=dim, q_len=q_len, kv_len=kv_len, ring=ring,
             window=window, mean_document=mean_document, std=std)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest call: a short fp32 sequence on a small model, where the latency of a call counts
        _case("forward", "causal", "float32", 1, 4, 64, 1024, 1024, 4, name="forward_1k_fp32"),
        # fine-tuning on packed short documents in fp32, many short shards
        _case("train", "causal+documents", "float32", 2, 4, 64, 2048, 2048, 8, mean_document=512, name="train_2k_packed_fp32"),
        # a small language model with ALiBi, head dim 64
        _case("train", "causal+alibi", "bfloat16", 2, 16, 64, 4096, 4096, 4, name="train_4k_alibi"),
        # cross attention of sequences that fit no tile, a head dim that needs padding, fp16
        _case("train", "none", "float16", 2, 8, 96, 1047, 4791, 3, name="train_cross_ragged_fp16"),
        # scoring with a bidirectional prefix
        _case("forward", "prefix", "bfloat16", 2, 16, 128, 4096, 4096, 4, name="forward_4k_prefix"),
        # 128 new tokens behind a context of 32768
        _case("continue", "causal", "bfloat16", 1, 32, 128, 128, 32768, 8, name="continue_32k"),
        # training at 8192 tokens, 8 shards of 1024
        _case("train", "causal", "bfloat16", 2, 16, 128, 8192, 8192, 8, name="train_8k_causal"),
        # long sequences with a sliding window of half a shard
        _case("train", "window", "bfloat16", 1, 8, 128, 65536, 65536, 8, window=4096, std=0.5, name="train_64k_window"),
        # packed documents with ALiBi
        _case("train", "documents+alibi", "bfloat16", 1, 16, 128, 32768, 32768, 4, mean_document=2048, name="train_32k_packed_alibi"),
        # the same documents through a Python callable that returns dense blocks
        _case("train", "callable", "bfloat16", 1, 16, 128, 32768, 32768, 4, mean_document=2048, name="train_32k_callable"),
        # one device of a ring: its diagonal shard pair and a full one
        _case("step", "causal", "bfloat16", 1, 16, 128, 8192, 8192, 2, name="step_8k"),
        # the largest: 131072 tokens, 32 heads, 8 shards of 16384
        _case("train", "causal", "bfloat16", 1, 32, 128, 131072, 131072, 8, name="train_128k_causal"),
    ]


def draw(rng):
    """One more case of the ranges above: lengths spread over their logarithm, most of them odd."""
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    most = work(listed()[-1])["flops"]
    while True:
        path = rng.choice(["forward", "train", "train", "train", "continue", "step"])
        dim = rng.choice([128, 128, 128, 64, 64, 96, 80, 32])
        heads, batch, ring = rng.choice([4, 8, 12, 16, 32]), rng.choice([1, 1, 2, 4]), rng.choice([1, 2, 3, 4, 8])
        dtype = rng.choice(["bfloat16", "bfloat16", "bfloat16", "float16", "float32"])
        shard = spread(max(16, 512 // ring), 65536 // ring)
        if rng.random() < 0.3:
            shard = -(-shard // 128) * 128
        length = ring * shard
        extra = dict(std=rng.choice([0.5, 1.0]))
        if path == "continue":
            mask, q_len, kv_len = "causal", ring * spread(1, max(2, 512 // ring)), length
            if q_len > kv_len:
                continue
        elif path == "step":
            mask, q_len, kv_len = rng.choice(["causal", "none"]), 2 * shard, 2 * shard
            ring, dim, dtype = 2, rng.choice([64, 128]), "bfloat16"
        else:
            mask = rng.choice(["causal", "causal", "none", "window", "causal+documents", "documents+alibi", "causal+alibi",
                               "prefix", "callable"])
            q_len = kv_len = length
            if mask == "none":
                q_len = ring * spread(16, shard)
            if mask == "callable" and length > 16384:
                continue
            if mask == "window":
                extra["window"] = spread(64, length)
            if mask in ("causal+documents", "documents+alibi", "callable"):
                extra["mean_document"] = spread(128, 4096)
        c = _case(path, mask, dtype, batch, heads, dim, q_len, kv_len, ring, **extra)
        if work(c)["flops"] <= most:
            return c


def _documents(case, length, gen):
    """Document ids of packed sequences, the documents' lengths geometric with the case's mean."""
    starts = torch.rand((case["batch"], length), generator=gen, device="cuda") < 1.0 / case["mean_document"]
    starts[:, 0] = False
    return starts.to(torch.int32).cumsum(1, dtype=torch.int32)


def _document_mask(q_segment_ids, kv_segment_ids):
    same = q_segment_ids[:, :, None] == kv_segment_ids[:, None, :]
    return torch.where(same, 0.0, float("-inf"))[:, None]


def prepare(case, seed):
    B, H, D, Sq, Sk = (case[x] for x in ("batch", "heads", "dim", "q_len", "kv_len"))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    train = case["path"] == "train"

    def normal(*shape, std=case["std"]):
        t = torch.empty(shape, device="cuda", dtype=dtype)
        return t.normal_(0.0, std, generator=gen)

    s = dict(case=case, axis=ra.RingAxis("sp", case["ring"]), q_kw=None, kv_kw=None, bias_fn=None, self_kw=None)
    if case["path"] == "step":
        # [b, h, l, d] views of one device's [b, l, h, d] arrays, its own key/value shard last
        L = Sq // 2
        def blocks(count):
            return [normal(B, L, H, D).permute(0, 2, 1, 3) for _ in range(count)]
        s["q"], s["do"] = blocks(2)
        s["kv"] = [blocks(2) for _ in range(2)]
        causal = case["mask"] == "causal"
        s["bias"] = [ra.BlockBias(ra.causal_bias(), L, 0), ra.BlockBias(ra.causal_bias(), L, L)] if causal else [None, None]
        return s
    s["q"], s["k"], s["v"] = normal(B, Sq, H, D), normal(B, Sk, H, D), normal(B, Sk, H, D)
    if train:
        s["do"] = normal(B, Sq, H, D, std=1.0)
        for x in "qkv":
            s[x].requires_grad_(True)
    mask = case["mask"]
    at = torch.arange(Sk, device="cuda")[None].expand(B, Sk)
    if case["path"] == "continue":
        s["bias_fn"] = ra.causal_bias()
        s["q_kw"], s["kv_kw"] = {"q_positions": at[:, Sk - Sq:]}, {"kv_positions": at}
    elif mask == "causal":
        s["self_kw"] = dict(causal=True, positions=at)
    elif mask == "causal+documents":
        s["self_kw"] = dict(causal=True, positions=at, segment_ids=_documents(case, Sk, gen))
    elif mask == "prefix":
        # a prompt of a quarter to half of each sequence
        ends = torch.randint(Sk // 4, Sk // 2 + 1, (B, 1), generator=gen, device="cuda")
        s["self_kw"] = dict(positions=at, prefix_mask=(at < ends).to(torch.int32))
    elif mask == "window":
        s["bias_fn"] = ra.sliding_window_bias(case["window"])
    elif mask == "causal+alibi":
        s["bias_fn"] = ra.causal_bias() + ra.alibi_bias(ra.alibi_slopes(H).cuda())
    elif mask in ("documents+alibi", "callable"):
        ids = _documents(case, Sk, gen)
        s["q_kw"], s["kv_kw"] = {"q_segment_ids": ids}, {"kv_segment_ids": ids}
        s["bias_fn"] = _document_mask if mask == "callable" else ra.segment_bias() + ra.alibi_bias(ra.alibi_slopes(H).cuda())
    return s


def _run_step(s):
    q, do = s["q"], s["do"]
    B, H, L, D = q.shape
    scale = 1.0 / math.sqrt(D)
    carry = ring_steps.init_carry(B, H, L, D, q.device)
    for (k, v), bias in zip(reversed(s["kv"]), reversed(s["bias"])):
        ra.fwd_block(q, k, v, bias, *carry, scale)
    out = torch.empty((B, L, H, D), dtype=q.dtype, device=q.device).permute(0, 2, 1, 3)
    lse = torch.empty((B, H, L), dtype=torch.float32, device=q.device)
    ring_steps.finalize_carry(*carry, out, lse)
    grads = [ra.bwd_block(q, k, v, bias, out, lse, do, scale) for (k, v), bias in zip(s["kv"], s["bias"])]
    return out, lse, grads


def run(state):
    s = state
    path = s["case"]["path"]
    if path == "step":
        return _run_step(s)
    if path == "continue":
        return ra.ring_attention_with_lse(s["q"], s["k"], s["v"], s["axis"], s["bias_fn"], s["q_kw"], s["kv_kw"])
    if s["self_kw"] is not None:
        out = ra.ring_self_attention(s["q"], s["k"], s["v"], s["axis"], **s["self_kw"])
    else:
        out = ra.ring_attention(s["q"], s["k"], s["v"], s["axis"], s["bias_fn"], s["q_kw"], s["kv_kw"])
    if path == "forward":
        return out
    return out, torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["do"])


def _pairs(case):
    """Unmasked (query, key) pairs of one batch row and head; where the seed draws the mask, their mean."""
    Sq, Sk, mask = case["q_len"], case["kv_len"], case["mask"]
    if case["path"] == "continue":
        return Sq * (Sk - Sq) + Sq * (Sq + 1) / 2
    if case["path"] == "step":
        L = Sq // 2
        return L * L + (L * (L + 1) / 2 if mask == "causal" else L * L)
    if mask == "none":
        return Sq * Sk
    if mask == "window":
        w = min(case["window"], Sq)
        return w * (w + 1) / 2 + (Sq - w) * w
    if mask in ("causal", "causal+alibi"):
        return Sq * (Sq + 1) / 2
    if mask == "prefix":
        lo, hi = Sk / 4, Sk / 2
        return Sq * (Sq + 1) / 2 + (lo * lo + lo * hi + hi * hi) / 6
    # documents: two tokens d apart share one with probability r^d; sum over d = 1 .. S - 1 of (S - d) r^d
    r = 1.0 - 1.0 / case["mean_document"]
    apart = r * (Sq * (1 - r) - 1 + r ** Sq) / (1 - r) ** 2
    return Sq + apart * (1 if mask.startswith("causal") else 2)


def work(case):
    B, H, D, Sq, Sk = (case[x] for x in ("batch", "heads", "dim", "q_len", "kv_len"))
    size = 4 if case["dtype"] == "float32" else 2
    backward = case["path"] in ("train", "step")
    if case["path"] == "step":
        L = Sq // 2
        # q, dO and both key/value shards in, the output, the logsumexp and the fp32 gradients of both pairs out
        data = B * H * L * (D * (2 * 6 + 2 + 4 * 6) + 4)
    else:
        # q and out, k and v; behind them dO and dq, dk and dv
        data = (4 if backward else 2) * B * H * D * size * (Sq + Sk)
        if case["mask"] == "callable":
            data += 2 * 4 * B * Sq * Sk  # what the callable returns, written once and read once
    return {"bytes": float(data), "flops": float((14 if backward else 4) * D * B * H * _pairs(case))}


def tolerance(case):
    # bf16 probabilities and bf16 products with fp32 sums.  Against the dense form in 64 bits the
    # cases read a relative error of 1.2e-3 to 2.7e-3 and a largest one of 0.01 to 0.14 (single small
    # gradients of the first tokens under a causal mask); the same kernels with the shards' sums in
    # another order differ by up to 3.0e-3 and 0.035.
    return {"rel": 1.0e-2, "max": 0.3}
