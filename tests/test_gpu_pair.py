"""The kernels for short and irregular pairs (csrc/ra_pair.hip) at the sizes where they can go wrong:
edges of their 128-row and 64-key tiles, single rows, rows whose keys several workgroups share (evenly, and
under masks that leave rows of different lengths, down to none), every bias term on the tile lists, and key
sequences longer than a list.  Tolerances as in test_gpu_parity.py."""
import numpy as np
import pytest
import torch

import ring_attention as ra
from ring_attention import bias as bias_module
from oracle import ring_oracle as R
from test_gpu_dense_map import _both_ways
from test_gpu_parity import _check

pytestmark = pytest.mark.gpu


def _bias(kind, B, Sq, Sk, H, seed=0):
    rng = np.random.default_rng(seed)
    sl = R.alibi_slopes(H)

    def documents(S):
        ids = np.zeros((B, S), np.int32)
        for b in range(B):
            for c in rng.integers(0, max(S, 2), 4):
                ids[b, c:] += 1
        return ids

    seg_q = documents(Sq)
    seg_k = seg_q if Sq == Sk else documents(Sk)
    pre_q = (np.arange(Sq)[None] < rng.integers(1, Sq + 1, (B, 1))).astype(np.int32)
    pre_k = pre_q if Sq == Sk else (np.arange(Sk)[None] < rng.integers(1, Sk + 1, (B, 1))).astype(np.int32)
    seg = {"q_segment_ids": seg_q}, {"kv_segment_ids": seg_k}
    pre = {"q_prefix_mask": pre_q}, {"kv_prefix_mask": pre_k}
    w = max(1, Sk // 7)
    return {
        "none": (None, None, None, None),
        "causal": (ra.causal_bias(), R.make_bias_fn(causal=True), None, None),
        "window": (ra.sliding_window_bias(w), R.make_bias_fn(causal=True, window=w), None, None),
        "window2": (ra.sliding_window_bias(w, causal=False), R.make_bias_fn(window=w), None, None),
        "documents": (ra.segment_bias(), R.make_bias_fn(use_segments=True), *seg),
        "documents+causal+alibi": (ra.segment_bias() + ra.causal_bias() + ra.alibi_bias(sl),
                                   R.make_bias_fn(use_segments=True, causal=True, alibi=sl), *seg),
        "alibi": (ra.alibi_bias(sl), R.make_bias_fn(alibi=sl), None, None),
        "prefix": (ra.prefix_lm_bias(), R.make_bias_fn(use_prefix=True), *pre),
        "prefix+documents": (ra.prefix_lm_bias() + ra.segment_bias(), R.make_bias_fn(use_prefix=True, use_segments=True),
                             {**seg[0], **pre[0]}, {**seg[1], **pre[1]}),
        "prefix+window": (ra.prefix_lm_bias() + ra.sliding_window_bias(w, causal=False),
                          R.make_bias_fn(use_prefix=True, window=w), *pre),
    }[kind]


@pytest.mark.parametrize("Sq,Sk,D,kind", [
    (1, 1, 64, "none"), (1, 5000, 128, "none"), (33, 63, 128, "causal"), (127, 64, 64, "causal"), (128, 65, 128, "window2"),
    (129, 129, 128, "causal"), (1000, 1000, 64, "causal"), (257, 3001, 128, "none"), (2048, 2048, 128, "causal"),
    (1500, 1500, 128, "window"), (700, 900, 64, "window2"), (1300, 1300, 128, "documents"), (130, 2500, 64, "documents"),
    (1100, 1100, 64, "documents+causal+alibi"), (900, 900, 128, "alibi"), (65, 1900, 128, "alibi"),
    (1200, 1200, 128, "prefix"), (300, 1000, 64, "prefix"), (1024, 1024, 64, "prefix+documents"), (777, 777, 128, "prefix+window"),
    (40, 65600, 64, "prefix"),
])
def test_pair_kernels_at_their_edges(device, Sq, Sk, D, kind):
    B, H = (1, 1) if Sk > 60000 else (2, 2)
    fn, ofn, qkw, kvkw = _bias(kind, B, Sq, Sk, H)
    _check(device, f"pair {kind}", B, Sq, Sk, H, D, 1, fn, ofn, qkw, kvkw, seed=Sq + Sk, impl="pallas")


def _spread(where, absolute, q_segment_ids, kv_segment_ids):
    """A dense block of values and -inf: rows whose id is a multiple of three see no key whose id is one."""
    d = q_segment_ids[:, :, None] - kv_segment_ids[:, None, :]
    return where(d % 3 == 0, float("-inf"), -0.1 * absolute(d))[:, None]


@pytest.mark.parametrize("Sq,Sk,D,n", [(1, 1, 64, 1), (33, 63, 128, 1), (129, 65, 64, 1), (387, 195, 128, 3), (64, 520, 64, 2),
                                       (260, 516, 128, 4)])
def test_pair_kernels_take_single_steps_on_dense_blocks(device, monkeypatch, Sq, Sk, D, n):
    # into a carry and fp32 accumulators; rows without a live key in the first shard (n = 1: in all)
    rng = np.random.default_rng(Sq + Sk)
    q_ids, k_ids = rng.integers(0, 7, (2, Sq)).astype(np.int32), rng.choice([0, 3, 6, 1], (2, Sk)).astype(np.int32)
    q_ids[:, 0] = 3
    k_ids[:, : Sk // n] = 3  # a shard of which these rows see nothing
    if n == 1:
        q_ids[:, Sq // 2:] = 4
    def torch_fn(q_segment_ids, kv_segment_ids):
        return _spread(torch.where, lambda d: d.abs().float(), q_segment_ids, kv_segment_ids)

    def numpy_fn(q_segment_ids, kv_segment_ids):
        return _spread(np.where, lambda d: np.abs(d).astype(np.float32), q_segment_ids, kv_segment_ids)

    _both_ways(device, monkeypatch, "dense steps", 2, Sq, Sk, 2, D, n, torch_fn, numpy_fn, {"q_segment_ids": q_ids},
               {"kv_segment_ids": k_ids}, seed=Sq)


def test_a_repeated_call_reads_nothing_of_the_one_before(device):
    # the workspace of shared rows comes back from the allocator with the last call's partial results
    q, k, v, _ = (torch.from_numpy(x).to(device, torch.bfloat16) for x in R.make_inputs(1, 1, 300, 300, 2, 64))
    first = ra.ring_attention(q, k, v, 1, ra.causal_bias())
    ra.ring_attention(*(torch.full_like(x, float("nan")) for x in (q, k, v)), 1, ra.causal_bias())
    assert torch.equal(ra.ring_attention(q, k, v, 1, ra.causal_bias()), first)


@pytest.mark.parametrize("summary", [True, False])
@pytest.mark.parametrize("D", [64, 128])
def test_rows_without_a_live_score_keep_their_carry(device, monkeypatch, D, summary):
    # bit for bit: queries 32..63 and 160..191 (one wave each) see nothing, their neighbours do
    monkeypatch.setattr(bias_module, "DENSE_SUMMARY", summary)
    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn((1, 300, 2, D), generator=g).to(device, torch.bfloat16).permute(0, 2, 1, 3) for _ in range(3))
    block = torch.randn((1, 1, 300, 300), generator=g)
    dead = torch.zeros(300, dtype=torch.bool)
    dead[32:64] = dead[160:192] = True
    block[:, :, dead] = -float("inf")
    o = torch.randn((1, 2, 300, D), generator=g).to(device)
    m, l = torch.randn((1, 2, 300), generator=g).to(device), torch.rand((1, 2, 300), generator=g).to(device) + 0.5
    before = [x.clone() for x in (o, m, l)]
    ra.fwd_block(q, k, v, block.to(device), o, m, l, 0.1)
    for x, was in zip((o, m, l), before):
        same = (x == was).reshape(1, 2, 300, -1).all(-1).cpu()
        assert same[:, :, dead].all() and not same[:, :, ~dead].all()
