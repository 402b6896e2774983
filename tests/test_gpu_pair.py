"""The kernels for short and irregular pairs (csrc/ra_pair.hip) at the sizes where they can go wrong:
edges of their 128-row and 64-key tiles, single rows, rows whose keys several workgroups share (evenly, and
under masks that leave rows of different lengths, down to none), every bias term on the tile lists, and key
sequences longer than a list.  Tolerances as in test_gpu_parity.py."""
import ctypes as C
import re

import numpy as np
import pytest
import torch

import ring_attention as ra
from ring_attention import _lib, bias as bias_module, ring as rr
from oracle import ring_oracle as R
from test_gpu_dense_map import _both_ways
from test_gpu_parity import GRAD_TOL, LSE_TOL, OUT_TOL, _check, _dev, _rel

pytestmark = pytest.mark.gpu


def _kernels(call):
    """What ``call`` returns, and the kernels of this library that it launched."""
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as run:
        got = call()
        torch.cuda.synchronize()
    return got, {m.group(1) for m in (re.search(r"ra::(\w+<[^>]*>)", e.key) for e in run.key_averages()) if m}


def _ran(launched, kernels):
    """Whether each of ``kernels`` was launched.  "both<D, MODE>": the kernels for short pairs made both gradients, in one launch or in two."""
    def one(name):
        if not name.startswith("both"):
            return name in launched
        at = name[4:]
        return f"bwd_pair_kernel{at}" in launched or {f"dq_pair_kernel{at}", f"dkdv_pair_kernel{at}"} <= launched

    return all(one(name) for name in kernels)


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


@pytest.mark.parametrize("S,D,kind", [(415, 64, "segments"), (415, 128, "segments"), (300, 128, "segments+causal+alibi"),
                                      (300, 64, "segments+alibi"), (415, 64, "prefix"), (300, 128, "prefix+segments"),
                                      (129, 128, "window+segments")])
def test_each_wave_decides_by_its_own_ids_and_flags(device, S, D, kind):
    """Ids and flags that change inside, at and across the 32 rows of a wave and the 64 (32) tokens of a tile, in no
    order; k and q with row strides of their own, v and the gradient with others."""
    B, H = 2, 2
    rng = np.random.default_rng(S + D)
    cuts = (np.arange(S)[None] // np.array([[32], [24]])) % 5  # whole waves and tiles, and shifted ones
    ids = np.where(rng.random((B, S)) < 0.02, 9, cuts * 7 - 3).astype(np.int32)
    flags = np.where(rng.random((B, S)) < 0.02, 0, np.array([0, 1, -5, 1, 0])[(cuts * 3) % 5]).astype(np.int32)
    sl = R.alibi_slopes(H)
    fn, kw, qkw, kvkw = None, {}, {}, {}
    for term in kind.split("+"):
        f, o = {"segments": (ra.segment_bias(), dict(use_segments=True)), "causal": (ra.causal_bias(), dict(causal=True)),
                "alibi": (ra.alibi_bias(sl), dict(alibi=sl)), "prefix": (ra.prefix_lm_bias(), dict(use_prefix=True)),
                "window": (ra.sliding_window_bias(40), dict(causal=True, window=40))}[term]
        fn = f if fn is None else fn + f
        kw.update(o)
    if "segments" in kind:
        qkw["q_segment_ids"], kvkw["kv_segment_ids"] = ids, ids
    if "prefix" in kind:
        qkw["q_prefix_mask"], kvkw["kv_prefix_mask"] = flags, flags
    q, k, v, do = R.make_inputs(S, B, S, S, H, D)
    at = np.broadcast_to(np.arange(S), (B, S))
    bias = R.make_bias_fn(**kw)(**qkw, **kvkw, q_positions=at, kv_positions=at)
    qk = torch.zeros((B, S, 2, H, D), dtype=torch.bfloat16, device=device)
    qk[:, :, 0], qk[:, :, 1] = _dev(q, device, torch.bfloat16), _dev(k, device, torch.bfloat16)
    leaves = [x.detach().requires_grad_(True) for x in (qk[:, :, 0], qk[:, :, 1], _dev(v, device, torch.bfloat16))]
    out, lse = ra.ring_attention_with_lse(*leaves, 1, fn, {a: _dev(x, device) for a, x in qkw.items()},
                                          {a: _dev(x, device) for a, x in kvkw.items()}, out_dtype=torch.float32)
    want, want_lse = R.mha_dense(q, k, v, bias)
    live = np.isfinite(want_lse).transpose(0, 2, 1)
    assert live.all(axis=2).any() and np.isnan(out.detach().cpu().numpy()[~live]).all()
    got = out.detach().cpu().numpy()
    assert np.abs(got - want)[live].max() <= OUT_TOL
    assert np.abs(lse.cpu().numpy() - want_lse)[np.isfinite(want_lse)].max() <= LSE_TOL
    rows = live.all(axis=2)
    do = np.where(rows[:, :, None, None], do, 0.0)
    bias = np.where(rows[:, None, :, None], bias, 0.0)
    grads = torch.autograd.grad(out, leaves, _dev(do, device))
    for g, ref, name in zip(grads, R.mha_dense_grads(q, k, v, do, bias), ("dq", "dk", "dv")):
        g = g.float().cpu().numpy()
        if name == "dq":
            g, ref = g[rows], ref[rows]
        assert max(_rel(g, ref)) <= GRAD_TOL, name


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


def _spaces(Sq, Sk, H, D, flags):
    """The workspaces of a forward and a backward call (B = 1) in bytes."""
    f, b = _lib.RaFwdStepParams(), _lib.RaBwdStepParams()
    for p in (f, b):
        p.B, p.H, p.Lq, p.Lk, p.D, p.sm_scale, p.bias.flags = 1, H, Sq, Sk, D, 0.1, flags
    return _lib.load().ra_fwd_pair_workspace(C.byref(f)), _lib.load().ra_bwd_pair_workspace(C.byref(b))


# rows of q and of k that share their work; q alone; k alone
@pytest.mark.parametrize("Sq,Sk,causal", [(2048, 2048, True), (64, 4096, False), (4096, 64, False)])
def test_a_repeated_call_reads_nothing_of_the_one_before(device, Sq, Sk, causal):
    # the workspaces come back from the allocator with the last call's statistics and partial results
    H, D = 2, 64
    forward, backward = _spaces(Sq, Sk, H, D, _lib.RA_BIAS_CAUSAL if causal else 0)
    assert (forward > 0) == (Sk > 64)
    shares = (8 * Sq * (Sk > 64) + 16 * Sk * (Sq > 64)) * H * D  # two shares of dq, of dk and dv, at least
    assert backward >= 12 * H * Sq + shares
    q, k, v, do = (torch.from_numpy(x).to(device, torch.bfloat16) for x in R.make_inputs(1, 1, Sq, Sk, H, D))

    def call(*inputs):
        q, k, v, do = inputs
        q, k, v = (x.clone().requires_grad_(True) for x in (q, k, v))
        out, lse = ra.ring_attention_with_lse(q, k, v, 1, ra.causal_bias() if causal else None)
        return out.detach(), lse, *torch.autograd.grad(out, (q, k, v), do)

    first = call(q, k, v, do)
    call(*(torch.full_like(x, float("nan")) for x in (q, k, v, do)))
    for a, b in zip(call(q, k, v, do), first):
        assert torch.isfinite(b).all() and torch.equal(a, b)


@pytest.mark.parametrize("Lq,Lk,D,summary", [(100, 3000, 64, True), (3000, 100, 128, True), (1000, 1000, 128, False)])
def test_finished_pairs_on_a_dense_block(device, Lq, Lk, D, summary):
    """ra_fwd_pair and ra_bwd_pair with RA_BIAS_DENSE, rows or keys shared, against the oracle."""
    H, scale = 2, 1 / np.sqrt(D)
    rng = np.random.default_rng(Lq)
    q, k, v, do = R.make_inputs(Lq, 1, Lq, Lk, H, D)
    block = rng.standard_normal((1, 1, Lq, Lk)).astype(np.float32)
    block[:, :, :, Lk // 3: Lk // 2] = -np.inf
    block[:, :, Lq // 2:] = 0.0
    tq, tk, tv, tdo = (_dev(x, device, torch.bfloat16) for x in (q, k, v, do))
    out, lse = torch.empty((1, Lq, H, D), device=device), torch.empty((1, H, Lq), device=device)
    grads = [torch.empty_like(x) for x in (tq, tk, tv)]
    lib, view = _lib.load(), rr._view_blhd
    dense = rr.BlockBias(dense=_dev(block, device))
    bias = dense.to_struct(tq.device, summary=summary)
    f = _lib.RaFwdStepParams(1, H, Lq, Lk, D, scale, view(tq), view(tk), view(tv), None, None, None, bias)
    size = lib.ra_fwd_pair_workspace(C.byref(f))
    b = _lib.RaBwdStepParams(1, H, Lq, Lk, D, scale, view(tq), view(tk), view(tv), view(tdo), lse.data_ptr(), None, None, None,
                             None, bias)
    size_b = lib.ra_bwd_pair_workspace(C.byref(b))
    assert size_b > 12 * H * Lq and (size > 0) == (Lk > 500)
    ws = torch.empty((max(size, size_b),), dtype=torch.uint8, device=device)
    _lib.check("ra_fwd_pair", lib.ra_fwd_pair(C.byref(f), out.data_ptr(), _lib.RA_DTYPE_F32, Lq * H * D, D, H * D, lse.data_ptr(),
                                              ws.data_ptr(), size, None))
    _lib.check("ra_bwd_pair", lib.ra_bwd_pair(
        C.byref(b), out.data_ptr(), _lib.RA_DTYPE_F32, Lq * H * D, D, H * D, grads[0].data_ptr(), Lq * H * D, D, H * D,
        grads[1].data_ptr(), grads[2].data_ptr(), Lk * H * D, D, H * D, ws.data_ptr(), size_b, None))
    torch.cuda.synchronize()
    want, want_lse = R.mha_dense(q, k, v, block)
    assert np.abs(out.cpu().numpy() - want).max() <= OUT_TOL and np.abs(lse.cpu().numpy() - want_lse).max() <= LSE_TOL
    for got, ref in zip(grads, R.mha_dense_grads(q, k, v, do, block)):
        assert max(_rel(got.float().cpu().numpy(), ref)) <= GRAD_TOL


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


@pytest.mark.parametrize("Lq,Lk,D", [(129, 193, 64), (300, 415, 128), (512, 320, 128)])
def test_each_wave_decides_by_its_own_cells_of_a_summary(device, Lq, Lk, D):
    # cells of 32 x 32 that are -inf, zero, constant or mixed, in no order; whole rows and columns of cells of one kind
    H, scale = 2, 1 / np.sqrt(D)
    rng = np.random.default_rng(Lq + D)
    nr, nc = -(-Lq // 32), -(-Lk // 32)
    kinds = rng.integers(0, 4, (nr, nc))
    kinds[1], kinds[:, 1], kinds[:, 2] = 1, 0, 1
    grid = np.repeat(np.repeat(kinds, 32, 0), 32, 1)[:Lq, :Lk]
    values = rng.standard_normal((Lq, Lk)).astype(np.float32)
    values[values > 1] = -np.inf
    block = np.select([grid == 0, grid == 1, grid == 2], [np.float32(-np.inf), np.float32(0), np.float32(0.7)], values)[None, None]
    q, k, v, do = R.make_inputs(Lq, 1, Lq, Lk, H, D)
    tq, tk, tv, tdo = (_dev(x, device, torch.bfloat16).permute(0, 2, 1, 3) for x in (q, k, v, do))
    carry = rr.init_carry(1, H, Lq, D, tq.device)
    ra.fwd_block(tq, tk, tv, _dev(block, device), *carry, scale)
    out, lse = torch.empty((1, H, Lq, D), device=device), torch.empty((1, H, Lq), device=device)
    rr.finalize_carry(*carry, out, lse)
    want, want_lse = R.mha_dense(q, k, v, block)
    assert np.isfinite(want_lse).all()
    assert np.abs(out.permute(0, 2, 1, 3).cpu().numpy() - want).max() <= OUT_TOL
    assert np.abs(lse.cpu().numpy() - want_lse).max() <= LSE_TOL
    grads = ra.bwd_block(tq, tk, tv, _dev(block, device), out, lse, tdo, scale)
    for got, ref in zip(grads, R.mha_dense_grads(q, k, v, do, block)):
        assert max(_rel(got.permute(0, 2, 1, 3).cpu().numpy(), ref)) <= GRAD_TOL


@pytest.mark.parametrize("Sq,Sk,D,kind", [
    (1, 1, 32, "none"), (129, 63, 96, "none"), (257, 3001, 96, "none"), (2048, 2048, 96, "causal"), (1000, 1000, 32, "causal"),
    (1500, 1500, 80, "window"), (700, 900, 20, "window2"), (1100, 1100, 96, "documents+causal+alibi"), (130, 2500, 32, "documents"),
    (65, 1900, 65, "alibi"), (1024, 1024, 96, "prefix+documents"), (777, 777, 32, "prefix+window"), (64, 2100, 8, "none"),
])
def test_pair_kernels_in_head_dims_of_their_own(device, Sq, Sk, D, kind):
    # computed in 32 and 96; D = 96 and 32 without padding, as views of a wider array whose other columns are not to be read
    fn, ofn, qkw, kvkw = _bias(kind, 2, Sq, Sk, 2)
    _check(device, f"pair {kind}", 2, Sq, Sk, 2, D, 1, fn, ofn, qkw, kvkw, seed=Sq + Sk, impl="pallas")


@pytest.mark.parametrize("D", [32, 96])
def test_narrow_rows_of_a_wider_array(device, D):
    B, S, H = 1, 300, 2
    q, k, v, do = R.make_inputs(D, B, S, S, H, D)
    wide = [torch.full((B, S, H, D + 8), float("nan"), dtype=torch.bfloat16, device=device) for _ in range(4)]
    for w, x in zip(wide, (q, k, v, do)):
        w[..., :D] = _dev(x, device, torch.bfloat16)
    leaves = [w[..., :D].detach().requires_grad_(True) for w in wide[:3]]
    out, lse = ra.ring_attention_with_lse(*leaves, 1, ra.causal_bias(), out_dtype=torch.float32)
    bias = R.make_bias_fn(causal=True)(q_positions=np.arange(S)[None], kv_positions=np.arange(S)[None])
    want, want_lse = R.mha_dense(q, k, v, bias)
    assert np.abs(out.detach().cpu().numpy() - want).max() <= OUT_TOL and np.abs(lse.cpu().numpy() - want_lse).max() <= LSE_TOL
    grads = torch.autograd.grad(out, leaves, wide[3][..., :D].float())
    for g, ref in zip(grads, R.mha_dense_grads(q, k, v, do, bias)):
        assert max(_rel(g.float().cpu().numpy(), ref)) <= GRAD_TOL


@pytest.mark.parametrize("Sq,Sk,D,kind", [(300, 415, 96, "none"), (2048, 130, 32, "none"), (640, 640, 96, "causal"),
                                          (300, 1000, 32, "documents")])
def test_one_head_whose_rows_are_closer_together_than_in_lds(device, Sq, Sk, D, kind):
    # 192 and 64 bytes from row to row, where an LDS tile has 256 and 128
    fn, ofn, qkw, kvkw = _bias(kind, 1, Sq, Sk, 1)
    _check(device, f"pair {kind}", 1, Sq, Sk, 1, D, 1, fn, ofn, qkw, kvkw, seed=Sq + Sk, impl="pallas")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("Sq,Sk,D,H", [(129, 65, 64, 2), (300, 1000, 96, 2), (2048, 130, 32, 1), (640, 640, 128, 40), (8200, 8200, 128, 1)])
def test_gradients_leave_the_kernels_in_the_callers_dtype(device, Sq, Sk, D, H, dtype):
    # rows and keys that several workgroups share, and some that they do not
    g = torch.Generator(device=device).manual_seed(Sq + D)
    q, k, v = (torch.randn((1, S, H, D), device=device, generator=g).to(torch.bfloat16).to(dtype).requires_grad_(True) for S in (Sq, Sk, Sk))
    do = torch.randn((1, Sq, H, D), device=device, generator=g).to(torch.bfloat16).to(dtype)
    causal = Sq == Sk
    out = ra.ring_attention(q, k, v, 1, ra.causal_bias() if causal else None)
    grads = torch.autograd.grad(out, (q, k, v), do)
    for x, got in zip((q, k, v), grads):
        assert got.dtype == dtype and got.shape == x.shape
    ref = [x.detach().float().requires_grad_(True) for x in (q, k, v)]
    for h in range(H):
        s = (ref[0][0, :, h] @ ref[1][0, :, h].T) / np.sqrt(D)
        if causal:
            s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -float("inf"))
        (torch.softmax(s, -1) @ ref[2][0, :, h]).backward(do[0, :, h].float())
    for got, x in zip(grads, ref):
        assert max(_rel(got.float().cpu().numpy(), x.grad.cpu().numpy())) <= GRAD_TOL


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("S,H,causal,kernels", [
    (640, 40, True, {"both<128, 0>"}),
    (4100, 17, True, {"both<128, 0>"}),
    (8190, 8, False, {"dkdv_kernel<128, 0, true>", "dq_pair_kernel<128, 0>"}),
    (10300, 8, False, {"dkdv_kernel<128, 0, true>", "dq_kernel<128, 0, true>"})])
def test_converted_gradients_are_the_bf16_ones_converted(device, S, H, causal, kernels, dtype):
    # bit for bit, on both kinds of kernels; the inputs are the same in bf16, fp16 and fp32
    g = torch.Generator(device=device).manual_seed(S)
    q, k, v, do = (torch.randn((1, S, H, 128), device=device, generator=g).to(torch.bfloat16) for _ in range(4))
    for x in (q, k, v, do):
        x[x.abs() < 1e-3] = 0  # (fp16 holds what is left exactly)

    def gradients(dtype, out_dtype):
        leaves = [x.to(dtype).requires_grad_(True) for x in (q, k, v)]
        out, _ = ra.ring_attention_with_lse(*leaves, 1, ra.causal_bias() if causal else None, out_dtype=out_dtype)
        return _kernels(lambda: torch.autograd.grad(out, leaves, do.to(out.dtype)))

    want, _ = gradients(torch.bfloat16, torch.float32 if dtype == torch.float32 else None)
    got, launched = gradients(dtype, None)
    assert _ran(launched, kernels), launched
    for a, b in zip(got, want):
        assert a.dtype == dtype and b.dtype == torch.bfloat16 and torch.isfinite(b).all() and b.any()
        assert torch.equal(a, b.to(dtype))


@pytest.mark.parametrize("Lq,Lk,H,D,offset", [(1, 1, 1, 64, None), (129, 200, 2, 128, 0), (257, 63, 3, 64, 100), (300, 300, 2, 128, 400),
                                              (1000, 700, 2, 128, -500), (3601, 3700, 32, 128, None), (3601, 3700, 32, 128, 4000),
                                              (2100, 2100, 32, 64, None), (4100, 4100, 17, 128, 0), (64, 64, 2, 128, -64), (130, 130, 1600, 64, 0), (8190, 8190, 8, 128, None),
                                              (10300, 10300, 8, 128, None)])
def test_single_steps_on_both_sides_of_the_rule(device, Lq, Lk, H, D, offset):
    """fwd_block on a carry that is not empty and bwd_block: pairs on the kernels for short pairs and on the long-stretch
    ones (the larger ones without a mask), a pair that sees nothing (-64), queries that see nothing (-500)."""
    g = torch.Generator(device=device).manual_seed(Lq + H)
    q, k, v, do, k0, v0 = (torch.randn((1, H, L, D), device=device, generator=g).to(torch.bfloat16)
                           for L in (Lq, Lk, Lk, Lq, 40, 40))
    scale = 1 / np.sqrt(D)
    bias = None if offset is None else ra.BlockBias(ra.causal_bias(), max(offset, 0), max(-offset, 0))
    carry = rr.init_carry(1, H, Lq, D, device)
    ra.fwd_block(q, k0, v0, None, *carry, scale)
    ra.fwd_block(q, k, v, bias, *carry, scale)
    out, lse = torch.empty((1, H, Lq, D), device=device), torch.empty((1, H, Lq), device=device)
    rr.finalize_carry(*carry, out, lse)
    grads = ra.bwd_block(q, k, v, bias, out, lse, do, scale)
    seen = None
    if offset is not None:
        seen = torch.arange(Lq, device=device)[:, None] + offset >= torch.arange(Lk, device=device)[None]
    for h in range(H):
        a = [x[0, h].float() for x in (q, k, v, do, k0, v0)]
        s = torch.cat([a[0] @ a[4].T, a[0] @ a[1].T], 1) * scale
        if seen is not None:
            s[:, 40:].masked_fill_(~seen, -float("inf"))
        p = torch.softmax(s, -1)
        o = p @ torch.cat([a[5], a[2]])
        assert (out[0, h] - o).abs().max() <= OUT_TOL and (lse[0, h] - torch.logsumexp(s, -1)).abs().max() <= LSE_TOL
        ds = p * (a[3] @ torch.cat([a[5], a[2]]).T - (o * a[3]).sum(-1, keepdim=True))
        want = ((ds[:, 40:] @ a[1]) * scale, (ds[:, 40:].T @ a[0]) * scale, p[:, 40:].T @ a[3])
        for got, ref in zip(grads, want):
            err = (got[0, h] - ref).abs().max() / max(ref.abs().max().item(), 1e-3)
            assert err <= GRAD_TOL, (h, err)


@pytest.mark.parametrize("bias", [None, "causal", "dense"])
def test_block_gradients_of_what_lies_beyond_the_call(device, bias):
    # more heads and batch rows of keys than of queries, values without a key: the gradients of the call cut to size, zeros around
    g = torch.Generator(device=device).manual_seed(5)
    q, k, v, do = (torch.randn(s, device=device, generator=g).to(torch.bfloat16) for s in ((2, 2, 70, 64), (3, 4, 90, 64), (2, 2, 130, 64), (2, 2, 70, 64)))
    bias = {"causal": ra.BlockBias(ra.causal_bias(), 50, 0), "dense": torch.randn((2, 1, 70, 90), device=device, generator=g)}.get(bias)
    cut = k[:2, :2].contiguous(), v[:, :, :90].contiguous()
    carry = ra.fwd_block(q, k, v, bias, *rr.init_carry(2, 2, 70, 64, device), 0.1)
    for a, b in zip(carry, ra.fwd_block(q, *cut, bias, *rr.init_carry(2, 2, 70, 64, device), 0.1)):
        assert torch.equal(a, b)
    out, lse = torch.empty((2, 2, 70, 64), device=device), torch.empty((2, 2, 70), device=device)
    rr.finalize_carry(*carry, out, lse)
    for got, want in zip(ra.bwd_block(q, k, v, bias, out, lse, do, 0.1), ra.bwd_block(q, *cut, bias, out, lse, do, 0.1)):
        B, H, L, _ = want.shape
        assert torch.equal(got[:B, :H, :L], want) and got.count_nonzero() == want.count_nonzero() > 0


@pytest.mark.parametrize("D,n", [(32, 1), (64, 1), (96, 1), (128, 1), (64, 3), (128, 3)])
@pytest.mark.parametrize("transposed", ["qk", "v"])
def test_keys_and_values_laid_out_differently(device, D, n, transposed):
    # [b, h, l, d] arrays seen as [b, l, h, d] (rotary embeddings leave q and k that way) beside contiguous ones; n = 3: shards whose
    # positions are not consecutive, a whole-ring launch of several shards
    B, S, H = 2, 129 * n, 2
    q, k, v, do = R.make_inputs(D, B, S, S, H, D)
    at = np.broadcast_to(np.concatenate([np.arange(129) + 200 * ((2 * i) % n) for i in range(n)]), (B, S))

    def leaf(x, name):
        t = _dev(x, device, torch.bfloat16)
        return (t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) if name in transposed else t).requires_grad_(True)

    leaves = [leaf(x, name) for x, name in zip((q, k, v), "qkv")]
    positions = _dev(at.copy(), device)
    out, lse = ra.ring_attention_with_lse(*leaves, n, ra.causal_bias(), {"q_positions": positions}, {"kv_positions": positions},
                                          out_dtype=torch.float32)
    bias = R.make_bias_fn(causal=True)(q_positions=at, kv_positions=at)
    want, want_lse = R.mha_dense(q, k, v, bias)
    assert np.abs(out.detach().cpu().numpy() - want).max() <= OUT_TOL and np.abs(lse.cpu().numpy() - want_lse).max() <= LSE_TOL
    for g, ref in zip(torch.autograd.grad(out, leaves, _dev(do, device)), R.mha_dense_grads(q, k, v, do, bias)):
        assert max(_rel(g.float().cpu().numpy(), ref)) <= GRAD_TOL


@pytest.mark.parametrize("L,H,D,causal,kernels", [
    (1000, 2, 128, True, {"fwd_pair_kernel<128, 0>", "both<128, 0>"}),
    (2100, 32, 64, False, {"fwd_step_kernel<64, 0, false, false>", "both<64, 0>"}),
    (3601, 32, 128, False, {"fwd_step_kernel<128, 0, false, false>", "dq_pair_kernel<128, 0>", "dkdv_kernel<128, 0, false>"}),
    (4100, 17, 128, True, {"fwd_pair_kernel<128, 0>", "both<128, 0>"}),
    (130, 1600, 64, True, {"dq_pair_kernel<64, 0>", "dkdv_pair_kernel<64, 0>"}),
    (8190, 8, 128, False, {"dq_pair_kernel<128, 0>", "dkdv_kernel<128, 0, false>"}),
    (10300, 8, 128, False, {"fwd_step_kernel<128, 0, false, false>", "dq_kernel<128, 0, false>", "dkdv_kernel<128, 0, false>"})])
def test_which_kernels_a_single_step_takes(device, L, H, D, causal, kernels):
    # ... so that the test above runs them all: fwd_block and bwd_block of its larger cases
    q = torch.randn((1, H, L, D), device=device).to(torch.bfloat16)
    bias = ra.BlockBias(ra.causal_bias(), 0, 0) if causal else None
    carry = rr.init_carry(1, H, L, D, device)
    lse = torch.zeros((1, H, L), device=device)

    def step():
        ra.fwd_block(q, q, q, bias, *carry, 0.1)
        ra.bwd_block(q, q, q, bias, q, lse + 100, q, 0.1)

    _, launched = _kernels(step)
    assert _ran(launched, kernels), launched


@pytest.mark.parametrize("q_off,kv_off", [(100000, 0), (0, 300000)])
def test_alibi_far_from_the_diagonal_on_the_long_stretch_kernels(device, q_off, kv_off):
    """Single steps of 4096 x 4096, H=32, whose bias reaches 6000 and 19000; the slopes are those of test_gpu_parity's smaller
    steps, which run on the kernels for short pairs.  Against float64, tolerances as there."""
    L, H, D = 4096, 32, 128
    g = torch.Generator(device=device).manual_seed(q_off)
    q, k, v, do = (torch.randn((1, H, L, D), device=device, generator=g).to(torch.bfloat16) for _ in range(4))
    slopes = torch.logspace(-4, -8, H, base=2, device=device)
    bias, scale = ra.BlockBias(ra.alibi_bias(slopes), q_off, kv_off), 1 / np.sqrt(D)
    carry = rr.init_carry(1, H, L, D, device)
    out, lse = torch.empty((1, H, L, D), device=device), torch.empty((1, H, L), device=device)
    grads = [torch.zeros((1, H, L, D), device=device) for _ in range(3)]

    def step():
        ra.fwd_block(q, k, v, bias, *carry, scale)
        rr.finalize_carry(*carry, out, lse)
        rr._bwd_step(q, k, v, do, lse, rr.precompute_delta(out, do), *grads, bias, scale)

    _, launched = _kernels(step)
    assert {"fwd_step_kernel<128, 1, false, false>", "dq_kernel<128, 1, false>", "dkdv_kernel<128, 1, false>"} <= launched, launched
    rel = (q_off + torch.arange(L, device=device)[:, None] - kv_off - torch.arange(L, device=device)[None]).abs().double()
    for h in range(H):
        a = [x[0, h].double() for x in (q, k, v, do)]
        s = a[0] @ a[1].T * scale - slopes[h].double() * rel
        p, ref_lse = torch.softmax(s, -1), torch.logsumexp(s, -1)
        o = p @ a[2]
        assert (out[0, h] - o).abs().max() <= OUT_TOL
        assert (lse[0, h] - ref_lse).abs().max() <= LSE_TOL + 4e-7 * ref_lse.abs().max(), h
        ds = p * (a[3] @ a[2].T - (o * a[3]).sum(-1, keepdim=True))
        for got, ref in zip(grads, (ds @ a[1] * scale, ds.T @ a[0] * scale, p.T @ a[3])):
            assert max(_rel(got[0, h].cpu().numpy(), ref.cpu().numpy())) <= GRAD_TOL, h


@pytest.mark.parametrize("mask,Sq,Sk,H,D,dtype", [
    ("causal", 300, 300, 171, 64, torch.bfloat16),         # 513 + 513 workgroups, heads that do not divide by eight
    ("none", 40, 3000, 43, 128, torch.bfloat16),           # few long rows: dQ's workgroups first, their keys shared
    ("documents", 2000, 2000, 8, 96, torch.float32),       # rows of both kinds shared, gradients converted
    ("causal", 700, 700, 86, 32, torch.float16),
    ("none", 894, 894, 8, 128, torch.bfloat16),            # a fraction of a round each, keys and queries shared
    ("none", 1, 64, 1, 128, torch.bfloat16),
    ("causal", 1000, 1000, 2, 128, torch.float32),         # small ones: shares of every row of both kinds
    ("none", 513, 513, 4, 64, torch.bfloat16),
    ("causal", 4090, 4090, 17, 128, torch.bfloat16),       # slabs of different lengths, a few more than places
    ("causal", 129, 129, 1, 64, torch.bfloat16),
    ("documents", 261, 261, 176, 128, torch.bfloat16)])
def test_both_gradients_in_one_launch(device, mask, Sq, Sk, H, D, dtype):
    g = torch.Generator(device=device).manual_seed(Sq + D)
    q, k, v = (torch.randn((1, S, H, D), device=device, generator=g).to(torch.bfloat16).to(dtype).requires_grad_(True) for S in (Sq, Sk, Sk))
    do = torch.randn((1, Sq, H, D), device=device, generator=g).to(torch.bfloat16).to(dtype)
    fn, q_kw, kv_kw, seen = None, None, None, torch.ones((Sq, Sk), dtype=torch.bool, device=device)
    if mask == "causal":
        fn, seen = ra.causal_bias(), seen.tril()
    elif mask == "documents":
        ids = (torch.arange(Sq, device=device) // 130).to(torch.int32)
        fn, q_kw, kv_kw, seen = ra.segment_bias(), {"q_segment_ids": ids[None]}, {"kv_segment_ids": ids[None]}, ids[:, None] == ids[None]
    out = ra.ring_attention(q, k, v, 1, fn, q_kw, kv_kw)
    grads, launched = _kernels(lambda: torch.autograd.grad(out, (q, k, v), do))
    assert f"bwd_pair_kernel<{D}, {int(mask == 'documents')}>" in launched, launched
    ref = [x.detach().float().permute(0, 2, 1, 3).contiguous().requires_grad_(True) for x in (q, k, v)]
    s = (ref[0] @ ref[1].transpose(2, 3)) / np.sqrt(D)
    (torch.softmax(s.masked_fill(~seen, -float("inf")), -1) @ ref[2]).backward(do.float().permute(0, 2, 1, 3))
    for got, x in zip(grads, ref):
        assert max(_rel(got.float().cpu().numpy(), x.grad.permute(0, 2, 1, 3).cpu().numpy())) <= GRAD_TOL


@pytest.mark.parametrize("mask,S,H,D,forward,backward", [
    # even rows on up to a quarter more workgroups than places: halved, an odd number of tiles among them
    ("none", 8100, 9, 128, "halved", "bwd_pair_kernel<128, 0>"), ("none", 4095, 18, 64, "halved", "bwd_pair_kernel<64, 0>"),
    ("alibi", 8100, 9, 128, "halved", "bwd_pair_kernel<128, 1>"), ("none", 7700, 9, 96, "halved", "bwd_pair_kernel<96, 0>"),
    # ... up to one and a half times the places: whole, on the same kernel
    ("none", 4090, 24, 128, "whole", None),
    # slabs of different lengths, all on their places at once or a few more than there are
    ("causal", 4090, 16, 128, "whole", "bwd_pair_kernel<128, 0>"), ("causal", 2047, 32, 128, "whole", "bwd_pair_kernel<128, 0>"),
    ("causal", 16300, 5, 128, "whole", "bwd_pair_kernel<128, 0>"), ("causal", 2300, 30, 128, None, "bwd_pair_kernel<128, 0>"),
    # slabs of one length, a few more than places; long ones that all have a place stay on the long-stretch kernel
    ("none", 4090, 18, 128, "halved", "bwd_pair_kernel<128, 0>"), ("none", 8190, 8, 128, "whole", "dkdv_kernel<128, 0, true>")])
def test_long_rows_about_as_many_as_places(device, mask, S, H, D, forward, backward):
    g = torch.Generator(device=device).manual_seed(S + H)
    leaves = [torch.randn((1, S, H, D), device=device, generator=g).to(torch.bfloat16).requires_grad_(True) for _ in range(3)]
    do = torch.randn((1, S, H, D), device=device, generator=g).to(torch.bfloat16)
    slopes = torch.logspace(-1, -8, H, base=2, device=device)
    fn = {"causal": ra.causal_bias(), "alibi": ra.alibi_bias(slopes)}.get(mask)
    with torch.no_grad():
        _, launched = _kernels(lambda: ra.ring_attention(*leaves, 1, fn))
    if forward:
        assert f"fwd_pair_kernel<{D}, {int(mask == 'alibi')}>" in launched
        assert any(x.startswith("pair_combine_kernel") for x in launched) == (forward == "halved"), launched
    out, lse = ra.ring_attention_with_lse(*leaves, 1, fn, out_dtype=torch.float32)
    grads, launched = _kernels(lambda: torch.autograd.grad(out, leaves, do.float()))
    assert backward is None or backward in launched, launched
    at = torch.arange(S, device=device)
    for h in (0, H // 2, H - 1):
        ref = [x.detach()[0, :, h].float().requires_grad_(True) for x in leaves]
        s = ref[0] @ ref[1].T / np.sqrt(D)
        if mask == "causal":
            s = s.masked_fill(at[:, None] < at[None], -float("inf"))
        elif mask == "alibi":
            s = s - slopes[h] * (at[:, None] - at[None]).abs()
        want = torch.softmax(s, -1) @ ref[2]
        assert (out[0, :, h] - want).abs().max() <= OUT_TOL and (lse[0, h] - torch.logsumexp(s, -1)).abs().max() <= LSE_TOL
        want.backward(do[0, :, h].float())
        for got, x in zip(grads, ref):
            assert max(_rel(got[0, :, h].float().cpu().numpy(), x.grad.cpu().numpy())) <= GRAD_TOL


@pytest.mark.parametrize("S", [63, 65, 1027, 2049, 4100, 16500])
@pytest.mark.parametrize("kind", ["documents", "prefix", "both"])
def test_tile_lists_of_any_length(device, S, kind):
    """Ids and flags that are read a kilobyte at a time, rows that are aligned and that are not, the last tiles of a row, ids in any
    order: documents that come back later, prefix flags in the middle."""
    B, H, D = 2, 1, 32
    g = torch.Generator(device=device).manual_seed(S)
    q, k, v, do = (torch.randn((B, S, H, D), device=device, generator=g).to(torch.bfloat16) for _ in range(4))
    at = torch.arange(S, device=device)
    ids = ((at[None] // 97 * torch.tensor([[5], [7]], device=device)) % 11).to(torch.int32)
    flags = ((at[None] // 150) % 3 == torch.tensor([[0], [1]], device=device)).to(torch.int32)
    seen = torch.ones((B, S, S), dtype=torch.bool, device=device)
    fn, kw = None, {}
    if kind != "prefix":
        fn, seen = ra.segment_bias(), seen & (ids[:, :, None] == ids[:, None])
        kw["segment_ids"] = ids
    if kind != "documents":
        fn = ra.prefix_lm_bias() if fn is None else fn + ra.prefix_lm_bias()
        seen = seen & ((at[:, None] >= at[None]) | ((flags[:, :, None] != 0) & (flags[:, None] != 0)))
        kw["prefix_mask"] = flags
    leaves = [x.clone().requires_grad_(True) for x in (q, k, v)]
    out = ra.ring_attention(*leaves, 1, fn, {"q_" + a: x for a, x in kw.items()}, {"kv_" + a: x for a, x in kw.items()})
    grads = torch.autograd.grad(out, leaves, do)
    for b in range(B):
        ref = [x[b, :, 0].float().requires_grad_(True) for x in (q, k, v)]
        s = (ref[0] @ ref[1].T / np.sqrt(D)).masked_fill(~seen[b], -float("inf"))
        want = torch.softmax(s, -1) @ ref[2]
        assert (out[b, :, 0].float() - want).abs().max() <= OUT_TOL
        want.backward(do[b, :, 0].float())
        for got, x in zip(grads, ref):
            assert max(_rel(got[b, :, 0].float().cpu().numpy(), x.grad.cpu().numpy())) <= GRAD_TOL


@pytest.mark.parametrize("summary", [True, False])
@pytest.mark.parametrize("Lq,Lk,D,columns", [(3, 40, 128, 40), (37, 130, 64, 131), (64, 64, 128, 64), (101, 33, 128, 200), (70, 300, 64, 300)])
def test_values_of_a_dense_block_on_both_gradients(device, monkeypatch, Lq, Lk, D, columns, summary):
    """More slabs than compute units: dkdv_pair_kernel reads the block's rows by a scalar address and the lanes' offset, and a tile that
    is not whole by an address per lane; rows that are further apart than they are long, masked entries among the values."""
    monkeypatch.setattr(bias_module, "DENSE_SUMMARY", summary)
    H = 270
    g = torch.Generator(device=device).manual_seed(Lq + D)
    q, k, v, do = (torch.randn((1, H, L, D), device=device, generator=g).to(torch.bfloat16) for L in (Lq, Lk, Lk, Lq))
    block = torch.randn((1, H, Lq, columns), device=device, generator=g)[..., :Lk]
    block[:, :, :, 1::5] = -float("inf")
    scale = 1 / np.sqrt(D)
    ref = [x.float().requires_grad_(True) for x in (q, k, v)]
    s = ref[0] @ ref[1].transpose(2, 3) * scale + block
    out = torch.softmax(s, -1) @ ref[2]
    out.backward(do.float())
    grads, launched = _kernels(lambda: ra.bwd_block(q, k, v, block, out.detach().to(torch.bfloat16), torch.logsumexp(s, -1).detach(), do, scale))
    assert f"bwd_pair_kernel<{D}, 2>" in launched, launched
    for got, x in zip(grads, ref):
        assert max(_rel(got.cpu().numpy(), x.grad.cpu().numpy())) <= GRAD_TOL
