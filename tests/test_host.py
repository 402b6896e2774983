"""CPU-only checks of the host-side mirror of the reference interface (no kernels run)."""
import ctypes as C

import numpy as np
import pytest
import torch

import ring_attention as ra
from ring_attention import ring as rr
from ring_attention.bias import BiasFn


def test_public_names_match_reference_package():
    # reference __init__.py:3 re-exports exactly these two
    assert callable(ra.ring_attention) and callable(ra.ring_self_attention)


def test_bias_composition_and_flags():
    b = ra.causal_bias() + ra.segment_bias()
    assert b.causal and b.segments and b.flags == 1 | 4
    w = ra.sliding_window_bias(128) + ra.sliding_window_bias(64)
    assert w.window == 64 and w.flags == 1 | 2
    a = ra.alibi_bias([0.5, 0.25]) + ra.alibi_bias([0.5, 0.25])
    assert torch.allclose(a.alibi_slopes, torch.tensor([1.0, 0.5]))
    with pytest.raises(ValueError):
        ra.causal_bias() + ra.prefix_lm_bias()  # ring.py:368-374
    with pytest.raises(ValueError):
        ra.sliding_window_bias(0)
    np.testing.assert_allclose(ra.alibi_slopes(8).numpy(), [2.0 ** -(i + 1) for i in range(8)])


def test_cpu_tensors_fail_loudly():
    q = torch.zeros(1, 64, 1, 64)
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        ra.ring_attention(q, q, q, 2)


def test_block_impl_and_bias_type_errors():
    q = torch.zeros(1, 64, 1, 64)
    with pytest.raises(ValueError):
        ra.ring_attention(q, q, q, 2, block_impl="triton")  # ring.py:312 raises ValueError too
    # the reference's own two values are both accepted (ring.py:296-311): they get past the
    # block_impl check and fail on the CPU tensors like any other call
    for impl in ("jax", "pallas", "hip", "hip_fused"):
        with pytest.raises(RuntimeError, match="no CPU fallback"):
            ra.ring_attention(q, q, q, 2, block_impl=impl)
    with pytest.raises(TypeError):
        ra.ring_attention(q, q, q, 2, bias_fn="causal")  # neither a BiasFn nor a callable
    with pytest.raises(TypeError):
        rr._axis_size("sp")
    assert rr._axis_size(ra.RingAxis("sp", 8)) == 8 and rr._axis_size(("sp", 4)) == 4


def test_ring_self_attention_argument_rules():
    q = torch.zeros(1, 64, 1, 64)
    pos = torch.arange(64)[None]
    with pytest.raises(AssertionError):
        ra.ring_self_attention(q, q, q, 2, causal=True)  # positions required (ring.py:369)
    with pytest.raises(AssertionError):
        ra.ring_self_attention(q, q, q, 2, causal=True, positions=pos, prefix_mask=pos)  # ring.py:370
    with pytest.raises(AssertionError):
        ra.ring_self_attention(q, q, q, 2, prefix_mask=pos)  # ring.py:373


def test_long_segment_shards_are_walked_as_a_finer_ring():
    seg, causal = ra.segment_bias(), ra.causal_bias()
    cap = rr._lib.RA_MAX_SEGMENT_SHARD
    assert cap == 65536
    assert rr._walked_ring_size(1, 98304, 98304, seg + causal) == 2      # 2 x 49152
    assert rr._walked_ring_size(2, 4 * cap, 4 * cap, seg) == 4           # shards of 2 x cap -> cap
    assert rr._walked_ring_size(2, 4 * cap + 6, 4 * cap + 6, seg) == 10  # shards of 131075 = 5 x 26215
    assert rr._walked_ring_size(1, 98304, 1024, seg) == 2                # the longer side decides
    assert rr._walked_ring_size(1, 98304, 1023, seg) == 3                # ... and both must divide
    assert rr._walked_ring_size(8, 8 * cap, 8 * cap, seg) == 8           # at the limit: untouched
    assert rr._walked_ring_size(1, 98304, 98304, causal) == 1            # no segment term: no limit
    assert rr._walked_ring_size(1, 98304, 98304, None) == 1
    assert rr._walked_ring_size(1, 2 * 65537, 2 * 65537, seg) == 1       # 2 x a prime: left to the library's check


def test_ring_plan_shards_and_offsets():
    q = torch.zeros(2, 64, 2, 64, dtype=torch.bfloat16)
    k = torch.zeros(2, 32, 2, 64, dtype=torch.bfloat16)
    seg_q = torch.arange(64)[None].repeat(2, 1) // 10
    seg_k = torch.arange(32)[None].repeat(2, 1) // 10
    plan = rr._RingPlan(q, k, 4, ra.causal_bias() + ra.segment_bias(),
                        {"q_segment_ids": seg_q, "q_positions": torch.arange(64)[None].repeat(2, 1) + 100},
                        {"kv_segment_ids": seg_k})
    assert (plan.Lq, plan.Lk) == (16, 8)
    assert plan.q_off == [100, 116, 132, 148] and plan.kv_off == [0, 8, 16, 24]
    bb = plan.block_bias(2, 3)
    assert bb.q_offset == 132 and bb.kv_offset == 24
    assert torch.equal(bb.q_segment_ids, seg_q[:, 32:48].to(torch.int32))
    assert torch.equal(bb.kv_segment_ids, seg_k[:, 24:32].to(torch.int32))
    # shards may restart their positions, but must be consecutive inside
    pos = torch.cat([torch.arange(16) + 7 * i for i in range(4)])[None].repeat(2, 1)
    plan = rr._RingPlan(q, k, 4, ra.causal_bias(), {"q_positions": pos}, {})
    assert plan.q_off == [0, 7, 14, 21]
    # any other positions are honoured through a dense block per ring step, built from the
    # position arrays exactly like the reference's mask builder (ring.py:393-409)
    plan = rr._RingPlan(q, k, 4, ra.causal_bias() + ra.segment_bias(),
                        {"q_positions": pos * 2, "q_segment_ids": seg_q}, {"kv_segment_ids": seg_k})
    assert plan.callable is not None and plan.fn is None
    bb = plan.block_bias(1, 2)
    assert tuple(bb.dense.shape) == (2, 1, 16, 8)
    qp, kp = (pos * 2)[:, 16:32], torch.arange(32)[None].repeat(2, 1)[:, 16:24]
    want = (kp[:, None, :] <= qp[:, :, None]) & (seg_q[:, 16:32, None] == seg_k[:, None, 16:24])
    assert torch.equal(bb.dense[:, 0] == 0, want) and torch.equal(torch.isneginf(bb.dense[:, 0]), ~want)
    # positions that differ across the batch take the same path
    pos_b = torch.stack([torch.arange(64), torch.arange(64) + 3])
    assert rr._RingPlan(q, k, 4, ra.causal_bias(), {"q_positions": pos_b}, {}).callable is not None
    with pytest.raises(ValueError):
        rr._RingPlan(q, k, 3, None, None, None)  # 64 % 3 != 0
    with pytest.raises(ValueError):
        rr._RingPlan(q, k, 4, ra.segment_bias(), {"q_segment_ids": seg_q}, {})
    with pytest.raises(ValueError):
        rr._RingPlan(q, k, 4, ra.causal_bias(), {"bogus": seg_q}, {})
    with pytest.raises(ValueError):
        rr._RingPlan(q, k, 4, None, {"q_segment_ids": seg_q}, {})


def test_ring_plan_counts_the_steps_that_cost_something():
    q = torch.zeros(1, 64, 1, 64, dtype=torch.bfloat16)
    plan = rr._RingPlan(q, q, 4, ra.causal_bias(), None, None)
    assert [plan.live_steps(r, None) for r in range(4)] == [1, 2, 3, 4]
    assert [plan.live_steps(None, r) for r in range(4)] == [4, 3, 2, 1]
    plan = rr._RingPlan(q, q, 4, ra.sliding_window_bias(18), None, None)  # shards of 16 tokens
    assert [plan.live_steps(r, None) for r in range(4)] == [1, 2, 3, 3]
    plan = rr._RingPlan(q, q, 4, ra.sliding_window_bias(5, causal=False), None, None)
    assert [plan.live_steps(r, None) for r in range(4)] == [2, 3, 3, 2]
    assert rr._RingPlan(q, q, 4, None, None, None).live_steps(2, None) == 4
    # agrees with the library's own classification of a step
    lib = rr._lib.load()
    for fn in (ra.causal_bias(), ra.sliding_window_bias(17), ra.sliding_window_bias(18), ra.sliding_window_bias(5, causal=False)):
        plan = rr._RingPlan(q, q, 4, fn, None, None)
        for r in range(4):
            live = 0
            for s in range(4):
                st = plan.block_bias(r, s).to_struct(torch.device("cpu"))
                live += not lib.ra_step_is_skippable(st, 16, 16)
            assert plan.live_steps(r, None) == live


@pytest.mark.parametrize("starts,want", [
    ([0, 16, 32, 48], (1, [0])),              # consecutive: one shard
    ([100, 116, 132, 148], (1, [100])),
    ([0, 16, 64, 80], (2, [0, 64])),          # two pieces of two shards each
    ([0, 64, 16, 80], (4, [0, 64, 16, 80])),  # nothing follows on
])
def test_consecutive_shards_are_joined(starts, want):
    q = torch.zeros(1, 64, 1, 64, dtype=torch.bfloat16)
    pos = torch.cat([torch.arange(16) + s for s in starts])[None]
    plan = rr._RingPlan(q, q, 4, ra.causal_bias(), {"q_positions": pos}, {"kv_positions": pos})
    joined = plan.joined()
    assert (joined.n, joined.q_off) == want and joined.kv_off == joined.q_off
    assert (joined.Lq, joined.Lk) == (64 // joined.n,) * 2
    assert plan.n == 4 and plan.joined() is joined and joined.joined() is joined
    # only one side consecutive, a shard that would outgrow the tile lists
    assert rr._RingPlan(q, q, 4, ra.causal_bias(), {"q_positions": pos}, None).joined().n == want[0]
    long = torch.zeros(1, 1, 1, 64, dtype=torch.bfloat16).expand(1, 4 * 32768, 1, 64)
    ids = torch.zeros(1, 1, dtype=torch.int32).expand(1, 4 * 32768)
    plan = rr._RingPlan(long, long, 4, ra.causal_bias() + ra.segment_bias(), {"q_segment_ids": ids}, {"kv_segment_ids": ids})
    assert plan.joined().n == 2


def test_joined_shards_stay_within_one_launch():
    # 4 shards of 2^23 tokens: the library takes two of them as one, not all four
    long = torch.zeros(1, 1, 1, 64, dtype=torch.bfloat16).expand(1, 4 << 23, 1, 64)
    plan = rr._RingPlan(long, long, 4, ra.sliding_window_bias(128), None, None)
    assert (plan.joined().n, plan.joined().Lq) == (2, 1 << 24)


def test_ring_plan_with_a_callable_bias_fn():
    # the reference's general form: the callable sees the shards of its kwargs (ring.py:107,186)
    q = torch.zeros(2, 64, 2, 64, dtype=torch.bfloat16)
    k = torch.zeros(2, 32, 2, 64, dtype=torch.bfloat16)
    feat_q = torch.arange(2 * 64 * 3, dtype=torch.float32).reshape(2, 64, 3)
    ids_k = torch.arange(32)[None].repeat(2, 1)
    seen = {}

    def fn(q_feat, kv_ids):
        seen["q"], seen["k"] = q_feat, kv_ids
        return torch.zeros(2, 1, q_feat.shape[1], kv_ids.shape[1])

    plan = rr._RingPlan(q, k, 4, fn, {"q_feat": feat_q}, {"kv_ids": ids_k})
    bb = plan.block_bias(2, 3)
    assert torch.equal(seen["q"], feat_q[:, 32:48]) and torch.equal(seen["k"], ids_k[:, 24:32])
    assert bb.dense.shape == (2, 1, 16, 8) and bb.fn.flags == 0
    bb.check_dense_shape(2, 2, 16, 8)
    with pytest.raises(ValueError):
        bb.check_dense_shape(2, 2, 16, 9)
    s = bb.to_struct(torch.device("cpu"))
    assert s.flags == 32 and s.dense_stride_h == 0 and s.dense_stride_q == 8 and s.dense_stride_b == 128
    with pytest.raises(ValueError):
        rr._RingPlan(q, k, 4, fn, {"q_feat": feat_q[:, :10]}, {"kv_ids": ids_k})
    with pytest.raises(TypeError):
        rr._RingPlan(q, k, 4, lambda **kw: None, {}, {}).block_bias(0, 0)


def test_shard_view_is_zero_copy():
    x = torch.arange(2 * 8 * 3 * 4).reshape(2, 8, 3, 4)
    s = rr._shard_bhld(x, 1, 4)
    assert s.shape == (2, 3, 4, 4) and s.data_ptr() == x[:, 4:].data_ptr()
    assert torch.equal(s[1, 2, 3], x[1, 7, 2])


def test_launch_scheme_per_block_impl():
    q = torch.zeros(1, 64, 1, 64, dtype=torch.bfloat16)
    plain = rr._RingPlan(q, q, 4, ra.causal_bias(), None, None)
    dense = rr._RingPlan(q, q, 4, lambda q_ids, kv_ids: torch.zeros(1, 1, 16, 16),
                         {"q_ids": torch.zeros(1, 64)}, {"kv_ids": torch.zeros(1, 64)})
    # the reference's default spelling picks the scheme; its "jax" is the plain per-step loop
    assert rr._launch_whole_ring("pallas", plain) and not rr._launch_whole_ring("pallas", dense)
    assert not rr._launch_whole_ring("jax", plain) and not rr._launch_whole_ring("hip", plain)
    assert rr._launch_whole_ring("hip_fused", plain) and rr._launch_whole_ring("hip_fused", dense)
    import inspect
    for f in (ra.ring_attention, ra.ring_self_attention, ra.ring_attention_with_lse):
        assert inspect.signature(f).parameters["block_impl"].default == "pallas"  # ring.py:255


def test_plans_are_cached_per_bias_arrays():
    ra.clear_plan_cache()
    q = torch.zeros(2, 64, 2, 64, dtype=torch.bfloat16)
    seg = torch.arange(64)[None].repeat(2, 1) // 10
    fn = ra.causal_bias() + ra.segment_bias()
    a = rr._plan_for(q, q, 4, fn, {"q_segment_ids": seg}, {"kv_segment_ids": seg})
    assert rr._plan_for(q, q, 4, fn, {"q_segment_ids": seg}, {"kv_segment_ids": seg}) is a
    assert rr._plan_for(q, q, 4, ra.causal_bias() + ra.segment_bias(), {"q_segment_ids": seg},
                        {"kv_segment_ids": seg}) is a           # an equal description, not the same object
    assert rr._plan_for(q, q, 2, fn, {"q_segment_ids": seg}, {"kv_segment_ids": seg}) is not a
    seg2 = seg.clone()
    assert rr._plan_for(q, q, 4, fn, {"q_segment_ids": seg2}, {"kv_segment_ids": seg2}) is not a
    seg += 1                                                    # in place: a new version of the same tensor
    b = rr._plan_for(q, q, 4, fn, {"q_segment_ids": seg}, {"kv_segment_ids": seg})
    assert b is not a and torch.equal(b.q_seg, seg.to(torch.int32))
    # positions are read back on the host when a plan is made: the offsets follow the array
    pos = torch.arange(64)[None].repeat(2, 1)
    p1 = rr._plan_for(q, q, 4, ra.causal_bias(), {"q_positions": pos}, {})
    pos += 5
    p2 = rr._plan_for(q, q, 4, ra.causal_bias(), {"q_positions": pos}, {})
    assert p1.q_off == [0, 16, 32, 48] and p2.q_off == [5, 21, 37, 53]
    for i in range(20):                                         # bounded
        rr._plan_for(q, q, 4, ra.sliding_window_bias(i + 1), None, None)
    assert len(rr._PLAN_CACHE) <= rr._PLAN_CACHE_SIZE
    ra.clear_plan_cache()
    assert not rr._PLAN_CACHE


def test_a_callable_bias_is_built_in_bounded_chunks():
    q = torch.zeros(1, 256, 1, 64, dtype=torch.bfloat16)
    calls = []

    def fn(q_ids, kv_ids):
        calls.append((int(q_ids[0, 0]), int(kv_ids[0, 0])))
        return torch.zeros(1, 1, q_ids.shape[1], kv_ids.shape[1])

    ids = torch.arange(256)[None]
    plan = rr._RingPlan(q, q, 32, fn, {"q_ids": ids}, {"kv_ids": ids})
    chunks = list(rr._row_chunks(plan, 3))
    assert [len(c) for c in chunks] == [16, 16]                 # what one launch walks
    assert [s for c in chunks for s, _ in c] == [(3 - t) % 32 for t in range(32)]   # ring order, ring.py:51-55
    assert len(calls) == 32 and all(a == 24 for a, _ in calls)  # one block per pair, each built once
    old = rr._DENSE_BLOCKS_BYTES
    try:
        rr._DENSE_BLOCKS_BYTES = 3 * 8 * 8 * 4                  # three 8 x 8 blocks
        assert [len(c) for c in rr._row_chunks(plan, 0)] == [3] * 10 + [2]
    finally:
        rr._DENSE_BLOCKS_BYTES = old


def test_views_the_kernels_cannot_take_are_copied():
    # a view is passed through when its rows are 16-byte aligned, do not overlap and lie within the
    # row stride of the C ABI; otherwise the host makes a contiguous copy
    base = torch.zeros((2, 16, 4, 64 + 8), dtype=torch.bfloat16)
    ready = lambda t: rr._kernel_inputs((t,), 64)[0]
    padded = base[..., :64]                       # row stride 4 * 72, inner stride 1
    assert ready(padded) is padded
    odd = torch.zeros((2, 16, 4, 65), dtype=torch.bfloat16)[..., :64]   # strides not multiples of 8
    assert ready(odd).is_contiguous()
    same_row = torch.zeros((2, 1, 4, 64), dtype=torch.bfloat16).expand(2, 16, 4, 64)   # row stride 0
    got = ready(same_row)
    assert got.is_contiguous() and got.shape == same_row.shape
    heads_interleaved = torch.zeros((2, 4, 16, 64), dtype=torch.bfloat16).permute(0, 2, 1, 3)  # [b, l, h, d] view, row stride 64
    assert ready(heads_interleaved) is heads_interleaved
    assert ready(torch.zeros((1, 8, 1, 64))).dtype == torch.bfloat16


@pytest.mark.parametrize("D", [32, 64, 96, 128])
def test_dk_and_dv_share_their_strides_whatever_those_of_k_and_v(monkeypatch, D):
    # k a transposed [b, h, l, d], v contiguous, and the other way round: the library stores both gradients with dk's strides.  The
    # native call on host arrays, with functions in the library's place
    calls = []
    addr, size = C.c_void_p, C.c_int64
    fwd = C.CFUNCTYPE(C.c_int, addr, C.c_int32, addr, addr, C.c_int32, size, size, size, addr, addr, size, addr)(lambda *args: 0)
    bwd = C.CFUNCTYPE(C.c_int, addr, C.c_int32, addr, addr, C.c_int32, size, size, size, C.c_int32, addr, size, size, size, addr, addr, size,
                      size, size, addr, size, addr)(lambda *args: calls.append(args) or 0)
    room = C.CFUNCTYPE(size, addr)(lambda p: 64)
    host, lib = rr._lib.host(), rr._lib.load()
    host.init(*(C.cast(f, addr).value for f in (fwd, bwd, room, lib.ra_convert)), rr._lib.check)
    try:
        B, L, H = 2, 48, 3
        rows = torch.zeros((B, L, H, D), dtype=torch.bfloat16)
        heads = torch.zeros((B, H, L, D), dtype=torch.bfloat16).permute(0, 2, 1, 3)
        plan = rr._RingPlan(rows, rows, 1, None, None, None).joined()
        assert plan.D == D
        for case in [(heads, heads, rows), (rows, rows, heads), (heads, heads, heads), (heads, rows, rows)]:
            leaves = [x.detach().requires_grad_(True) for x in case]
            out, lse = host.attend(*leaves, plan.native(rows), 0.1, torch.bfloat16, torch.bfloat16)
            node = torch.autograd.grad(out, leaves, rows)
            plain = host.backward(*case, rows, lse, rows, plan.native(rows), 0.1)
            for dq, dk, dv in (plain, node):
                k, v = case[1:]
                assert dk.stride() == dv.stride() and (dk.stride() == k.stride() or k.stride() != v.stride())
                assert dq.stride() == case[0].stride()
                sb, sl, sh, _ = dk.stride()
                assert calls.pop()[-8:-3] == (dk.data_ptr(), dv.data_ptr(), sb, sh, sl)
    finally:
        monkeypatch.setattr(rr._lib, "_host", None)
        rr._lib.host()
    # the launches of a ring of several shards take their gradients from the same place
    grads = rr._empty_gradients(heads, heads, rows)
    assert grads[1].stride() == grads[2].stride() and grads[0].stride() == heads.stride()


@pytest.mark.parametrize("what", ["shape", "dtype", "head dim", "output", "gradient", "logsumexp"])
def test_the_native_calls_refuse_what_is_not_an_operand(what):
    x = torch.zeros((2, 48, 3, 64), dtype=torch.bfloat16)
    lse = torch.zeros((1, 2, 3, 48))
    plan = rr._RingPlan(x, x, 1, None, None, None).joined().native(x)
    host = rr._lib.host()
    q = {"shape": x[:, :40], "dtype": x.float(), "head dim": x[..., :32]}.get(what, x)
    if q is not x:
        with pytest.raises(RuntimeError, match="operands"):
            host.forward(q, x, x, plan, 0.1, torch.bfloat16)
    with pytest.raises(RuntimeError, match="operands|are not those of q"):
        host.backward(q, x, x, x[:1] if what == "output" else x, lse[:, :1] if what == "logsumexp" else lse, x[..., :32] if what == "gradient" else x, plan, 0.1)
    for args in [((x,) * 5, 64), ((), 64), ((x[0],), 64)]:
        with pytest.raises(RuntimeError, match="arrays"):
            host.operands(*args)


@pytest.mark.parametrize("D", [16, 32, 80, 96, 160])
def test_blocks_take_head_dims_64_and_128_only(monkeypatch, D):
    # forward and backward alike: the head dims of whole sequences (multiples of 32) are no head dims of a ring step
    monkeypatch.setattr(rr, "_require_gpu", lambda t: None)
    monkeypatch.setattr(rr, "_stream", lambda: None)
    x = torch.zeros((1, 2, 128, D), dtype=torch.bfloat16)
    rows = torch.zeros((1, 2, 128))
    acc = torch.zeros((1, 2, 128, D))
    with pytest.raises(RuntimeError, match=f"head dim {D} unsupported .64 or 128"):
        ra.fwd_block(x, x, x, None, acc, rows.clone(), rows.clone(), 0.1)
    for bias in (None, ra.BlockBias(ra.causal_bias()), torch.zeros((1, 1, 128, 128))):
        with pytest.raises(RuntimeError, match=f"head dim {D} unsupported .64 or 128"):
            ra.bwd_block(x, x, x, bias, acc, rows, x, 0.1)


@pytest.mark.parametrize("k_shape,v_shape", [((1, 64, 4, 64), None), ((2, 64, 1, 64), None), ((2, 64, 4, 64), (1, 64, 4, 64)),
                                             ((2, 64, 4, 64), (2, 64, 2, 64)), ((2, 64, 4, 64), (2, 32, 4, 64))])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_operands_smaller_than_the_call_are_refused(monkeypatch, k_shape, v_shape, dtype):
    # one head or batch row of keys for several of queries, values of another length: nothing broadcasts, and the kernels do
    # not look at the end of an array
    monkeypatch.setattr(rr, "_require_gpu", lambda t: None)
    q, k, v = (torch.zeros(s, dtype=dtype) for s in ((2, 64, 4, 64), k_shape, v_shape or k_shape))
    with pytest.raises(ValueError, match="do not hold the batch and heads"):
        ra.ring_attention(q, k, v, 2)


@pytest.mark.parametrize("k_shape,v_shape", [((3, 64, 2, 64), (2, 64, 2, 64)), ((2, 64, 3, 64), (2, 64, 2, 64)), ((2, 64, 2, 64), (2, 80, 2, 64)),
                                             ((3, 64, 4, 64), (4, 70, 3, 64))])
@pytest.mark.parametrize("impl,scheme", [("pallas", "attend"), ("hip", "_RingAttentionFn")])
def test_what_lies_beyond_the_call_does_not_reach_the_kernels(monkeypatch, k_shape, v_shape, impl, scheme):
    # more batch rows or heads than q has, values longer than the keys: dk and dv are stored with the same strides, so k and v that
    # differ in shape would have one of them written past its end
    seen = []

    class Host:
        def plan(self, *args):
            return None

        def attend(self, q, k, v, *args):
            seen.append((q, k, v))
            return q, q

    monkeypatch.setattr(rr, "_require_gpu", lambda t: None)
    monkeypatch.setattr(rr._lib, "host", Host)
    monkeypatch.setattr(rr._RingAttentionFn, "apply", Host().attend)
    q, k, v = (torch.zeros(s, dtype=torch.bfloat16, requires_grad=True) for s in ((2, 64, 2, 64), k_shape, v_shape))
    ra.ring_attention(q, k, v, 1, block_impl=impl)
    (_, k1, v1), = seen
    assert k1.shape == v1.shape == (2, 64, 2, 64) and k1.data_ptr() == k.data_ptr() and v1.data_ptr() == v.data_ptr()
    # the rest has a gradient: zeros
    dk, dv = torch.autograd.grad((k1 * 2 + v1 * 3).sum(), (k, v))
    for g, x in ((dk, 2), (dv, 3)):
        assert g.sum() == x * q.numel() and (g[:2, :64, :2] == x).all()


def test_operands_of_another_plan_are_refused():
    q = torch.zeros((2, 64, 2, 64), dtype=torch.bfloat16)
    bias = bytes(C.sizeof(rr._lib.RaBias))
    plan = rr._lib.host().plan(2, 2, 64, 64, 64, bias, 0, q, ())
    for k, v in [(q[:1], q[:1]), (q, q[:, :32]), (q, torch.cat([q, q], 2)), (q[..., :32], q[..., :32])]:
        with pytest.raises(RuntimeError, match="not the operands of this plan"):
            rr._lib.host().attend(q, k, v, plan, 0.1, torch.bfloat16, torch.bfloat16)


@pytest.mark.parametrize("k_shape,v_shape", [((1, 2, 32, 64), (2, 2, 32, 64)), ((2, 2, 32, 64), (2, 1, 32, 64)), ((2, 2, 32, 64), (2, 2, 31, 64)),
                                             ((2, 2, 32, 32), (2, 2, 32, 64))])
def test_blocks_refuse_keys_and_values_smaller_than_the_call(monkeypatch, k_shape, v_shape):
    monkeypatch.setattr(rr, "_require_gpu", lambda t: None)
    q, k, v = (torch.zeros(s, dtype=torch.bfloat16) for s in ((2, 2, 32, 64), k_shape, v_shape))
    rows, acc = torch.zeros((2, 2, 32)), torch.zeros((2, 2, 32, 64))
    for call in (lambda: ra.fwd_block(q, k, v, None, acc, rows, rows.clone(), 0.1), lambda: ra.bwd_block(q, k, v, None, acc, rows, q, 0.1),
                 lambda: rr.fwd_blocks(q, [(k, v)], [None], acc, rows, rows.clone(), 0.1)):
        with pytest.raises(ValueError, match="do not hold the batch, heads and head dim"):
            call()


@pytest.mark.parametrize("k_shape,v_shape", [((3, 2, 32, 64), (2, 2, 32, 64)), ((2, 3, 32, 64), (2, 2, 32, 64)), ((2, 2, 32, 64), (2, 2, 40, 128)),
                                             ((2, 4, 32, 128), (4, 3, 33, 64))])
@pytest.mark.parametrize("dense", [False, True])
def test_block_gradients_of_what_lies_beyond_the_call(monkeypatch, k_shape, v_shape, dense):
    # dk and dv are stored with the same strides: arrays of one shape, the call's, and zeros around what comes back
    class Library:
        def __getattr__(self, name):
            return lambda *args: 64

        def ra_bwd_step_check(self, p):
            return 0

        def ra_bwd_whole(self, p, *args):
            assert (p._obj.B, p._obj.H, p._obj.Lk, p._obj.D) == (2, 2, 32, 64) and args[-6:-3] == (2 * 32 * 64, 32 * 64, 64)
            for at, x in ((args[-8], 2.0), (args[-7], 3.0)):
                torch.frombuffer((C.c_float * (2 * 2 * 32 * 64)).from_address(at), dtype=torch.float32).fill_(x)
            return 0

    def step(q, k, v, do, lse, delta, dq, dk, dv, *_):
        assert k.shape == v.shape == q.shape
        dk.fill_(2.0)
        dv.fill_(3.0)

    monkeypatch.setattr(rr, "_require_gpu", lambda t: None)
    monkeypatch.setattr(rr, "_stream", lambda: None)
    monkeypatch.setattr(rr, "precompute_delta", lambda o, do: None)
    monkeypatch.setattr(rr, "_bwd_step", step)
    rr._lib.host()
    monkeypatch.setattr(rr._lib, "load", Library)
    q, k, v = (torch.zeros(s, dtype=torch.bfloat16) for s in ((2, 2, 32, 64), k_shape, v_shape))
    dq, *grads = ra.bwd_block(q, k, v, torch.zeros((2, 1, 32, 32)) if dense else None, torch.zeros(q.shape), torch.zeros((2, 2, 32)), q, 0.1)
    for got, x, value in zip(grads, (k, v), (2, 3)):
        assert got.shape == x.shape and got.sum() == value * q.numel() and (got[:2, :2, :32, :64] == value).all()


@pytest.mark.parametrize("elsewhere", ["k", "v", "kv"])
def test_operands_on_another_device_go_to_that_of_the_queries(monkeypatch, elsewhere):
    # a pointer into host memory would fault the GPU; "meta" stands for the other device here (the native call does the same on the GPU)
    seen = []
    monkeypatch.setattr(rr, "_require_gpu", lambda t: None)
    monkeypatch.setattr(rr._RingAttentionFn, "apply", lambda q, k, v, *a: seen.append((k, v)) or (q, q))
    q, k, v = (torch.zeros((1, 64, 2, 64), dtype=torch.bfloat16, device="cpu" if name in elsewhere else "meta") for name in "qkv")
    ra.ring_attention(q, k, v, 1, block_impl="hip")
    assert [x.device.type for x in seen[0]] == ["meta", "meta"]


@pytest.mark.parametrize("at", range(6))
def test_blocks_refuse_arrays_on_another_device(monkeypatch, at):
    monkeypatch.setattr(rr, "_require_gpu", lambda t: None)
    x, rows, acc = torch.zeros((1, 1, 32, 64), dtype=torch.bfloat16), torch.zeros((1, 1, 32)), torch.zeros((1, 1, 32, 64))
    there = lambda *args: [t.to("meta") if i == at else t for i, t in enumerate(args)]
    calls = []
    if at < 5:
        k, v, o, m, l = there(x, x, acc, rows, rows.clone())
        calls += [lambda: ra.fwd_block(x, k, v, None, o, m, l, 0.1), lambda: rr.fwd_blocks(x, [(k, v)], [None], o, m, l, 0.1)]
    if at != 2:
        k1, v1, _, o1, L, do = there(x, x, None, acc, rows, x)
        calls.append(lambda: ra.bwd_block(x, k1, v1, None, o1, L, do, 0.1))
    for call in calls:
        with pytest.raises(ValueError, match="on the device of q"):
            call()


def _build_module():
    import importlib.util
    import os

    spec = importlib.util.spec_from_file_location("ra_build", os.path.join(os.path.dirname(os.path.dirname(rr.__file__)), "build.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.mark.parametrize("torch_is", ["absent", "of another platform"])
def test_the_c_libraries_are_built_without_torch(monkeypatch, tmp_path, torch_is):
    # a host that binds the C ABI or the XLA FFI handlers only
    import sys

    build = _build_module()
    include = tmp_path / "xla" / "ffi" / "api"
    include.mkdir(parents=True)
    (include / "ffi.h").touch()
    ran = []
    monkeypatch.setenv("XLA_FFI_INCLUDE_DIR", str(tmp_path))
    monkeypatch.setattr(build, "OBJ_DIR", str(tmp_path / "build"))
    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(build.subprocess, "run", lambda cmd, **_: ran.append(cmd) or type("Result", (), {"returncode": 0})())
    if torch_is == "absent":
        monkeypatch.setitem(sys.modules, "torch", None)
        monkeypatch.setitem(sys.modules, "torch.utils", None)
    else:
        monkeypatch.setattr(torch.version, "hip", None)
    assert build.build() == build.LIB_PATH
    made = [cmd[cmd.index("-o") + 1] for cmd in ran]
    assert build.LIB_PATH in made and build.FFI_LIB_PATH in made and build.HOST_LIB_PATH not in made


def test_a_call_without_gradients_does_not_plan_a_backward(monkeypatch):
    class Library:
        def ra_fwd_whole_workspace(self, p):
            return 96

    made = []
    q = torch.zeros((1, 64, 2, 64), dtype=torch.bfloat16)
    plan = rr._RingPlan(q, q, 1, ra.causal_bias(), None, None).joined()
    monkeypatch.setattr(rr._lib, "load", Library)
    monkeypatch.setattr(rr._lib, "host", lambda: type("Host", (), {"plan": lambda s, *args: made.append(args)})())
    plan.native(q)
    assert made[0][:5] == (1, 2, 64, 64, 64) and made[0][6:] == (96, q, ())
