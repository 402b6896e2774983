"""The autograd node of a call on a whole sequence (csrc/ra_host.cc): what autograd asks of one beyond the gradients, and
operands that need more than a conversion of all three."""
import numpy as np
import pytest
import torch

import ring_attention as ra
from ring_attention import _lib
from test_gpu_parity import GRAD_TOL, OUT_TOL, _rel

pytestmark = pytest.mark.gpu


def _arrays(device, D=64, dtypes=(torch.bfloat16,) * 3, S=130):
    g = torch.Generator(device=device).manual_seed(D)
    return [torch.randn((2, S, 2, D), device=device, generator=g).to(torch.bfloat16).to(t).requires_grad_(True) for t in dtypes]


def _check(out, leaves, do, got):
    ref = [x.detach().float().permute(0, 2, 1, 3).contiguous().requires_grad_(True) for x in leaves]
    s = (ref[0] @ ref[1].transpose(2, 3)) / np.sqrt(ref[0].shape[-1])
    want = torch.softmax(s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -float("inf")), -1) @ ref[2]
    assert (out.float() - want.permute(0, 2, 1, 3)).abs().max() <= OUT_TOL
    want.backward(do.float().permute(0, 2, 1, 3))
    for x, r, g in zip(leaves, ref, got):
        if g is None:
            continue
        assert g.dtype == x.dtype and g.shape == x.shape
        assert max(_rel(g.float().cpu().numpy(), r.grad.permute(0, 2, 1, 3).cpu().numpy())) <= GRAD_TOL


@pytest.mark.parametrize("kind", ["mixed dtypes", "double", "inner stride", "rows too close", "gradient of another dtype", "expanded gradient",
                                  "padded head dim", "two of three", "retained"])
def test_operands_and_gradients_of_any_form(device, kind):
    b, f, h = torch.bfloat16, torch.float32, torch.float16
    leaves = _arrays(device, 40 if kind == "padded head dim" else 64,
                     {"mixed dtypes": (b, f, h), "double": (torch.float64,) * 3, "two of three": (f, f, f)}.get(kind, (b, b, b)))
    q, k, v = leaves
    if kind == "inner stride":
        q, k, v = (x.transpose(2, 3).contiguous().transpose(2, 3) for x in (q, k, v))
    elif kind == "rows too close":
        k = torch.cat([k, k[..., :4]], -1)[..., :64]  # rows of 68 elements
    if kind == "two of three":
        k = k.detach()
    out = ra.ring_attention(q, k, v, 1, ra.causal_bias())
    do = torch.randn(out.shape, device=device).to(out.dtype)
    if kind == "gradient of another dtype":
        do = torch.randn(out.shape, device=device)
        out_ = out.float()
    elif kind == "expanded gradient":
        do = torch.randn((1, 1, 1, 64), device=device).to(b).expand(out.shape)
    wanted = [x for x in (leaves if kind != "two of three" else (leaves[0], leaves[2]))]
    for _ in range(2 if kind == "retained" else 1):
        got = list(torch.autograd.grad(out_ if kind == "gradient of another dtype" else out, wanted, do, retain_graph=kind == "retained"))
    if kind == "two of three":
        got.insert(1, None)
    _check(out, leaves, do, got)


def test_what_autograd_asks_of_a_node(device):
    q, k, v = _arrays(device)
    do = torch.randn(q.shape, device=device).to(torch.bfloat16)
    call = lambda *x: ra.ring_attention(*x, 1, ra.causal_bias())
    want = torch.autograd.grad(call(q, k, v), (q, k, v), do)
    # tensors saved for the backward go through the hooks in force, here to host memory and back
    with torch.autograd.graph.save_on_cpu():
        out = call(q, k, v)
    for a, b in zip(want, torch.autograd.grad(out, (q, k, v), do)):
        assert torch.equal(a, b)
    # ... and are recomputed by a checkpoint
    out = torch.utils.checkpoint.checkpoint(call, q, k, v, use_reentrant=False)
    for a, b in zip(want, torch.autograd.grad(out, (q, k, v), do)):
        assert torch.equal(a, b)
    # an operand changed in place after the call is refused, as is a second backward
    x = q.detach().clone().requires_grad_(True)
    y = x * 1
    out = call(y, k, v)
    with torch.no_grad():
        y.mul_(2)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(out, x, do)
    out = call(q, k, v)
    torch.autograd.grad(out, q, do)
    with pytest.raises(RuntimeError, match="second time"):
        torch.autograd.grad(out, q, do)
    # the logsumexp carries no gradient, and a backward without one for the output gives zeros
    out, lse = ra.ring_attention_with_lse(q, k, v, 1)
    assert out.requires_grad and not lse.requires_grad
    # transforms that the node does not know stay refused
    with pytest.raises(RuntimeError):
        torch.func.vmap(call)(q[None], k[None], v[None])
    with pytest.raises(RuntimeError):
        torch.func.jvp(call, (q, k, v), (q, k, v))
    with torch.no_grad():
        assert not call(q, k, v).requires_grad
    with torch.inference_mode():
        assert torch.equal(call(q, k, v), call(q.detach(), k, v))


def test_errors_of_the_library_reach_the_caller(device):
    q, k, v = _arrays(device)
    with pytest.raises(_lib.RingAttentionHipError, match="sm_scale"):
        ra.ring_attention(q, k, v, 1, sm_scale=-1.0)


def test_tracing_stays_refused(device):
    # a trace would hold the allocations and not the kernels
    with pytest.raises(RuntimeError):
        torch.jit.trace(lambda *x: ra.ring_attention(*x, 1), [x.detach() for x in _arrays(device)], check_trace=False)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("impl", ["pallas", "hip"])
@pytest.mark.parametrize("k_shape,v_shape", [((2, 130, 3, 64), (2, 130, 2, 64)), ((2, 130, 2, 64), (3, 200, 4, 64)), ((4, 130, 2, 64), (4, 130, 2, 64))])
def test_keys_and_values_beyond_the_call(device, k_shape, v_shape, impl, dtype):
    # they take no part: the output is that of the operands cut to size, and the gradients there are zeros
    g = torch.Generator(device=device).manual_seed(k_shape[2])
    q, k, v = (torch.randn(s, device=device, generator=g).to(torch.bfloat16).to(dtype).requires_grad_(True) for s in ((2, 130, 2, 64), k_shape, v_shape))
    out = ra.ring_attention(q, k, v, 1, ra.causal_bias(), block_impl=impl)
    do = torch.randn(out.shape, device=device, generator=g).to(torch.bfloat16).to(out.dtype)
    grads = torch.autograd.grad(out, (q, k, v), do)
    cut = [x.detach()[:2, :130, :2].contiguous().requires_grad_(True) for x in (q, k, v)]
    want = ra.ring_attention(*cut, 1, ra.causal_bias(), block_impl=impl)
    assert torch.equal(out, want)
    for got, x in zip(grads, torch.autograd.grad(want, cut, do)):
        assert torch.equal(got[:2, :130, :2], x) and got.count_nonzero() == x.count_nonzero()


@pytest.mark.parametrize("impl", ["pallas", "hip"])
def test_keys_and_values_from_host_memory(device, impl):
    q, k, v = _arrays(device)
    do = torch.randn(q.shape, device=device).to(torch.bfloat16)
    at_home = [x.detach().cpu().requires_grad_(True) for x in (k, v)]
    out, want = (ra.ring_attention(q, *kv, 1, ra.causal_bias(), block_impl=impl) for kv in (at_home, (k, v)))
    assert torch.equal(out, want)
    for got, x in zip(torch.autograd.grad(out, (q, *at_home), do), torch.autograd.grad(want, (q, k, v), do)):
        assert torch.equal(got.to(device), x)
    assert got.device.type == "cpu"
