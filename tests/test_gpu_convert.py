"""ra_convert (csrc/ra_convert.hip): casts and pads between a caller's arrays and the kernels' operands, bit for bit
what torch's cast, pad and slice give, over head dims, dtypes, alignments and strides; and the calls that take it."""
import pytest
import torch

import ring_attention as ra
from ring_attention import ring as rr

DTYPES = [torch.bfloat16, torch.float16, torch.float32]


def _arrays(device, dtype, d):
    g = torch.Generator().manual_seed(d)
    base = torch.randn((3, 37, 5, 2 * d + 3), generator=g) * torch.logspace(-42, 30, 37)[None, :, None, None]
    base[0, 0, 0, :4] = torch.tensor([float("inf"), float("-inf"), float("nan"), -0.0])
    base = base.to(dtype).to(device)
    return {
        "contiguous": base[..., :d].contiguous(),
        "odd start and pitch": base[..., 1:1 + d],
        "heads first": base[..., :d].contiguous().permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3),
        "broadcast batch": base[:1, ..., :d].expand(3, -1, -1, -1),
        "inner stride 2": base[..., :2 * d:2],
    }


def _same(a, b):
    both_nan = torch.isnan(a) & torch.isnan(b)
    return a.dtype == b.dtype and bool(((a == b) & (torch.signbit(a) == torch.signbit(b)) | both_nan).all())


def _check_convert(device, src, dst, d, to_d):
    arrays = _arrays(device, src, d)
    for names in [list(arrays)[:3], list(arrays)[3:]]:
        got = rr._convert([arrays[n] for n in names], [dst] * len(names), to_d)
        for n, o in zip(names, got):
            t = arrays[n]
            want = (t[..., :to_d] if to_d <= d else torch.nn.functional.pad(t, (0, to_d - d))).to(dst)
            assert o.is_contiguous() and _same(o, want), n


@pytest.mark.gpu
@pytest.mark.parametrize("d,to_d", [(1, 64), (7, 64), (32, 64), (64, 64), (80, 128), (96, 128), (127, 128), (128, 128),
                                    (128, 80), (128, 99), (64, 1)])
@pytest.mark.parametrize("src", DTYPES)
@pytest.mark.parametrize("dst", DTYPES)
def test_convert_is_cast_and_pad(device, src, dst, d, to_d):
    _check_convert(device, src, dst, d, to_d)


@pytest.mark.parametrize("src", DTYPES + [torch.float64])
def test_what_the_kernel_does_not_take_goes_through_torch(src):
    _check_convert("cpu", src, torch.bfloat16, 96, 128)
    _check_convert("cpu", src, torch.bfloat16, 64, 64)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [24, 64, 72, 128])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("grad", [(True, True, True), (True, False, True), (False, False, False)])
def test_calls_equal_the_same_call_on_operands_cast_by_hand(device, dtype, d, grad):
    # cast and pad are exact on both sides, so everything between must be the same bits
    g = torch.Generator().manual_seed(d)
    q, k, v, do = (torch.randn((2, 200, 3, d), generator=g).to(device, dtype) for _ in range(4))
    pad = rr._kernel_dim(d) - d
    hand = [torch.nn.functional.pad(x.to(torch.bfloat16), (0, pad)) for x in (q, k, v, do)]
    for xs in (q, k, v), hand[:3]:
        for x, need in zip(xs, grad):
            x.requires_grad_(need)
    kw = dict(bias_fn=ra.causal_bias(), sm_scale=0.17)
    out, lse = ra.ring_attention_with_lse(q, k, v, 2, **kw)
    want, want_lse = ra.ring_attention_with_lse(*hand[:3], 2, out_dtype=torch.float32 if dtype == torch.float32 else None, **kw)
    want = want[..., :d].to(dtype)
    assert out.shape == q.shape and _same(out, want) and torch.equal(lse, want_lse)
    assert out.requires_grad == any(grad)
    if any(grad):
        out.backward(do)
        want.backward(hand[3][..., :d].to(dtype))
        for x, y, need in zip((q, k, v), hand, grad):
            assert (x.grad is not None) == need
            if need:
                assert x.grad.shape == x.shape and _same(x.grad, y.grad[..., :d].to(dtype))


class _Cut(torch.autograd.Function):
    """Passes its input on and no gradient back."""
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, g):
        return None


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.float16, 72), (torch.float32, 128)])
def test_a_missing_gradient_of_the_output_counts_as_zero(device, dtype, d):
    q, k, v = (torch.randn((1, 200, 2, d), device=device, dtype=dtype, requires_grad=True) for _ in range(3))
    grads = torch.autograd.grad(_Cut.apply(ra.ring_attention(q, k, v, 2)).sum(), (q, k, v))
    for g, x in zip(grads, (q, k, v)):
        assert g.shape == x.shape and g.dtype == x.dtype and not g.any()
