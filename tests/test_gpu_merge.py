"""merge_attention_partials in one HIP launch (mfa_merge) against the same
merge in float64 and against the torch ops it stands in for: sizes around the
kernel's 16-position x 4-head tiles, part counts around its groups of four,
strided parts, rows without a key in some or all parts, +inf and NaN.

Bars: the kernel sums n products in fp32 (relative error <= (n + 2) * 2^-24 of
sum |w_i o_i| plus the weights' exp error, a few 2^-24), then rounds once to
the output type (half an ulp: 2^-8 for the 8 significant bits of
bf16, 2^-11 for the 11 of fp16)."""
from __future__ import annotations

import pytest
import torch

import mtlflashattn_amd as mfa
from mtlflashattn_amd import _kernel

ROUND = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11, torch.float32: 0.0}


def parts_of(shape, n, dtype, dev, seed=0):
    *lead, L, H, D = shape
    g = torch.Generator().manual_seed(seed)
    outs = [torch.randn(shape, generator=g).to(dev, dtype) for _ in range(n)]
    lses = [(4 * torch.randn(*lead, H, L, generator=g)).to(dev) for _ in range(n)]
    return outs, lses


def exact(outs, lses):
    l = torch.stack([x.double() for x in lses])
    lse = torch.logsumexp(l, 0)
    w = torch.exp(l - lse.masked_fill(torch.isinf(lse), 0)).masked_fill(torch.isinf(lse), 0)
    terms = [o.double() * w[i].transpose(-1, -2).unsqueeze(-1) for i, o in enumerate(outs)]
    return sum(terms), sum(t.abs() for t in terms), lse


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape,n", [((1, 1, 1, 8), 1), ((2, 15, 3, 40), 2), ((1, 16, 4, 64), 3), ((1, 17, 5, 128), 4),
                                     ((33, 6, 80), 5), ((3, 2, 9, 128), 8), ((40, 4, 16), 16)])
def test_matches_float64(dtype, shape, n):
    outs, lses = parts_of(shape, n, dtype, "cuda", seed=n)
    lses[-1][..., ::3] = float("-inf")  # rows without a key in the last part
    for l in lses:
        l[..., :1, :1] = float("-inf")  # ... and in every part
    # strided parts (views with a wider row) beside contiguous ones
    if n > 1:
        wide = torch.randn(*shape[:-1], shape[-1] + 8, device="cuda").to(dtype)
        wide[..., :shape[-1]] = outs[1]
        outs[1] = wide[..., :shape[-1]]
        lses[1] = lses[1].transpose(-1, -2).contiguous().transpose(-1, -2)
    assert _kernel.merge_partials(outs, lses) is not None
    out, lse = mfa.merge_attention_partials(outs, lses)
    ref, mag, ref_lse = exact(outs, lses)
    assert out.dtype == dtype and out.shape == outs[0].shape and lse.dtype == torch.float32
    bar = ROUND[dtype] * ref.abs() + (n + 16) * 2.0 ** -24 * mag + (2.0 ** -24 if dtype == torch.float16 else 1e-38)
    assert ((out.double() - ref).abs() <= bar).all()
    assert torch.equal(torch.isneginf(lse), torch.isneginf(ref_lse))
    f = torch.isfinite(ref_lse)
    assert ((lse.double() - ref_lse).abs()[f] <= 4e-6 * ref_lse.abs()[f].clamp(min=1)).all()


@pytest.mark.gpu
def test_infinite_and_nan_rows_follow_the_torch_ops(monkeypatch):
    outs, lses = parts_of((1, 8, 2, 16), 3, torch.float32, "cuda", seed=3)
    lses[0][0, 0, 0] = float("inf")
    lses[1][0, 0, 1] = float("nan")
    outs[2][0, 2, 0, 0] = float("inf")
    outs[2][0, 3, 0, 0] = float("nan")
    lses[2][0, 0, 3] = float("-inf")
    got = mfa.merge_attention_partials(outs, lses)
    monkeypatch.setattr(_kernel, "merge_partials", lambda o, l: None)
    ref = mfa.merge_attention_partials(outs, lses)
    for a, b in zip(got, ref):
        torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-6, equal_nan=True)


@pytest.mark.gpu
def test_calls_outside_the_kernel_keep_the_torch_ops():
    outs, lses = parts_of((1, 9, 2, 16), 2, torch.bfloat16, "cuda")
    take = _kernel.merge_partials
    assert take(outs, lses) is not None
    assert take(outs * 9, lses * 9) is None  # more parts than one launch takes
    assert take([o.float() for o in outs[:1]] + outs[1:], lses) is None
    assert take([o.transpose(1, 2).contiguous().transpose(1, 2) for o in outs], lses) is None
    assert take(outs, [l.double() for l in lses]) is None
    assert take([o[..., :12].contiguous() for o in outs], lses) is None  # rows of 24 bytes
    req = [o.clone().requires_grad_() for o in outs]
    assert take(req, lses) is None
    with torch.no_grad():
        assert take(req, lses) is not None
    out, _ = mfa.merge_attention_partials(outs * 9, lses * 9)
    ref, mag, _ = exact(outs * 9, lses * 9)
    assert ((out.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 64 * 2.0 ** -24 * mag).all()


def test_transforms_and_cpu_tensors_run_the_torch_ops():
    outs, lses = parts_of((2, 5, 2, 8), 2, torch.float32, "cpu")
    assert _kernel.merge_partials(outs, lses) is None
    assert _kernel._plain(*outs)
    seen = []
    ref, _ = mfa.merge_attention_partials(outs, lses)

    def one(o0, o1, l0, l1):
        seen.append(_kernel._plain(o0))
        return mfa.merge_attention_partials([o0, o1], [l0, l1])[0]

    torch.testing.assert_close(torch.vmap(one)(*outs, *lses), ref)
    with torch.autograd.forward_ad.dual_level():
        seen.append(_kernel._plain(outs[0]))
    torch.jit.trace(lambda x: (seen.append(_kernel._plain(x)), x + 1)[1], outs[0], check_trace=False)

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    with Mode():
        seen.append(_kernel._plain(outs[0]))

    class Sub(torch.Tensor):
        pass

    seen.append(_kernel._plain(outs[0].as_subclass(Sub)))
    assert len(seen) == 5 and not any(seen)
