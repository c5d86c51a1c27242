"""Gradients of the packed entry points, written in place in one packed tensor:
bit-identical to the gradients of the same call on separate tensors, for dense
and ragged batches, packed qkv and kv, head dims that need padding (which go
through tensors of their own), grouped heads, non-contiguous inputs, empty
batches, and inputs of which only one needs a gradient."""
from __future__ import annotations

import pytest
import torch

import mtlflashattn_amd as mfa
from gpu_util import DEV

pytestmark = pytest.mark.gpu

CASES = [(torch.bfloat16, 64), (torch.float16, 128), (torch.bfloat16, 33), (torch.float32, 40)]


def rand(*shape, dtype):
    return torch.randn(*shape, device=DEV).to(dtype)


def grad(f, ts, dout):
    ts = [t.detach().requires_grad_() for t in ts]
    return torch.autograd.grad(f(*ts), ts, dout)


@pytest.mark.parametrize("dtype,d", CASES)
@pytest.mark.parametrize("strided", [False, True])
def test_dense(dtype, d, strided):
    torch.manual_seed(d)
    qkv = rand(2, 70, 3, 4, d, dtype=dtype)
    if strided:
        qkv = rand(2, 70, 3, 4, 2 * d, dtype=dtype)[..., :d]
    dout = rand(2, 70, 4, d, dtype=dtype)
    (g,) = grad(lambda x: mfa.flash_attn_qkvpacked_func(x, causal=True), [qkv], dout)
    ref = grad(lambda q, k, v: mfa.flash_attn_func(q, k, v, causal=True), qkv.unbind(2), dout)
    assert g.shape == qkv.shape and torch.equal(g, torch.stack(ref, 2))

    q, kv = rand(2, 50, 8, d, dtype=dtype), rand(2, 90, 2, 2, d, dtype=dtype)
    dout = rand(2, 50, 8, d, dtype=dtype)
    got = grad(lambda a, b: mfa.flash_attn_kvpacked_func(a, b, 0.0, None, True), [q, kv], dout)
    ref = grad(lambda q, k, v: mfa.flash_attn_func(q, k, v, causal=True), [q, *kv.unbind(2)], dout)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], torch.stack(ref[1:], 2))


@pytest.mark.parametrize("dtype,d", CASES)
def test_ragged(dtype, d):
    torch.manual_seed(d)
    lens = [40, 0, 1, 130]
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    qkv, dout = rand(sum(lens), 3, 4, d, dtype=dtype), rand(sum(lens), 4, d, dtype=dtype)
    (g,) = grad(lambda x: mfa.flash_attn_varlen_qkvpacked_func(x, cu, 130, causal=True), [qkv], dout)
    ref = grad(lambda q, k, v: mfa.flash_attn_varlen_func(q, k, v, cu, cu, 130, 130, causal=True), qkv.unbind(1), dout)
    assert torch.equal(g, torch.stack(ref, 1))
    kv = rand(sum(lens), 2, 2, d, dtype=dtype)
    got = grad(lambda a, b: mfa.flash_attn_varlen_kvpacked_func(a, b, cu, cu, 130, 130), [qkv[:, 0], kv], dout)
    ref = grad(lambda q, k, v: mfa.flash_attn_varlen_func(q, k, v, cu, cu, 130, 130), [qkv[:, 0], *kv.unbind(1)], dout)
    assert torch.equal(got[0], ref[0]) and torch.equal(got[1], torch.stack(ref[1:], 1))


def test_one_input_needs_a_gradient_and_empty_batches():
    q, kv = rand(1, 20, 4, 64, dtype=torch.bfloat16), rand(1, 20, 2, 4, 64, dtype=torch.bfloat16)
    dout = rand(1, 20, 4, 64, dtype=torch.bfloat16)
    both = grad(mfa.flash_attn_kvpacked_func, [q, kv], dout)
    for i in range(2):
        ts = [q.detach(), kv.detach()]
        ts[i].requires_grad_()
        (g,) = torch.autograd.grad(mfa.flash_attn_kvpacked_func(*ts), ts[i], dout)
        assert torch.equal(g, both[i])
    (g,) = grad(mfa.flash_attn_qkvpacked_func, [rand(0, 20, 3, 4, 64, dtype=torch.bfloat16)], dout[:0])
    assert g.shape == (0, 20, 3, 4, 64)


def test_prepared_parameters_follow_layout_and_alignment():
    # the same shapes again as other views: gradients are those of contiguous copies
    torch.manual_seed(1)
    shape = (2, 40, 4, 64)
    q, k, v, dout = (rand(*shape, dtype=torch.bfloat16) for _ in range(4))
    ref = grad(mfa.flash_attn_func, [q, k, v], dout)

    def off(t):  # contiguous, 2 bytes past an aligned address
        b = torch.empty(t.numel() + 8, dtype=t.dtype, device=DEV)[1:1 + t.numel()].view(t.shape)
        return b.copy_(t)

    def strided(t):
        b = torch.empty(*t.shape[:-1], 72, dtype=t.dtype, device=DEV)[..., :64]
        return b.copy_(t)

    def heads_second(t):
        return t.transpose(1, 2).contiguous().transpose(1, 2)

    for change in (off, strided, heads_second):
        for i in range(4):
            ts = [q, k, v, dout]
            ts[i] = change(ts[i])
            got = grad(mfa.flash_attn_func, ts[:3], ts[3])
            assert all(torch.equal(a, b) for a, b in zip(got, ref)), (change.__name__, i)
    again = grad(mfa.flash_attn_func, [q, k, v], dout)
    assert all(torch.equal(a, b) for a, b in zip(again, ref))
