"""The single-row (decode) kernel at the sizes where its split can go wrong:
key counts around its 32-key blocks, 256-key chunks and the lengths at which the
chunk grows, 1 to 33 query heads per K/V head (16 per workgroup), every padded
head dim, windows, ALiBi and soft-cap on grouped heads, log-sum-exps, ragged and
empty sequences.

A sequence's chunks depend on its own key count alone and every rescale is by a
power of two, so walking the chunks in one workgroup, splitting them over several
and merging, and any mixture must give the same bits; the oracle bars are the
16-bit ones of the other kernels."""
from __future__ import annotations

import pytest
import torch

import mtlflashattn_amd as mfa
from mtlflashattn_amd import _hip, _kernel
from oracle import chunked
from gpu_util import DEV, REL_16, REL_16_OUT, default_scale, make_qkv, make_varlen, max_err

pytestmark = pytest.mark.gpu


def both_ways(monkeypatch, f):
    """f() with a workspace (the library splits the chunks where it likes) and
    without one (one workgroup walks them)."""
    monkeypatch.setattr(_kernel, "_SPLIT_KEYS", None)
    a = f()
    monkeypatch.setattr(_kernel, "_SPLIT_KEYS", 0)
    b = f()
    monkeypatch.setattr(_kernel, "_SPLIT_KEYS", None)
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    return a


def check(monkeypatch, q, k, v, what, **kw):
    out, lse = both_ways(monkeypatch, lambda: mfa.flash_attn_func_with_lse(q, k, v, **kw))
    ref, ref_lse = chunked.flash_attn_func(q.cpu(), k.cpu(), v.cpu(), return_lse=True,
                                           **{x: (y.cpu() if torch.is_tensor(y) else y) for x, y in kw.items()})
    rmax = ref.abs().max().item()
    assert max_err(out, ref) <= REL_16_OUT * rmax, what
    fin = torch.isfinite(ref_lse)
    assert torch.equal(torch.isfinite(lse.cpu()), fin), what
    assert (lse.cpu() - ref_lse).abs()[fin].max().item() <= 4e-3, what
    ws = kw.get("window_size", (-1, -1))
    o32 = _kernel.forward_bshd(q, k, v, default_scale(q.shape[-1]), kw.get("causal", False), kw.get("softcap", 0.0),
                               ws[0], ws[1], kw.get("alibi_slopes"), out_dtype=torch.float32)
    assert max_err(o32, ref) <= REL_16 * rmax, what


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lk", [1, 31, 33, 127, 129, 255, 256, 257, 513, 1025, 4096, 16384, 16385])
def test_key_counts(dtype, lk, monkeypatch):
    for d, hq, hkv in ((128, 8, 2), (64, 4, 4)):
        q, k, v = make_qkv(2, 1, lk, hq, hkv, d, dtype, seed=lk)
        check(monkeypatch, q, k, v, f"Lk={lk} D={d}", causal=True)


@pytest.mark.parametrize("d", [8, 32, 40, 64, 72, 96, 128])
@pytest.mark.parametrize("r", [1, 3, 8, 16, 17, 33])
def test_head_dims_and_groups(d, r, monkeypatch):
    q, k, v = make_qkv(1, 1, 700, 2 * r, 2, d, torch.bfloat16, seed=d + r)
    check(monkeypatch, q, k, v, f"D={d} R={r}")


@pytest.mark.parametrize("d", [64, 96, 128])
def test_features_on_grouped_heads(d, monkeypatch):
    q, k, v = make_qkv(2, 1, 1500, 8, 2, d, torch.bfloat16, seed=d)
    slopes = torch.linspace(0.05, 0.4, 8, device=DEV)
    for kw in (dict(window_size=(100, 0), causal=True), dict(window_size=(700, 3)), dict(window_size=(0, 0)),
               dict(alibi_slopes=slopes), dict(alibi_slopes=slopes.expand(2, 8).contiguous(), softcap=5.0),
               dict(softcap=3.0, window_size=(900, -1), alibi_slopes=slopes)):
        check(monkeypatch, q, k, v, f"D={d} {sorted(kw)}", **kw)
        # grouped heads equal repeated K/V heads
        out = mfa.flash_attn_func(q, k, v, **kw)
        assert torch.equal(out, mfa.flash_attn_func(q, k.repeat_interleave(4, 2), v.repeat_interleave(4, 2), **kw)), kw


def test_long_sequences_and_their_chunk_lengths(monkeypatch):
    # chunks of 256 to 2048 keys in one ragged batch, each sequence as alone
    lens = [70000, 300, 33000, 17000, 0, 16384, 1]
    q, k, v, cu_q, cu_k = make_varlen([1] * len(lens), lens, 4, 1, 64, torch.bfloat16, seed=9)
    out, lse = both_ways(monkeypatch, lambda: mfa.flash_attn_varlen_func_with_lse(q, k, v, cu_q, cu_k, 1, max(lens)))
    ends = torch.tensor(lens).cumsum(0).tolist()
    for i, (n, e) in enumerate(zip(lens, ends)):
        if n == 0:
            assert (out[i] == 0).all() and torch.isneginf(lse[:, i]).all()
            continue
        alone, l1 = mfa.flash_attn_func_with_lse(q[None, i:i + 1], k[None, e - n:e], v[None, e - n:e])
        assert torch.equal(alone[0, 0], out[i]) and torch.equal(l1[0, :, 0], lse[:, i]), n
        ref = chunked.flash_attn_func(q[None, i:i + 1].cpu(), k[None, e - n:e].cpu(), v[None, e - n:e].cpu())
        assert max_err(alone, ref) <= REL_16_OUT * ref.abs().max().item(), n


def test_batches_that_walk_and_batches_that_split():
    # the same sequence in batches of every launch shape
    q, k, v = make_qkv(1, 1, 2000, 8, 8, 128, torch.bfloat16, seed=4)
    want = mfa.flash_attn_func(q, k, v)
    for b in (3, 20, 32, 33, 70):
        out = mfa.flash_attn_func(q.expand(b, -1, -1, -1), k.expand(b, -1, -1, -1), v.expand(b, -1, -1, -1))
        assert torch.equal(out, want.expand(b, -1, -1, -1)), b


def test_infinite_and_nan_inputs_stay_visible():
    q, k, v = make_qkv(1, 1, 900, 4, 2, 64, torch.bfloat16, seed=5)
    v2 = v.clone()
    v2[0, 5, 0, 3] = float("inf")
    out = mfa.flash_attn_func(q, k, v2)
    # (not finite: the two terms of a weight may differ in sign)
    assert not torch.isfinite(out[0, 0, :2, 3]).any() and torch.isfinite(out[0, 0, 2:]).all()
    k2 = k.clone()
    k2[0, 700, 1] = float("nan")
    out = mfa.flash_attn_func(q, k2, v)
    assert torch.isnan(out[0, 0, 2:]).all() and torch.isfinite(out[0, 0, :2]).all()
    # a key whose scores are all -inf drops out; equal scores far below zero do not
    big = torch.full_like(k[:, :1], -1e4)
    ones = torch.ones_like(q)
    out = mfa.flash_attn_func(ones, torch.cat([big] * 600, 1), v[:, :600])
    assert max_err(out, v[:, :600].float().mean(1, keepdim=True).repeat_interleave(2, 2).cpu()) <= 2e-3


def test_static_scratch_beyond_its_size_walks():
    # a request whose own chunks fit the static scratch is taken, whatever the
    # single-row kernel's chunks would need
    B, Lk, H, D = 64, 4096, 64, 128
    q = torch.randn(B, 1, H, D, device=DEV).bfloat16()
    k = torch.randn(1, Lk, 4, D, device=DEV).bfloat16().expand(B, -1, -1, -1)
    ref = mfa.flash_attn_func(q, k, k)
    out = torch.empty_like(q)
    p = _hip.MfaFwdParams()
    p.q, p.k, p.v, p.o = q.data_ptr(), k.data_ptr(), k.data_ptr(), out.data_ptr()
    p.q_batch_stride, p.q_seq_stride, p.q_head_stride = q.stride()[:3]
    p.k_batch_stride, p.k_seq_stride, p.k_head_stride = k.stride()[:3]
    p.v_batch_stride, p.v_seq_stride, p.v_head_stride = k.stride()[:3]
    p.o_batch_stride, p.o_seq_stride, p.o_head_stride = out.stride()[:3]
    p.batch, p.heads_q, p.heads_kv, p.seqlen_q, p.seqlen_k, p.head_dim = B, H, 4, 1, Lk, D
    p.scale, p.window_left, p.window_right = default_scale(D), -1, -1
    p.dtype_in = p.dtype_out = _hip.MFA_DTYPE_BF16
    _hip.fwd_splitkv_static(p, 2048, torch.cuda.current_stream().cuda_stream)
    assert torch.equal(out, ref)
