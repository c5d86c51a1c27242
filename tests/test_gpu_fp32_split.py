"""The key-split fp32 forward kernel (32 query rows per workgroup, each wavefront
its own key blocks) where its split can go wrong: lengths around 32 rows and 32
keys, fewer key blocks than wavefronts, walks of several blocks each, every
padded head dim, masks, biases, grouped heads, paging and the log-sum-exp; and
both sides of the rule that chooses it.  Oracle bars: the fp32 ones."""
from __future__ import annotations

import pytest
import torch

import mtlflashattn_amd as mfa
from mtlflashattn_amd import _hip, _kernel
from oracle import chunked
from gpu_util import DEV, assert_parity, make_qkv, make_varlen

pytestmark = pytest.mark.gpu

F32 = torch.float32


def kernel(q, k, **kw):
    return _kernel.launch_info(q, k, k, **kw).kernel_name


def check(q, k, v, what, **kw):
    out, lse = mfa.flash_attn_func_with_lse(q, k, v, **kw)
    cpu = {x: (y.cpu() if torch.is_tensor(y) else y) for x, y in kw.items()}
    ref, ref_lse = chunked.flash_attn_func(q.cpu(), k.cpu(), v.cpu(), return_lse=True, **cpu)
    assert_parity(out, ref, F32, what)
    fin = torch.isfinite(ref_lse)
    assert torch.equal(torch.isfinite(lse.cpu()), fin), what
    if fin.any():
        assert (lse.cpu() - ref_lse)[fin].abs().max().item() <= 1e-5 * max(1.0, ref_lse[fin].abs().max().item()), what


@pytest.mark.parametrize("d", [8, 32, 64, 72, 96, 128])
@pytest.mark.parametrize("lq,lk", [(1, 1), (31, 33), (32, 32), (33, 257), (65, 31), (97, 289), (5, 1000)])
def test_tile_edges(d, lq, lk):
    q, k, v = make_qkv(2, lq, lk, 4, 2, d, F32, seed=lq + lk + d)
    assert b"split" in kernel(q, k)
    check(q, k, v, f"D={d} {lq}x{lk}")
    check(q, k, v, f"D={d} {lq}x{lk} causal", causal=True)
    check(q, k, v, f"D={d} {lq}x{lk} window", window_size=(40, 17))
    check(q, k, v, f"D={d} {lq}x{lk} soft-cap + ALiBi", softcap=5.0, alibi_slopes=torch.linspace(0.02, 0.3, 4, device=DEV))


def test_paged_and_ragged_equal_dense():
    from test_gpu_lse_paged import paginate

    lens_q, lens_k = [5, 0, 130, 1, 64], [9, 7, 600, 0, 300]
    q, k, v, cu_q, cu_k = make_varlen(lens_q, lens_k, 4, 2, 64, F32, seed=3)
    args = (cu_q, cu_k, max(lens_q), max(lens_k))
    out = mfa.flash_attn_varlen_func(q, k, v, *args, causal=True)
    pk, pv, table = paginate(k, v, lens_k, 256, seed=4)
    assert torch.equal(out, mfa.flash_attn_varlen_func(q, pk, pv, *args, causal=True, block_table=table))
    sq, sk = ([0] + torch.tensor(x).cumsum(0).tolist() for x in (lens_q, lens_k))
    for i in range(len(lens_q)):
        if lens_q[i]:
            one = mfa.flash_attn_func(q[None, sq[i]:sq[i + 1]], k[None, sk[i]:sk[i + 1]], v[None, sk[i]:sk[i + 1]],
                                      causal=True)[0]
            assert torch.equal(out[sq[i]:sq[i + 1]], one), i


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("B,L,H,causal,split", [(2, 300, 8, True, True), (40, 256, 8, False, False),
                                                (8, 1000, 16, True, False), (3, 700, 4, False, True),
                                                (16, 256, 16, True, False)])
def test_both_sides_of_the_rule(d, B, L, H, causal, split):
    q, k, v = make_qkv(B, L, L, H, H, d, F32, seed=L)
    assert (b"split" in kernel(q, k, causal=causal)) == split
    check(q[:2], k[:2], v[:2], "part of the batch", causal=causal)
    out = mfa.flash_attn_func(q, k, v, causal=causal)
    ref = chunked.flash_attn_func(q[-1:].cpu(), k[-1:].cpu(), v[-1:].cpu(), causal=causal)
    assert_parity(out[-1:], ref, F32, "last of the batch")


# A row's sums are taken in the same order by both kernels, so the choice between
# them -- which depends on how much work the whole call has -- shows in no bit.
@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("kw", [dict(), dict(causal=True), dict(window_size=(100, 30)),
                                dict(causal=True, window_size=(333, 0)), dict(softcap=5.0, alibi=True),
                                dict(causal=True, alibi=True)])
def test_both_kernels_give_the_same_bits(d, kw):
    kw = dict(kw)
    if kw.pop("alibi", False):
        kw["alibi_slopes"] = torch.linspace(0.02, 0.3, 16, device=DEV)
    # (lengths around the 32-key blocks and 32-row tiles, walks of fewer blocks
    # than the key-split kernel has wavefronts, of one each and of several)
    lens_q = [256, 1, 31, 33, 200, 290, 127, 0, 64, 250] * 8
    lens_k = [256, 1, 33, 31, 200, 290, 520, 40, 600, 0] * 8
    q, k, v, cu_q, cu_k = make_varlen(lens_q, lens_k, 16, 8, d, F32, seed=d)
    args = (cu_q, cu_k, max(lens_q), max(lens_k))
    info = {x: y for x, y in kw.items() if x != "alibi_slopes" and x != "window_size"}
    wl, wr = kw.get("window_size", (-1, -1))
    info.update(alibi="alibi_slopes" in kw, window_left=wl, window_right=wr)
    name = _kernel.launch_info_varlen(q, k, len(lens_q), max(lens_q), max(lens_k), **info).kernel_name
    assert b"split" not in name
    out, lse = mfa.flash_attn_varlen_func_with_lse(q, k, v, *args, **kw)
    sq, sk = ([0] + torch.tensor(x).cumsum(0).tolist() for x in (lens_q, lens_k))
    for i in range(10):
        a = (q[None, sq[i]:sq[i + 1]], k[None, sk[i]:sk[i + 1]], v[None, sk[i]:sk[i + 1]])
        if lens_q[i] == 0 or lens_k[i] == 0:
            assert (out[sq[i]:sq[i + 1]] == 0).all()
            continue
        assert b"split" in kernel(a[0], a[1], **info), i
        one, l1 = mfa.flash_attn_func_with_lse(*a, **kw)
        assert torch.equal(out[sq[i]:sq[i + 1]], one[0]), i
        assert torch.equal(lse[:, sq[i]:sq[i + 1]], l1[0]), i


@pytest.mark.parametrize("d,L", [(64, 1500), (128, 1100)])
def test_long_rows_alone_and_in_a_batch_give_the_same_bits(d, L):
    q, k, v = make_qkv(24, L, L, 16, 4, d, F32, seed=d)
    assert b"split" not in kernel(q, k, causal=True) and b"split" in kernel(q[:1, :, :2], k[:1, :, :1], causal=True)
    whole = mfa.flash_attn_func(q, k, v, causal=True)
    one = mfa.flash_attn_func(q[5:6, :, 4:6], k[5:6, :, 1:2], v[5:6, :, 1:2], causal=True)
    assert torch.equal(whole[5:6, :, 4:6], one)


def test_infinite_and_nan_inputs_stay_visible_in_both_kernels():
    for B in (1, 40):
        q, k, v = make_qkv(B, 256, 256, 8, 8, 64, F32, seed=6)
        assert (b"split" in kernel(q, k)) == (B == 1)
        k2 = k.clone()
        k2[0, 200, 1] = float("nan")
        out = mfa.flash_attn_func(q, k2, v)
        assert torch.isnan(out[0, :, 1]).all() and torch.isfinite(out[0, :, 0]).all()
        v2 = v.clone()
        v2[0, 5, 0, 3] = float("inf")
        out = mfa.flash_attn_func(q, k, v2)
        assert torch.isinf(out[0, :, 0, 3]).all() and torch.isfinite(out[0, :, 1:]).all()
