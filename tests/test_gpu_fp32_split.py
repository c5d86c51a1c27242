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
