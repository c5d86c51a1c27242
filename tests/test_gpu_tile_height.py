"""The two heights of the 4-wavefront 16-bit tiles at head dims up to 64 (256
and 128 query rows): row counts around both tile edges, every mask, packed
heads, paging and split keys give the same bits at either height, and both
sides of the rule that chooses between them."""
from __future__ import annotations

import pytest
import torch

import mtlflashattn_amd as mfa
from mtlflashattn_amd import _hip, _kernel
from oracle import chunked
from gpu_util import DEV, assert_output, make_qkv, make_varlen


def name(B, L, H, Hk, d, **kw):
    q, k = (torch.empty(B, L, h, d, dtype=torch.bfloat16) for h in (H, Hk))
    return _kernel.launch_info(q, k, k, **kw).kernel_name.decode().replace(" ", "")


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("B,L,H,Hk,causal,rows", [
    (32, 197, 12, 12, False, 128),   # 384 tiles of 256 rows
    (64, 197, 12, 12, False, 256),   # 768, each row tile full to the same 256
    (64, 300, 16, 16, False, 128),   # 512 padded rows against 384
    (64, 512, 16, 16, False, 256),
    (64, 512, 16, 16, True, 128),    # a causal tile of 256 walks 1/5 more keys
    (16, 2048, 16, 16, True, 256),   # 1/17 more
    (16, 1024, 32, 8, True, 256),    # 4 heads in a tile: 64 positions
    (1, 4096, 20, 20, False, 128),   # 320 tiles: a quarter past one round
    (5, 1024, 16, 16, True, 128),
])
def test_rule(monkeypatch, d, B, L, H, Hk, causal, rows):
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the rule is stated for 256 compute units")
    assert name(B, L, H, Hk, d, causal=causal) == f"mfa_fwd16<bf16,d{d},{rows // 128},2>"
    # the hint that names the tall tiles gets them
    monkeypatch.setattr(_kernel, "_TILE_HINT", _hip.MFA_TILE_256)
    assert name(B, L, H, Hk, d, causal=causal) == f"mfa_fwd16<bf16,d{d},2,2>"


def both_heights(monkeypatch, run):
    auto = run()
    with monkeypatch.context() as m:
        m.setattr(_kernel, "_TILE_HINT", _hip.MFA_TILE_256)
        tall = run()
    for x, y in zip(auto, tall):
        assert torch.equal(x, y)
    return auto[0]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [24, 32, 64])
@pytest.mark.parametrize("lq,lk", [(2, 2), (127, 130), (128, 64), (129, 257), (255, 90), (257, 1000), (385, 385), (40, 5000)])
def test_same_bits_at_either_height(monkeypatch, dtype, d, lq, lk):
    q, k, v = make_qkv(2, lq, lk, 4, 2, d, dtype, seed=lq + lk + d)
    kws = [{}, {"causal": True}, {"window_size": (40, 17)}, {"causal": True, "window_size": (100, 0)}]
    if d <= 32:
        kws.append({"softcap": 5.0, "alibi_slopes": torch.linspace(0.02, 0.3, 4, device=DEV)})
    for kw in kws:
        out = both_heights(monkeypatch, lambda: mfa.flash_attn_func_with_lse(q, k, v, **kw))
        cpu = {x: (y.cpu() if torch.is_tensor(y) else y) for x, y in kw.items()}
        ref = chunked.flash_attn_func(q.cpu(), k.cpu(), v.cpu(), **cpu)
        assert_output(out, ref, dtype, f"D={d} {lq}x{lk} {list(kw)}")


@pytest.mark.gpu
@pytest.mark.parametrize("d", [32, 64])
def test_ragged_and_paged(monkeypatch, d):
    from test_gpu_lse_paged import paginate

    lens_q, lens_k = [5, 0, 130, 2, 300], [9, 7, 600, 0, 3000]
    q, k, v, cu_q, cu_k = make_varlen(lens_q, lens_k, 4, 2, d, torch.bfloat16, seed=3)
    args = (cu_q, cu_k, max(lens_q), max(lens_k))
    out = both_heights(monkeypatch, lambda: (mfa.flash_attn_varlen_func(q, k, v, *args, causal=True),))
    pk, pv, table = paginate(k, v, lens_k, 256, seed=4)
    paged = both_heights(
        monkeypatch, lambda: (mfa.flash_attn_varlen_func(q, pk, pv, *args, causal=True, block_table=table),))
    assert torch.equal(out, paged)
    ref = chunked.flash_attn_varlen_func(q.cpu(), k.cpu(), v.cpu(), cu_q.cpu(), cu_k.cpu(), causal=True)
    assert_output(out, ref, torch.bfloat16, "ragged")
