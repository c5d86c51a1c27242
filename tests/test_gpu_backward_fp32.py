"""The fp32 backward's matrix-core kernels where their split can go wrong:
lengths around the 32-row / 32-key tiles and around the four wavefronts' share
of a walk, every padded head dim, grouped heads, masks, grids that fold, and
rows too far apart for 32-bit offsets.  Reference: float64 autograd of the
oracle.

Bar: 5e-6 of max|grad| (the bar of the fp32 gradients elsewhere), plus
D * 2^-23 * max|dout| * max|v| * max|k or q| * scale for the rounding of the
two sums dO.V and dO.O, each of D products, whose difference is 0 where a row
sees one key."""
from __future__ import annotations

import pytest
import torch

import mtlflashattn_amd as mfa
from mtlflashattn_amd import _kernel
from oracle import chunked
from gpu_util import DEV, make_qkv

pytestmark = pytest.mark.gpu


def grads(q, k, v, dout, **kw):
    q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
    return torch.autograd.grad(mfa.flash_attn_func(q, k, v, **kw), (q, k, v), dout)


def check(q, k, v, dout, what, **kw):
    got = grads(q, k, v, dout, **kw)
    ref = chunked.attention_grads(q, k, v, dout, causal=kw.get("causal", False),
                                  window_size=kw.get("window_size", (-1, -1)), softcap=kw.get("softcap", 0.0),
                                  dtype=torch.float64)
    D = q.shape[-1]
    top = [t.abs().max().item() for t in (dout, v, q, k)]
    for name, g, r, other in zip(("dq", "dk", "dv"), got, ref, (top[3], top[2], 0.0)):
        bar = 5e-6 * r.abs().max().item() + D ** 0.5 * 2.0 ** -23 * top[0] * top[1] * other
        err = (g.double().cpu() - r).abs().max().item()
        assert err <= bar, f"{what} {name}: {err:.2e} > {bar:.2e}"


@pytest.mark.parametrize("D", [8, 32, 64, 72, 96, 128])
@pytest.mark.parametrize("Lq,Lk", [(1, 1), (31, 33), (32, 32), (33, 31), (97, 128), (129, 161), (5, 300)])
def test_tile_edges(D, Lq, Lk):
    q, k, v = make_qkv(2, Lq, Lk, 6, 2, D, torch.float32, seed=Lq + Lk)
    dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(D)).to(DEV)
    check(q, k, v, dout, f"D={D} {Lq}x{Lk}")
    check(q, k, v, dout, f"D={D} {Lq}x{Lk} causal", causal=True)
    check(q, k, v, dout, f"D={D} {Lq}x{Lk} window + soft-cap", window_size=(40, 17), softcap=4.0)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_grids_of_one_to_two_workgroups_per_cu(D):
    # 12 units x 31 tiles (the reversed slots of a causal grid) and both
    # sides of it
    for L in (600, 961, 1100):
        q, k, v = make_qkv(1, L, L, 12, 12, D, torch.float32, seed=L)
        dout = torch.randn(q.shape, generator=torch.Generator().manual_seed(L)).to(DEV)
        check(q, k, v, dout, f"D={D} L={L}", causal=True)


def test_rows_beyond_32_bit_offsets():
    # 32 rows span more than 2 GiB: the same gradients, bit for bit
    L, D, stride = 35, 64, (1 << 24) + 4
    base = torch.empty((L - 1) * stride + 2 * D, device=DEV)
    q, k, v = make_qkv(1, L, L, 2, 2, D, torch.float32, seed=1)
    dout = torch.randn(q.shape, device=DEV)

    def wide(t):
        w = base.as_strided(t.shape, (0, stride, D, 1))
        w.copy_(t)
        return w

    # (the backward itself: the forward takes such strides in q only)
    out, lse = mfa.flash_attn_func_with_lse(q, k, v, causal=True)

    def bwd(q, k, v, dout):
        return _kernel._run_bwd(q, k, v, out, dout, lse, scale=0.125, causal=True, softcap=0.0, window_left=-1,
                                window_right=-1, alibi=None, alibi_bstride=0)

    ref = bwd(q, k, v, dout)
    for i in range(4):
        ts = [q, k, v, dout]
        ts[i] = wide(ts[i])
        assert all(torch.equal(a, b) for a, b in zip(bwd(*ts), ref)), i


@pytest.mark.parametrize("d", [64, 128])
def test_gradients_do_not_depend_on_the_batch(d):
    # (the forward's two kernels give the same output and log-sum-exp, and the
    # backward's order of sums is the sequence's own)
    q, k, v = make_qkv(40, 256, 256, 8, 2, d, torch.float32, seed=d)
    dout = torch.randn(q.shape, device=DEV)
    names = [_kernel.launch_info(t[:n], u[:n], u[:n], causal=True).kernel_name for t, u, n in ((q, k, 40), (q, k, 1))]
    assert b"split" not in names[0] and b"split" in names[1]
    whole = grads(q, k, v, dout, causal=True)
    alone = grads(q[7:8], k[7:8], v[7:8], dout[7:8], causal=True)
    for a, b in zip(whole, alone):
        assert torch.equal(a[7:8], b)
