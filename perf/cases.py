"""The work this package is timed on: the attention calls its users make.

A case is one call (or one forward and backward) through a public entry point,
described by plain values.  `listed()` holds the fixed ones, `draw(rng)` makes
more of the same ranges, `prepare` builds what a program holds before the
call, `run` is one pass, `work` what the pass cannot do without, `tolerance`
how far two correct implementations may differ and `exact` the result in 64
bits from plain torch.

The kinds, and what each stands for:

  decode       one new token per sequence against a contiguous K/V cache
               (flash_attn_func, causal); grouped-query and plain heads, from
               one sequence to a serving batch.  The smallest calls.
  decode_paged one new token per sequence against a paged K/V cache of ragged
               lengths (flash_attn_varlen_func with a block table).
  dense        prompt processing / encoders: flash_attn_func over equal
               lengths, causal or not, with and without window, soft-cap and
               ALiBi; query and key lengths may differ.
  varlen       the same over a ragged batch packed without padding
               (flash_attn_varlen_func).
  train        forward and backward of flash_attn_func (output and the three
               gradients).
  train_varlen forward and backward of flash_attn_varlen_qkvpacked_func, the
               ragged training batch of a packed projection.
  merge        merge_attention_partials over the shards of a key range
               (context parallelism, cache + new tokens).
"""
from __future__ import annotations

import math

import torch

import mtlflashattn_amd as mfa

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_DEV = "cuda"


# --------------------------------------------------------------------------
# the cases


def listed():
    return [
        # One user's next token: a single sequence, grouped-query heads, a
        # short and odd context.  Latency and idle compute units decide it.
        dict(name="decode_one_gqa_d128", kind="decode", dtype="bf16", B=1, Lk=3001, Hq=32, Hkv=8, D=128),
        # A small batch of plain heads at head dim 64.
        dict(name="decode_batch_d64", kind="decode", dtype="fp16", B=6, Lk=1500, Hq=16, Hkv=16, D=64),
        # A serving batch over a paged cache: ragged contexts, pages of 256.
        dict(name="decode_paged_gqa_d128", kind="decode_paged", dtype="bf16", nseq=24, len_min=128, len_max=4096,
             len_seed=24, page=256, Hq=32, Hkv=8, D=128),
        # The headline shape: long rows, head dim 64, no mask.
        dict(name="dense_d64_8k", kind="dense", dtype="bf16", B=1, Lq=8192, Lk=8192, Hq=16, Hkv=16, D=64,
             causal=False, left=-1, right=-1, softcap=0.0, alibi=False),
        # A batch of short, odd rows (patch sequences, sentence encoders).
        dict(name="dense_short_d64", kind="dense", dtype="fp16", B=32, Lq=197, Lk=197, Hq=12, Hkv=12, D=64,
             causal=False, left=-1, right=-1, softcap=0.0, alibi=False),
        # Every score option at once over a long row: sliding window,
        # soft-cap and ALiBi, head dim 128.
        dict(name="dense_window_bias_d128", kind="dense", dtype="bf16", B=1, Lq=32768, Lk=32768, Hq=16, Hkv=16, D=128,
             causal=True, left=2048, right=0, softcap=30.0, alibi=True),
        # Ragged prompts packed without padding, grouped-query heads.
        dict(name="varlen_gqa_d128", kind="varlen", dtype="bf16", nseq=8, len_min=256, len_max=4096, len_seed=3, Hq=32,
             Hkv=8, D=128, causal=True),
        # Training on long rows: forward and backward, causal, head dim 128.
        # The largest case.
        dict(name="train_causal_d128_8k", kind="train", dtype="fp16", B=1, L=8192, Hq=16, Hkv=16, D=128, causal=True),
        # Training on a ragged packed batch, head dim 64.
        dict(name="train_varlen_d64", kind="train_varlen", dtype="bf16", nseq=12, len_min=200, len_max=2048,
             len_seed=12, H=12, D=64, causal=True),
        # Full-precision training.
        dict(name="train_fp32_d64", kind="train", dtype="fp32", B=2, L=1024, Hq=8, Hkv=8, D=64, causal=True),
        # Full-precision inference on a small batch.
        dict(name="dense_fp32_d64", kind="dense", dtype="fp32", B=1, Lq=512, Lk=512, Hq=2, Hkv=2, D=64, causal=False,
             left=-1, right=-1, softcap=0.0, alibi=False),
        # Partial results of four key shards of one long row.
        dict(name="merge_4_d128", kind="merge", dtype="bf16", parts=4, B=1, L=4096, H=16, D=128),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    """Rough seconds of a pass, to bound what is drawn."""
    w = work(case)
    rate = 4e13 if case["dtype"] == "fp32" else 6e14
    return w["flops"] / rate + w["bytes"] / 4e12


def draw(rng):
    bound = max(_cost(c) for c in listed())
    while True:
        case = _draw(rng)
        if _cost(case) <= bound:
            return case


def _draw(rng):
    kind = rng.choice(["decode", "decode", "decode_paged", "dense", "dense", "varlen", "train", "train_varlen",
                       "train_fp32", "dense_fp32", "merge"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    heads = rng.choice([(32, 8), (16, 16), (64, 8), (32, 4), (12, 12), (16, 8)])
    d = rng.choice([64, 128, 128, 96, 80])
    seed = rng.randrange(1 << 20)
    if kind == "decode":
        return dict(kind=kind, dtype=half, B=_log_int(rng, 1, 48), Lk=_log_int(rng, 200, 16384), Hq=heads[0],
                    Hkv=heads[1], D=rng.choice([64, 128]))
    if kind == "decode_paged":
        top = _log_int(rng, 600, 8192)
        return dict(kind=kind, dtype=half, nseq=_log_int(rng, 1, 48), len_min=max(1, top // 16), len_max=top,
                    len_seed=seed, page=rng.choice([256, 512]), Hq=heads[0], Hkv=heads[1], D=rng.choice([64, 128]))
    if kind == "dense":
        lq = _log_int(rng, 100, 16384)
        lk = lq if rng.random() < 0.7 else _log_int(rng, 100, 16384)
        causal = rng.random() < 0.5 and lk >= lq
        option = rng.choice(["none", "none", "none", "window", "softcap", "alibi", "all"])
        window = option in ("window", "all") and lk >= lq and lk >= 1024
        return dict(kind=kind, dtype=half, B=_log_int(rng, 1, 32), Lq=lq, Lk=lk, Hq=heads[0], Hkv=heads[1], D=d,
                    causal=causal, left=rng.randrange(256, 3000) if window else -1,
                    right=(0 if causal else rng.randrange(0, 1024)) if window else -1,
                    softcap=rng.choice([20.0, 30.0, 50.0]) if option in ("softcap", "all") else 0.0,
                    alibi=option in ("alibi", "all"))
    if kind == "varlen":
        top = _log_int(rng, 300, 8192)
        return dict(kind=kind, dtype=half, nseq=_log_int(rng, 2, 48), len_min=max(2, top // 16), len_max=top,
                    len_seed=seed, Hq=heads[0], Hkv=heads[1], D=d, causal=rng.random() < 0.7)
    if kind == "train":
        return dict(kind=kind, dtype=half, B=_log_int(rng, 1, 16), L=_log_int(rng, 200, 8192), Hq=heads[0],
                    Hkv=heads[1], D=d, causal=rng.random() < 0.7)
    if kind == "train_varlen":
        top = _log_int(rng, 300, 4096)
        return dict(kind=kind, dtype=half, nseq=_log_int(rng, 2, 32), len_min=max(2, top // 10), len_max=top,
                    len_seed=seed, H=rng.choice([12, 16]), D=d, causal=rng.random() < 0.7)
    if kind == "train_fp32":
        return dict(kind="train", dtype="fp32", B=_log_int(rng, 1, 8), L=_log_int(rng, 100, 2500),
                    Hq=(h := rng.choice([(8, 8), (8, 2), (16, 16)]))[0], Hkv=h[1], D=rng.choice([32, 64, 96, 128]),
                    causal=rng.random() < 0.7)
    if kind == "dense_fp32":
        lq = _log_int(rng, 100, 4096)
        return dict(kind="dense", dtype="fp32", B=_log_int(rng, 1, 8), Lq=lq, Lk=lq,
                    Hq=(h := rng.choice([(2, 2), (8, 8), (8, 2), (16, 16)]))[0], Hkv=h[1],
                    D=rng.choice([32, 64, 96, 128]), causal=rng.random() < 0.5, left=-1, right=-1,
                    softcap=rng.choice([0.0, 0.0, 20.0]), alibi=rng.random() < 0.25)
    return dict(kind="merge", dtype=rng.choice(["bf16", "fp16", "fp32"]), parts=rng.randrange(2, 9),
                B=_log_int(rng, 1, 4), L=_log_int(rng, 1, 8192), H=rng.choice([8, 16, 32]), D=rng.choice([64, 80, 128]))


# --------------------------------------------------------------------------
# inputs


def _lens(case):
    """Ragged lengths, uniform between the bounds, the same for every input seed."""
    g = torch.Generator().manual_seed(case["len_seed"])
    return torch.randint(case["len_min"], case["len_max"] + 1, (case["nseq"],), generator=g).tolist()


def _cu(lens):
    return torch.tensor([0] + lens, dtype=torch.int64).cumsum(0).to(device=_DEV, dtype=torch.int32)


def _slopes(h):
    return torch.tensor([2 ** (-8 * (i + 1) / h) for i in range(h)], dtype=torch.float32, device=_DEV)


def _randn(g, *shape, dtype):
    return torch.randn(*shape, generator=g, device=_DEV).to(dtype)


def prepare(case, seed):
    """Inputs ~ N(0, 1) from the seed alone, on the GPU."""
    g = torch.Generator(device=_DEV).manual_seed(seed)
    dt = _DTYPES[case["dtype"]]
    kind = case["kind"]
    s = dict(case=case)
    if kind == "decode":
        B, Lk, Hq, Hkv, D = (case[x] for x in ("B", "Lk", "Hq", "Hkv", "D"))
        s["q"] = _randn(g, B, 1, Hq, D, dtype=dt)
        s["k"], s["v"] = (_randn(g, B, Lk, Hkv, D, dtype=dt) for _ in range(2))
    elif kind == "decode_paged":
        lens, page = _lens(case), case["page"]
        Hq, Hkv, D = case["Hq"], case["Hkv"], case["D"]
        need = [-(-n // page) for n in lens]
        pages = sum(need) + 4  # (a pool holds pages that no sequence uses)
        s["q"] = _randn(g, len(lens), Hq, D, dtype=dt)
        s["k"], s["v"] = (_randn(g, pages, page, Hkv, D, dtype=dt) for _ in range(2))
        ids = torch.randperm(pages, generator=torch.Generator().manual_seed(seed)).tolist()
        table = torch.zeros(len(lens), max(need), dtype=torch.int32)
        for b, n in enumerate(need):
            table[b, :n] = torch.tensor([ids.pop() for _ in range(n)], dtype=torch.int32)
        s["table"], s["lens"], s["max_k"] = table.to(_DEV), lens, max(lens)
        s["cu_q"], s["cu_k"] = _cu([1] * len(lens)), _cu(lens)
    elif kind == "dense":
        B, Lq, Lk, Hq, Hkv, D = (case[x] for x in ("B", "Lq", "Lk", "Hq", "Hkv", "D"))
        s["q"] = _randn(g, B, Lq, Hq, D, dtype=dt)
        s["k"], s["v"] = (_randn(g, B, Lk, Hkv, D, dtype=dt) for _ in range(2))
        s["slopes"] = _slopes(Hq) if case["alibi"] else None
    elif kind == "varlen":
        lens = _lens(case)
        s["q"] = _randn(g, sum(lens), case["Hq"], case["D"], dtype=dt)
        s["k"], s["v"] = (_randn(g, sum(lens), case["Hkv"], case["D"], dtype=dt) for _ in range(2))
        s["cu"], s["lens"], s["max"] = _cu(lens), lens, max(lens)
    elif kind == "train":
        B, L, Hq, Hkv, D = (case[x] for x in ("B", "L", "Hq", "Hkv", "D"))
        s["q"] = _randn(g, B, L, Hq, D, dtype=dt).requires_grad_()
        s["k"], s["v"] = (_randn(g, B, L, Hkv, D, dtype=dt).requires_grad_() for _ in range(2))
        s["dout"] = _randn(g, B, L, Hq, D, dtype=dt)
    elif kind == "train_varlen":
        lens = _lens(case)
        s["qkv"] = _randn(g, sum(lens), 3, case["H"], case["D"], dtype=dt).requires_grad_()
        s["dout"] = _randn(g, sum(lens), case["H"], case["D"], dtype=dt)
        s["cu"], s["lens"], s["max"] = _cu(lens), lens, max(lens)
    else:  # merge
        B, L, H, D = (case[x] for x in ("B", "L", "H", "D"))
        s["outs"] = [_randn(g, B, L, H, D, dtype=dt) for _ in range(case["parts"])]
        # log-sum-exps of a few thousand keys each; a causal shard leaves the
        # first rows of the last part without a key
        s["lses"] = [8.0 + torch.randn(B, H, L, generator=g, device=_DEV) for _ in range(case["parts"])]
        s["lses"][-1][:, :, :L // 8] = float("-inf")
        s["outs"][-1][:, :L // 8] = 0
    return s


# --------------------------------------------------------------------------
# one pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        with torch.no_grad():
            return mfa.flash_attn_func(s["q"], s["k"], s["v"], causal=True)
    if kind == "decode_paged":
        with torch.no_grad():
            return mfa.flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu_q"], s["cu_k"], 1, s["max_k"], causal=True,
                                              block_table=s["table"])
    if kind == "dense":
        with torch.no_grad():
            return mfa.flash_attn_func(s["q"], s["k"], s["v"], causal=case["causal"],
                                       window_size=(case["left"], case["right"]), softcap=case["softcap"],
                                       alibi_slopes=s["slopes"])
    if kind == "varlen":
        with torch.no_grad():
            return mfa.flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["max"], s["max"],
                                              causal=case["causal"])
    if kind == "train":
        out = mfa.flash_attn_func(s["q"], s["k"], s["v"], causal=case["causal"])
        return (out.detach(), *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"]))
    if kind == "train_varlen":
        out = mfa.flash_attn_varlen_qkvpacked_func(s["qkv"], s["cu"], s["max"], causal=case["causal"])
        return (out.detach(), *torch.autograd.grad(out, (s["qkv"],), s["dout"]))
    with torch.no_grad():
        return mfa.merge_attention_partials(s["outs"], s["lses"])


# --------------------------------------------------------------------------
# what a pass cannot do without


def _pairs(lq, lk, causal=False, left=-1, right=-1):
    """Valid (query, key) pairs of one head (bottom-right aligned masks)."""
    i = torch.arange(lq, dtype=torch.int64) + lk - lq
    lo = (i - left).clamp(min=0) if left >= 0 else torch.zeros_like(i)
    hi = torch.full_like(i, lk - 1)
    if causal:
        hi = torch.minimum(hi, i)
    if right >= 0:
        hi = torch.minimum(hi, i + right)
    return int((hi - lo + 1).clamp(min=0).sum())


def work(case):
    """Each input read once, each output written once; 4 D operations per
    valid (query, key) pair forward, 10 D more backward."""
    kind = case["kind"]
    es = 4 if case["dtype"] == "fp32" else 2
    D = case["D"]
    if kind == "merge":
        rows = case["B"] * case["L"] * case["H"]
        return {"bytes": (case["parts"] + 1) * rows * (D * es + 4), "flops": case["parts"] * rows * (2 * D + 4)}
    if kind == "train_varlen":
        lens, Hq, Hkv = _lens(case), case["H"], case["H"]
    else:
        Hq, Hkv = case["Hq"], case["Hkv"]
        lens = _lens(case) if kind in ("varlen", "decode_paged") else None
    if kind == "decode":
        pairs, tq, tk = case["B"] * case["Lk"], case["B"], case["B"] * case["Lk"]
    elif kind == "decode_paged":
        pairs, tq, tk = sum(lens), len(lens), sum(lens)
    elif kind == "dense":
        pairs = case["B"] * _pairs(case["Lq"], case["Lk"], case["causal"], case["left"], case["right"])
        tq, tk = case["B"] * case["Lq"], case["B"] * case["Lk"]
    elif kind == "train":
        pairs = case["B"] * _pairs(case["L"], case["L"], case["causal"])
        tq = tk = case["B"] * case["L"]
    else:
        pairs = sum(_pairs(n, n, case["causal"]) for n in lens)
        tq = tk = sum(lens)
    fwd = (2 * tq * Hq + 2 * tk * Hkv) * D * es
    if kind in ("train", "train_varlen"):
        # backward: q, k, v, out and dout in, the three gradients out
        return {"bytes": fwd + (4 * tq * Hq + 4 * tk * Hkv) * D * es, "flops": 14 * D * pairs * Hq}
    return {"bytes": fwd, "flops": 4 * D * pairs * Hq}


# --------------------------------------------------------------------------
# how far correct results may differ


def tolerance(case):
    """Set from measurement: about four times the distance of the outputs to
    the 64-bit result (the rounding of the outputs and, for 16-bit types, of
    the probabilities that the matrix products take)."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    if case["kind"] in ("train", "train_varlen"):
        return {"rel": 1.6e-2} if case["dtype"] == "bf16" else {"rel": 3e-3}
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 2e-3}


# --------------------------------------------------------------------------
# the result in 64 bits


def _attend64(q, k, v, causal=False, left=-1, right=-1, softcap=0.0, slope=0.0, dout=None):
    """One head in float64: q [Lq, D], k/v [Lk, D] -> out (and dq, dk, dv)."""
    lq, lk = q.shape[0], k.shape[0]
    scale = 1.0 / math.sqrt(q.shape[1])
    out = torch.empty_like(q)
    grads = None if dout is None else [torch.zeros_like(t) for t in (q, k, v)]
    step = max(1, min(lq, (1 << 25) // lk))
    for r0 in range(0, lq, step):
        r1 = min(lq, r0 + step)
        centre = torch.arange(r0, r1, device=q.device) + (lk - lq)
        # the keys that some row of this slice can see
        j0 = max(0, int(centre[0]) - left) if left >= 0 else 0
        j1 = min(lk, int(centre[-1]) + 1) if causal else lk
        if right >= 0:
            j1 = min(j1, int(centre[-1]) + right + 1)
        if j1 <= j0:
            out[r0:r1] = 0
            continue
        j = torch.arange(j0, j1, device=q.device)
        d = j[None, :] - centre[:, None]
        ok = torch.ones_like(d, dtype=torch.bool)
        if causal:
            ok &= d <= 0
        if left >= 0:
            ok &= d >= -left
        if right >= 0:
            ok &= d <= right
        kk, vv = k[j0:j1], v[j0:j1]
        s = (q[r0:r1] @ kk.t()) * scale
        if softcap > 0:
            s = softcap * torch.tanh(s / softcap)
        if slope:
            s = s - slope * d.abs()
        s = s.masked_fill(~ok, float("-inf"))
        p = torch.softmax(s, dim=-1)
        p = torch.where(ok.any(-1, keepdim=True), p, torch.zeros_like(p))
        out[r0:r1] = p @ vv
        if dout is not None:  # (training cases use neither soft-cap nor ALiBi)
            go = dout[r0:r1]
            ds = p * (go @ vv.t() - (go * out[r0:r1]).sum(-1, keepdim=True)) * scale
            grads[0][r0:r1] = ds @ kk
            grads[1][j0:j1] += ds.t() @ q[r0:r1]
            grads[2][j0:j1] += p.t() @ go
    return (out,) if dout is None else (out, *grads)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "merge":
        lses = torch.stack([x.double() for x in s["lses"]])
        lse = torch.logsumexp(lses, dim=0)
        w = torch.exp(lses - lse)
        out = sum(o.double() * w[i].transpose(-1, -2).unsqueeze(-1) for i, o in enumerate(s["outs"]))
        return out, lse
    if kind in ("varlen", "decode_paged", "train_varlen"):
        lens = s["lens"]
        ends = torch.tensor(lens).cumsum(0).tolist()
    if kind == "train_varlen":
        qkv, dout = s["qkv"].detach().double(), s["dout"].double()
        out, grad = torch.empty_like(dout), torch.empty_like(qkv)
        for n, e in zip(lens, ends):
            for h in range(case["H"]):
                q, k, v = (qkv[e - n:e, i, h].contiguous() for i in range(3))
                out[e - n:e, h], grad[e - n:e, 0, h], grad[e - n:e, 1, h], grad[e - n:e, 2, h] = _attend64(
                    q, k, v, causal=case["causal"], dout=dout[e - n:e, h].contiguous())
        return out, grad
    r = case["Hq"] // case["Hkv"]
    q = s["q"].detach().double()
    if kind == "decode_paged":
        out = torch.empty_like(q)
        for b, n in enumerate(lens):
            ids = s["table"][b, :-(-n // case["page"])].long()
            k, v = (s[x][ids].flatten(0, 1)[:n].double() for x in ("k", "v"))
            for h in range(case["Hq"]):
                out[b:b + 1, h] = _attend64(q[b:b + 1, h].contiguous(), k[:, h // r].contiguous(),
                                            v[:, h // r].contiguous(), causal=True)[0]
        return out
    k, v = s["k"].detach().double(), s["v"].detach().double()
    if kind == "varlen":
        out = torch.empty_like(q)
        for n, e in zip(lens, ends):
            for h in range(case["Hq"]):
                out[e - n:e, h] = _attend64(q[e - n:e, h].contiguous(), k[e - n:e, h // r].contiguous(),
                                            v[e - n:e, h // r].contiguous(), causal=case["causal"])[0]
        return out
    out = torch.empty_like(q)
    train = kind == "train"
    if train:
        dout = s["dout"].double()
        dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    opts = dict(causal=True) if kind == "decode" else dict(causal=case["causal"])
    if kind == "dense":
        opts.update(left=case["left"], right=case["right"], softcap=case["softcap"])
    for b in range(case["B"]):
        for h in range(case["Hq"]):
            args = (q[b, :, h].contiguous(), k[b, :, h // r].contiguous(), v[b, :, h // r].contiguous())
            if train:
                o, gq, gk, gv = _attend64(*args, dout=dout[b, :, h].contiguous(), **opts)
                out[b, :, h], dq[b, :, h] = o, gq
                dk[b, :, h // r] += gk
                dv[b, :, h // r] += gv
            else:
                slope = float(s["slopes"][h]) if s.get("slopes") is not None else 0.0
                out[b, :, h] = _attend64(*args, slope=slope, **opts)[0]
    return (out, dq, dk, dv) if train else out
