"""What a user of this framework has it do, as cases to be timed and compared.

A case is a dict of plain values; `prepare` makes its inputs on the GPU, `run`
takes them once through the public entry points (flash_attn_func,
flash_attn_varlen_func, flash_attn_with_kvcache), `work` states what the pass
cannot do without, `exact` is the same result from plain torch in 64 bits.

Six kinds of call stand for the framework's range:
  dense    flash_attn_func, inference: the prompt of a batch of equal sequences
  train    flash_attn_func and its backward: one attention layer of a training step
  packed   flash_attn_varlen_func with RoPE tables: prompts of many lengths, packed
  decode   flash_attn_with_kvcache, one new token per sequence over a paged pool
  verify   the same with a window of draft tokens per sequence (speculative decoding)
  chunk    the same with a packed chunk per sequence (chunked prefill over the pool)
Ragged lengths come from the case's own "lens" number, everything else from the
seed: values and new tokens N(0, 1), the block table a random permutation of
the pool's pages.
"""

import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "flywheel-tpu_amd"))

from flywheel_tpu import (  # noqa: E402
    flash_attn_func,
    flash_attn_varlen_func,
    flash_attn_with_kvcache,
)

DEVICE = "cuda"
K_DESCALE, V_DESCALE = 0.8, 1.25  # per-tensor descales of the e4m3 pools


def listed():
    return [
        # a short prompt on a small attention layer (8/2 heads, 512 tokens):
        # what an interactive call costs, launches and host path included
        dict(name="prefill_short", kind="dense", b=1, h=8, hk=2, sq=512, sk=512, d=128, dv=128,
             causal=True),
        # the benchmark's headline: a 4K prompt, 32/4 heads
        dict(name="prefill_gqa", kind="dense", b=1, h=32, hk=4, sq=4096, sk=4096, d=128, dv=128,
             causal=True),
        # head dim 64, a batch of prompts of a length that fills no tile
        dict(name="prefill_d64", kind="dense", b=4, h=32, hk=8, sq=1999, sk=1999, d=64, dv=64,
             causal=True),
        # head dim 256, the reference's published dense shape
        dict(name="prefill_d256", kind="dense", b=1, h=32, hk=4, sq=4096, sk=4096, d=256, dv=256,
             causal=True),
        # query/key heads wider than the value heads (192/128), one head per KV
        # head, a chunk of queries behind a prefix
        dict(name="prefill_192_128", kind="dense", b=1, h=16, hk=16, sq=2048, sk=3000, d=192,
             dv=128, causal=True),
        # a serving engine's prefill batch: prompts from a few tokens to 2K, packed, with RoPE
        dict(name="packed_rope", kind="packed", n=16, lo=5, hi=2048, lens=1, h=32, hk=8, d=128,
             rope=True, causal=True),
        # one attention layer of a training step at the headline shape
        dict(name="train_gqa", kind="train", b=1, h=32, hk=4, sq=4096, sk=4096, d=128, dv=128,
             causal=True),
        # the same at head dim 64 with one head per KV head and a batch
        dict(name="train_d64", kind="train", b=4, h=16, hk=16, sq=2000, sk=2000, d=64, dv=64,
             causal=True),
        # one user generating: a single sequence, one token a call
        dict(name="decode_one", kind="decode", n=1, lo=4001, hi=4001, lens=0, h=32, hk=8, d=128,
             page=16, fp8=False),
        # a full serving batch: 64 sequences of 1K to 32K tokens
        dict(name="decode_batch", kind="decode", n=64, lo=1024, hi=32768, lens=0, h=32, hk=8,
             d=128, page=16, fp8=False),
        # speculative decoding on an fp8 pool: 128 sequences of 4K to 64K, 4 draft tokens each
        dict(name="verify_fp8", kind="verify", n=128, lo=4096, hi=65536, lens=0, h=32, hk=8,
             d=128, page=16, fp8=True, sq=4),
        # chunked prefill: 8 requests, chunks of 256 to 2048 tokens behind up to
        # 16K tokens of context, a sliding window of 4096 and softcap 50
        dict(name="chunk_window", kind="chunk", n=8, lo=256, hi=2048, prior=16384, lens=0, h=32,
             hk=8, d=128, page=16, fp8=False, window=4096, softcap=50.0),
    ]


# ------------------------------------------------------------------ drawing


def _log(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def _heads(rng):
    hk = rng.choice((1, 2, 4, 8, 8, 16))
    return hk * rng.choice((1, 1, 2, 4, 8)) if hk < 16 else hk, hk


def _draw(rng):
    kind = rng.choice(("dense", "dense", "train", "packed", "decode", "verify", "chunk"))
    h, hk = _heads(rng)
    if kind in ("dense", "train"):
        d, dv = rng.choice(((64, 64), (128, 128), (128, 128), (256, 256), (192, 128))
                           if kind == "dense" else ((64, 64), (128, 128)))
        sq = _log(rng, 16 if kind == "dense" else 128, 6000)
        sk = sq if rng.random() < 0.7 else sq + _log(rng, 1, 4000)
        return dict(kind=kind, b=_log(rng, 1, 8), h=h, hk=hk, sq=sq, sk=sk, d=d, dv=dv,
                    causal=rng.random() < 0.75)
    lens = rng.randrange(1 << 30)
    if kind == "packed":
        return dict(kind=kind, n=_log(rng, 1, 32), lo=rng.randint(1, 16), hi=_log(rng, 64, 4096),
                    lens=lens, h=h, hk=hk, d=rng.choice((64, 128, 128)),
                    rope=rng.random() < 0.6, causal=rng.random() < 0.8)
    page, fp8 = rng.choice((16, 16, 64, 128)), rng.random() < 0.4
    if kind == "chunk":
        window = rng.choice((0, 1024, 4096))
        return dict(kind=kind, n=_log(rng, 1, 12), lo=rng.randint(1, 256), hi=_log(rng, 256, 2048),
                    prior=_log(rng, 64, 16384), lens=lens, h=h, hk=hk, d=128, page=page, fp8=fp8,
                    window=window, softcap=rng.choice((0.0, 30.0, 50.0)))
    hi = _log(rng, 100, 65536)
    case = dict(kind=kind, n=_log(rng, 1, 128), lo=max(1, hi // rng.choice((1, 4, 32))), hi=hi,
                lens=lens, h=h, hk=hk, d=rng.choice((64, 128, 128, 256)), page=page, fp8=fp8)
    if kind == "verify":
        case["sq"] = rng.randint(2, 8)
    return case


def draw(rng):
    """One more case: the same kinds over their whole ranges, none dearer than
    the largest listed ones (the pool of verify_fp8, the products of train_gqa)."""
    most = work(listed()[6])["flops"]
    while True:
        case = _draw(rng)
        w = work(case)
        bound = most if case["kind"] == "train" else most / 3.5
        if w["flops"] <= bound and w["bytes"] <= 5e9:
            return case


# ------------------------------------------------------------------ the cases' sizes


def _lens(case):
    """The ragged lengths of a case: (new tokens, tokens before them) per sequence."""
    rng = np.random.default_rng(case["lens"])
    a = rng.integers(case["lo"], case["hi"] + 1, case["n"])
    if case["kind"] == "packed":
        return a, np.zeros_like(a)
    if case["kind"] == "chunk":
        return a, rng.integers(0, case["prior"] + 1, case["n"])
    return np.full(case["n"], case.get("sq", 1)), a


def _pairs(sq, sk, causal, window=0):
    """Visible (query, key) pairs of one head, the mask aligned to the last key."""
    if not causal:
        return sq * sk
    last = np.arange(sq, dtype=np.int64) + sk - sq
    first = np.maximum(last - window + 1, 0) if window else np.zeros_like(last)
    return int(np.maximum(last - first + 1, 0).sum())


def work(case):
    h, hk, d = case["h"], case["hk"], case["d"]
    if case["kind"] in ("dense", "train"):
        b, sq, sk, dv = case["b"], case["sq"], case["sk"], case["dv"]
        nq, nk, no = b * h * sq * d, b * hk * sk * (d + dv), b * h * sq * dv
        flops = 2.0 * b * h * (d + dv) * _pairs(sq, sk, case["causal"])
        if case["kind"] == "dense":
            return {"bytes": 2.0 * (nq + nk + no), "flops": flops}
        # q, k, v, dout read; out and the three gradients written; backward = 2.5 forwards
        return {"bytes": 4.0 * (nq + nk + no), "flops": 3.5 * flops}
    new, prior = _lens(case)
    tokens, q_bytes = int(new.sum()), 2.0 * int(new.sum()) * h * d
    if case["kind"] == "packed":
        pairs = sum(_pairs(int(s), int(s), case["causal"]) for s in new)
        table = 4.0 * int(new.max()) * d if case["rope"] else 0.0
        return {"bytes": 2 * q_bytes + 4.0 * tokens * hk * d + table, "flops": 4.0 * h * d * pairs}
    item = 1 if case["fp8"] else 2
    window = case.get("window", 0)
    row = 2.0 * hk * d * item
    seen = prior if not window else np.minimum(prior, window - 1)
    pairs = sum(_pairs(int(a), int(a + p), True, window) for a, p in zip(new, prior))
    # the pool's visible rows and the new rows read, the new rows written
    return {"bytes": row * (int(seen.sum()) + 2 * tokens) + 2 * q_bytes,
            "flops": 4.0 * h * d * pairs}


# ------------------------------------------------------------------ inputs


def _normal(gen, shape):
    return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.bfloat16)


def _rope_tables(rows, d):
    freq = 10000.0 ** (-torch.arange(0, d, 2, device=DEVICE, dtype=torch.float64) / d)
    angle = torch.arange(rows, device=DEVICE, dtype=torch.float64)[:, None] * freq
    return angle.cos().float(), angle.sin().float()


def _pool(case, gen, totals):
    """The paged pool (fp8: N(0, 1) over the descale) and its block table."""
    page, hk, d = case["page"], case["hk"], case["d"]
    need = [-(-int(t) // page) for t in totals]
    pages = sum(need) + 8
    heads = 2 * (hk + hk % 2) if case["fp8"] else 2 * hk
    if case["fp8"]:
        pool = torch.empty((pages, page, heads, d), dtype=torch.float8_e4m3fn, device=DEVICE)
        step = max(1, (1 << 28) // (page * heads * d))
        for i in range(0, pages, step):
            x = torch.randn((min(step, pages - i), page, heads, d), generator=gen, device=DEVICE)
            x[:, :, 0:2 * hk:2] /= K_DESCALE
            x[:, :, 1:2 * hk:2] /= V_DESCALE
            x[:, :, 2 * hk:] = 0
            pool[i:i + step] = x.to(torch.float8_e4m3fn)
    else:
        pool = _normal(gen, (pages, page, heads, d))
    perm = torch.randperm(pages, generator=gen, device=DEVICE).to(torch.int32)
    table = torch.zeros((len(need), max(need)), dtype=torch.int32, device=DEVICE)
    at = 0
    for r, c in enumerate(need):
        table[r, :c] = perm[at:at + c]
        at += c
    return pool, table


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed))
    h, hk, d = case["h"], case["hk"], case["d"]
    s = {"case": dict(case)}
    if case["kind"] in ("dense", "train"):
        b, sq, sk, dv = case["b"], case["sq"], case["sk"], case["dv"]
        s["q"] = _normal(gen, (b, h, sq, d))
        s["k"] = _normal(gen, (b, hk, sk, d))
        s["v"] = _normal(gen, (b, hk, sk, dv))
        if case["kind"] == "train":
            for name in ("q", "k", "v"):
                s[name].requires_grad_(True)
            s["dout"] = _normal(gen, (b, h, sq, dv))
        return s
    new, prior = _lens(case)
    tokens = int(new.sum())
    if case["kind"] == "packed":
        s["q"] = _normal(gen, (h, tokens, d))
        s["k"] = _normal(gen, (hk, tokens, d))
        s["v"] = _normal(gen, (hk, tokens, d))
        s["cu"] = torch.tensor(np.concatenate([[0], np.cumsum(new)]), dtype=torch.int32,
                               device=DEVICE)
        s["longest"] = int(new.max())
        s["cos"], s["sin"] = _rope_tables(s["longest"], d) if case["rope"] else (None, None)
        return s
    s["pool"], s["table"] = _pool(case, gen, new + prior)
    s["lens"] = torch.tensor(prior, dtype=torch.int32, device=DEVICE)
    lead = (tokens,) if case["kind"] == "chunk" else (case["n"], case.get("sq", 1))
    s["q"] = _normal(gen, (*lead, h, d))
    k, v = _normal(gen, (*lead, hk, d)), _normal(gen, (*lead, hk, d))
    s["extra"] = {}
    if case["fp8"]:
        k = (k.float() / K_DESCALE).to(torch.float8_e4m3fn)
        v = (v.float() / V_DESCALE).to(torch.float8_e4m3fn)
        s["extra"] = dict(k_descale=K_DESCALE, v_descale=V_DESCALE, nheads_k=hk)
    s["k"], s["v"] = k, v
    if case["kind"] == "chunk":
        s["cu"] = torch.tensor(np.concatenate([[0], np.cumsum(new)]), dtype=torch.int32,
                               device=DEVICE)
        window = case["window"]
        s["extra"].update(cu_seqlens_q=s["cu"], max_seqlen_q=int(new.max()), causal=True,
                          window_size=(window - 1, 0) if window else (-1, -1),
                          softcap=case["softcap"])
    elif case["kind"] == "verify":
        s["extra"]["causal"] = True
    return s


# ------------------------------------------------------------------ one pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "dense":
        return flash_attn_func(s["q"], s["k"], s["v"], causal=case["causal"])
    if kind == "train":
        out = flash_attn_func(s["q"], s["k"], s["v"], causal=case["causal"])
        grads = torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"])
        return (out.detach(), *grads)
    if kind == "packed":
        return flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["longest"],
                                      s["longest"], causal=case["causal"], rotary_cos=s["cos"],
                                      rotary_sin=s["sin"])
    return flash_attn_with_kvcache(s["q"], s["pool"], None, s["k"], s["v"],
                                   cache_seqlens=s["lens"], block_table=s["table"], **s["extra"])


# ------------------------------------------------------------------ results in 64 bits


def _attend(q, k, v, causal, window=0, softcap=0.0, dout=None):
    """Attention of (h, sq, d) queries over (hk, sk, .) keys and values in 64
    bits, the mask aligned to the last key: (out, dq, dk, dv), the gradients
    only with dout.  One KV head and its query heads at a time, and a block of
    rows at a time."""
    h, sq, d = q.shape
    hk, sk, dv = v.shape
    n = h // hk
    out = torch.empty((h, sq, dv), dtype=torch.float64, device=q.device)
    dq = torch.zeros_like(q) if dout is not None else None
    dk = torch.zeros_like(k) if dout is not None else None
    dvv = torch.zeros_like(v) if dout is not None else None
    scale, key = 1.0 / math.sqrt(d), torch.arange(sk, device=q.device)
    step = max(1, min(sq, (1 << 25) // (sk * n)))
    for g in range(hk):
        heads = slice(g * n, g * n + n)
        for r in range(0, sq, step):
            rows = slice(r, min(sq, r + step))
            qr = q[heads, rows].reshape(-1, d)
            x = qr @ k[g].T * scale
            if softcap:
                x = torch.tanh(x / softcap) * softcap
            if causal:
                last = torch.arange(rows.start, rows.stop, device=q.device)[:, None] + sk - sq
                hidden = key > last
                if window:
                    hidden |= key <= last - window
                x.masked_fill_(hidden.repeat(n, 1), -math.inf)
            p = torch.softmax(x, dim=-1)
            o = p @ v[g]
            out[heads, rows] = o.reshape(n, -1, dv)
            if dout is not None:
                go = dout[heads, rows].reshape(-1, dv)
                ds = p * (go @ v[g].T - (go * o).sum(-1, keepdim=True))
                dq[heads, rows] = (ds @ k[g] * scale).reshape(n, -1, d)
                dk[g] += ds.T @ qr * scale
                dvv[g] += p.T @ go
    return out, dq, dk, dvv


def _rotated(x, s):
    """(heads, t, d) rows at positions 0.., the two halves of a head paired."""
    cos, sin = s["cos"][:x.shape[1]].double(), s["sin"][:x.shape[1]].double()
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, a * sin + b * cos], dim=-1)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    wide = {n: s[n].detach().double() for n in ("q", "k", "v", "dout") if n in s}
    q, k, v = wide["q"], wide["k"], wide["v"]
    if kind in ("dense", "train"):
        each = [_attend(q[i], k[i], v[i], case["causal"],
                        dout=wide["dout"][i] if kind == "train" else None)
                for i in range(case["b"])]
        got = [torch.stack(x) for x in zip(*each) if x[0] is not None]
        return tuple(got) if kind == "train" else got[0]
    new, prior = _lens(case)
    at = np.concatenate([[0], np.cumsum(new)])
    if kind == "packed":
        out = torch.empty_like(q)
        for i in range(case["n"]):
            rows = slice(int(at[i]), int(at[i + 1]))
            qi, ki = q[:, rows], k[:, rows]
            if case["rope"]:
                qi, ki = _rotated(qi, s), _rotated(ki, s)
            out[:, rows] = _attend(qi, ki, v[:, rows], case["causal"])[0]
        return out
    hk, d, page = case["hk"], case["d"], case["page"]
    kd, vd = (K_DESCALE, V_DESCALE) if case["fp8"] else (1.0, 1.0)
    flat = q.reshape(-1, case["h"], d)
    k, v = k.reshape(-1, hk, d), v.reshape(-1, hk, d)
    out = torch.empty_like(flat)
    for i in range(case["n"]):
        rows, n = slice(int(at[i]), int(at[i + 1])), int(prior[i])
        pages = s["table"][i, :-(-n // page)].long() if n else s["table"][i, :0].long()
        old = s["pool"][pages].reshape(-1, *s["pool"].shape[2:])[:n, :2 * hk].double()
        ki = torch.cat([old[:, 0::2], k[rows]]).transpose(0, 1) * kd
        vi = torch.cat([old[:, 1::2], v[rows]]).transpose(0, 1) * vd
        out[rows] = _attend(flat[rows].transpose(0, 1), ki, vi, True, case.get("window", 0),
                            case.get("softcap", 0.0))[0].transpose(0, 1)
    return out.reshape(q.shape), None


def tolerance(case):
    """bf16 results of bf16 products.  Measured against `exact` over the listed
    and 16 drawn cases: a forward is 2.0e-3 to 3.7e-3 off (the bf16 rounding of
    the result and of the probabilities; RoPE adds that of rotated q and k), a
    gradient 2.5e-3 to 3.4e-3, and a single value at most 0.14 of the result's
    root mean square."""
    return {"rel": 0.013 if case["kind"] in ("train", "packed") else 0.011, "max": 0.5}
