"""GPU parity of the MFMA prefill kernel (dense, packed varlen, paged varlen,
and chunked prefill through flash_attn_with_kvcache) against the oracle."""

import math

import numpy as np
import pytest
import torch

from flywheel_tpu import flash_attn_func, flash_attn_varlen_func, flash_attn_with_kvcache
from flywheel_tpu import _native as N
from oracle import attention as A
from oracle import paged as P
from tests.gpu_util import (DEV, FP8, PagedCase, announce, assert_close, assert_lse, codes_of,
                            dev_from_codes, randn, to_dev_bf16)

pytestmark = pytest.mark.gpu
FORMS = ["LARGE", "MID", "SMALL", "FREE", "GENERAL"]


def head_major(x):  # (B, S, H, D) -> (B, H, S, D)
    return np.ascontiguousarray(x.transpose(0, 2, 1, 3))


def dense_form(q, k, v, causal, window=(-1, -1)):
    """The kernel form flash_attn_func takes for contiguous head-major q, k, v."""
    p = N.PrefillParams()
    p.kv_mode, p.kv_dtype, p.causal = N.FW_KV_DENSE, N.FW_BF16, int(causal)
    p.k, p.v = N.ptr(k), N.ptr(v)
    p.batch, p.nheads, p.seqlen_q, p.head_dim = q.shape
    p.nheads_k, p.seqlen_k, p.head_dim_v = k.shape[1], k.shape[2], v.shape[3]
    p.k_stride_t, p.v_stride_t = p.head_dim, p.head_dim_v
    p.window_left, p.window_right = window[0], 0 if causal else window[1]
    return FORMS[N.lib().fw_prefill_form(p)]


@pytest.mark.parametrize(
    "b,h,hk,sq,sk,causal,window,softcap,sinks",
    [
        (1, 8, 2, 512, 512, True, (-1, -1), 0.0, False),
        (2, 4, 4, 200, 333, True, (-1, -1), 0.0, False),
        (1, 4, 1, 333, 200, True, (-1, -1), 0.0, False),  # leading rows see nothing
        (1, 8, 2, 300, 300, False, (-1, -1), 0.0, False),
        (2, 4, 2, 257, 257, False, (64, 17), 0.0, False),
        (1, 4, 2, 384, 384, True, (100, -1), 30.0, False),
        # softcap tanh paths (N(0,1) scores, |s| < 6): exact (|s/5| > 0.3 somewhere in every
        # tile), degree-5 polynomial (0.12 < max |s/20| <= 0.3), degree-3 (max |s/50| <= 0.12)
        (1, 4, 1, 512, 512, True, (-1, -1), 5.0, False),
        (1, 4, 1, 512, 512, True, (-1, -1), 20.0, False),
        (1, 4, 1, 512, 512, True, (-1, -1), 50.0, False),
        (1, 4, 2, 130, 130, True, (-1, -1), 0.0, True),
        # head packing: 3 (one head per workgroup), 6 (two), 16 (8 per workgroup, two
        # workgroups per KV head) query heads per KV head
        (1, 6, 2, 300, 300, True, (-1, -1), 0.0, False),
        (2, 12, 2, 200, 260, True, (40, -1), 0.0, True),
        (1, 16, 1, 100, 400, True, (-1, -1), 50.0, False),
        (1, 16, 2, 77, 77, False, (-1, -1), 0.0, False),
    ],
)
def test_flash_attn_func(b, h, hk, sq, sk, causal, window, softcap, sinks):
    announce(f"dense b{b} h{h}/{hk} sq{sq} sk{sk} causal={causal} window={window} softcap={softcap}")
    rng = np.random.default_rng(10)
    q, k, v = randn(rng, (b, sq, h, 128)), randn(rng, (b, sk, hk, 128)), randn(rng, (b, sk, hk, 128))
    s = rng.standard_normal(h).astype(np.float32) if sinks else None
    out, lse = flash_attn_func(
        to_dev_bf16(head_major(q)), to_dev_bf16(head_major(k)), to_dev_bf16(head_major(v)),
        causal=causal, window_size=window, softcap=softcap, return_softmax_lse=True,
        learnable_sink=None if s is None else torch.tensor(s, device=DEV))
    torch.cuda.synchronize()
    ro, rl = A.attention_ref(q, k, v, causal=causal, window_size=window, softcap=softcap, sinks=s,
                             round_scaled_q=True)
    assert_close(out.float().cpu().numpy(), head_major(ro))
    assert_lse(lse.cpu().numpy(), rl)


def test_flash_attn_func_layouts():
    """token_major and heads_outer_fold address the same math in place."""
    announce("dense layouts")
    rng = np.random.default_rng(11)
    b, h, hk, s, d = 2, 4, 2, 160, 128
    q, k, v = randn(rng, (b, s, h, d)), randn(rng, (b, s, hk, d)), randn(rng, (b, s, hk, d))
    ro, _ = A.attention_ref(q, k, v, causal=True, round_scaled_q=True)
    out = flash_attn_func(to_dev_bf16(q.reshape(b, s, h * d)), to_dev_bf16(k.reshape(b, s, hk * d)),
                          to_dev_bf16(v.reshape(b, s, hk * d)), causal=True, head_dim=d,
                          token_major=True)
    assert_close(out.float().cpu().numpy().reshape(b, s, h, d), ro)
    hof = lambda x: np.ascontiguousarray(x.transpose(2, 0, 1, 3))  # (H, B, S, D)
    out = flash_attn_func(to_dev_bf16(hof(q)), to_dev_bf16(hof(k)), to_dev_bf16(hof(v)),
                          causal=True, heads_outer_fold=True)
    assert_close(out.float().cpu().numpy(), hof(ro))


def test_flash_attn_func_c2_full_size():
    """BASELINE config 2 at full size; the oracle checks 4 of the 32 heads."""
    announce("dense C2 1x32/4x4096")
    rng = np.random.default_rng(12)
    q, k, v = randn(rng, (1, 4096, 32, 128)), randn(rng, (1, 4096, 4, 128)), randn(rng, (1, 4096, 4, 128))
    out, lse = flash_attn_func(to_dev_bf16(head_major(q)), to_dev_bf16(head_major(k)),
                               to_dev_bf16(head_major(v)), causal=True, return_softmax_lse=True)
    torch.cuda.synchronize()
    heads = [0, 9, 18, 31]  # query head h reads KV head h // 8
    outs = out.float().cpu().numpy()
    lses = lse.cpu().numpy()
    for hh in heads:
        ro, rl = A.attention_ref(q[:, :, [hh]], k[:, :, [hh // 8]], v[:, :, [hh // 8]], causal=True,
                                 round_scaled_q=True)
        assert_close(outs[:, hh], ro[:, :, 0], what=f"head {hh}")
        assert_lse(lses[:, [hh]], rl)


@pytest.mark.parametrize("b,h,hk,sq,sk,causal,window,softcap,sinks", [
    (1, 32, 4, 4096, 4096, True, (-1, -1), 0.0, False),     # C2
    (1, 32, 4, 4096, 4096, False, (-1, -1), 0.0, False),
    (1, 32, 4, 4096, 4096, True, (1000, 0), 0.0, True),
    (1, 32, 4, 4096, 4096, True, (-1, -1), 30.0, False),
    (1, 32, 4, 4096, 6000, True, (-1, -1), 0.0, False),     # keys past the queries
    (2, 32, 32, 4096, 4096, True, (-1, -1), 0.0, False),    # MHA: XCD-aware head groups
])
@pytest.mark.parametrize("d", [128, 256])
def test_pair_kernel_matches_one_tile_kernel(d, b, h, hk, sq, sk, causal, window, softcap, sinks,
                                             monkeypatch):
    """Dense grids whose q tiles pair up and whose half still covers every CU
    run fw_prefill_pp_pair_kernel / fw_prefill_d256_pair_kernel (a heavy q
    tile, then its mirror of the same head group, per workgroup);
    FW_PREFILL_PAIR=0 runs one q tile per workgroup.  Both compute every tile the same way: bitwise equal out and
    lse, and the C2 full-size test above checks the pair kernel against the
    oracle."""
    announce(f"pair kernel d{d} b{b} h{h}/{hk} sq{sq} sk{sk} causal={causal} window={window}"
             f" softcap={softcap} sinks={sinks}")
    gen = torch.Generator(device=DEV).manual_seed(21)
    q = torch.randn((b, h, sq, d), generator=gen, device=DEV, dtype=torch.bfloat16)
    k = torch.randn((b, hk, sk, d), generator=gen, device=DEV, dtype=torch.bfloat16)
    v = torch.randn((b, hk, sk, d), generator=gen, device=DEV, dtype=torch.bfloat16)
    kw = dict(causal=causal, window_size=window, softcap=softcap, return_softmax_lse=True)
    if sinks:
        kw["learnable_sink"] = torch.randn((h,), generator=gen, device=DEV, dtype=torch.float32)
    out_p, lse_p = flash_attn_func(q, k, v, **kw)
    monkeypatch.setenv("FW_PREFILL_PAIR", "0")
    out_1, lse_1 = flash_attn_func(q, k, v, **kw)
    torch.cuda.synchronize()
    assert torch.isfinite(out_p.float()).all()
    assert torch.equal(out_p, out_1)
    assert torch.equal(lse_p, lse_1)


@pytest.mark.parametrize("causal,window,softcap", [(True, (-1, -1), 0.0), (False, (-1, -1), 0.0),
                                                   (True, (50, -1), 20.0)])
def test_flash_attn_varlen_packed(causal, window, softcap):
    announce(f"varlen packed causal={causal} window={window}")
    rng = np.random.default_rng(13)
    qlens, klens = [5, 130, 1, 300], [9, 130, 40, 512]
    h, hk, d = 8, 2, 128
    cu_q = np.concatenate([[0], np.cumsum(qlens)]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(klens)]).astype(np.int32)
    pad = 7
    q = randn(rng, (h, cu_q[-1] + pad, d))
    k = randn(rng, (hk, cu_k[-1] + 3, d))
    v = randn(rng, (hk, cu_k[-1] + 3, d))
    out, lse = flash_attn_varlen_func(
        to_dev_bf16(q), to_dev_bf16(k), to_dev_bf16(v), torch.tensor(cu_q, device=DEV),
        torch.tensor(cu_k, device=DEV), max(qlens), max(klens), causal=causal, window_size=window,
        softcap=softcap, return_softmax_lse=True)
    torch.cuda.synchronize()
    outs, lses = out.float().cpu().numpy(), lse.cpu().numpy()
    for s in range(4):
        qs = q[:, cu_q[s]:cu_q[s + 1]].transpose(1, 0, 2)[None]
        ks = k[:, cu_k[s]:cu_k[s + 1]].transpose(1, 0, 2)[None]
        vs = v[:, cu_k[s]:cu_k[s + 1]].transpose(1, 0, 2)[None]
        ro, rl = A.attention_ref(qs, ks, vs, causal=causal, window_size=window, softcap=softcap,
                                 round_scaled_q=True)
        got = outs[:, cu_q[s]:cu_q[s + 1]].transpose(1, 0, 2)
        rows_ok = np.isfinite(rl[0]).all(axis=0)  # rows with no visible key are unspecified
        assert_close(got[rows_ok], ro[0][rows_ok], what=f"seq {s}")
        assert_lse(lses[:, cu_q[s]:cu_q[s + 1]][:, rows_ok], rl[0][:, rows_ok])
    assert not outs[:, cu_q[-1]:].any()
    assert np.isneginf(lses[:, cu_q[-1]:]).all()


@pytest.mark.parametrize("nseq", [300, 2100])
def test_flash_attn_varlen_many_sequences(nseq):
    """Many short packed sequences: the tile schedule orders up to 2048 q tiles
    by cost (300) and keeps the sequence order beyond that (2100)."""
    announce(f"varlen packed many sequences n={nseq}")
    rng = np.random.default_rng(15)
    qlens = rng.integers(1, 5, nseq)
    qlens[::97] = 300  # a few multi-tile sequences among the short ones
    klens = qlens + rng.integers(0, 40, nseq)
    h, hk, d = 2, 1, 128
    cu_q = np.concatenate([[0], np.cumsum(qlens)]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(klens)]).astype(np.int32)
    q = randn(rng, (h, cu_q[-1], d))
    k = randn(rng, (hk, cu_k[-1], d))
    v = randn(rng, (hk, cu_k[-1], d))
    out = flash_attn_varlen_func(
        to_dev_bf16(q), to_dev_bf16(k), to_dev_bf16(v), torch.tensor(cu_q, device=DEV),
        torch.tensor(cu_k, device=DEV), int(qlens.max()), int(klens.max()), causal=True)
    torch.cuda.synchronize()
    outs = out.float().cpu().numpy()
    for s in range(nseq):
        qs = q[:, cu_q[s]:cu_q[s + 1]].transpose(1, 0, 2)[None]
        ks = k[:, cu_k[s]:cu_k[s + 1]].transpose(1, 0, 2)[None]
        vs = v[:, cu_k[s]:cu_k[s + 1]].transpose(1, 0, 2)[None]
        ro, _ = A.attention_ref(qs, ks, vs, causal=True, round_scaled_q=True)
        assert_close(outs[:, cu_q[s]:cu_q[s + 1]].transpose(1, 0, 2), ro[0], what=f"seq {s}")


@pytest.mark.parametrize("dtype", ["bf16", "e4m3", "e5m2"])
@pytest.mark.parametrize("h,hk", [(4, 2), (8, 1), (16, 2), (6, 3)])
def test_paged_varlen_read_only(dtype, h, hk):
    """flash_attn_varlen_func(block_table=...) over a merged pool; reference
    edge case random_ragged_case lengths (3, 0, 5) on prefixes (127, 0, 251).
    Heads: 2 or 8 query heads per KV head (one workgroup serves 2 or 8), and
    an odd KV head count (the fp8 pool's zero pad head)."""
    announce(f"paged varlen {dtype} h{h}/{hk}")
    rng = np.random.default_rng(14)
    dt = torch.bfloat16 if dtype == "bf16" else FP8[dtype]
    ks, vs = (1.0, 1.0) if dtype == "bf16" else (0.5, 2.0)
    qlens = [3, 0, 5, 200]
    prefix = [127, 0, 251, 1000]
    totals = np.array(qlens) + np.array(prefix)
    case = PagedCase(rng, batch=4, nheads=h, nheads_k=hk, lengths=totals, new_tokens=[0] * 4,
                     dtype=dt, k_descale=ks, v_descale=vs)
    cu = np.concatenate([[0], np.cumsum(qlens)]).astype(np.int32)
    q = randn(rng, (cu[-1] + 7, h, 128))
    out, lse = flash_attn_varlen_func(
        to_dev_bf16(np.ascontiguousarray(q.transpose(1, 0, 2))), case.pool(), None,
        torch.tensor(cu, device=DEV), None, max(qlens), int(totals.max()), causal=True,
        return_softmax_lse=True, block_table=torch.tensor(case.table, device=DEV),
        seqused_k=torch.tensor(totals, dtype=torch.int32, device=DEV), k_descale=ks,
        v_descale=vs, nheads_k=hk)
    torch.cuda.synchronize()
    kp, vp = case.kv_pages(case.pool_codes)
    ro, rl = A.ragged_reference(q, kp, vp, cu, totals, case.table, causal=True, k_descale=ks,
                                v_descale=vs, round_scaled_q=True)
    assert_close(out.float().cpu().numpy().transpose(1, 0, 2), ro, fp8=dtype != "bf16")
    assert_lse(lse.cpu().numpy(), rl)


@pytest.mark.parametrize("dtype", ["bf16", "e4m3"])
def test_chunked_prefill_kvcache(dtype):
    """BASELINE config 4's call at reduced size: packed chunks appended to the
    paged cache then attended causally with a sliding window and softcap;
    num_active leaves the last request out."""
    announce(f"chunked prefill {dtype}")
    rng = np.random.default_rng(15)
    dt = torch.bfloat16 if dtype == "bf16" else FP8[dtype]
    ks, vs = (1.0, 1.0) if dtype == "bf16" else (1.5, 0.7)
    chunks = [256, 700, 1, 129, 64]
    prior = [0, 3000, 17, 999, 50]
    case = PagedCase(rng, batch=5, nheads=8, nheads_k=2, lengths=prior, new_tokens=chunks,
                     dtype=dt, k_descale=ks, v_descale=vs)
    cu = case.cu
    q = randn(rng, (cu[-1] + 5, 8, 128))
    k_dev = dev_from_codes(np.concatenate([case.k_codes, np.zeros((5, 2, 128), case.k_codes.dtype)]), dt)
    v_dev = dev_from_codes(np.concatenate([case.v_codes, np.zeros((5, 2, 128), case.v_codes.dtype)]), dt)
    pool = case.pool()
    out, lse, pool2 = flash_attn_with_kvcache(
        to_dev_bf16(q), pool, None, k_dev, v_dev,
        cache_seqlens=torch.tensor(prior, dtype=torch.int32, device=DEV),
        block_table=torch.tensor(case.table, device=DEV),
        cu_seqlens_q=torch.tensor(cu, device=DEV), max_seqlen_q=max(chunks), causal=True,
        window_size=(4095 // 8, 0), softcap=50.0, return_softmax_lse=True, num_active=4,
        k_descale=ks, v_descale=vs)
    torch.cuda.synchronize()
    assert pool2 is pool
    exp_pool = case.expected_pool(num_active=4)
    np.testing.assert_array_equal(codes_of(pool), exp_pool)
    kp, vp = case.kv_pages(exp_pool)
    totals = case.lengths + case.new_tokens
    ro, rl = A.ragged_reference(q, kp, vp, cu, totals, case.table, causal=True,
                                window_left=4095 // 8, softcap=50.0, k_descale=ks, v_descale=vs,
                                round_scaled_q=True, num_active=4)
    assert_close(out.float().cpu().numpy(), ro, fp8=dtype != "bf16")
    assert_lse(lse.cpu().numpy(), rl)
    assert not out[cu[4]:].float().abs().sum().item()


def test_prefill_bitwise_repeat():
    """test_prefill.py:827-875's race check: repeats are bitwise equal."""
    announce("dense repeat")
    rng = np.random.default_rng(16)
    q = to_dev_bf16(randn(rng, (1, 8, 1024, 128)))
    k = to_dev_bf16(randn(rng, (1, 2, 1024, 128)))
    v = to_dev_bf16(randn(rng, (1, 2, 1024, 128)))
    ref = flash_attn_func(q, k, v, causal=True)
    for _ in range(20):
        assert torch.equal(flash_attn_func(q, k, v, causal=True), ref)


# ---------------------------------------------------------------- head_dim 256
# The reference benchmarks and accepts head_dim 256 (multiples of 128,
# inputs.py:100-140, fwd_paged.py:1186); its published shapes are d256
# (docs/v7x.md:49-60, 157-169).


# Head dims of q/k and v: the d256 kernel, the free-running one at 64 and
# 192/128, the register-staged kernel at 96, 192 and the other head_dim_v !=
# head_dim (inputs.py:193-207); the reference's compiled set
# (test_prefill.py:52,205-208), 384 and 512 (multiples of 128,
# inputs.py:100-140) plus 128/256 and 256/128.  A head_dim_v above 256 runs as
# launches over chunks of v and out.
HEAD_DIMS = [(256, 256), (64, 64), (128, 256), (256, 128), (96, 96), (192, 192), (192, 128),
             (64, 256), (64, 512), (384, 384), (512, 512)]


@pytest.mark.parametrize("d,dv", HEAD_DIMS)
@pytest.mark.parametrize(
    "b,h,hk,sq,sk,causal,window,softcap",
    [
        (1, 8, 2, 512, 512, True, (-1, -1), 0.0),
        (2, 4, 4, 200, 333, True, (-1, -1), 0.0),
        (1, 4, 1, 333, 200, True, (-1, -1), 0.0),
        (1, 4, 2, 257, 257, False, (64, 17), 0.0),
        (1, 8, 1, 384, 384, True, (100, -1), 30.0),
    ],
)
def test_flash_attn_func_head_dims(d, dv, b, h, hk, sq, sk, causal, window, softcap):
    announce(f"dense d{d}/{dv} b{b} h{h}/{hk} sq{sq} sk{sk} causal={causal} window={window}")
    rng = np.random.default_rng(70)
    q, k, v = randn(rng, (b, sq, h, d)), randn(rng, (b, sk, hk, d)), randn(rng, (b, sk, hk, dv))
    out, lse = flash_attn_func(
        to_dev_bf16(head_major(q)), to_dev_bf16(head_major(k)), to_dev_bf16(head_major(v)),
        causal=causal, window_size=window, softcap=softcap, return_softmax_lse=True)
    torch.cuda.synchronize()
    ro, rl = A.attention_ref(q, k, v, causal=causal, window_size=window, softcap=softcap,
                             round_scaled_q=True)
    assert_close(out.float().cpu().numpy(), head_major(ro))
    assert_lse(lse.cpu().numpy(), rl)


@pytest.mark.parametrize("g", [1, 2, 4, 6])  # heads a workgroup serves: 1, 2, 4, 2
@pytest.mark.parametrize("sq,sk,causal,window,softcap", [
    (1, 1, True, (-1, -1), 0.0),
    (31, 65, True, (-1, -1), 0.0),      # one key past a tile
    (33, 63, False, (-1, -1), 0.0),
    (129, 128, True, (-1, -1), 0.0),    # a row that sees nothing, a row past a q tile
    (97, 193, True, (70, -1), 0.0),     # four key tiles: every buffer reused
    (64, 450, False, (300, 5), 50.0),
])
def test_head_dim_64_tile_edges(g, sq, sk, causal, window, softcap):
    announce(f"d64 g{g} sq{sq} sk{sk} causal={causal} window={window} softcap={softcap}")
    rng = np.random.default_rng(71)
    b, hk = 2, 2
    h = g * hk
    q, k, v = randn(rng, (b, sq, h, 64)), randn(rng, (b, sk, hk, 64)), randn(rng, (b, sk, hk, 64))
    s = rng.standard_normal(h).astype(np.float32) if g == 2 else None
    out, lse = flash_attn_func(
        to_dev_bf16(head_major(q)), to_dev_bf16(head_major(k)), to_dev_bf16(head_major(v)),
        causal=causal, window_size=window, softcap=softcap, return_softmax_lse=True,
        learnable_sink=None if s is None else torch.tensor(s, device=DEV))
    ro, rl = A.attention_ref(q, k, v, causal=causal, window_size=window, softcap=softcap, sinks=s,
                             round_scaled_q=True)
    assert_close(out.float().cpu().numpy(), head_major(ro))
    assert_lse(lse.cpu().numpy(), rl)


@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128), (192, 128)])
@pytest.mark.parametrize("b,h,hk,sq,sk,causal,window,softcap", [
    # one wave per key group and 32 rows (8 key tiles or more)
    (1, 2, 1, 1, 1100, True, (-1, -1), 0.0),    # more key tiles than groups by one or two
    (1, 3, 1, 33, 512, True, (-1, -1), 30.0),   # a row past a q tile; group sizes equal
    (1, 4, 2, 600, 600, True, (-1, -1), 0.0),   # leading q tiles with fewer tiles than groups
    (1, 2, 2, 600, 520, True, (-1, -1), 0.0),   # rows that see nothing
    (2, 2, 2, 70, 900, False, (700, 3), 0.0),
    # three key tiles: too few to split (the four-wave form at 128)
    (1, 4, 1, 65, 130, True, (-1, -1), 0.0),
    # two key groups of four waves
    (3, 24, 6, 129, 700, True, (-1, -1), 0.0),  # 4 heads a workgroup, 11 key tiles
    (3, 30, 15, 300, 513, False, (-1, -1), 50.0),
    # up to two such workgroups per CU
    (1, 20, 20, 2050, 2100, True, (-1, -1), 0.0),
])
def test_dense_forms(d, dv, b, h, hk, sq, sk, causal, window, softcap):
    """Dense calls whose grid leaves CUs idle: the key tiles of a q tile split
    over waves and merged (prefill_form)."""
    announce(f"dense form d{d}/{dv} b{b} h{h}/{hk} sq{sq} sk{sk} causal={causal} window={window}")
    rng = np.random.default_rng(72)
    q, k, v = randn(rng, (b, sq, h, d)), randn(rng, (b, sk, hk, d)), randn(rng, (b, sk, hk, dv))
    s = rng.standard_normal(h).astype(np.float32) if sq % 2 else None
    out, lse = flash_attn_func(
        to_dev_bf16(head_major(q)), to_dev_bf16(head_major(k)), to_dev_bf16(head_major(v)),
        causal=causal, window_size=window, softcap=softcap, return_softmax_lse=True,
        learnable_sink=None if s is None else torch.tensor(s, device=DEV))
    check = slice(0, h) if sq * sk < 1 << 20 else slice(h - 1, h)  # the oracle's time
    kv = slice(0, hk) if sq * sk < 1 << 20 else slice(hk - 1, hk)
    ro, rl = A.attention_ref(q[:, :, check], k[:, :, kv], v[:, :, kv], causal=causal,
                             window_size=window, softcap=softcap,
                             sinks=None if s is None else s[check], round_scaled_q=True)
    assert_close(out.float().cpu().numpy()[:, check], head_major(ro))
    assert_lse(lse.cpu().numpy()[:, check], rl)


@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128), (192, 128)])
@pytest.mark.parametrize("sq,sk,causal,window", [
    (600, 600, True, (-1, -1)),     # leading q tiles with one key tile: none for the second group
    (600, 520, True, (-1, -1)),     # rows that see nothing: both groups' maxima -inf
    (600, 700, False, (300, 200)),  # waves that skip their group's first tile
    (600, 700, True, (480, -1)),
])
def test_two_key_groups(d, dv, sq, sk, causal, window):
    announce(f"two key groups d{d}/{dv} sq{sq} sk{sk} causal={causal} window={window}")
    rng = np.random.default_rng(80)
    h = 16  # 304 workgroups of 32 rows, 80 of 128
    q, k, v = randn(rng, (1, sq, h, d)), randn(rng, (1, sk, h, d)), randn(rng, (1, sk, h, dv))
    qt, kt, vt = (to_dev_bf16(head_major(x)) for x in (q, k, v))
    assert dense_form(qt, kt, vt, causal, window) == "MID"
    out, lse = flash_attn_func(qt, kt, vt, causal=causal, window_size=window, return_softmax_lse=True)
    ro, rl = A.attention_ref(q, k, v, causal=causal, window_size=window, round_scaled_q=True)
    assert_close(out.float().cpu().numpy(), head_major(ro))
    assert_lse(lse.cpu().numpy(), rl)


# One call per kernel form: (d, dv, h, sq, sk, form)
FORM_CALLS = [
    (64, 64, 4, 256, 768, "SMALL"), (64, 64, 60, 256, 768, "MID"), (64, 64, 132, 256, 768, "LARGE"),
    (128, 128, 4, 256, 768, "SMALL"), (128, 128, 60, 256, 768, "MID"),
    (128, 128, 132, 256, 768, "FREE"), (128, 128, 132, 256, 1728, "LARGE"),
    (128, 128, 256, 512, 1728, "LARGE"),  # pairs of q tiles
    (192, 128, 4, 256, 768, "SMALL"), (192, 128, 60, 256, 768, "MID"),
    (192, 128, 132, 256, 768, "LARGE"),
    (256, 256, 256, 256, 768, "LARGE"),  # pairs of q tiles
]


@pytest.mark.parametrize("b,h,hk,sq,sk,causal,window,softcap,sinks", [
    # the ping-pong kernel (many rows, at least 1,600 keys a row): ragged ends
    # on both sides, 1, 2 and 8 heads a workgroup
    (1, 30, 30, 1150, 2305, False, (-1, -1), 0.0, True),
    (2, 18, 9, 1055, 2113, False, (1800, 700), 50.0, False),
    (1, 64, 8, 2309, 3457, True, (-1, -1), 0.0, False),
    # softcap tanh: exact, and the degree-5 polynomial
    (1, 64, 8, 1055, 2113, False, (-1, -1), 5.0, False),
    (1, 64, 8, 1055, 2113, False, (-1, -1), 20.0, False),
    # the four-wave form: tile edges, 1, 2 and 4 heads a workgroup
    (5, 24, 8, 257, 257, True, (-1, -1), 0.0, True),
    (9, 10, 5, 129, 191, False, (64, 17), 30.0, False),
    (16, 16, 4, 97, 65, True, (-1, -1), 0.0, False),
])
def test_dense_large_and_free_forms(b, h, hk, sq, sk, causal, window, softcap, sinks):
    announce(f"dense form b{b} h{h}/{hk} sq{sq} sk{sk} causal={causal} window={window}")
    rng = np.random.default_rng(73)
    q, k, v = randn(rng, (b, sq, h, 128)), randn(rng, (b, sk, hk, 128)), randn(rng, (b, sk, hk, 128))
    s = rng.standard_normal(h).astype(np.float32) if sinks else None
    out, lse = flash_attn_func(
        to_dev_bf16(head_major(q)), to_dev_bf16(head_major(k)), to_dev_bf16(head_major(v)),
        causal=causal, window_size=window, softcap=softcap, return_softmax_lse=True,
        learnable_sink=None if s is None else torch.tensor(s, device=DEV))
    hs, ks = slice(h - h // hk, h), slice(hk - 1, hk)  # the last KV head's group, last batch
    ro, rl = A.attention_ref(q[-1:, :, hs], k[-1:, :, ks], v[-1:, :, ks], causal=causal,
                             window_size=window, softcap=softcap,
                             sinks=None if s is None else s[hs], round_scaled_q=True)
    assert_close(out[-1:, hs].float().cpu().numpy(), head_major(ro))
    assert_lse(lse[-1:, hs].cpu().numpy(), rl)


@pytest.mark.parametrize("d,dv", [(64, 64), (128, 128), (192, 128), (256, 256)])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("step", [1 << 23, -(1 << 10), 1 << 10])
def test_kv_token_strides(d, dv, packed, step):
    """Token strides of K and V through the C-ABI: 16 MiB and more, and
    negative (rows in reverse), which the register-staged kernel takes, and a
    plain stride beside them."""
    announce(f"kv strides d{d}/{dv} packed={packed} step {step}")
    from flywheel_tpu import _native as N
    rng = np.random.default_rng(76)
    b, h, hk, sq, sk = 1, 4, 2, 45, 67
    q, k, v = randn(rng, (b, sq, h, d)), randn(rng, (b, sk, hk, d)), randn(rng, (b, sk, hk, dv))
    qd, out = to_dev_bf16(head_major(q)), torch.empty((b, h, sq, dv), dtype=torch.bfloat16, device=DEV)
    buf = torch.zeros(((sk - 1) * abs(step) + 2 * hk * 256,), dtype=torch.bfloat16, device=DEV)
    at = torch.arange(sk) * abs(step) if step > 0 else torch.arange(sk - 1, -1, -1) * -step
    rows = buf.as_strided((buf.numel() - 4 * 256 + 1, 2 * hk * 256), (1, 1))  # [start, element]
    for x, off in ((k, 0), (v, hk * 256)):  # K heads at 0 and 256, V heads after them
        for i in range(hk):
            w = x.shape[-1]
            for t in range(sk):
                rows[int(at[t]), off + 256 * i:off + 256 * i + w] = to_dev_bf16(x[0, t, i])
    first = buf.data_ptr() + 2 * int(at[0])
    cu_q = torch.tensor([0, sq], dtype=torch.int32, device=DEV)
    cu_k = torch.tensor([0, sk], dtype=torch.int32, device=DEV)
    p = N.PrefillParams()
    p.kv_mode = N.FW_KV_VARLEN if packed else N.FW_KV_DENSE
    p.q, p.out, p.k, p.v = N.ptr(qd), N.ptr(out), first, first + 2 * hk * 256
    p.cu_seqlens_q, p.cu_seqlens_k = N.ptr(cu_q), N.ptr(cu_k)
    p.q_stride_h, p.q_stride_t, p.o_stride_h, p.o_stride_t = sq * d, d, sq * dv, dv
    p.k_stride_h = p.v_stride_h = 256
    p.k_stride_t = p.v_stride_t = step
    p.batch, p.nheads, p.nheads_k, p.head_dim, p.head_dim_v = b, h, hk, d, dv
    p.seqlen_q, p.seqlen_k, p.max_seqlen_q = sq, sk, sq
    p.kv_dtype, p.softmax_scale, p.causal = N.FW_BF16, d ** -0.5, 1
    p.window_left = p.window_right = -1
    p.k_descale = p.v_descale = 1.0
    wide = not 0 <= step < 1 << 23
    assert (N.lib().fw_prefill_form(p) == N.FORM_GENERAL) == wide
    ws = torch.empty(max(1, N.lib().fw_prefill_workspace_bytes(p)), dtype=torch.uint8, device=DEV)
    p.workspace, p.workspace_bytes = N.ptr(ws), ws.numel()
    N.check(N.lib().fw_prefill(p, N.stream_of(qd)))
    ro, _ = A.attention_ref(q, k, v, causal=True, round_scaled_q=True)
    assert_close(out.float().cpu().numpy(), head_major(ro))


@pytest.mark.parametrize("d,dv", [(64, 64), (192, 128)])
def test_kv_rows_off_16_bytes(d, dv):
    """Contiguous K and V that start one value into their storage."""
    announce(f"kv off 16 bytes d{d}/{dv}")
    rng = np.random.default_rng(77)
    b, h, hk, sq, sk = 2, 4, 2, 70, 133
    q, k, v = randn(rng, (b, sq, h, d)), randn(rng, (b, sk, hk, d)), randn(rng, (b, sk, hk, dv))

    def shifted(x):
        x = to_dev_bf16(head_major(x))
        y = torch.empty(x.numel() + 1, dtype=x.dtype, device=DEV)[1:].view(x.shape)
        return y.copy_(x)

    out = flash_attn_func(to_dev_bf16(head_major(q)), shifted(k), shifted(v), causal=True)
    ro, _ = A.attention_ref(q, k, v, causal=True, round_scaled_q=True)
    assert_close(out.float().cpu().numpy(), head_major(ro))


def schedule_of(qlens, klens, h, hk, causal, num_rows, *, window=-1, num_active=None, codes_at=None):
    """The (sequence, first row) pairs fw_prefill's schedule holds for packed
    sequences (head dim 128), read back from the workspace; with the slots' split
    codes, held after codes_at slots, beside them."""
    from flywheel_tpu import _native as N
    dev = lambda x: torch.tensor(np.concatenate([[0], np.cumsum(x)]), dtype=torch.int32, device=DEV)
    cu_q, cu_k = dev(qlens), dev(klens)
    q = torch.zeros((h, num_rows, 128), dtype=torch.bfloat16, device=DEV)
    k = torch.zeros((hk, max(1, sum(klens)), 128), dtype=torch.bfloat16, device=DEV)
    out = torch.empty_like(q)
    p = N.PrefillParams()
    p.kv_mode, p.q, p.out, p.k, p.v = N.FW_KV_VARLEN, N.ptr(q), N.ptr(out), N.ptr(k), N.ptr(k)
    p.cu_seqlens_q, p.cu_seqlens_k = N.ptr(cu_q), N.ptr(cu_k)
    for x, t in (("q", q), ("o", q), ("k", k), ("v", k)):
        setattr(p, x + "_stride_h", t.shape[1] * 128)
        setattr(p, x + "_stride_t", 128)
    p.batch, p.nheads, p.nheads_k, p.head_dim = len(qlens), h, hk, 128
    p.seqlen_q, p.seqlen_k, p.max_seqlen_q = num_rows, sum(klens), max(qlens)
    p.kv_dtype, p.softmax_scale, p.causal = N.FW_BF16, 0.1, int(causal)
    p.window_left, p.window_right = window, -1
    p.k_descale = p.v_descale = 1.0
    active = None if num_active is None else torch.tensor([num_active], dtype=torch.int32, device=DEV)
    p.num_active = N.ptr(active)
    ws = torch.zeros(N.lib().fw_prefill_workspace_bytes(p), dtype=torch.uint8, device=DEV)
    p.workspace, p.workspace_bytes = N.ptr(ws), ws.numel()
    N.check(N.lib().fw_prefill(p, N.stream_of(q)))
    w = ws[:ws.numel() // 4 * 4].view(torch.int32).cpu().numpy()
    slots = [(int(w[1 + 2 * i]), int(w[2 + 2 * i])) for i in range(w[0])]
    if codes_at is None:
        return slots
    codes = -(-(1 + 2 * codes_at) * 4 // 256) * 64
    return slots, [int(x) for x in w[codes:codes + w[0]]]


@pytest.mark.parametrize("n,lo,hi,extra", [
    (1, 1, 1, 0), (70, 0, 90, 0), (64, 64, 64, 33),
    (40, 300, 1700, 0),    # ~1,250 tiles of 32 rows: 20 runs of 64
    (1500, 0, 40, 100),    # more sequences than threads
    (45, 1800, 2000, 0),   # more than 2,048 tiles: sequence order
    (2100, 0, 3, 0),       # more than 2,048 sequences: sequence order
])
def test_schedule_order(n, lo, hi, extra):
    """Every tile once, heaviest first, equal costs in sequence order."""
    announce(f"schedule n{n} {lo}..{hi} + {extra}")
    rng = np.random.default_rng(75)
    lens = [int(x) for x in rng.integers(lo, hi + 1, n)]
    rows = sum(lens)
    got = schedule_of(lens, lens, 4, 1, True, rows + extra)  # 4 heads of 32 rows
    tiles = [(s, r) for s in range(n) for r in range(0, lens[s], 32)]
    if n <= 2048 and len(tiles) <= 2048:
        # exact buckets below 64 key tiles, the longest here 32
        tiles.sort(key=lambda t: -min(t[1] + 32, lens[t[0]]) // 64)  # -ceil(keys / 64)
    assert got == tiles + [(-1, r) for r in range(rows, rows + extra, 32)]


def cost_bucket(cost):
    """The schedule's cost buckets: exact below 64 key tiles, 32 an octave above."""
    if cost < 64:
        return cost
    e = cost.bit_length() - 1
    return 64 + 32 * (e - 6) + (cost >> (e - 5)) - 32


def tile_cost(qlen, klen, row, rows, causal, window):
    last, off = min(row + rows, qlen) - 1, klen - qlen
    lo = max(0, row + off - window) if window >= 0 else 0
    hi = min(klen, last + off + 1) if causal else klen
    return -(-hi // 64) - lo // 64 if hi > lo else 0


def test_schedule_order_many_sequences():
    """More than 2,048 sequences, most of them without rows: ordered as well."""
    announce("schedule of 2600 sequences")
    rng = np.random.default_rng(78)
    lens = [int(x) if rng.random() < 0.3 else 0 for x in rng.integers(1, 121, 2600)]
    tiles = [(s, r) for s in range(2600) for r in range(0, lens[s], 32)]
    assert 1000 < len(tiles) <= 2048
    got = schedule_of(lens, lens, 4, 1, True, sum(lens))
    tiles.sort(key=lambda t: -tile_cost(lens[t[0]], lens[t[0]], t[1], 32, True, -1))
    assert got == tiles


@pytest.mark.parametrize("n,qlo,qhi,klo,khi,h,hk,causal,window,active", [
    (40, 0, 200, 1500, 9000, 8, 1, True, -1, None),    # costs on both sides of 64 and 128
    (40, 0, 200, 1500, 9000, 8, 1, False, -1, 33),     # sequences past num_active are padding
    (24, 1, 400, 2000, 6000, 16, 2, True, 1500, None), # two head groups, a window
    (3, 1, 300, 2000, 40000, 8, 1, True, -1, None),
    (9, 100, 300, 2000, 2400, 64, 4, True, 100, None), # too few key tiles to split any
])
def test_schedule_split_slots(n, qlo, qhi, klo, khi, h, hk, causal, window, active):
    """The ping-pong kernel's schedule: the heaviest tiles first, the first
    ranks among them split in two (as many as even the last round of the CUs),
    their second halves after every sequence tile, padding last."""
    announce(f"schedule with splits n{n} h{h}/{hk} causal={causal} window={window} active={active}")
    rng = np.random.default_rng(79)
    qlens = [int(x) for x in rng.integers(qlo, qhi + 1, n)]
    klens = [q + int(x) for q, x in zip(qlens, rng.integers(klo, khi + 1, n))]
    rows, nact = 32, n if active is None else active  # 8 heads x 32 rows a workgroup
    ng, total = h // 8, sum(qlens)
    most = min(32, max(1, 256 // ng))
    got, codes = schedule_of(qlens, klens, h, hk, causal, total, window=window, num_active=active,
                             codes_at=-(-total // rows) + n + 1 + most)
    cost = lambda t: tile_cost(qlens[t[0]], klens[t[0]], t[1], rows, causal, window)
    tiles = [(s, r) for s in range(nact) for r in range(0, qlens[s], rows)]
    tiles.sort(key=lambda t: -cost_bucket(cost(t)))
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    nsplit = 0
    if len(tiles) * ng < 16 * cus:
        nsplit = min(most, sum(cost(t) >= 8 for t in tiles), -(-(-len(tiles) * ng % cus) // ng))
    assert (nsplit > 0) == (window != 100)
    padding = [(-1, r) for r in range(sum(qlens[:nact]), total, rows)]
    assert got == tiles + tiles[:nsplit] + padding
    assert codes == ([2 * i for i in range(nsplit)] + [-1] * (len(tiles) - nsplit) +
                     [2 * i + 1 for i in range(nsplit)] + [-1] * len(padding))


@pytest.mark.parametrize("wide", [False, True])  # the four-wave form, the ping-pong kernel
@pytest.mark.parametrize("dense_kv", [False, True])
def test_ragged_forms(wide, dense_kv):
    """Packed varlen and paged rows on both sides of prefill_form's line (mean
    length, block-table width), the same sequences on each."""
    announce(f"ragged forms wide={wide} packed={dense_kv}")
    rng = np.random.default_rng(74)
    qlens, prior = [65, 1, 256, 33, 0, 130], [0, 300, 17, 64, 5, 129]
    h, hk = 8, 2
    cu = torch.tensor(np.concatenate([[0], np.cumsum(qlens)]), dtype=torch.int32, device=DEV)
    if not dense_kv:
        case = PagedCase(rng, batch=6, nheads=h, nheads_k=hk, lengths=prior, new_tokens=qlens,
                         max_pages=200 if wide else 25)
        q = randn(rng, (sum(qlens), h, 128))
        pool = case.pool()
        out, lse, _ = flash_attn_with_kvcache(
            to_dev_bf16(q), pool, None, dev_from_codes(case.k_codes, case.dtype),
            dev_from_codes(case.v_codes, case.dtype),
            cache_seqlens=torch.tensor(prior, dtype=torch.int32, device=DEV),
            block_table=torch.tensor(case.table, device=DEV), cu_seqlens_q=cu,
            max_seqlen_q=max(qlens), causal=True, return_softmax_lse=True)
        exp = case.expected_pool()
        np.testing.assert_array_equal(codes_of(pool), exp)
        krows, vrows = case.rows(exp)
        out, lse = out.float().cpu().numpy(), lse.cpu().numpy()
        for i, (n, p) in enumerate(zip(qlens, prior)):
            if n == 0:
                continue
            rows = slice(int(cu[i]), int(cu[i + 1]))
            ro, rl = A.attention_ref(q[None, rows], krows[None, i, :n + p], vrows[None, i, :n + p],
                                     causal=True, round_scaled_q=True)
            assert_close(out[rows], ro[0])
            assert_lse(lse[:, rows], rl[0])
        return
    klens = [n + p for n, p in zip(qlens, prior)]
    if wide:
        klens[2] += 12000
    cuk = np.concatenate([[0], np.cumsum(klens)])
    q = randn(rng, (sum(qlens), h, 128))
    k, v = randn(rng, (sum(klens), hk, 128)), randn(rng, (sum(klens), hk, 128))
    hm = lambda x: to_dev_bf16(x.transpose(1, 0, 2))
    out, lse = flash_attn_varlen_func(hm(q), hm(k), hm(v), cu,
                                      torch.tensor(cuk, dtype=torch.int32, device=DEV), max(qlens),
                                      max(klens), causal=True, return_softmax_lse=True)
    out, lse = out.float().cpu().numpy(), lse.cpu().numpy()
    for i, n in enumerate(qlens):
        if n == 0:
            continue
        rows, keys = slice(int(cu[i]), int(cu[i + 1])), slice(int(cuk[i]), int(cuk[i + 1]))
        ro, rl = A.attention_ref(q[None, rows], k[None, keys], v[None, keys], causal=True,
                                 round_scaled_q=True)
        assert_close(out[:, rows], ro[0].transpose(1, 0, 2))
        assert_lse(lse[:, rows], rl[0])


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("jump", [40.0, 600.0])
def test_flash_attn_func_anchor_rescale(d, jump):
    """The slow path of the static anchor (new row maximum, O and l rescaled)
    taken twice per row: keys in thirds score 0, J/2 and J (log2 units), values
    1, 2, 3.  J = 40 rescales by 2^-20 twice (the rescale must reach every O
    register: one left unscaled moves out by ~1); J = 600 underflows the
    factor to 0 (as the reference's anchor-change test,
    test_regression.py:1035-1063).  Out is ~3 in closed form."""
    announce(f"dense d{d} anchor rescale jump {jump}")
    sk, sq, h = 768, 256, 2
    y = jump / (math.sqrt(d) * A.LOG2E)  # q = 1: score(log2) = y * sqrt(d) * log2(e)
    q = np.ones((1, sq, h, d), np.float32)
    k = np.zeros((1, sk, 1, d), np.float32)
    v = np.ones((1, sk, 1, d), np.float32)
    k[:, 256:512], k[:, 512:] = y / 2, y
    v[:, 256:512], v[:, 512:] = 2.0, 3.0
    q, k, v = (np.asarray(torch.tensor(x).to(torch.bfloat16).float()) for x in (q, k, v))
    out, lse = flash_attn_func(to_dev_bf16(head_major(q)), to_dev_bf16(head_major(k)),
                               to_dev_bf16(head_major(v)), return_softmax_lse=True)
    torch.cuda.synchronize()
    o = out.float().cpu().numpy()
    np.testing.assert_allclose(o, 3.0, atol=2e-2)
    ro, rl = A.attention_ref(q, k, v, round_scaled_q=True)
    assert_close(o, head_major(ro))
    assert_lse(lse.cpu().numpy(), rl)


@pytest.mark.parametrize("d,dv,h,sq,sk,form", FORM_CALLS)
@pytest.mark.parametrize("jump", [40.0, 600.0])
def test_anchor_rescale_forms(d, dv, h, sq, sk, form, jump):
    """The rescale of test_flash_attn_func_anchor_rescale in every form of the
    prefill kernels: scores 0, J/2 and J and values 1, 2 and 3 by thirds of the
    keys, out ~3 and lse = J ln 2 + ln(sk / 3) in closed form."""
    announce(f"anchor rescale d{d}/{dv} h{h} sq{sq} sk{sk} {form} jump {jump}")
    y = jump / (math.sqrt(d) * A.LOG2E)
    third = torch.arange(sk, device=DEV) // (sk // 3)
    rows = lambda w, x: x.to(torch.bfloat16).reshape(1, 1, sk, 1).expand(1, 1, sk, w).contiguous()
    q = torch.ones((1, h, sq, d), dtype=torch.bfloat16, device=DEV)
    k, v = rows(d, third * (y / 2)), rows(dv, third + 1)
    assert dense_form(q, k, v, False) == form
    out, lse = flash_attn_func(q, k, v, return_softmax_lse=True)
    # the last third's score with q scaled and rounded, and k, as bf16 (2^-8 each)
    qs = torch.tensor(d ** -0.5 * A.LOG2E).to(torch.bfloat16).double()
    score = float(qs * k[0, 0, -1, 0].double().cpu()) * d / A.LOG2E
    assert (out.float() - 3.0).abs().max() <= 2e-2
    assert (lse - (score + math.log(sk // 3))).abs().max() <= 1e-3


@pytest.mark.parametrize("d,dv,h,sq,sk,form", FORM_CALLS)
def test_bitwise_repeat_forms(d, dv, h, sq, sk, form):
    """Repeats are bitwise equal in every form (a race on the shared LDS
    buffers would show as a difference)."""
    announce(f"repeat d{d}/{dv} h{h} sq{sq} sk{sk} {form}")
    gen = torch.Generator(device=DEV).manual_seed(81)
    q, k, v = (torch.randn(x, generator=gen, device=DEV, dtype=torch.bfloat16)
               for x in ((1, h, sq, d), (1, h // 2, sk, d), (1, h // 2, sk, dv)))
    assert dense_form(q, k, v, False) == form
    ref = flash_attn_func(q, k, v)
    for _ in range(20):
        assert torch.equal(flash_attn_func(q, k, v), ref)


@pytest.mark.parametrize("d,dv", [(64, 64), (192, 128)])
@pytest.mark.parametrize("h,s,form", [(8, 512, "SMALL"), (16, 2048, "MID"), (96, 2048, "LARGE")])
def test_peaked_softmax_precision(d, dv, h, s, form):
    """Queries four times N(0, 1): most of a row's weight lies on a few keys,
    and with the row maximum as the anchor the largest weight is exactly 1.
    The error against 64 bits is then little more than the output's rounding to
    8 bits, 2^-7 / sqrt(12) over the root mean square of a log-uniform mantissa
    (1.47): 1.53e-3, and 1.70e-3 to 1.73e-3 with P's rounding of the other keys
    (emulated and measured); an anchor that lags the maximum gives 2.17e-3 and more."""
    announce(f"peaked softmax d{d}/{dv} h{h} s{s} {form}")
    gen = torch.Generator(device=DEV).manual_seed(5)
    randn = lambda *shape: torch.randn(shape, device=DEV, generator=gen)
    q, k, v = (4 * randn(1, h, s, d)).bfloat16(), randn(1, h, s, d).bfloat16(), randn(1, h, s, dv).bfloat16()
    assert dense_form(q, k, v, True) == form
    out = flash_attn_func(q, k, v, causal=True)
    qs = (q.float() * (d ** -0.5 * A.LOG2E)).bfloat16()  # the scaled queries as the kernel rounds them
    for i in range(0, h, max(1, h // 4)):
        w = (qs[0, i].double() @ k[0, i].double().T) / A.LOG2E
        w = w.masked_fill(~torch.ones_like(w, dtype=torch.bool).tril(), -math.inf)
        ref = torch.softmax(w, -1) @ v[0, i].double()
        assert (out[0, i].double() - ref).norm() <= 1.95e-3 * ref.norm()


@pytest.mark.parametrize("d,dv", HEAD_DIMS)
def test_flash_attn_func_head_dims_sinks(d, dv):
    """learnable_sink through the d256 and register-staged kernels (rows that
    see no key return the sink-only result: out 0, lse = the sink)."""
    announce(f"dense d{d}/{dv} sinks")
    rng = np.random.default_rng(74)
    b, h, hk, sq, sk = 1, 8, 2, 200, 150
    q, k, v = randn(rng, (b, sq, h, d)), randn(rng, (b, sk, hk, d)), randn(rng, (b, sk, hk, dv))
    sinks = rng.standard_normal(h).astype(np.float32)
    out, lse = flash_attn_func(
        to_dev_bf16(head_major(q)), to_dev_bf16(head_major(k)), to_dev_bf16(head_major(v)),
        causal=True, return_softmax_lse=True, learnable_sink=torch.tensor(sinks, device=DEV))
    torch.cuda.synchronize()
    ro, rl = A.attention_ref(q, k, v, causal=True, sinks=sinks, round_scaled_q=True)
    assert_close(out.float().cpu().numpy(), head_major(ro))
    assert_lse(lse.cpu().numpy(), rl)


def test_flash_attn_func_token_major_paired_d64():
    """Token-major head_dim 64 (the reference's paired form: MHA, even head
    count, inputs.py:106-147)."""
    announce("dense token-major d64")
    rng = np.random.default_rng(73)
    b, h, s, d = 2, 6, 300, 64
    q, k, v = randn(rng, (b, s, h, d)), randn(rng, (b, s, h, d)), randn(rng, (b, s, h, d))
    out = flash_attn_func(to_dev_bf16(q.reshape(b, s, h * d)), to_dev_bf16(k.reshape(b, s, h * d)),
                          to_dev_bf16(v.reshape(b, s, h * d)), causal=True, head_dim=d,
                          token_major=True)
    torch.cuda.synchronize()
    ro, _ = A.attention_ref(q, k, v, causal=True, round_scaled_q=True)
    assert_close(out.float().cpu().numpy().reshape(b, s, h, d), ro)


@pytest.mark.parametrize("d,dv", HEAD_DIMS)
def test_flash_attn_varlen_head_dims(d, dv):
    announce(f"varlen packed d{d}/{dv}")
    rng = np.random.default_rng(71)
    qlens, klens = [1, 130, 77, 256], [1, 200, 77, 300]
    h, hk = 4, 2
    cu_q = np.concatenate([[0], np.cumsum(qlens)]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(klens)]).astype(np.int32)
    q = randn(rng, (h, cu_q[-1] + 5, d))
    k = randn(rng, (hk, cu_k[-1], d))
    v = randn(rng, (hk, cu_k[-1], dv))
    out, lse = flash_attn_varlen_func(
        to_dev_bf16(q), to_dev_bf16(k), to_dev_bf16(v), torch.tensor(cu_q, device=DEV),
        torch.tensor(cu_k, device=DEV), max(qlens), max(klens), causal=True,
        return_softmax_lse=True)
    torch.cuda.synchronize()
    outs, lses = out.float().cpu().numpy(), lse.cpu().numpy()
    for s in range(4):
        qs = q[:, cu_q[s]:cu_q[s + 1]].transpose(1, 0, 2)[None]
        ks = k[:, cu_k[s]:cu_k[s + 1]].transpose(1, 0, 2)[None]
        vs = v[:, cu_k[s]:cu_k[s + 1]].transpose(1, 0, 2)[None]
        ro, rl = A.attention_ref(qs, ks, vs, causal=True, round_scaled_q=True)
        assert_close(outs[:, cu_q[s]:cu_q[s + 1]].transpose(1, 0, 2), ro[0], what=f"seq {s}")
        assert_lse(lses[:, cu_q[s]:cu_q[s + 1]], rl[0])
    assert not outs[:, cu_q[-1]:].any()


@pytest.mark.parametrize("hd", [256, 64, 384, 512])
@pytest.mark.parametrize("dtype", ["bf16", "e4m3"])
def test_chunked_prefill_kvcache_head_dims(dtype, hd):
    """The chunked-prefill call (append + paged varlen, window, softcap,
    num_active) at head_dim 256, 64, 384 and 512 (the reference's paged
    prefill takes any multiple of 128 shared by q and the pool,
    kernels/fwd_paged.py:1186-1190)."""
    announce(f"chunked prefill d{hd} {dtype}")
    rng = np.random.default_rng(72)
    dt = torch.bfloat16 if dtype == "bf16" else FP8[dtype]
    ks, vs = (1.0, 1.0) if dtype == "bf16" else (1.5, 0.7)
    chunks = [256, 300, 1, 129]
    prior = [0, 1000, 17, 500]
    case = PagedCase(rng, batch=4, nheads=8, nheads_k=2, lengths=prior, new_tokens=chunks,
                     head_dim=hd, dtype=dt, k_descale=ks, v_descale=vs)
    cu = case.cu
    q = randn(rng, (cu[-1], 8, hd))
    pool = case.pool()
    out, lse, pool2 = flash_attn_with_kvcache(
        to_dev_bf16(q), pool, None, dev_from_codes(case.k_codes, dt),
        dev_from_codes(case.v_codes, dt),
        cache_seqlens=torch.tensor(prior, dtype=torch.int32, device=DEV),
        block_table=torch.tensor(case.table, device=DEV),
        cu_seqlens_q=torch.tensor(cu, device=DEV), max_seqlen_q=max(chunks), causal=True,
        window_size=(400, 0), softcap=30.0, return_softmax_lse=True, num_active=3,
        k_descale=ks, v_descale=vs)
    torch.cuda.synchronize()
    assert pool2 is pool
    exp_pool = case.expected_pool(num_active=3)
    np.testing.assert_array_equal(codes_of(pool), exp_pool)
    kp, vp = case.kv_pages(exp_pool)
    totals = case.lengths + case.new_tokens
    ro, rl = A.ragged_reference(q, kp, vp, cu, totals, case.table, causal=True, window_left=400,
                                softcap=30.0, k_descale=ks, v_descale=vs, round_scaled_q=True,
                                num_active=3)
    assert_close(out.float().cpu().numpy(), ro, fp8=dtype != "bf16")
    assert_lse(lse.cpu().numpy(), rl)


@pytest.mark.parametrize("hd", [384, 512])
@pytest.mark.parametrize("dtype", ["bf16", "e4m3", "e5m2"])
def test_paged_varlen_read_only_wide_heads(dtype, hd):
    """flash_attn_varlen_func(block_table=...) over a merged pool at head dims
    384 and 512 (launched as 128-dim chunks of V, each chunk reading its dims
    of the merged row's V head): random_ragged_case's (3, 0, 5) on prefixes
    (127, 0, 251), plus a longer request, with an odd KV head count."""
    announce(f"paged varlen d{hd} {dtype}")
    rng = np.random.default_rng(91 + hd)
    dt = torch.bfloat16 if dtype == "bf16" else FP8[dtype]
    ks, vs = (1.0, 1.0) if dtype == "bf16" else (0.5, 2.0)
    h, hk = 6, 3
    qlens = [3, 0, 5, 300]
    prefix = [127, 0, 251, 700]
    totals = np.array(qlens) + np.array(prefix)
    case = PagedCase(rng, batch=4, nheads=h, nheads_k=hk, lengths=totals, new_tokens=[0] * 4,
                     dtype=dt, k_descale=ks, v_descale=vs, head_dim=hd)
    cu = np.concatenate([[0], np.cumsum(qlens)]).astype(np.int32)
    q = randn(rng, (cu[-1] + 7, h, hd))
    out, lse = flash_attn_varlen_func(
        to_dev_bf16(np.ascontiguousarray(q.transpose(1, 0, 2))), case.pool(), None,
        torch.tensor(cu, device=DEV), None, max(qlens), int(totals.max()), causal=True,
        window_size=(200, 0), softcap=20.0,
        return_softmax_lse=True, block_table=torch.tensor(case.table, device=DEV),
        seqused_k=torch.tensor(totals, dtype=torch.int32, device=DEV), k_descale=ks,
        v_descale=vs, nheads_k=hk)
    torch.cuda.synchronize()
    kp, vp = case.kv_pages(case.pool_codes)
    ro, rl = A.ragged_reference(q, kp, vp, cu, totals, case.table, causal=True, window_left=200,
                                softcap=20.0, k_descale=ks, v_descale=vs, round_scaled_q=True)
    got = out.float().cpu().numpy().transpose(1, 0, 2)
    assert_close(got[:cu[-1]], ro[:cu[-1]], fp8=dtype != "bf16")
    assert_lse(lse.cpu().numpy()[:, :cu[-1]], rl[:, :cu[-1]])
    assert not got[cu[-1]:].any()


@pytest.mark.parametrize("dtype,window,softcap,sinks", [
    ("bf16", -1, 0.0, False), ("bf16", 1000, 30.0, True), ("e4m3", -1, 50.0, False),
    ("bf16", 300, 0.0, True)])
def test_key_split_slots(dtype, window, softcap, sinks):
    """Few heavy q tiles over long prior contexts: the schedule splits the
    heaviest slots in two along their keys (fewer workgroups than CUs), each
    half stores an (m, l, O) partial and the second to finish merges them.
    Windows leave rows with no key in one half; sinks fold in after the
    merge."""
    announce(f"key split {dtype} window {window} softcap {softcap} sinks {sinks}")
    rng = np.random.default_rng(400 + window)
    dt = torch.bfloat16 if dtype == "bf16" else FP8[dtype]
    ks, vs = (1.0, 1.0) if dtype == "bf16" else (0.8, 1.25)
    h, hk = 32, 8
    qlens = [300, 100, 64]
    prefix = [4000, 700, 2500]
    totals = np.array(qlens) + np.array(prefix)
    case = PagedCase(rng, batch=3, nheads=h, nheads_k=hk, lengths=totals, new_tokens=[0] * 3,
                     dtype=dt, k_descale=ks, v_descale=vs)
    cu = np.concatenate([[0], np.cumsum(qlens)]).astype(np.int32)
    q = randn(rng, (cu[-1], h, 128))
    sk = rng.standard_normal(h).astype(np.float32) if sinks else None
    w2 = (window, 0) if window >= 0 else (-1, -1)
    out, lse = flash_attn_varlen_func(
        to_dev_bf16(np.ascontiguousarray(q.transpose(1, 0, 2))), case.pool(), None,
        torch.tensor(cu, device=DEV), None, max(qlens), int(totals.max()), causal=True,
        window_size=w2, softcap=softcap, return_softmax_lse=True,
        block_table=torch.tensor(case.table, device=DEV),
        seqused_k=torch.tensor(totals, dtype=torch.int32, device=DEV), k_descale=ks,
        v_descale=vs, nheads_k=hk, learnable_sink=None if sk is None else torch.tensor(sk, device=DEV))
    torch.cuda.synchronize()
    kp, vp = case.kv_pages(case.pool_codes)
    ro, rl = A.ragged_reference(q, kp, vp, cu, totals, case.table, causal=True,
                                window_left=None if window < 0 else window, softcap=softcap,
                                sinks=sk, k_descale=ks, v_descale=vs, round_scaled_q=True)
    assert_close(out.float().cpu().numpy().transpose(1, 0, 2), ro, fp8=dtype != "bf16")
    assert_lse(lse.cpu().numpy(), rl)
    # the same call again: the arrival counters start from zero every call
    out2 = flash_attn_varlen_func(
        to_dev_bf16(np.ascontiguousarray(q.transpose(1, 0, 2))), case.pool(), None,
        torch.tensor(cu, device=DEV), None, max(qlens), int(totals.max()), causal=True,
        window_size=w2, softcap=softcap, block_table=torch.tensor(case.table, device=DEV),
        seqused_k=torch.tensor(totals, dtype=torch.int32, device=DEV), k_descale=ks,
        v_descale=vs, nheads_k=hk, learnable_sink=None if sk is None else torch.tensor(sk, device=DEV))
    torch.cuda.synchronize()
    assert torch.equal(out, out2)


def test_key_split_packed_varlen():
    """The packed-varlen (non-paged) mode of the same kernel with split slots."""
    announce("key split packed varlen")
    rng = np.random.default_rng(410)
    h, hk, d = 16, 4, 128
    ql = np.array([256, 70]); kl = np.array([3000, 1500])
    cu_q = np.concatenate([[0], np.cumsum(ql)]).astype(np.int32)
    cu_k = np.concatenate([[0], np.cumsum(kl)]).astype(np.int32)
    q, k, v = randn(rng, (h, cu_q[-1], d)), randn(rng, (hk, cu_k[-1], d)), randn(rng, (hk, cu_k[-1], d))
    out, lse = flash_attn_varlen_func(to_dev_bf16(q), to_dev_bf16(k), to_dev_bf16(v),
                                      torch.tensor(cu_q, device=DEV), torch.tensor(cu_k, device=DEV),
                                      int(ql.max()), int(kl.max()), causal=True,
                                      return_softmax_lse=True)
    torch.cuda.synchronize()
    outs, lses = out.float().cpu().numpy(), lse.cpu().numpy()
    for s in range(2):
        qs_ = q[:, cu_q[s]:cu_q[s + 1]].transpose(1, 0, 2)[None]
        ks_ = k[:, cu_k[s]:cu_k[s + 1]].transpose(1, 0, 2)[None]
        vs_ = v[:, cu_k[s]:cu_k[s + 1]].transpose(1, 0, 2)[None]
        ro, rl = A.attention_ref(qs_, ks_, vs_, causal=True, round_scaled_q=True)
        assert_close(outs[:, cu_q[s]:cu_q[s + 1]].transpose(1, 0, 2), ro[0], what=f"seq {s}")
        assert_lse(lses[:, cu_q[s]:cu_q[s + 1]], rl[0])


@pytest.mark.parametrize("h,hk,q_len,kv_len,offset,fold", [
    (8, 2, 300, 1000, 0, False), (8, 2, 300, 1000, 700, False), (4, 4, 129, 700, 333, True),
    (16, 2, 1024, 4096, 2048, False)])
def test_runtime_causal_offset(h, hk, q_len, kv_len, offset, fold):
    """The dense forward with a device-side causal offset (reference
    prefill.py:344-434): query i sees keys 0 .. offset + i; against the oracle
    on the first offset + q_len keys with bottom-right causal alignment."""
    from flywheel_tpu.prefill import _flash_attn_func_pcp_causal_offset
    announce(f"runtime causal offset h{h}/{hk} q{q_len} kv{kv_len} off{offset} fold{fold}")
    rng = np.random.default_rng(500 + offset)
    q, k, v = randn(rng, (1, q_len, h, 128)), randn(rng, (1, kv_len, hk, 128)), randn(rng, (1, kv_len, hk, 128))
    hm = lambda x: np.ascontiguousarray(x.transpose(0, 2, 1, 3))
    dev = [to_dev_bf16(hm(x)) for x in (q, k, v)]
    if fold:
        dev = [t.transpose(0, 1).contiguous() for t in dev]
    out, lse = _flash_attn_func_pcp_causal_offset(
        *dev, torch.tensor(offset, dtype=torch.int32, device=DEV), return_softmax_lse=True,
        heads_outer_fold=fold)
    torch.cuda.synchronize()
    if fold:
        out = out.transpose(0, 1)
    assert lse.shape == (1, h, q_len)
    n = offset + q_len
    ro, rl = A.attention_ref(q, k[:, :n], v[:, :n], causal=True, round_scaled_q=True)
    assert_close(out.float().cpu().numpy().transpose(0, 2, 1, 3), ro)
    assert_lse(lse.cpu().numpy(), rl)
