"""GPU parity of multi-query attention under bool array masks (the masks
makeMask and createBatchCausalMask build), packed to bits and run on the
matrix-core kernel: against the oracle's SDPA / quantized SDPA and against the
generic kernel, over broadcast and per-row / per-head masks, strided and
unaligned mask rows, edges of the 32-key tile, of the 256-key packing chunk
and of the row block, whole tiles hidden or visible, rows and blocks that see
no key, sinks, several key splits, key windows of the gather, and rows of
unequal length."""
import numpy as np
import pytest
import torch

import oracle as O
import vkv
from gpu_util import (OPTIONS, assert_within, attn_tol, dev, qattn_tol, qref, rand_bits, values)

pytestmark = pytest.mark.gpu


def window_mask(L, T, win):
    pos = np.arange(T - L, T)[:, None]
    key = np.arange(T)[None]
    return (key <= pos) & (key > pos - win)


def masks(rng, kind, B, Hq, L, T):
    """-> (numpy mask, torch mask as the caller would hold it)"""
    if kind == "window":                       # [L, T], whole tiles hidden
        m = window_mask(L, T, max(2, T // 3))
    elif kind == "batch":                      # [B, 1, L, T], padded rows
        m = np.stack([window_mask(L, T, T) & (np.arange(T) < T - 17 * b) for b in range(B)])[:, None]
    elif kind == "head":                       # [B, Hq, L, T], random holes
        m = rng.random((B, Hq, L, T)) < 0.6
    elif kind == "nothing":                    # most rows see no key
        m = np.zeros((L, T), bool)
        m[L // 2, T // 2:T // 2 + 3] = True
    elif kind == "all":
        m = np.ones((1, T), bool)              # broadcast over the queries
    else:                                      # "strided": key stride 2, odd row pitch
        m = window_mask(L, T, max(2, T // 2))
        wide = torch.zeros((L, 2 * T + 1), dtype=torch.bool, device="cuda")
        wide[:, 1::2] = torch.from_numpy(m).cuda()
        return m, wide[:, 1::2]
    return m, torch.from_numpy(m).cuda()


@pytest.mark.parametrize("kind", ["window", "batch", "head", "nothing", "all", "strided"])
@pytest.mark.parametrize("dtype,D,Hq,Hkv,L,T", [
    (O.BF16, 128, 32, 8, 70, 301), (O.F16, 256, 16, 8, 65, 257), (O.BF16, 64, 12, 4, 2, 33),
    (O.BF16, 128, 3, 1, 300, 1031), (O.F16, 128, 8, 8, 129, 31)])
def test_dense_array_mask(kind, dtype, D, Hq, Hkv, L, T, monkeypatch):
    rng = np.random.default_rng(D + L + T + len(kind))
    B, f = 2, lambda a: O.to_f32(a, dtype)
    T = max(T, L) if kind in ("window", "batch", "strided") else T
    q = rand_bits(rng, (B, Hq, L, D), dtype)
    k, v = (rand_bits(rng, (B, Hkv, T, D), dtype) for _ in range(2))
    sinks = rand_bits(rng, (Hq,), dtype) if L == 70 else None
    m, mt = masks(rng, kind, B, Hq, L, T)
    run = lambda: values(vkv.scaled_dot_product_attention(
        dev(q, dtype), dev(k, dtype), dev(v, dtype), D ** -0.5, mask=mt,
        sinks=None if sinks is None else dev(sinks, dtype)), dtype)
    got = run()
    ref = O.sdpa(f(q), f(k), f(v), D ** -0.5, mask=m, q_dtype=dtype,
                 sinks=None if sinks is None else f(sinks))
    assert_within(got, ref, attn_tol(dtype, ref), "oracle")
    monkeypatch.setattr(OPTIONS, "generic_attention", 1)
    assert_within(got, run(), attn_tol(dtype, ref), "generic")


@pytest.mark.parametrize("kind", ["window", "batch", "head", "nothing"])
@pytest.mark.parametrize("bits,D,L,T,gather", [(4, 128, 48, 333, 0), (8, 256, 16, 600, 0),
                                               (4, 64, 130, 1100, 256)])
def test_quantized_array_mask(kind, bits, D, L, T, gather, monkeypatch):
    """Quantized tuples; gather > 0: the keys gathered in several windows."""
    dtype, B, Hq, Hkv = O.BF16, 2, 8, 4
    monkeypatch.setattr(OPTIONS, "gather_tokens", gather)
    rng = np.random.default_rng(bits + D + L + T + len(kind))
    f = lambda a: O.to_f32(a, dtype)
    q = rand_bits(rng, (B, Hq, L, D), dtype)
    kx, vx = (rand_bits(rng, (B, Hkv, T, D), dtype) for _ in range(2))
    kq, ks, kb, _ = O.quantize(kx, dtype, 64, bits)
    vq, vs, vb, _ = O.quantize(vx, dtype, 64, bits)
    m, mt = masks(rng, kind, B, Hq, L, T)
    t = lambda a: torch.from_numpy(a.view(np.int32)).cuda()
    run = lambda: values(vkv.quantized_scaled_dot_product_attention(
        dev(q, dtype), (t(kq), dev(ks, dtype), dev(kb, dtype)),
        (t(vq), dev(vs, dtype), dev(vb, dtype)), D ** -0.5, mask=mt, group_size=64, bits=bits), dtype)
    got = run()
    ref, wb = qref(f(q), dtype, kq, f(ks), f(kb), vq, f(vs), f(vb), D ** -0.5, 64, bits, mask=m,
                   rounding=O.REF_CHUNK)
    assert_within(got, ref, qattn_tol(dtype, ref, wb), "oracle", wb)
    monkeypatch.setattr(OPTIONS, "generic_attention", 1)
    assert_within(got, run(), attn_tol(dtype, ref) + 2 * wb, "generic", wb)


@pytest.mark.parametrize("per_row", [False, True])
def test_quantized_pool_rows_of_unequal_length(per_row, monkeypatch):
    """A pool view with per-sequence lengths under one mask for all rows or
    one each: keys past a row's length stay hidden though the mask shows
    them, and a row whose visible keys all lie past its length averages V."""
    dtype, B, Hq, Hkv, D, L, bs = O.BF16, 3, 8, 2, 128, 40, 32
    lens, Tm = [300, 64, 31], 320
    rng = np.random.default_rng(7 + per_row)
    pool = vkv.PagedPool(40, bs, 1, Hkv, D, dtype=vkv.BF16, bits=4)
    nb = Tm // bs
    table = torch.randperm(39, device="cuda")[:B * nb].int().view(B, nb).contiguous()
    k, v = (torch.randn((B, Tm, Hkv, D), device="cuda").bfloat16() for _ in range(2))
    slots = (table[:, :, None] * bs + torch.arange(bs, device="cuda")).view(-1).int()
    pool.append(0, k.view(-1, Hkv, D), v.view(-1, Hkv, D), slots)
    view = pool.view(0, table, torch.tensor(lens, dtype=torch.int32, device="cuda"), Tm)
    m = rng.random((B, 1, L, Tm) if per_row else (L, Tm)) < 0.5
    m[..., 3, :] = False
    m[..., 3, 310:] = True
    q = torch.randn((B, Hq, L, D), device="cuda").bfloat16()
    run = lambda: vkv.quantized_paged_attention(q, view, D ** -0.5,
                                                mask=torch.from_numpy(m).cuda()).float().cpu().numpy()
    got = run()
    monkeypatch.setattr(OPTIONS, "generic_attention", 1)
    ref = run()
    # both paths round scores to bf16: 2e-2 each side of the exact value
    assert_within(got, ref, 2 * attn_tol(dtype, ref), "generic")
