"""Attention sinks of -inf and of the type's lowest value (a logit that adds
nothing) where the first keys a kernel takes are hidden: the running max has
no finite value yet.  One-token decodes and prompt chunks, bool and additive
masks, the float-decode, matrix-core and generic kernels, against the oracle.
NaN keys in one-token decodes.  Short rows, whose heads are dealt to several
workgroups, and chunks of little work under a bool mask, at the lines of their
rules.  The values that a masked chunk over a quantized cache attends."""
import numpy as np
import pytest
import torch

import oracle as O
import vkv
from gpu_util import OPTIONS, assert_within, attn_tol, dev, rand_bits, values

pytestmark = pytest.mark.gpu

LOWEST = {O.F32: -3.4028234e38, O.F16: -65504.0, O.BF16: -3.3895314e38}


@pytest.mark.parametrize("generic", [0, 1])
@pytest.mark.parametrize("dtype,D,Hq,Hkv,L,T", [
    (O.BF16, 128, 8, 2, 1, 20), (O.F16, 64, 12, 4, 1, 700), (O.BF16, 256, 4, 2, 1, 2100),
    (O.F32, 128, 4, 2, 1, 300), (O.BF16, 128, 8, 2, 70, 301), (O.F16, 256, 4, 2, 65, 65),
    (O.BF16, 64, 4, 4, 200, 200)])
@pytest.mark.parametrize("additive", [False, True])
def test_sinks_that_add_nothing(additive, dtype, D, Hq, Hkv, L, T, generic, monkeypatch):
    monkeypatch.setattr(OPTIONS, "generic_attention", generic)
    rng = np.random.default_rng(D + L + T)
    B, f = 2, lambda a: O.to_f32(a, dtype)
    q = rand_bits(rng, (B, Hq, L, D), dtype)
    k, v = (rand_bits(rng, (B, Hkv, T, D), dtype) for _ in range(2))
    s = rng.standard_normal(Hq).astype(np.float32)
    s[0::4], s[1::4] = -np.inf, LOWEST[dtype]
    sinks = O.from_f32(s, dtype)
    # decode: the first keys hidden; chunk: a window of 20, so that later rows
    # see none of the first tile that the first rows see
    key, pos = np.arange(T)[None], np.arange(T - L, T)[:, None]
    m = (key >= min(T - 3, 170)) if L == 1 else (key <= pos) & (key > pos - 20)
    mt = torch.from_numpy(m).cuda()
    if additive:
        m = np.where(m, 0.0, -np.inf).astype(np.float32)
        mt = torch.from_numpy(m).cuda()
    ref = O.sdpa(f(q), f(k), f(v), D ** -0.5, mask=m, q_dtype=dtype, sinks=f(sinks))
    got = values(vkv.scaled_dot_product_attention(dev(q, dtype), dev(k, dtype), dev(v, dtype),
                                                  D ** -0.5, mask=mt, sinks=dev(sinks, dtype)), dtype)
    assert_within(got, ref, attn_tol(dtype, ref), "oracle")


@pytest.mark.parametrize("dtype", [O.BF16, O.F16])
@pytest.mark.parametrize("D,Hq,Hkv,T", [(256, 4, 2, 20), (128, 8, 2, 300), (64, 4, 4, 5000)])
def test_a_nan_key_shows(dtype, D, Hq, Hkv, T):
    """A NaN in one key makes its head's outputs NaN, not zeros, in launches
    of one part and of several; the other heads stay as they are."""
    rng = np.random.default_rng(D + T)
    f = lambda a: O.to_f32(a, dtype)
    q = rand_bits(rng, (1, Hq, 1, D), dtype)
    k, v = (rand_bits(rng, (1, Hkv, T, D), dtype) for _ in range(2))
    ref = O.sdpa(f(q), f(k), f(v), D ** -0.5, q_dtype=dtype)
    kd = dev(k, dtype)
    kd[0, 0, T // 2, 3] = float("nan")
    got = values(vkv.scaled_dot_product_attention(dev(q, dtype), kd, dev(v, dtype), D ** -0.5), dtype)
    rep = Hq // Hkv
    assert np.isnan(got[:, :rep]).all()
    assert_within(got[:, rep:], ref[:, rep:], attn_tol(dtype, ref[:, rep:]), "other heads")


@pytest.mark.parametrize("dtype,D", [(O.BF16, 128), (O.F16, 64), (O.BF16, 256)])
@pytest.mark.parametrize("B,Hq,Hkv", [(1, 32, 8), (1, 24, 8), (2, 12, 1), (8, 16, 2), (5, 64, 8), (40, 8, 8)])
def test_short_rows(B, Hq, Hkv, dtype, D):
    """The edges of one part (32768 / D tokens), of the rows whose heads are
    split (768 tokens) and of a wave's step, plain and masked."""
    f = lambda a: O.to_f32(a, dtype)
    for T in (1, 16, 17, 128, 129, 32768 // D, 32768 // D + 1, 768, 769):
        rng = np.random.default_rng(B + Hq + D + T)
        q = rand_bits(rng, (B, Hq, 1, D), dtype)
        k, v = (rand_bits(rng, (B, Hkv, T, D), dtype) for _ in range(2))
        m = rng.random((B, 1, 1, T)) < 0.7
        for mask in (None, m):
            ref = O.sdpa(f(q), f(k), f(v), D ** -0.5, mask=mask, q_dtype=dtype)
            got = vkv.scaled_dot_product_attention(
                dev(q, dtype), dev(k, dtype), dev(v, dtype), D ** -0.5,
                mask=None if mask is None else torch.from_numpy(mask).cuda())
            assert_within(values(got, dtype), ref, attn_tol(dtype, ref), f"T {T}")


@pytest.mark.parametrize("Hq,Hkv,D", [(32, 8, 128), (64, 8, 128), (12, 1, 64), (16, 2, 256)])
def test_a_step_writes_its_token_once_for_all_head_groups(Hq, Hkv, D):
    """Decode steps through a cache: the token that the decode launch writes is
    read by every head group of its kv head and is in the cache afterwards."""
    torch.manual_seed(Hq + D)
    T, c = 30, vkv.KVCacheSimple()
    k, v = (torch.randn((2, Hkv, T + 4, D), device="cuda").bfloat16() for _ in range(2))
    c.update(k[:, :, :T].contiguous(), v[:, :, :T].contiguous())
    for t in range(T, T + 4):
        q = torch.randn((2, Hq, 1, D), device="cuda").bfloat16()
        out = vkv.attention_with_cache_update(q, k[:, :, t:t + 1].contiguous(),
                                              v[:, :, t:t + 1].contiguous(), c, D ** -0.5)
        n = lambda x: x.float().cpu().numpy()
        ref = O.sdpa(n(q), n(k[:, :, :t + 1]), n(v[:, :, :t + 1]), D ** -0.5, q_dtype=O.BF16)
        assert_within(n(out), ref, attn_tol(O.BF16, ref), f"step {t}")
    for got, want in zip(c.state, (k, v)):
        assert torch.equal(vkv.to_torch(got) if not torch.is_tensor(got) else got, want)


@pytest.mark.parametrize("Hq,Hkv,D,L,T", [(8, 8, 128, 4, 1024), (16, 8, 256, 4, 1024),
                                          (32, 8, 64, 2, 1024), (24, 8, 128, 3, 1024)])
def test_little_masked_chunks_take_the_generic_kernel(Hq, Hkv, D, L, T, monkeypatch):
    """The longest rows of chunks that the generic kernel takes, bit for bit;
    with one key more they are packed, and agree with the oracle."""
    rng = np.random.default_rng(D + L + T)
    f = lambda a: O.to_f32(a, O.BF16)
    for n in (T, T + 1):
        q = rand_bits(rng, (1, Hq, L, D), O.BF16)
        k, v = (rand_bits(rng, (1, Hkv, n, D), O.BF16) for _ in range(2))
        m = rng.random((L, n)) < 0.6
        run = lambda: values(vkv.scaled_dot_product_attention(
            *(dev(x, O.BF16) for x in (q, k, v)), D ** -0.5, mask=torch.from_numpy(m).cuda()), O.BF16)
        monkeypatch.setattr(OPTIONS, "generic_attention", 0)
        got = run()
        ref = O.sdpa(f(q), f(k), f(v), D ** -0.5, mask=m, q_dtype=O.BF16)
        assert_within(got, ref, attn_tol(O.BF16, ref), f"T {n}")
        monkeypatch.setattr(OPTIONS, "generic_attention", 1)
        if n == T:
            assert np.array_equal(got, run())


@pytest.mark.parametrize("bits,D", [(4, 128), (8, 64), (8, 256)])
def test_masked_quantized_chunks_attend_what_causal_ones_do(bits, D):
    """K and V dequantized and rounded to the dtype: the causal mask as an array
    gives the causal mode's output (up to the order of the merge: one unit)."""
    torch.manual_seed(bits + D)
    B, Hq, Hkv, L, T = 2, 8, 4, 48, 300
    q = torch.randn((B, Hq, L, D), device="cuda").bfloat16()
    k, v = (vkv.quantized(torch.randn((B, Hkv, T, D), device="cuda").bfloat16(), 64, bits) for _ in range(2))
    m = torch.ones((L, T), dtype=torch.bool, device="cuda").tril(T - L)
    run = lambda mask: vkv.quantized_scaled_dot_product_attention(
        q, k, v, D ** -0.5, mask=mask, group_size=64, bits=bits).float().cpu().numpy()
    a, b = run(m), run("causal")
    assert_within(a, b, 2.0 ** -8 * np.abs(b) + 1e-6, "causal")
