"""Attention sinks of -inf and of the type's lowest value (a logit that adds
nothing) where the first keys a kernel takes are hidden: the running max has
no finite value yet.  One-token decodes and prompt chunks, bool and additive
masks, the float-decode, matrix-core and generic kernels, against the oracle.
NaN keys in one-token decodes."""
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
