"""Edges of the affine append and of the code gather: quantization by
reciprocal and corrections against the oracle's divisions on groups of equal
values, of one sign, near-tie codes, tiny and huge scales, scales with an
all-ones mantissa, infinities and NaN; 8-token value groups that are aligned,
ragged or split by a page; gathers of token windows at every offset."""
import numpy as np
import pytest
import torch

import oracle as O
import vkv
from gpu_util import dev, host

pytestmark = pytest.mark.gpu


def hard_rows(rng, n, D, bits, dtype):
    x = rng.standard_normal((n, D)).astype(np.float32)
    bins = (1 << bits) - 1
    for i in range(n):
        k = i % 8
        if k == 0:
            x[i] = x[i, 0]                                   # equal values
        elif k == 1:
            x[i] = np.abs(x[i]) + 3                           # one sign
        elif k == 2:                                          # codes at ties
            x[i] = (rng.integers(0, bins + 1, D) + 0.5) * 0.25
            x[i, 0], x[i, 1] = 0.0, bins * 0.25
        elif k == 3:
            x[i] *= 1e-30 if dtype == O.F32 else 1e-4         # tiny
        elif k == 4 and dtype != O.F16:
            x[i] *= 1e37                                      # huge
        elif k == 5:                                          # all-ones scale mantissa
            s = np.uint32(0x3EFFFFFF + (rng.integers(0, 8) << 23)).view(np.float32)
            x[i] = rng.uniform(0, 1, D) * s * bins
            x[i, 0], x[i, 1] = 0.0, s * bins
        elif k == 6:
            x[i, 3] = 0.0
            x[i, 4:] = -np.abs(x[i, 4:])
    return O.from_f32(x, dtype) if dtype != O.F32 else x


@pytest.mark.parametrize("group", [32, 64, 128])
@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("dtype", [O.BF16, O.F16, O.F32])
def test_hard_groups_bit_exact(dtype, bits, group):
    rng = np.random.default_rng(bits + group + dtype)
    x = hard_rows(rng, 4096, 128, bits, dtype)
    wq, s, b, _ = O.quantize(x, dtype, group, bits)
    g = vkv.quantized(dev(x, dtype), group, bits)
    assert np.array_equal(host(g[0]), wq.view(np.uint32).reshape(host(g[0]).shape))
    for got, want in zip(g[1:], (s, b)):
        assert np.array_equal(host(got).view(np.uint16 if dtype != O.F32 else np.uint32),
                              np.asarray(want).view(np.uint16 if dtype != O.F32 else np.uint32))


@pytest.mark.parametrize("bits", [4, 8])
def test_infinities_and_nan_follow_the_division(bits):
    """A wave with such a group divides, as all groups did: the codes equal
    the formula's in fp32."""
    rng = np.random.default_rng(bits)
    x = rng.standard_normal((64, 64)).astype(np.float32)
    x[3, 5], x[9, 0], x[17, 63], x[30, 1] = np.inf, -np.inf, np.nan, np.inf
    x[30, 2] = -np.inf
    n = np.float32((1 << bits) - 1)
    with np.errstate(all="ignore"):
        lo = np.fmin.reduce(x, 1, initial=np.float32(3.402823466e38))[:, None]
        hi = np.fmax.reduce(x, 1, initial=np.float32(0))[:, None]
        scale = np.fmax((hi - lo) / n, np.float32(1e-7))
        side = np.abs(lo) > np.abs(hi)
        scale = np.where(side, scale, -scale).astype(np.float32)
        edge = np.where(side, lo, hi)
        half = lambda t: np.sign(t) * np.floor(np.abs(t) + np.float32(0.5))
        q0 = half(edge / scale)
        z = q0 == 0
        scale = np.where(z, scale, edge / np.where(z, np.float32(1), q0)).astype(np.float32)
        bias = np.where(z, np.float32(0), edge)
        c = np.fmin(half((x - bias) / scale), n)
        c = np.where(c > 0, c, 0).astype(np.uint32)
    wq, _, _ = vkv.quantized(torch.from_numpy(x).cuda(), 64, bits)
    w = host(wq)
    got = np.stack([(w[:, i // (32 // bits)] >> np.uint32(bits * (i % (32 // bits)))) & np.uint32(n)
                    for i in range(64)], 1)
    keep = np.isfinite(x).all(1)
    assert np.array_equal(got[keep], c[keep])
    assert np.array_equal(got[[3, 9, 17, 30]], c[[3, 9, 17, 30]])


@pytest.mark.parametrize("bits", [4, 8])
@pytest.mark.parametrize("D,group,dtype", [(128, 64, O.BF16), (64, 32, O.F32), (256, 128, O.F16),
                                           (32, 32, O.BF16)])
def test_appends_and_code_windows(bits, D, group, dtype):
    """updateQuantized in pieces that leave value groups ragged, the tuples
    brought up to date in windows, the whole state, and toQuantized."""
    rng = np.random.default_rng(D + bits)
    B, H = 2, 3
    total = 0
    c = vkv.QuantizedKVCache(group_size=group, bits=bits)
    simple = vkv.KVCacheSimple()
    ks, vs = [], []
    for n in (5, 3, 8, 1, 1, 30, 17, 64):
        k, v = (rng.standard_normal((B, H, n, D)).astype(np.float32) for _ in range(2))
        k, v = ((O.from_f32(a, dtype) if dtype != O.F32 else a) for a in (k, v))
        ks.append(k)
        vs.append(v)
        tup = c.update_quantized_tuples(dev(k, dtype), dev(v, dtype))
        simple.update(dev(k, dtype), dev(v, dtype))
        total += n
        for got, rows in zip(tup, (ks, vs)):
            want = O.quantize(np.ascontiguousarray(np.concatenate(rows, 2)), dtype, group, bits)
            for a, w in zip(got, want[:3]):
                g = host(vkv.to_torch(a))
                assert np.array_equal(g.view(np.uint8), np.ascontiguousarray(w).view(np.uint8).reshape(
                    g.view(np.uint8).shape)), (total, n)
    for a, b in zip(c.state, simple.to_quantized(group, bits).state):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
