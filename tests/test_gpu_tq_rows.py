"""TurboQuant's row kernels (head dims 64, 128, 256) where they can go wrong:
partial tiles of 32 vectors, vectors of zeros, of tiny and of huge
values (the division by reciprocal gives way to the true one) and of values
that cancel in the rotation.  Codes, signs, norms and decoded values equal the
oracle's bit for bit."""
import numpy as np
import pytest
import torch

import oracle as O
import vkv
from gpu_util import values
from test_gpu_turboquant import _check_record, _simple, _state

pytestmark = pytest.mark.gpu


def _bits(x, dtype):
    if dtype == O.F32:
        return x.astype(np.float32)
    return O.from_f32(x.astype(np.float32), dtype)


def _vectors(rng, B, H, T, D, dtype, kind):
    x = rng.standard_normal((B, H, T, D)).astype(np.float32)
    if kind == "scales":  # bf16 / f32: from denormal squares to norms past 2^20
        low, top = (-4, 5) if dtype == O.F16 else (-110, 30)
        x *= np.exp2(rng.integers(low, top, (B, H, T, 1))).astype(np.float32)
    elif kind == "sparse":  # zeros, equal magnitudes that cancel, one tiny value
        x = np.where(rng.random(x.shape) < 0.5, 0.0, np.sign(x)).astype(np.float32)
        x[..., 3] *= np.float32(6e-5 if dtype == O.F16 else 2.0 ** -104)
        if dtype != O.F16:  # (f16's divisor of a zero vector is zero)
            x[:, :, ::3] = 0.0
    return x


def _same(t, want, dtype):
    # a norm past 65504 is stored infinite (f16): its product with a zero
    # coordinate is NaN, here and in the oracle
    assert {torch.float16: O.F16, torch.float32: O.F32, torch.bfloat16: O.BF16}[t.dtype] == dtype
    assert np.array_equal(values(t, dtype), want, equal_nan=True)


@pytest.mark.parametrize("kind", ["normal", "scales", "sparse"])
@pytest.mark.parametrize("dtype", [O.BF16, O.F16, O.F32])
@pytest.mark.parametrize("B,H,T,D,kb,vb", [(1, 1, 8, 128, 3, 3), (1, 1, 31, 64, 4, 2), (1, 3, 11, 128, 3, 4),
                                           (1, 1, 65, 256, 5, 3), (2, 2, 17, 256, 4, 8)])
def test_edges_match_the_oracle_bit_for_bit(B, H, T, D, kb, vb, dtype, kind):
    rng = np.random.default_rng(1000 * D + T)
    k, v = (_bits(_vectors(rng, B, H, T, D, dtype, kind), dtype) for _ in range(2))
    tq = vkv.TurboQuantKVCache.from_simple_cache(_simple(k, v, dtype), kb, vb, 0, 0)
    st = _state(D, kb, vb)
    f = (lambda x: x) if dtype == O.F32 else (lambda x: O.to_f32(x, dtype))
    ek, ev = O.tq_encode(f(k), dtype, st, True, 0, 0), O.tq_encode(f(v), dtype, st, False, 0, 0)
    gk, gv = tq.encoded()
    _check_record(gk, ek, True, dtype)
    _check_record(gv, ev, False, dtype)
    sk, sv = tq.state
    _same(sk, *O.tq_decode(ek, st, True))
    _same(sv, *O.tq_decode(ev, st, False))
