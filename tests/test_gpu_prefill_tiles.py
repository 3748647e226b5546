"""Chunks whose key range is 1 to 9 tiles of 32 keys, the last one partial or
whole: the edges of the tile loop (the first and last steps of the staggered
wave groups, the unrolled part of four tiles and its remainder, the masked
tiles behind the open ones), against the oracle with the tolerance of the
other chunk tests."""
import numpy as np
import pytest

import oracle as O
from test_gpu_prefill import run_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 128, 256])
@pytest.mark.parametrize("mask", [None, "causal"])
@pytest.mark.parametrize("T", [32, 33, 64, 95, 128, 130, 160, 191, 224, 256, 288])
def test_tile_counts(T, mask, D):
    rng = np.random.default_rng(1000 + T + D)
    run_case(rng, O.BF16 if T % 2 else O.F16, 1, 8, 2, 20, T, mask, D=D)
