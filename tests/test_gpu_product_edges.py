"""Products at the edges of their kernels' tiles, k-tiles and slices, against
float64: integer operands small enough that every F32 sum is exact, so any
order gives the same bits, or random ones within a derived bound.
"""
import numpy as np
import pytest

import miburn
from miburn import bf16_bits, bf16_to_f32

pytestmark = pytest.mark.gpu

RNG = np.random.default_rng(41)


def _ints(shape, lo=-2, hi=3):
    return RNG.integers(lo, hi, shape).astype(np.float32)


@pytest.mark.parametrize("m,n,k", [(640, 320, 4000), (64, 64, 2080), (128, 192, 1056)])
def test_bf16_split_k_of_a_half_k_tile(engine, m, n, k):
    """k a multiple of 32 and not of the 64-wide k-tile, split over k: the last
    slice ends inside its k-tile and reads nothing past it."""
    a, b = _ints((m, k)), _ints((k, n))
    ia, ib = engine.upload_bf16(bf16_bits(a)), engine.upload_bf16(bf16_bits(b))
    o = engine.matmul_dram(ia, False, ib, False)
    got = engine.download(o)
    for t in (ia, ib, o):
        engine.free(t)
    assert np.array_equal(got, (a.astype(np.float64) @ b).astype(np.float32))
