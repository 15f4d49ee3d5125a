"""The momentum adjoint forms (1 + t) * tt in one fused operation with the addition that follows: the same bits as long as the
product is exact in 53 bits, 1 + t having at most 29."""
from fractions import Fraction

import pytest


@pytest.mark.parametrize("its", [2, 3, 10, 50, 100, 200, 1000])
def test_one_plus_every_step_size_has_at_most_29_bits(its):
    from customnetworklayers_amd.cudaTV import tvInpaint_cuda_ext as ext

    steps = ext.step_sizes(its)
    assert len(steps) == its and steps[0] == 0.0
    for t in steps:
        assert t == 0.0 or 0.25 <= t < 1.0
        assert (1 + Fraction(t)).numerator.bit_length() <= 29
