"""Candidates whose levels are of every length that a chain of 16 bins at a time tells apart: none to
three pieces of 16 and every rest, all lanes alike, some lanes a bin longer, or (few levels) neither."""
import numpy as np
import pytest

from mxnet_amd import capi
from test_gpu_entropy import divergence, histogram

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["gaps", "fractions", "large"])
@pytest.mark.parametrize("levels,bins", [(3, 257), (40, 2049), (130, 8001), (255, 8191)])
def test_bounds_hold_at_every_length(kind, levels, bins):
    h = histogram(kind, bins, np.random.default_rng(levels))
    half, zero = levels // 2, bins // 2
    bounds = capi.entropy_bounds([h], [levels])
    for i in sorted({*range(half, zero, max(1, zero // 90)), zero - 1, zero}):
        lower, upper = bounds[i - half]
        exact = divergence(h, i, levels)
        if exact is None:
            assert (lower, upper) == (-np.inf, np.inf)
        elif np.isinf(exact):
            assert lower == upper == np.inf
        else:
            assert lower <= exact <= upper
            # a rounding of the largest running sum per bin, each way, and a few of the terms: a bin
            # more or less in a sum is past it
            assert upper - lower <= 2 ** -23 * 1.1 * (2 * i + 12) * max(1.0, 2 * abs(exact))
