"""Uncalibrated casts of tensors that one work-group holds: the same bytes and ranges as the
reduction and cast of two launches, which unaligned data takes (its own parity with the oracle is
tested beside it)."""
import numpy as np
import pytest
import torch

from mxnet_amd import capi, contrib

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 3, 4, 5, 255, 256, 257, 1023, 4095, 4096, 4097, 4099, 16381, 16383, 16384, 16385]


def aligned(values):
    t = torch.empty(len(values) + 4, dtype=torch.from_numpy(values).dtype, device="cuda")
    assert t.data_ptr() % 16 == 0
    t[:len(values)] = torch.from_numpy(values)
    return t[:len(values)]


def unaligned(values):
    t = torch.empty(len(values) + 1, dtype=torch.from_numpy(values).dtype, device="cuda")
    t[1:] = torch.from_numpy(values)
    return t[1:]


def same(a, b):
    for x, y in zip(a, b):
        assert x.dtype == y.dtype
        x, y = x.cpu().numpy(), y.cpu().numpy()
        assert x.tobytes() == y.tobytes()


@pytest.mark.parametrize("special", [None, np.nan, np.inf, -np.inf, "zeros", "one value"])
@pytest.mark.parametrize("n", SIZES)
def test_float(n, special):
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n).astype(np.float32)
    if special == "zeros":  # of both signs
        x = np.copysign(np.float32(0), x)
    elif special == "one value":
        x[:] = -1.25
    elif special is not None:
        x[rng.integers(n)] = special
    for place in (0, n - 1):  # the extreme in the first or the last element
        if special is None:
            x[place] = 9 if place else -9
        for cast in (lambda v: capi.quantize_v2(v, "int8"), lambda v: capi.quantize_v2(v, "uint8"),
                     contrib.quantize_asym):
            same(cast(aligned(x)), cast(unaligned(x)))


@pytest.mark.parametrize("n", SIZES)
def test_int32(n):
    rng = np.random.default_rng(n)
    lo, hi = (torch.tensor([v], device="cuda") for v in (-3.5, 3.0))
    for limit in (5, 2 ** 31 - 1):
        x = rng.integers(-limit - 1, limit, n, endpoint=True).astype(np.int32)
        for place in (0, n - 1):
            x[place] = -limit - 1 if place else limit
            same(capi.requantize(aligned(x), lo, hi), capi.requantize(unaligned(x), lo, hi))
