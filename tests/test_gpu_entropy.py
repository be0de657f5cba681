"""The entropy calibration's bounds from the GPU: they hold for what the definition's float sums
give, candidate by candidate, and the search that starts from them is the host's own search."""
import time

import numpy as np
import pytest
import torch

from mxnet_amd import capi
from mxnet_amd import quantization as Q
from test_calibrate_entropy import _libm, running_sum, smooth

pytestmark = pytest.mark.gpu

f32 = np.float32
KINDS = ["gaps", "one_sided", "large", "fractions", "flat", "few"]


def histogram(kind, bins, rng):
    x = np.abs(np.arange(bins) - bins // 2) / (bins / 8)
    if kind == "gaps":  # runs of empty bins, a few values far out
        h = np.floor(3000 * np.exp(-x * x)) * (rng.random(bins) < 0.7)
        h[[0, bins // 9, bins - 2]] = 1, 3, 2
    elif kind == "one_sided":
        h = np.floor(50 * rng.random(bins) / (1 + x ** 4)) * (np.arange(bins) > bins // 2)
    elif kind == "large":  # past 2^24 in all: the order of the edge entries' sums counts
        h = np.floor(2e5 * rng.random(bins) * np.exp(-x))
    elif kind == "fractions":
        h = 40 * rng.random(bins) * np.exp(-x) * (rng.random(bins) < 0.9)
    elif kind == "flat":
        h = np.full(bins, 7.0)
    elif kind == "few":  # no narrow candidate has a quantized distribution
        h = np.zeros(bins)
        h[bins // 2 + 40] = 9
    return h.astype(f32)


def divergence(hist, i, levels):
    """None: the definition has none (its logarithm's argument is not positive)."""
    zero = len(hist) // 2
    start, stop = zero - i, zero + i + 1
    p = hist[start:stop].copy()
    sliced = hist[start:stop].astype(np.int64)
    sliced[0] = 0
    p[0] = running_sum(hist[:start + 1])
    p[-1] = running_sum(hist[stop:], p[-1])
    merged = len(p) // levels
    q = np.zeros(len(p), f32)
    for j in range(levels):
        lo, end = j * merged, len(p) if j == levels - 1 else (j + 1) * merged
        level = f32(sliced[lo:lo + merged].sum())
        if j == levels - 1:
            level = f32(level + f32(sliced[lo + merged:].sum()))
        filled = int((sliced[lo:end] != 0).sum())
        if filled:
            q[lo:end] = np.where(p[lo:end] != 0, level / f32(filled), 0)
    ps, qs = smooth(p), smooth(q)
    if qs is None:
        return np.inf
    if ps is None:
        return None
    ps, qs = ps / running_sum(ps), qs / running_sum(qs)
    if not ((ps > 0).all() and (qs > 0).all()):
        return None
    return running_sum(ps * np.array([_libm.logf(r) for r in (ps / qs).astype(f32)], f32))


@pytest.mark.parametrize("levels", [3, 64, 255, 511])
@pytest.mark.parametrize("kind", KINDS)
def test_bounds_hold(kind, levels):
    h = histogram(kind, 1601, np.random.default_rng(7))
    bounds = capi.entropy_bounds([h], [levels])
    half, zero = levels // 2, 800
    assert bounds.shape == (zero + 1 - half, 2)
    for i in [*range(half, zero, 17), zero]:
        lower, upper = bounds[i - half]
        exact = divergence(h, i, levels)
        if exact is None:
            assert (lower, upper) == (-np.inf, np.inf)
        elif np.isinf(exact):
            assert lower == upper == np.inf
        else:
            assert lower <= exact <= upper
            # a rounding of the largest running sum per bin, each way, and a few of the terms
            assert upper - lower <= 2 ** -23 * 1.1 * (2 * i + 12) * max(1.0, 2 * abs(exact))


@pytest.mark.parametrize("levels", [3, 64, 255, 511])
@pytest.mark.parametrize("kind", KINDS)
def test_search_is_the_host_search(kind, levels, monkeypatch):
    rng = np.random.default_rng(levels)
    sizes = [511, 513, 1023, 4001, 8001] + [601] * 14  # more than one call takes
    problems = [(histogram(kind, n, rng), np.linspace(-3, 3, n + 1).astype(f32), levels)
                for n in sizes]
    good, want = [], []
    for p in problems:
        with monkeypatch.context() as m:
            m.setattr(Q, "_entropy_bounds", lambda hists, levels: None)
            try:
                want.append(Q._calibrate_entropy_many([p])[0])
                good.append(p)
                continue
            except Exception as e:
                kind_of_error, text = type(e), str(e)
        with pytest.raises(kind_of_error) as raised:
            Q._calibrate_entropy_many([p])
        assert str(raised.value).splitlines()[-1] == text.splitlines()[-1]
    assert [Q._calibrate_entropy_many([p])[0] for p in good] == want
    assert Q._calibrate_entropy_many(good) == want


def test_what_stays_on_the_host():
    good = np.ones(601, f32)
    assert Q._entropy_bounds([good], [255]) is not None
    assert Q._entropy_bounds([], []) is None
    for h, levels in ((good[1:], 255), (good, 2), (good, 602), (-good, 255),
                      (np.full(601, np.nan, f32), 255), (np.full(601, np.inf, f32), 255),
                      (np.full(601, 2.0 ** 23, f32), 255), (np.ones(32769, f32), 255)):
        assert Q._entropy_bounds([good, h], [255, levels]) is None
    assert Q._entropy_bounds([np.ones(32767, f32)], [255]).shape == (16384 - 127, 2)


def test_histograms_that_are_not_exact_take_no_round_trip_a_bin():
    """Counts of 2^24 and more are added up in the order of the bins: with reads ahead of the
    additions a quarter more than an exact histogram takes, with an access at a time three times
    as much."""
    bins = 8001
    x = np.arange(bins) - bins // 2
    exact = np.floor(60 * np.exp(-(x / 1200.0) ** 2)).astype(f32)
    took = []
    for h in (exact, exact * f32(5000)):
        runs = []
        for _ in range(8):
            torch.cuda.synchronize()
            start = time.perf_counter()
            capi.entropy_bounds([h], [255])
            runs.append(time.perf_counter() - start)
        took.append(min(runs))
    assert took[1] < 1.8 * took[0], took


@pytest.mark.parametrize("bins,count,device", [([201, 201], 30, True), ([201], 30, False),
                                               ([227], 30, False), ([229], 30, True)])
def test_few_candidates_stay_on_the_host(bins, count, device):
    """99 candidates and fewer, in all: the host's threads are through before the launches are."""
    found = Q._entropy_bounds([np.ones(b, f32) for b in bins], [count] * len(bins))
    assert (found is not None) == device


@pytest.mark.parametrize("room", [1, 3 << 20, 1 << 30])
def test_histograms_beyond_a_workspace_take_further_calls(room, monkeypatch):
    rng = np.random.default_rng(room)
    hists = [histogram(KINDS[i % len(KINDS)], 401 + 200 * i, rng) for i in range(11)]
    levels = [255, 3, 64] * 3 + [31, 401]
    want = np.concatenate([capi.entropy_bounds([h], [n]) for h, n in zip(hists, levels)])
    calls, run = [], capi.lib.mxq_entropy_bounds

    def bounds(stream, count, *args):
        calls.append((count, args[-1]))
        return run(stream, count, *args)

    monkeypatch.setattr(capi, "_ENTROPY_WS_BYTES", room)
    monkeypatch.setattr(capi.lib, "mxq_entropy_bounds", bounds)
    assert np.array_equal(capi.entropy_bounds(hists, levels), want)
    assert all(count == 1 or size <= room for count, size in calls)
    assert len(calls) == (11 if room == 1 else 1) or 1 < len(calls) < 11
