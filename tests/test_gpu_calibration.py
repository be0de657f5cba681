"""The calibration collectors' device reductions against numpy: extreme values and histogram
counts are the same numbers, at the edges of the vector loads, of the LDS bins and of the bins
themselves."""
import numpy as np
import pytest
import torch

from mxnet_amd import capi
from mxnet_amd import quantization as Q

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 4, 5, 1023, 4097, 100003])
@pytest.mark.parametrize("offset", [0, 1])
def test_minmax(n, offset):
    x = np.random.default_rng(n).standard_normal(n + offset).astype(np.float32)
    got = capi.minmax(torch.from_numpy(x).cuda()[offset:]).cpu().numpy()
    assert tuple(got) == (x[offset:].min(), x[offset:].max())


def test_minmax_nan():
    x = torch.randn(1000, device="cuda")
    x[777] = float("nan")
    assert torch.isnan(capi.minmax(x)).all()


@pytest.mark.parametrize("n", [1, 511, 513, 70001, 1 << 20])
@pytest.mark.parametrize("bins", [1, 2, 255, 8001, 16384, 16385, 30001])
def test_histogram_counts_as_numpy(n, bins):
    rng = np.random.default_rng(n + bins)
    x = rng.standard_normal(n).astype(np.float32)
    x[:: 3] = np.maximum(x[:: 3], 0)
    th = np.max(np.abs(x)) * np.float32(0.9 if n % 2 else 1.0)  # values outside, too
    got = Q._Values(torch.from_numpy(x).cuda()).counts(bins, th)
    assert np.array_equal(got, np.histogram(x, bins=bins, range=(-th, th))[0])


def test_histogram_of_values_on_the_edges():
    edges = np.linspace(-2, 2, 8002).astype(np.float32)
    x = np.concatenate([edges, np.nextafter(edges, np.float32(9)),
                        np.nextafter(edges, np.float32(-9)), [np.nan]]).astype(np.float32)
    got = capi.histogram(torch.from_numpy(x).cuda(), torch.from_numpy(edges).cuda())
    inside = x[(x >= edges[0]) & (x <= edges[-1])]
    at = np.minimum(np.searchsorted(edges, inside, side="right") - 1, 8000)
    assert np.array_equal(got.cpu().numpy(), np.bincount(at, minlength=8001))


def test_collector_on_device_tensors_is_the_host_collector():
    rng = np.random.default_rng(1)
    batches = [rng.standard_normal((64, 33)).astype(np.float32) * s for s in (1.0, 3.0, 0.5)]
    on_host, on_device = (Q._LayerHistogramCollector("int8", include_layers=["t"])
                          for _ in range(2))
    for b in batches:
        on_host.collect("t", "op", b)
        on_device.collect("t", "op", torch.from_numpy(b).cuda())
    for h, d in zip(on_host.hist_dict["t"], on_device.hist_dict["t"]):
        assert np.array_equal(h, d)
    assert on_host.post_collect() == on_device.post_collect()


@pytest.mark.parametrize("bins", [1, 2, 255, 8001, 16384, 20001])
@pytest.mark.parametrize("th", [None, 1e-33, 0.7, 1.6e38])  # bins of normal width: numpy has no others
def test_symmetric_histogram_is_the_two_calls(bins, th):
    """Values on numpy's edges and beside them, so that an edge one last place off would show."""
    top = np.float32(2.7 if th is None else th)
    edges = np.histogram_bin_edges(np.empty(0, np.float32), bins=bins, range=(-top, top))
    assert edges.dtype == np.float32
    x = np.concatenate([edges, np.nextafter(edges, np.float32(0)), edges[::3] * np.float32(0.3)])
    if th is not None and top < 1e38:
        x = np.append(x, 2 * top).astype(np.float32)
    v = Q._Values(torch.from_numpy(x).cuda())
    v.measure(bins, None if th is None else top)
    assert v.extremes() == (x.min(), x.max())
    assert v._counts is not None
    got = v.counts(bins, top)
    assert np.array_equal(got, Q._Values(torch.from_numpy(x).cuda()).counts(bins, top))
    assert np.array_equal(got, np.histogram(x, bins=bins, range=(-top, top))[0])


@pytest.mark.parametrize("value", [0.0, float("nan"), float("inf")])
def test_symmetric_histogram_without_a_range(value):
    x = torch.full((1000,), value, device="cuda")
    v = Q._Values(x)
    v.measure(101)
    assert v._counts is None
    lo, hi = v.extremes()
    assert (np.isnan(lo) and np.isnan(hi)) if np.isnan(value) else (lo, hi) == (value, value)


@pytest.mark.parametrize("bins", [101, 8001, 20001])
@pytest.mark.parametrize("value, th", [(0.0, None), (1e-44, None), (0.5, np.float32(0)),
                                       (0.5, np.float32(1e-44))])
def test_nothing_is_counted_without_edges(bins, value, th):
    """Edges that do not increase: looking for a bin between them would walk through all of them, so
    no value is looked at."""
    x = torch.full((70001,), value, device="cuda")
    x[::2] *= -1
    found = capi.symmetric_histogram(x, bins, th).cpu().numpy()
    assert tuple(found[:2].view(np.float32)) == (-np.float32(value), np.float32(value))
    assert found[2] == 0 and not found[3:].any()


@pytest.mark.parametrize("bins", [101, 8001, 20001])
@pytest.mark.parametrize("value, counted", [(0.5, True), (np.nextafter(np.float32(0.5), 1), False),
                                            (-0.6, False), (np.inf, False)])
def test_nothing_is_counted_of_a_batch_that_reaches_further(bins, value, counted):
    x = np.random.default_rng(bins).uniform(-0.5, 0.5, 70001).astype(np.float32)
    x[777] = value
    t = torch.from_numpy(x).cuda()
    found = capi.symmetric_histogram(t, bins, np.float32(0.5), inside=True).cpu().numpy()
    assert tuple(found[:2].view(np.float32)) == (x.min(), x.max())
    assert found[2] == counted
    plain = capi.symmetric_histogram(t, bins, np.float32(0.5)).cpu().numpy()
    assert plain[2] == 1 and plain[3:].sum() == 70001 - (not counted)
    assert np.array_equal(found[3:], plain[3:] if counted else 0 * plain[3:])
