"""The host's side of the calibration collectors' device histograms, without a GPU."""
import numpy as np
import torch

from mxnet_amd import capi
from mxnet_amd import quantization as Q


def edges_of_numpy_1(a, bins, range):
    """numpy.histogram_bin_edges as it was with its former rules of promotion: in float64."""
    lo, hi = (float(v) for v in range)
    edges = np.arange(bins + 1, dtype=np.float64) * ((hi - lo) / bins) + lo
    edges[-1] = hi
    return edges.astype(np.result_type(a.dtype, np.float32))


def test_edges_of_the_installed_numpy_are_looked_at(monkeypatch):
    made = Q._edges_in_float32()
    assert made == (int(np.__version__.split(".")[0]) >= 2) == Q._EDGES_IN_FLOAT32
    monkeypatch.setattr(np, "histogram_bin_edges", edges_of_numpy_1)
    assert not Q._edges_in_float32()


def test_edges_that_numpy_makes_otherwise_come_from_numpy(monkeypatch):
    x = torch.linspace(-2.7, 2.7, 30001)
    values = Q._Values(x)
    values._device = x  # as a tensor on the device
    monkeypatch.setattr(Q, "_EDGES_IN_FLOAT32", False)
    monkeypatch.setattr(np, "histogram_bin_edges", edges_of_numpy_1)

    def not_asked(*args):
        raise AssertionError("edges in float32")

    monkeypatch.setattr(capi, "symmetric_histogram", not_asked)
    asked = []

    def histogram(data, edges):
        asked.append(edges.numpy())
        return torch.zeros(len(edges) - 1, dtype=torch.int32)

    monkeypatch.setattr(capi, "histogram", histogram)
    th = np.float32(2.7)
    values.measure(8001)
    values.measure(8001, th)
    values.counts(8001, th)
    want = edges_of_numpy_1(np.empty(0, np.float32), 8001, (-th, th))
    assert len(asked) == 1 and np.array_equal(asked[0], want)
