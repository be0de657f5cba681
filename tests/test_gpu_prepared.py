"""Layers with what they derive from constant ranges computed once (mxq_prepare_layer): the same
bytes as the calls that compute it themselves, on every kind of kernel the choosers take, with and
without a bias."""
import pytest
import torch

from mxnet_amd import _lib, capi

pytestmark = pytest.mark.gpu


def scalars(*v):
    return [torch.tensor([x], dtype=torch.float32, device="cuda") for x in v]


def stream():
    return torch.cuda.current_stream().cuda_stream


def draw(g, *shape):
    return torch.randint(-128, 128, shape, device="cuda", generator=g, dtype=torch.int8)


def prepare(bias, n, ranges, calib):
    out = torch.full((64 + 4 * n,), 77, dtype=torch.int8, device="cuda")
    at = [None if r is None else r.data_ptr() for r in ranges]
    _lib.check(_lib.lib.mxq_prepare_layer(stream(), None if bias is None else bias.data_ptr(), n,
                                          *at, *calib, out.data_ptr()))
    return out


def setting(g, n, with_bias):
    bias = draw(g, n) if with_bias else None
    ranges = scalars(-1.0, 0.9, -2.0, 2.1) + (scalars(-40.0, 39.0) if with_bias else [None, None])
    return bias, ranges


@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("m,n,k", [
    (1, 16, 16), (49, 512, 2048), (300, 48, 64), (8193, 512, 64),   # few tiles, streamed
    (1024, 1024, 1024), (2048, 768, 768), (130, 33, 96), (513, 70, 45)])
def test_fully_connected(m, n, k, with_bias):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    data, weight, res = draw(g, m, k), draw(g, n, k), draw(g, m, n)
    bias, ranges = setting(g, n, with_bias)
    calib = (-2.0 * k ** 0.5, 1.9 * k ** 0.5)
    ready = prepare(bias, n, ranges, calib)
    ws_bytes = _lib.lib.mxq_quantized_fc_workspace(m, n, k, 1)
    ws = torch.zeros(max(ws_bytes, 16), dtype=torch.uint8, device="cuda")
    head = [stream(), data.data_ptr(), weight.data_ptr(), ready.data_ptr(), m, n, k]
    tail = [ws.data_ptr(), ws_bytes]
    for relu in (0, 1):
        want = capi.quantized_fc(data, weight, bias, *ranges, want_int32=False, calib=calib,
                                 relu=bool(relu))["out8"]
        got = torch.empty_like(want)
        _lib.check(_lib.lib.mxq_quantized_fc_prepared(*head, got.data_ptr(), None, relu, *calib,
                                                      *tail))
        assert torch.equal(got, want)
        want = capi.quantized_fc_f32(data, weight, bias, *ranges, calib=calib,
                                     relu=bool(relu))["outf"]
        got = torch.empty_like(want)
        _lib.check(_lib.lib.mxq_quantized_fc_prepared(*head, None, got.data_ptr(), relu, *calib,
                                                      *tail))
        assert torch.equal(got, want)
    res_range = scalars(-2.0, 2.0)
    for requant in (0, 1):
        want = capi.quantized_fc_sum(data, weight, bias, res, *ranges, *res_range, calib,
                                     (-4.0, 4.0), sum_relu=True, requant=bool(requant))["out8"]
        pairs = capi.sum_requant_pairs(calib, (-2.0, 2.0), (-4.0, 4.0))
        got = torch.empty_like(want)
        _lib.check(_lib.lib.mxq_quantized_fc_sum_prepared(
            *head, res.data_ptr(), res_range[0].data_ptr(), res_range[1].data_ptr(),
            got.data_ptr(), *calib, -4.0, 4.0, 1, requant, pairs.data_ptr(), *tail))
        assert torch.equal(got, want)


@pytest.mark.parametrize("with_bias", [False, True])
@pytest.mark.parametrize("n,h,w,c,o,k,s", [
    (16, 56, 56, 64, 64, 3, 1), (48, 28, 28, 128, 128, 3, 1),   # weights / patch kept in LDS
    (8, 60, 61, 16, 48, 4, 1), (1, 7, 7, 512, 64, 3, 1),        # few taps, few tiles
    (8, 14, 14, 256, 256, 3, 1), (2, 9, 9, 48, 20, 3, 2), (4, 20, 20, 22, 30, 3, 1),
    (8, 28, 28, 128, 64, 1, 2), (8, 14, 14, 64, 128, 1, 1)])
def test_convolution(n, h, w, c, o, k, s, with_bias):
    g = torch.Generator(device="cuda").manual_seed(c + o)
    data, weight = draw(g, n, h, w, c), draw(g, o, k, k, c)
    bias, ranges = setting(g, o, with_bias)
    calib = (-2.0 * c ** 0.5 * k, 1.9 * c ** 0.5 * k)
    ready = prepare(bias, o, ranges, calib)
    geo = (n, h, w, c, o, k, k, s, s, k // 2, k // 2, 1, 1)
    ws_bytes = _lib.lib.mxq_quantized_conv_workspace(*geo, 1)
    ws = torch.zeros(max(ws_bytes, 16), dtype=torch.uint8, device="cuda")
    for relu in (0, 1):
        want = capi.quantized_conv_nhwc(data, weight, bias, *ranges, stride=(s, s),
                                        pad=(k // 2, k // 2), want_int32=False, calib=calib,
                                        relu=bool(relu))["out8"]
        got = torch.empty_like(want)
        _lib.check(_lib.lib.mxq_quantized_conv_nhwc_prepared(
            stream(), data.data_ptr(), weight.data_ptr(), ready.data_ptr(), *geo, got.data_ptr(),
            relu, *calib, ws.data_ptr(), ws_bytes))
        assert torch.equal(got, want)
