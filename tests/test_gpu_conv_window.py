"""The convolution over 16 channels whose window and pixels are resident in LDS, against float64 products (exact
for these lengths) and, requantized, against the smallest tile pinned."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import mxnet_amd
    return mxnet_amd.capi


# images, rows, columns, channels out, window, stride, padding, dilation: tiles that pass from image to image,
# rows shorter and longer than a tile, one pixel out, odd taps, windows as large as the image
GEOMETRIES = [(1, 7, 7, 8, (3, 3), (1, 1), (1, 1), (1, 1)), (9, 5, 6, 33, (3, 3), (1, 1), (1, 1), (1, 1)),
              (3, 51, 51, 12, (7, 7), (1, 1), (3, 3), (1, 1)), (2, 33, 140, 70, (5, 5), (1, 1), (2, 2), (1, 1)),
              (5, 29, 30, 64, (5, 5), (2, 2), (2, 2), (1, 1)), (4, 40, 17, 27, (3, 5), (2, 1), (0, 2), (1, 2)),
              (7, 9, 9, 31, (6, 6), (1, 1), (0, 0), (1, 1)), (13, 8, 8, 40, (5, 5), (2, 2), (2, 2), (1, 1)),
              (2, 64, 3, 96, (2, 1), (1, 1), (0, 0), (1, 1)), (300, 3, 3, 16, (3, 3), (1, 1), (0, 0), (1, 1)),
              (40, 4, 4, 65, (3, 3), (4, 4), (2, 2), (1, 1)), (2, 30, 31, 20, (3, 3), (1, 1), (2, 2), (2, 2))]


@pytest.mark.parametrize("n,h,w,o,window,stride,pad,dilate", GEOMETRIES)
def test_every_tile(capi, n, h, w, o, window, stride, pad, dilate):
    g = torch.Generator(device="cuda").manual_seed(n * h + w)
    d = torch.randint(-128, 128, (n, h, w, 16), dtype=torch.int8, device="cuda", generator=g)
    k = torch.randint(-128, 128, (o,) + window + (16,), dtype=torch.int8, device="cuda", generator=g)
    ranges = [torch.tensor([v], device="cuda") for v in (-1.0, 1.0, -0.1, 0.1)]
    want = torch.nn.functional.conv2d(d.permute(0, 3, 1, 2).double().cpu(), k.permute(0, 3, 1, 2).double().cpu(),
                                      stride=stride, padding=pad, dilation=dilate)
    kw = dict(stride=stride, pad=pad, dilate=dilate)
    for cfg in (None, 66, 67):
        force = None if cfg is None else (cfg, 1)
        got = capi.quantized_conv_nhwc(d, k, None, *ranges, want_int32=True, force=force, **kw)["out32"]
        assert torch.equal(got.permute(0, 3, 1, 2).double().cpu(), want), cfg
        for relu in (False, True):
            fused = dict(want_int32=False, calib=(-2.0, 2.0), relu=relu, **kw)
            assert torch.equal(capi.quantized_conv_nhwc(d, k, None, *ranges, force=force, **fused)["out8"],
                               capi.quantized_conv_nhwc(d, k, None, *ranges, force=(25, 1), **fused)["out8"]), cfg


# through the rule: the operator's int32 planes as well, rows that leave int8 rows ragged
@pytest.mark.parametrize("n,c,h,o,k,s", [(64, 16, 28, 29, 5, 1), (9, 3, 31, 87, 7, 1), (40, 11, 41, 24, 3, 1),
                                         (40, 16, 61, 13, 3, 1), (15, 16, 66, 75, 5, 1), (5, 8, 78, 88, 7, 2),
                                         (12, 16, 20, 108, 3, 1), (2, 16, 100, 33, 7, 1)])
def test_operator(capi, n, c, h, o, k, s):
    from mxnet_amd import contrib
    g = torch.Generator(device="cuda").manual_seed(n * h + o)
    d = torch.randint(-128, 128, (n, c, h, h), dtype=torch.int8, device="cuda", generator=g)
    w = torch.randint(-128, 128, (o, c, k, k), dtype=torch.int8, device="cuda", generator=g)
    ranges = [torch.tensor([v], device="cuda") for v in (-1.0, 1.0, -0.1, 0.1)]
    want = torch.nn.functional.conv2d(d.double().cpu(), w.double().cpu(), stride=s, padding=k // 2)
    acc = contrib.quantized_conv(d, w, None, *ranges, None, None, kernel=(k, k), stride=(s, s), pad=(k // 2, k // 2),
                                 num_filter=o, no_bias=True)[0]
    assert torch.equal(acc.double().cpu(), want)
    pixels = [x.permute(0, 2, 3, 1).contiguous() for x in (d, w)]
    got = capi.quantized_conv_nhwc(*pixels, None, *ranges, stride=(s, s), pad=(k // 2, k // 2), want_int32=True)
    assert torch.equal(got["out32"].permute(0, 3, 1, 2).double().cpu(), want)
