"""The few-tiles kernel and the padded copies in front of the tiled ones, at the sizes where they
can go wrong: rows and columns around the 32 x 32 tile, reductions around the 128-byte block and
the 16-byte piece, operands off every mark up to the last byte of their buffer.  Products are
exact in float64, so the int32 output is compared with one; the other outputs with the operators
behind it."""
import ctypes

import pytest
import torch

from mxnet_amd import _lib, capi

pytestmark = pytest.mark.gpu


def scalars(*v):
    return [torch.tensor([x], dtype=torch.float32, device="cuda") for x in v]


def int8(g, offset, *shape):
    """A tensor `offset` bytes into its buffer, whose last byte is the buffer's last."""
    n = 1
    for s in shape:
        n *= s
    flat = torch.randint(-128, 128, (n + offset,), device="cuda", generator=g, dtype=torch.int8)
    return flat[offset:].view(*shape)


def exact(x, w):
    return (x.double() @ w.double().t()).round().to(torch.int64).to(torch.int32)


RANGES = (-1.0, 1.0, -2.0, 2.0)


@pytest.mark.parametrize("waves", [0, 2, 4, 8, 16, -4, -8])
@pytest.mark.parametrize("m,n,k,off", [
    (1, 1, 16, 0), (1, 16, 17, 0), (31, 33, 127, 0), (32, 32, 128, 0), (33, 31, 129, 1),
    (65, 48, 256, 0), (3, 70, 45, 3), (17, 20, 1237, 5), (49, 64, 4096, 0), (64, 5, 2049, 2),
    (2, 130, 16, 1), (40, 40, 6160, 0)])
def test_products_and_epilogues(m, n, k, off, waves):
    g = torch.Generator(device="cuda").manual_seed(m * n + k)
    x, w, b = int8(g, off, m, k), int8(g, (off * 3) % 16, n, k), int8(g, 0, n)
    args = scalars(*RANGES)
    force = (71, waves, 0)
    plain = capi.quantized_fc(x, w, None, *args, force=force)
    assert torch.equal(plain["out32"], exact(x, w))
    bias = scalars(-0.5, 0.5)
    r = 3.0 * k ** 0.5
    for relu in (False, True):
        got = capi.quantized_fc(x, w, b, *args, *bias, calib=(-r, 0.5 * r), relu=relu, force=force)
        ref = capi.quantized_fc(x, w, b, *args, *bias, calib=(-r, 0.5 * r), relu=relu,
                                force=(4, 1, 0))
        for key in ("out32", "out8", "omin", "omax", "rmin", "rmax"):
            assert torch.equal(got[key], ref[key]), key
        f = capi.quantized_fc_f32(x, w, b, *args, *bias, calib=(-r, 0.5 * r), relu=relu,
                                  force=(71, waves))
        assert torch.equal(f["outf"], capi.dequantize(got["out8"], got["rmin"], got["rmax"]))
    res = int8(g, off, m, n)
    for requant in (False, True):
        sums = [capi.quantized_fc_sum(x, w, b, res, *args, *bias, *scalars(-2.0, 2.0), (-r, r),
                                      (-r, r), sum_relu=True, requant=requant, force=f)["out8"]
                for f in (force, (4, 1, 0))]
        assert torch.equal(*sums)


@pytest.mark.parametrize("m,n,k", [(257, 1024, 1237), (1024, 1024, 435), (1500, 520, 65),
                                   (4100, 260, 77), (700, 1100, 31)])
def test_unaligned_rows_of_many_tiles(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(k)
    x, w = int8(g, 1, m, k), int8(g, 7, n, k)
    got = capi.quantized_fc(x, w, None, *scalars(*RANGES), calib=(-50.0, 50.0))
    assert torch.equal(got["out32"], exact(x, w))
    want = capi.requantize(got["out32"], got["omin"], got["omax"], -50.0, 50.0)[0]
    assert torch.equal(got["out8"], want)
    only8 = capi.quantized_fc(x, w, None, *scalars(*RANGES), want_int32=False, calib=(-50.0, 50.0))
    assert torch.equal(only8["out8"], want)


def conv_exact(x, w, stride, pad, dilate):
    """NHWC int8 convolution as a float64 product of unfolded patches."""
    n, h, wd, c = x.shape
    o, kh, kw, _ = w.shape
    patches = torch.nn.functional.unfold(x.permute(0, 3, 1, 2).float(), (kh, kw), stride=stride,
                                         padding=pad, dilation=dilate)  # [n, c kh kw, L]
    flat = w.permute(0, 3, 1, 2).reshape(o, -1).double()
    out = (flat @ patches.double()).round().to(torch.int64).to(torch.int32)
    oh = (h + 2 * pad[0] - dilate[0] * (kh - 1) - 1) // stride[0] + 1
    return out.view(n, o, oh, -1).permute(0, 2, 3, 1).contiguous()


@pytest.mark.parametrize("n,h,w,c,o,k,stride,pad,dilate", [
    (1, 7, 7, 512, 64, 3, 1, 1, 1), (1, 14, 13, 48, 33, 3, 2, 1, 1), (2, 9, 9, 16, 20, 5, 1, 2, 2),
    (1, 5, 6, 32, 17, 1, 2, 0, 1), (3, 4, 4, 64, 40, 4, 1, 2, 1), (1, 1, 1, 272, 32, 1, 1, 1, 1)])
@pytest.mark.parametrize("waves", [0, 2, 4, 8, 16, -4, -8])
def test_convolutions(n, h, w, c, o, k, stride, pad, dilate, waves):
    g = torch.Generator(device="cuda").manual_seed(c + k)
    x, wt = int8(g, 0, n, h, w, c), int8(g, 0, o, k, k, c)
    got = capi.quantized_conv_nhwc(x, wt, None, *scalars(*RANGES), stride=(stride,) * 2,
                                   pad=(pad,) * 2, dilate=(dilate,) * 2, calib=(-40.0, 40.0),
                                   relu=True, force=(63, waves))
    assert torch.equal(got["out32"], conv_exact(x, wt, (stride,) * 2, (pad,) * 2, (dilate,) * 2))
    q = capi.requantize(got["out32"], got["omin"], got["omax"], -40.0, 40.0)[0]
    assert torch.equal(got["out8"], q.clamp_min(0))


@pytest.mark.parametrize("n,h,w,c,o,k,stride,off", [
    (1, 6, 5, 1, 4, 3, 1, 0), (2, 9, 8, 17, 64, 7, 1, 1), (1, 20, 20, 22, 30, 5, 1, 3),
    (3, 11, 7, 3, 16, 3, 2, 0), (8, 12, 12, 77, 130, 3, 1, 2)])
def test_convolutions_over_unaligned_channels(n, h, w, c, o, k, stride, off):
    g = torch.Generator(device="cuda").manual_seed(c)
    x, wt = int8(g, off, n, h, w, c), int8(g, off, o, k, k, c)
    got = capi.quantized_conv_nhwc(x, wt, None, *scalars(*RANGES), stride=(stride,) * 2,
                                   pad=(k // 2,) * 2, calib=(-20.0, 20.0))
    want = conv_exact(x, wt, (stride,) * 2, (k // 2,) * 2, (1, 1))
    assert torch.equal(got["out32"], want)
    q = capi.requantize(got["out32"], got["omin"], got["omax"], -20.0, 20.0)[0]
    assert torch.equal(got["out8"], q)


@pytest.mark.parametrize("n,h,w,o,k,stride,pad,dilate", [
    (3, 13, 11, 64, (4, 4), 1, 1, 1), (2, 9, 40, 48, (3, 3), 1, 1, 1), (1, 33, 1, 16, (2, 1), 1, 0, 1),
    (5, 7, 6, 128, (4, 4), 2, 3, 1), (2, 21, 19, 112, (3, 2), 1, 2, 3), (4, 1, 16, 32, (1, 16), 1, 5, 1),
    (7, 1, 1, 96, (3, 3), 1, 1, 1), (6, 80, 77, 64, (4, 4), 1, 1, 1)])
def test_convolutions_of_few_taps(n, h, w, o, k, stride, pad, dilate):
    g = torch.Generator(device="cuda").manual_seed(h * w + o)
    x, wt, b = int8(g, 0, n, h, w, 16), int8(g, 0, o, *k, 16), int8(g, 0, o)
    args = scalars(*RANGES, -0.5, 0.5)
    conv = dict(stride=(stride,) * 2, pad=(pad,) * 2, dilate=(dilate,) * 2, calib=(-30.0, 20.0))
    ref = capi.quantized_conv_nhwc(x, wt, None, *args[:4], **conv)
    assert torch.equal(ref["out32"], conv_exact(x, wt, *(conv[a] for a in ("stride", "pad", "dilate"))))
    for bias, relu in ((None, True), (b, False), (b, True)):
        a = args if bias is not None else args[:4]
        ref = capi.quantized_conv_nhwc(x, wt, bias, *a, relu=relu, force=(4, 1), **conv)
        got = capi.quantized_conv_nhwc(x, wt, bias, *a, relu=relu, want_int32=False, force=(64, 1),
                                       **conv)
        for key in ("out8", "omin", "omax", "rmin", "rmax"):
            assert torch.equal(got[key], ref[key]), key


@pytest.mark.parametrize("c", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n,h,w,off", [(2, 7, 6, 1), (1, 8, 8, 0), (3, 5, 9, 1), (1, 1, 1, 0)])
def test_quantize_with_space_to_depth(c, n, h, w, off):
    g = torch.Generator(device="cuda").manual_seed(c * h * w)
    x = torch.randn(n, c, h, w, device="cuda", generator=g) * 2
    q = capi.quantize_v2(x, "int8", -3.0, 3.0)[0]
    cp = (4 * c + 15) // 16 * 16
    oh, ow = (h + off + 1) // 2, (w + off + 1) // 2
    out = torch.empty(n, oh, ow, cp, dtype=torch.int8, device="cuda")
    ranges = torch.empty(2, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib.mxq_quantize_to_nhwc(
        stream, x.data_ptr(), out.data_ptr(), ranges.data_ptr(), ranges.data_ptr() + 4, n, c, h, w,
        cp, 1, off, off, -3.0, 3.0))
    want = torch.empty_like(out)
    _lib.check(_lib.lib.mxq_nchw_to_s2d_nhwc_i8(stream, q.data_ptr(), want.data_ptr(), n, c, h, w,
                                                off, off, cp))
    assert torch.equal(out, want)
