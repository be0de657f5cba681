"""A stem in one launch: the bytes of the convolution and the pooling on their own, at the edges of
its strips and bands, with every edge of the image, widths that are no multiple of a strip, and
biases that the sums wrap around with."""
import pytest
import torch

from mxnet_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def pooled(extent, full):
    over = extent + 2 - 3
    return (over + 1) // 2 + 1 if full else over // 2 + 1


# (images, height, width, channels, padding down, across)
@pytest.mark.parametrize("shape", [(2, 115, 115, 64, 0, 0), (1, 4, 4, 16, 0, 0), (3, 5, 9, 32, 0, 1),
                                   (1, 33, 31, 48, 1, 0), (5, 17, 60, 64, 2, 3), (2, 7, 59, 80, 3, 2),
                                   (70, 31, 45, 64, 1, 1), (1, 3, 200, 128, 1, 1),
                                   (9, 200, 3, 16, 1, 1)])
@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("full", [False, True])
@pytest.mark.parametrize("far", [False, True])
def test_stem_is_convolution_and_pooling(shape, relu, full, far):
    n, h, w, o, ph, pw = shape
    oh, ow = h + 2 * ph - 3, w + 2 * pw - 3
    p_h, p_w = pooled(oh, full), pooled(ow, full)
    g = torch.Generator(device="cuda").manual_seed(h * w + o)
    draw = lambda s: torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight, bias = draw((n, h, w, 16)), draw((o, 4, 4, 16)), draw((o,))
    # an output level of 2^-14 * 0.12 against a bias level of 0.008: a bias beyond 2^31 levels is
    # the largest integer
    reach = 1e9 if far else 1.0
    ranges = [torch.tensor([v], device="cuda") for v in (-3.0, 2.5, -0.5, 0.75, -reach, reach)]
    prepared = torch.empty(64 + 4 * o, dtype=torch.int8, device="cuda")
    calib = (-3e5, 2e5) if far else (-20.0, 18.0)
    stream = torch.cuda.current_stream().cuda_stream
    check(lib.mxq_prepare_layer(stream, bias.data_ptr(), o, *[r.data_ptr() for r in ranges], *calib,
                                prepared.data_ptr()))
    if far:
        assert prepared[64:].view(torch.int32).abs().max().item() > 2 ** 31 - 2 ** 22
    conv = torch.empty((n, oh, ow, o), dtype=torch.int8, device="cuda")
    check(lib.mxq_quantized_conv_nhwc_prepared(
        stream, data.data_ptr(), weight.data_ptr(), prepared.data_ptr(), n, h, w, 16, o, 4, 4, 1, 1,
        ph, pw, 1, 1, conv.data_ptr(), relu, *calib, None, 0))
    size = n * p_h * p_w * o
    want, got = (torch.full((size + 64,), 77, dtype=torch.int8, device="cuda") for _ in range(2))
    check(lib.mxq_quantized_pooling_nhwc(stream, conv.data_ptr(), n, oh, ow, o, 3, 3, 2, 2, 1, 1,
                                         p_h, p_w, 0, 1, want.data_ptr()))
    assert lib.mxq_quantized_conv_pool_fits(n, h, w, 16, o, 4, 4, ph, pw, p_h, p_w)
    check(lib.mxq_quantized_conv_pool(stream, data.data_ptr(), weight.data_ptr(),
                                      prepared.data_ptr(), n, h, w, 16, o, 4, 4, ph, pw, p_h, p_w,
                                      got.data_ptr(), relu))
    assert len(want[:size].unique()) > 1
    assert torch.equal(got, want)


def test_rows_outside_the_image_do_not_overtake():
    """Bands of one pooled row at the image's lower edge, where the rows sent for ahead are zeros
    that arrive at once: the same bytes every time."""
    n, h, w, o, p_h, p_w = 64, 33, 33, 64, 16, 16
    g = torch.Generator(device="cuda").manual_seed(5)
    draw = lambda s: torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight, bias = draw((n, h, w, 16)), draw((o, 4, 4, 16)), draw((o,))
    ranges = [torch.tensor([v], device="cuda") for v in (-3.0, 2.5, -0.5, 0.75, -1.0, 1.0)]
    prepared = torch.empty(64 + 4 * o, dtype=torch.int8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    check(lib.mxq_prepare_layer(stream, bias.data_ptr(), o, *[r.data_ptr() for r in ranges], -20.0,
                                18.0, prepared.data_ptr()))
    conv = torch.empty((n, 32, 32, o), dtype=torch.int8, device="cuda")
    check(lib.mxq_quantized_conv_nhwc_prepared(
        stream, data.data_ptr(), weight.data_ptr(), prepared.data_ptr(), n, h, w, 16, o, 4, 4, 1, 1,
        1, 1, 1, 1, conv.data_ptr(), 1, -20.0, 18.0, None, 0))
    want = torch.empty((n, p_h, p_w, o), dtype=torch.int8, device="cuda")
    check(lib.mxq_quantized_pooling_nhwc(stream, conv.data_ptr(), n, 32, 32, o, 3, 3, 2, 2, 1, 1,
                                         p_h, p_w, 0, 1, want.data_ptr()))
    for _ in range(100):
        got = torch.empty_like(want)
        check(lib.mxq_quantized_conv_pool(stream, data.data_ptr(), weight.data_ptr(),
                                          prepared.data_ptr(), n, h, w, 16, o, 4, 4, 1, 1, p_h, p_w,
                                          got.data_ptr(), 1))
        assert torch.equal(got, want)


def test_what_does_not_fit():
    fits = lib.mxq_quantized_conv_pool_fits
    assert fits(1, 115, 115, 16, 64, 4, 4, 0, 0, 56, 56)
    assert not fits(1, 115, 115, 32, 64, 4, 4, 0, 0, 56, 56)
    assert not fits(1, 115, 115, 16, 64, 3, 4, 0, 0, 56, 56)
    assert not fits(1, 115, 115, 16, 60, 4, 4, 0, 0, 56, 56)
    assert not fits(1, 115, 115, 16, 64, 4, 4, 0, 0, 58, 56)   # a window outside the image
    assert not fits(1, 3, 115, 16, 64, 4, 4, 0, 0, 1, 56)      # no output
