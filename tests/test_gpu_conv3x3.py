"""3 x 3 convolutions over many channels with their weights laid out: the bytes of the general path at
ragged rows, columns short of a tile, planes of a pixel, a row or a column, and both ways to
requantize."""
import pytest
import torch

from mxnet_amd._lib import check, lib

pytestmark = pytest.mark.gpu


# (images, height, width, channels, output channels)
@pytest.mark.parametrize("shape", [(64, 7, 7, 512, 512), (33, 7, 7, 512, 144), (64, 14, 14, 256, 256),
                                   (3, 5, 9, 768, 272), (40, 1, 13, 256, 16), (40, 13, 1, 512, 48),
                                   (70, 1, 1, 512, 128), (1, 3, 3, 1024, 32), (2, 17, 100, 256, 240)])
@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("forms", [False, True])
def test_bytes_of_the_general_path(shape, relu, forms):
    n, h, w, c, o = shape
    g = torch.Generator(device="cuda").manual_seed(h * w + o)
    draw = lambda s: torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight, bias = draw((n, h, w, c)), draw((o, 3, 3, c)), draw((o,))
    ranges = [torch.tensor([v], device="cuda") for v in (-3.0, 2.5, -0.5, 0.75, -1.0, 1.0)]
    prepared = torch.empty(64 + 4 * o, dtype=torch.int8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for step in range(20):
        calib = (-60.0 - 0.1 * step, 54.0)
        check(lib.mxq_prepare_layer(stream, bias.data_ptr(), o, *[r.data_ptr() for r in ranges],
                                    *calib, prepared.data_ptr()))
        if not forms:
            break
        check(lib.mxq_prepare_forms(stream, prepared.data_ptr()))
        if prepared[32:36].view(torch.int32).item() == 3:  # as for nine ranges out of ten
            break
    else:
        pytest.fail("no short forms for any of these ranges")
    size = n * h * w * o
    want, got = (torch.full((size + 64,), 77, dtype=torch.int8, device="cuda") for _ in range(2))
    check(lib.mxq_quantized_conv_nhwc_prepared(
        stream, data.data_ptr(), weight.data_ptr(), prepared.data_ptr(), n, h, w, c, o, 3, 3, 1, 1,
        1, 1, 1, 1, want.data_ptr(), relu, *calib, None, 0))
    laid = torch.empty(lib.mxq_quantized_conv3x3_weights(c, o), dtype=torch.int8, device="cuda")
    check(lib.mxq_pack_conv3x3_weights(stream, weight.data_ptr(), c, o, laid.data_ptr()))
    check(lib.mxq_quantized_conv3x3(stream, data.data_ptr(), laid.data_ptr(), prepared.data_ptr(),
                                    n, h, w, c, o, got.data_ptr(), relu))
    assert len(want[:size].unique()) > 1
    assert torch.equal(got, want)


def test_what_does_not_fit():
    fits = lib.mxq_quantized_conv3x3_fits
    assert fits(64, 7, 7, 512, 512)
    assert not fits(8, 7, 7, 512, 512)      # few work-groups
    assert not fits(256, 7, 7, 512, 512)    # many
    assert not fits(64, 14, 14, 256, 48)    # columns for two waves of four
    assert not fits(64, 7, 7, 384, 512)     # half of the channels a wave, in groups of four steps
    assert not fits(64, 7, 7, 512, 520)     # 16 | O
    assert not fits(64, 56, 56, 1024, 512)  # the pixels of a tile exceed the LDS
