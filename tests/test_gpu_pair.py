"""Two 1 x 1 convolutions of one tensor in one launch: the bytes of two launches, on each way the
pair can go out (a few output tiles, 64 x 64 and 128 x 128 tiles, weights in registers) and where it
falls back to two, with ragged rows, strides, and columns short of a tile on either side."""
import pytest
import torch

from mxnet_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def layer(o, c, seed, forms):
    g = torch.Generator(device="cuda").manual_seed(seed)
    draw = lambda s: torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int8)
    weight, bias = draw((o, c)), draw((o,))
    ranges = [torch.tensor([v], device="cuda") for v in (-3.0, 2.5, -0.5, 0.75, -1.0, 1.0)]
    prepared = torch.empty(64 + 4 * o, dtype=torch.int8, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    for step in range(20):
        calib = (-20.0 - seed - 0.1 * step, 18.0)
        check(lib.mxq_prepare_layer(stream, bias.data_ptr(), o, *[r.data_ptr() for r in ranges],
                                    *calib, prepared.data_ptr()))
        assert prepared[32:36].view(torch.int32).item() == 0
        if not forms:
            break
        check(lib.mxq_prepare_forms(stream, prepared.data_ptr()))
        if prepared[32:36].view(torch.int32).item() == 3:  # as for nine ranges out of ten
            break
    else:
        pytest.fail("no short forms for any of these ranges")
    return weight, prepared, calib


# (images, height, width, channels, first width, second width, stride)
SHAPES = [(1, 14, 14, 512, 256, 1024, 1), (1, 15, 13, 512, 272, 48, 2), (1, 7, 7, 1024, 512, 2048, 1),
          (2, 9, 5, 256, 16, 32, 1), (1, 14, 14, 2064, 64, 16, 2),        # few tiles
          (1, 56, 56, 64, 64, 256, 1), (3, 29, 31, 48, 80, 16, 2),        # 64 x 64 tiles
          (5, 14, 14, 1024, 512, 208, 1),                                 # ... on deep stages
          (64, 14, 14, 1024, 512, 2048, 2), (31, 9, 11, 1040, 528, 1040, 1),  # 128 x 128 tiles
          (64, 56, 56, 256, 128, 512, 2), (64, 28, 28, 512, 256, 1024, 2),    # weights in registers
          (33, 57, 29, 256, 512, 144, 1), (50, 31, 33, 512, 240, 1008, 2),
          (64, 56, 56, 64, 64, 256, 1), (65, 57, 55, 64, 48, 208, 1),         # ... of 64 bytes
          (64, 16, 16, 64, 64, 256, 1), (80, 14, 15, 64, 64, 240, 1),
          (64, 56, 56, 128, 64, 256, 1)]                                  # two launches


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("relu", [(1, 0), (0, 1)])
@pytest.mark.parametrize("off", [0, 1])  # unaligned images: two launches
@pytest.mark.parametrize("forms", [False, True])
def test_pair_is_two_convolutions(shape, relu, off, forms):
    n, h, w, c, o1, o2, s = shape
    if off and n > 5:
        pytest.skip("the fallback does not depend on the size")
    m = n * ((h - 1) // s + 1) * ((w - 1) // s + 1)
    data = torch.randint(-127, 128, (n * h * w * c + 16,), device="cuda", dtype=torch.int8)
    data = data[off:off + n * h * w * c]
    stream = torch.cuda.current_stream().cuda_stream
    layers, outs, wants = [layer(o1, c, 1, forms), layer(o2, c, 2, forms)], [], []
    for (weight, prepared, calib), o, r in zip(layers, (o1, o2), relu):
        # a guard behind every output
        outs.append(torch.full((m * o + 64,), 77, dtype=torch.int8, device="cuda"))
        want = torch.full((m * o + 64,), 77, dtype=torch.int8, device="cuda")
        check(lib.mxq_quantized_conv_nhwc_prepared(
            stream, data.data_ptr(), weight.data_ptr(), prepared.data_ptr(), n, h, w, c, o, 1, 1,
            s, s, 0, 0, 1, 1, want.data_ptr(), r, *calib, None, 0))
        wants.append(want)
    args = []
    for (weight, prepared, calib), o, r, out in zip(layers, (o1, o2), relu, outs):
        args += [weight.data_ptr(), prepared.data_ptr(), o, out.data_ptr(), r, *calib]
    check(lib.mxq_quantized_conv_pair_prepared(stream, data.data_ptr(), n, h, w, c, s, s, *args))
    for out, want in zip(outs, wants):
        assert torch.equal(out, want)


def test_which_shapes_pair():
    fits = [lib.mxq_quantized_conv_pair_fits(n, h, w, c, o1, o2, s, s)
            for n, h, w, c, o1, o2, s in SHAPES]
    assert fits == [1] * (len(SHAPES) - 1) + [0]
    assert not lib.mxq_quantized_conv_pair_fits(1, 14, 14, 24, 16, 16, 1, 1)   # 16 | C
    assert not lib.mxq_quantized_conv_pair_fits(1, 14, 14, 64, 24, 16, 1, 1)   # 16 | O
    assert not lib.mxq_quantized_conv_pair_fits(0, 14, 14, 64, 32, 16, 1, 1)   # no pixels
