"""1 x 1 convolutions of NCHW tensors whose pixels are gathered first: the integers of the general
path at planes whose bytes are odd, channel groups and images that are left over, strides that
differ, single rows and columns, and planes that go through LDS one by one or not at all."""
import pytest
import torch

from mxnet_amd._lib import check, lib

pytestmark = pytest.mark.gpu


# (images, channels, height, width, output channels, strides)
@pytest.mark.parametrize("shape", [(64, 512, 7, 7, 2048, 1, 1), (3, 48, 7, 7, 32, 1, 1),
                                   (64, 512, 28, 28, 1024, 2, 2), (64, 1024, 14, 14, 2048, 2, 2),
                                   (5, 80, 9, 13, 48, 2, 1), (2, 16, 45, 45, 16, 1, 2),
                                   (70, 16, 1, 5, 16, 1, 3), (33, 32, 5, 1, 16, 2, 1),
                                   (130, 16, 1, 1, 64, 1, 1), (1, 32, 181, 181, 16, 2, 2),
                                   (2, 16, 40, 51, 32, 3, 2), (1, 16, 128, 256, 16, 1, 3),
                                   (1, 16, 129, 256, 16, 1, 3), (9, 96, 3, 3, 16, 1, 1),
                                   (64, 128, 28, 28, 512, 2, 2), (16, 256, 57, 57, 528, 2, 2),
                                   (25, 272, 46, 46, 512, 2, 2),
                                   # the longest groups that go through LDS, and the next ones
                                   (1, 16, 128, 256, 16, 8, 8), (2, 16, 43, 45, 32, 4, 4),
                                   (2, 16, 43, 45, 32, 3, 4), (3, 64, 21, 21, 32, 1, 1),
                                   (3, 64, 23, 23, 32, 1, 1), (2, 48, 35, 35, 64, 2, 2)])
def test_integers_of_the_general_path(shape):
    n, c, h, w, o, sh, sw = shape
    oh, ow = (h - 1) // sh + 1, (w - 1) // sw + 1
    g = torch.Generator(device="cuda").manual_seed(h * w + o)
    draw = lambda s: torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight = draw((n, c, h, w)), draw((o, c, 1, 1))
    ranges = [torch.tensor([v], device="cuda") for v in (-3.0, 2.5, -0.5, 0.75)]
    size, outs = n * o * oh * ow, []
    stream = torch.cuda.current_stream().cuda_stream
    for cfg in (0, 1):  # 1: NHWC copies of both operands
        out = torch.full((size + 64,), 77, dtype=torch.int32, device="cuda")
        span = torch.empty(2, device="cuda")
        need = lib.mxq_quantized_conv_nchw_workspace(n, c, h, w, o, 1, 1, sh, sw, 0, 0, 1, 1, 0)
        space = torch.full((need + 64,), 55, dtype=torch.int8, device="cuda")
        check(lib.mxq_test_quantized_conv_nchw(
            stream, data.data_ptr(), weight.data_ptr(), None, n, c, h, w, o, 1, 1, sh, sw, 0, 0, 1,
            1, *[r.data_ptr() for r in ranges], None, None, out.data_ptr(), span.data_ptr(),
            span.data_ptr() + 4, space.data_ptr(), need, cfg))
        assert (space[need:] == 55).all()
        outs.append(out)
    assert torch.equal(*outs)


def test_many_tiles_without_a_workspace():
    """Layers that gather beforehand only because it is faster (256 channels, 12544 pixels of 512
    outputs; 128 channels from 32768 pixels on) do without the room for it."""
    n, c, h, o = 64, 256, 28, 512
    data = torch.randint(-127, 128, (n, c, h, h), device="cuda", dtype=torch.int8)
    weight = torch.randint(-127, 128, (o, c, 1, 1), device="cuda", dtype=torch.int8)
    ranges = [torch.tensor([v], device="cuda") for v in (-3.0, 2.5, -0.5, 0.75)]
    span = torch.empty(2, device="cuda")
    need = lib.mxq_quantized_conv_nchw_workspace(n, c, h, h, o, 1, 1, 2, 2, 0, 0, 1, 1, 1)
    space, outs = torch.empty(need, dtype=torch.int8, device="cuda"), []
    assert need >= n * c * (h // 2) ** 2
    for room in (need, 0):
        out = torch.full((n, o, h // 2, h // 2), 77, dtype=torch.int32, device="cuda")
        check(lib.mxq_quantized_conv_nchw(
            torch.cuda.current_stream().cuda_stream, data.data_ptr(), weight.data_ptr(), None, n, c,
            h, h, o, 1, 1, 2, 2, 0, 0, 1, 1, *[r.data_ptr() for r in ranges], None, None,
            out.data_ptr(), span.data_ptr(), span.data_ptr() + 4,
            space.data_ptr() if room else None, room))
        outs.append(out)
    assert torch.equal(*outs)


@pytest.mark.parametrize("n,c,gathers", [(64, 128, False), (168, 128, True), (64, 256, True),
                                         (61, 256, False)])
def test_which_layers_gather_beforehand(n, c, gathers):
    """28 x 28 / 2 -> 512: where the second launch is worth it.  (Behind it the workspace holds the
    pixels the layer reads.)"""
    need = lib.mxq_quantized_conv_nchw_workspace(n, c, 28, 28, 512, 1, 1, 2, 2, 0, 0, 1, 1, 1)
    assert (need >= n * c * 14 * 14) == gathers
