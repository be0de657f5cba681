"""3 x 3 convolutions over 64 channels into int32 planes by the kernel of whole rows: the integers of
the tiled kernel, at the shortest and longest rows, single rows, and an odd last one."""
import pytest
import torch

from mxnet_amd._lib import check, lib

pytestmark = pytest.mark.gpu


# (images, height, width)
@pytest.mark.parametrize("shape", [(64, 56, 56), (28, 28, 28), (32, 25, 24), (385, 2, 58),
                                   (800, 1, 33), (70, 11, 57), (300, 13, 32), (17, 61, 49)])
@pytest.mark.parametrize("with_bias", [False, True])
def test_planes_of_the_tiled_kernel(shape, with_bias):
    n, h, w = shape
    g = torch.Generator(device="cuda").manual_seed(h * w)
    draw = lambda s: torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight, bias = draw((n, h, w, 64)), draw((64, 3, 3, 64)), draw((64,))
    ranges = [torch.tensor([v], device="cuda") for v in (-3.0, 2.5, -0.5, 0.75, -9.0, 9.0)]
    given = [r.data_ptr() if i < 4 or with_bias else None for i, r in enumerate(ranges)]
    size = n * h * w * 64
    rows, planes = (torch.full((size + 64,), 77, dtype=torch.int32, device="cuda")
                    for _ in range(2))
    spans = torch.empty(4, device="cuda")
    at = [spans.data_ptr() + 4 * i for i in range(4)]
    stream = torch.cuda.current_stream().cuda_stream
    head = (stream, data.data_ptr(), weight.data_ptr(), bias.data_ptr() if with_bias else None, n,
            h, w, 64, 64, 3, 3, 1, 1, 1, 1, 1, 1, *given)
    check(lib.mxq_quantized_conv_nhwc(*head, rows.data_ptr(), at[0], at[1], None, None, None, 0,
                                      0.0, 0.0, None, 0))
    check(lib.mxq_quantized_conv_nhwc_out_nchw(*head, planes.data_ptr(), at[2], at[3], None, 0))
    want = rows[:size].view(n, h * w, 64).transpose(1, 2)
    assert len(want.unique()) > 1000
    assert torch.equal(planes[:size].view(n, 64, h * w), want)
    assert (planes[size:] == 77).all() and torch.equal(spans[:2], spans[2:])
