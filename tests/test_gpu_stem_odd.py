"""Stems over images of odd extents: the space-to-depth form with a row or column of zeros more, and
plans whose last windows reach it, against the quantize operator and the graph walked operator by
operator."""
import pytest
import torch

from mxnet_amd import capi
from mxnet_amd import symbol as S
from mxnet_amd._lib import MXQError, check, lib
from test_gpu_plan import check as check_plan, conv, quantized, relu

pytestmark = pytest.mark.gpu


def to_s2d(x, off, rows, columns, padded):
    n, c, h, w = x.shape
    out = torch.full((n * rows * columns * padded + 64,), 99, dtype=torch.int8, device="cuda")
    lo, hi = torch.zeros(1, device="cuda"), torch.zeros(1, device="cuda")
    check(lib.mxq_quantize_to_s2d(torch.cuda.current_stream().cuda_stream, x.data_ptr(),
                                  out.data_ptr(), lo.data_ptr(), hi.data_ptr(), n, c, h, w, padded,
                                  *off, rows, columns, -2.5, 3.0))
    assert (out[-64:] == 99).all()
    return out[:-64].view(n, rows, columns, padded)


# one pixel, one column, lanes that run on from image to image (below 1024 pixels) and those that do
# not, more than one chunk of channels
@pytest.mark.parametrize("n,c,h,w", [(1, 3, 1, 1), (3, 1, 9, 1), (5, 2, 7, 4), (2, 3, 63, 65),
                                     (9, 3, 15, 17), (2, 4, 31, 66), (2, 5, 9, 11)])
@pytest.mark.parametrize("off", [(0, 0), (1, 1), (0, 1)])
@pytest.mark.parametrize("more", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_form_with_another_row_or_column(n, c, h, w, off, more):
    g = torch.Generator(device="cuda").manual_seed(h * w + c)
    x = torch.randn((n, c, h, w), device="cuda", generator=g) * 2
    rows, columns = (h + off[0] + 1) // 2 + more[0], (w + off[1] + 1) // 2 + more[1]
    got = to_s2d(x, off, rows, columns, (4 * c + 15) // 16 * 16)
    q, _, _ = capi.quantize_v2(x, "int8", min_calib_range=-2.5, max_calib_range=3.0)
    want = torch.zeros((n, 2 * rows, 2 * columns, c), dtype=torch.int8, device="cuda")
    want[:, off[0]:off[0] + h, off[1]:off[1] + w] = q.permute(0, 2, 3, 1)
    want = want.view(n, rows, 2, columns, 2, c).permute(0, 1, 3, 2, 4, 5)
    assert torch.equal(got[..., :4 * c], want.reshape(n, rows, columns, 4 * c))
    assert not got[..., 4 * c:].any()


@pytest.mark.parametrize("rows,columns", [(3, 5), (6, 5), (4, 4), (4, 7)])
def test_rows_the_image_does_not_give_are_refused(rows, columns):
    with pytest.raises(MXQError):
        to_s2d(torch.zeros((1, 3, 7, 9), device="cuda"), (1, 1), rows, columns, 16)


@pytest.mark.parametrize("h,w", [(33, 33), (47, 32), (32, 47), (7, 9), (61, 3)])
@pytest.mark.parametrize("k", [3, 5, 7, 4])
@pytest.mark.parametrize("pool", [False, True])
def test_plan_of_a_stem(h, w, k, pool):
    x = relu(conv(S.Variable("data"), "stem", 40, k, 2), "stem_relu")
    if pool:
        x = S.Pooling(x, kernel=(3, 3), stride=(2, 2), pad=(1, 1), pool_type="max", name="pool")
    x = conv(x, "next", 24)
    ex = quantized(x, {"stem_weight": (40, 3, k, k), "stem_bias": (40,),
                       "next_weight": (24, 40, 1, 1), "next_bias": (24,)})
    g = torch.Generator(device="cuda").manual_seed(h + w)
    check_plan(ex, data=torch.randn((3, 3, h, w), device="cuda", generator=g))
