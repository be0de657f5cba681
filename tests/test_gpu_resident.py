"""The 1 x 1 convolution / fully-connected kernel that holds its weights in registers: the bytes of
the tiled kernels (pinned; their parity with the oracle is tested beside them) at its edges: ragged
rows, columns short of a group, strides, images inside a tile, with and without bias and relu."""
import pytest
import torch

from mxnet_amd import capi
from mxnet_amd._lib import MXQError

pytestmark = pytest.mark.gpu


def operands(shape, o, k, bias, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    draw = lambda s: torch.randint(-127, 128, s, device="cuda", generator=g, dtype=torch.int8)
    ranges = [torch.tensor([v], device="cuda") for v in (-3.0, 2.5, -0.5, 0.75, -1.0, 1.0)]
    return draw(shape + (k,)), draw((o, k)), draw((o,)) if bias else None, ranges


def same(got, want):
    for name in ("out8", "omin", "omax", "rmin", "rmax"):
        assert torch.equal(got[name], want[name])


# what launches the kernel: 3 (K = 256) or 6 (K = 512) tiles per CU and column group
def rows_for(k, n):
    wide, high = (64, 64) if k == 256 and n <= 64 else (128, 32) if n <= 128 else (256, 32)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    groups = -(-n // wide)
    return -(-(3 if k == 256 else 6) * cus // groups) * high


@pytest.mark.parametrize("k,n", [(256, 48), (256, 64), (256, 96), (256, 128), (256, 192),
                                 (256, 256), (256, 464), (512, 96), (512, 128), (512, 256),
                                 (512, 400)])
@pytest.mark.parametrize("relu,bias", [(True, True), (False, True), (True, False)])
def test_rows(k, n, relu, bias):
    least = rows_for(k, n)
    for m in (least, least + 1, least + 31, 2 * least + 17):
        x, w, b, r = operands((1, 1, m), n, k, bias, m)
        x = x.view(1, 1, m, k)
        args = (x, w.view(n, 1, 1, k), b, *r[:4], *(r[4:] if bias else (None, None)))
        kw = dict(want_int32=False, calib=(-20.0, 18.0), relu=relu)
        got = capi.quantized_conv_nhwc(*args, **kw)
        want = capi.quantized_conv_nhwc(*args, force=(25, 1), **kw)
        same(got, want)
        # it is this kernel that was chosen: pinned, any other choice is an error
        flat = (x.view(m, k), w, *args[2:])
        pinned = capi.quantized_fc(*flat, force=(65, 1, 0), **kw)
        assert torch.equal(pinned["out8"], want["out8"].view(m, n))
    with pytest.raises(MXQError):
        capi.quantized_fc(x.view(m, k)[:least // 2], w, *args[2:], force=(65, 1, 0), **kw)


# (images, height, width, strides): odd planes, images smaller than a tile, one output line
@pytest.mark.parametrize("images,h,w,sh,sw", [(40, 57, 55, 2, 2), (3000, 9, 7, 2, 2),
                                              (9000, 5, 4, 2, 3), (26000, 2, 2, 2, 2),
                                              (2, 199, 299, 2, 1), (3, 2, 65000, 2, 3),
                                              # planes the kernel leaves to the tiled ones
                                              (2, 301, 300, 2, 1)])
@pytest.mark.parametrize("k,n", [(256, 64), (256, 128), (256, 512), (512, 128), (512, 512)])
def test_strided(images, h, w, sh, sw, k, n):
    oh, ow = (h - 1) // sh + 1, (w - 1) // sw + 1
    images = max(images, -(-rows_for(k, n) // (oh * ow)))
    x, wt, b, r = operands((images, h, w), n, k, True, h * w)
    args = (x, wt.view(n, 1, 1, k), b, *r)
    kw = dict(want_int32=False, calib=(-20.0, 18.0), relu=True, stride=(sh, sw))
    got = capi.quantized_conv_nhwc(*args, **kw)
    want = capi.quantized_conv_nhwc(*args, force=(25, 1), **kw)
    same(got, want)
    if oh * ow < 30000:
        same(capi.quantized_conv_nhwc(*args, force=(65, 1), **kw), want)
    else:
        with pytest.raises(MXQError):
            capi.quantized_conv_nhwc(*args, force=(65, 1), **kw)
