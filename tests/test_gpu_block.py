"""A residual block's tail as one launch (mxq_quantized_block) against the launches it stands for,
byte for byte: tile edges in pixels and in channels, rows and images that end inside a tile, sums
and layers with and without their short forms; and the plans that take it."""
import pytest
import torch

from mxnet_amd import _lib, capi
from mxnet_amd import symbol as S
from tests.test_gpu_plan import check, conv, quantized, relu

pytestmark = pytest.mark.gpu
lib = _lib.lib


def stream():
    return torch.cuda.current_stream().cuda_stream


def scalar(v):
    return torch.tensor([v], dtype=torch.float32, device="cuda")


class Layer:
    """Weights of `taps` taps, a bias and ranges, over a calibrated range that some saturate."""

    def __init__(self, g, o, c, taps, spread=1.0):
        self.o, self.c, self.taps = o, c, taps
        self.weight = torch.randint(-128, 128, (o, taps * c), device="cuda", generator=g,
                                    dtype=torch.int8)
        self.bias = torch.randint(-128, 128, (o,), device="cuda", generator=g, dtype=torch.int8)
        self.ranges = [scalar(v) for v in (-1.0, 0.9, -2.0, 2.1, -40.0, 39.0)]
        # a level of the data is about 1/127, one of the weights 2/127, both about 70 levels
        self.reach = spread * 1.5 * (taps * c) ** 0.5
        self.prepared = torch.empty(64 + 4 * o, dtype=torch.int8, device="cuda")
        _lib.check(lib.mxq_prepare_layer(stream(), self.bias.data_ptr(), o,
                                         *[r.data_ptr() for r in self.ranges], -self.reach,
                                         self.reach, self.prepared.data_ptr()))


def blocks(n, h, w, c, mid, out, after, relu1=1, relu3=1, residual=(-3.0, 3.0), total=None,
           spread=1.0, seed=0):
    """(the launch's outputs, the separate launches' outputs, the forms' flags)"""
    g = torch.Generator(device="cuda").manual_seed(seed + n + 3 * h + 5 * w + 7 * c + 11 * mid + out)
    data = torch.randint(-128, 128, (n, h, w, c), device="cuda", generator=g, dtype=torch.int8)
    m = n * h * w
    shortcut = torch.randint(-128, 128, (m, out), device="cuda", generator=g, dtype=torch.int8)
    first, second = Layer(g, mid, c, 9, spread), Layer(g, out, mid, 1, spread)
    third = Layer(g, after, out, 1, spread) if after else None
    total = total or 0.8 * (second.reach + 3.0)
    rmin, rmax = scalar(residual[0]), scalar(residual[1])
    layers = [first, second, third]
    at = [None if l is None else l.prepared.data_ptr() for l in layers]
    weights = torch.full((lib.mxq_quantized_block_weights(c, mid, out, after),), 99,
                         dtype=torch.int8, device="cuda")
    _lib.check(lib.mxq_pack_block_weights(
        stream(), *[None if l is None else l.weight.data_ptr() for l in layers], c, mid, out,
        after, weights.data_ptr()))
    forms = torch.full((lib.mxq_quantized_block_forms(),), 99, dtype=torch.int8, device="cuda")
    _lib.check(lib.mxq_prepare_block(stream(), *at, rmin.data_ptr(), rmax.data_ptr(),
                                     -second.reach, second.reach, -total, total,
                                     forms.data_ptr()))
    # room on both sides that has to stay as it is
    got = torch.full((m * out + 64,), 77, dtype=torch.int8, device="cuda")
    nxt = torch.full((m * after + 64,), 77, dtype=torch.int8, device="cuda")
    _lib.check(lib.mxq_quantized_block(
        stream(), data.data_ptr(), weights.data_ptr(), forms.data_ptr(), *at, n, h, w, c, mid, out,
        after, shortcut.data_ptr(), got[32:].data_ptr(),
        nxt[32:].data_ptr() if after else None, relu1, relu3))

    x = capi.quantized_conv_nhwc(data, first.weight.reshape(mid, 3, 3, c), first.bias,
                                 *first.ranges, pad=(1, 1), want_int32=False,
                                 calib=(-first.reach, first.reach), relu=bool(relu1))["out8"]
    y = capi.quantized_fc_sum(x.reshape(m, mid), second.weight, second.bias, shortcut,
                              *second.ranges, rmin, rmax, (-second.reach, second.reach),
                              (-total, total), sum_relu=True, requant=True)["out8"]
    for t, size in ((got, m * out), (nxt, m * after)):
        assert torch.all(t[:32] == 77) and torch.all(t[32 + size:] == 77)
    have = [got[32:32 + m * out].reshape(m, out)]
    want = [y.reshape(m, out)]
    if after:
        have.append(nxt[32:32 + m * after].reshape(m, after))
        want.append(capi.quantized_fc(y.reshape(m, out), third.weight, third.bias, *third.ranges,
                                      want_int32=False, calib=(-third.reach, third.reach),
                                      relu=bool(relu3))["out8"])
    return have, want, int(forms[:192].view(torch.int32)[35])


SHAPES = [
    (1, 4, 4, 16, 16, 16, 16), (1, 8, 8, 32, 64, 256, 64), (1, 5, 13, 48, 48, 80, 0),
    (2, 7, 9, 64, 64, 256, 48), (3, 13, 5, 16, 32, 144, 16), (1, 3, 43, 80, 16, 16, 272),
    (2, 56, 56, 64, 64, 256, 64), (1, 112, 9, 16, 32, 48, 16),          # up to 64 in the middle
    (2, 14, 14, 128, 128, 512, 128), (1, 9, 7, 96, 80, 336, 80), (5, 28, 28, 128, 112, 64, 0),
    (3, 7, 5, 144, 96, 32, 160),                                         # up to 128
    (1, 14, 14, 256, 256, 1024, 256), (4, 14, 13, 256, 144, 592, 144), (2, 9, 31, 160, 256, 16, 0),
    (1, 1, 65, 16, 176, 48, 512)]                                        # up to 256


@pytest.mark.parametrize("n,h,w,c,mid,out,after", SHAPES)
def test_block(n, h, w, c, mid, out, after):
    have, want, _ = blocks(n, h, w, c, mid, out, after)
    for a, b in zip(have, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,h,w,c,mid,out,after", SHAPES)
def test_block_on_whole_tiles(n, h, w, c, mid, out, after):
    """Enough pixels for tiles of 64, which fewer images than fill half of the chip do not take."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    have, want, _ = blocks(n + cus * 32 // (h * w) + 1, h, w, c, mid, out, after)
    for a, b in zip(have, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,h,w,c,mid,out,after", SHAPES[8:])
@pytest.mark.parametrize("more", [1, 700, 5000])
def test_block_that_ends_in_halves(n, h, w, c, mid, out, after, more):
    """A few tiles more than the chip has CUs: what is left over goes in tiles of 32."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    have, want, _ = blocks((cus * 64 + more) // (h * w) + 1, h, w, c, mid, out, after)
    for a, b in zip(have, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("whole", [False, True])
@pytest.mark.parametrize("n,h,w,c,mid,out,after", [
    (1, 6, 11, 64, 48, 16, 16), (2, 9, 10, 64, 64, 1040, 0), (1, 5, 5, 128, 16, 16, 48),
    (2, 9, 10, 128, 96, 208, 16), (1, 7, 10, 256, 256, 16, 32), (2, 7, 7, 256, 240, 1040, 80)])
def test_block_whose_taps_are_constants(n, h, w, c, mid, out, after, whole):
    """Exactly the channels that a kernel instance is made for, with one piece a row and with many."""
    if whole:
        n += torch.cuda.get_device_properties(0).multi_processor_count * 32 // (h * w) + 1
    have, want, _ = blocks(n, h, w, c, mid, out, after)
    for a, b in zip(have, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("n,h,w,c,mid,out,after", [
    (1, 7, 7, 128, 256, 2048, 256), (1, 8, 8, 96, 192, 2048, 0), (2, 10, 10, 1232, 112, 768, 0),
    (1, 4, 4, 704, 256, 512, 256), (1, 11, 11, 528, 112, 512, 0)])
@pytest.mark.parametrize("whole", [False, True])
def test_block_that_lds_just_holds(n, h, w, c, mid, out, after, whole):
    if whole:
        n += torch.cuda.get_device_properties(0).multi_processor_count * 32 // (h * w) + 1
    have, want, _ = blocks(n, h, w, c, mid, out, after)
    for a, b in zip(have, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("relu1,relu3", [(0, 0), (1, 0), (0, 1)])
@pytest.mark.parametrize("mid,spread", [(48, 0.02), (128, 40.0), (160, 1.0)])
def test_block_ranges_on_whole_tiles(mid, spread, relu1, relu3):
    have, want, _ = blocks(90, 10, 11, 64, mid, 96, 32, relu1, relu3, spread=spread)
    for a, b in zip(have, want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("kwargs", [
    {"relu1": 0}, {"relu3": 0}, {"spread": 0.02}, {"spread": 40.0}, {"residual": (-1e-3, 1e-3)},
    {"residual": (-4000.0, 0.0)}, {"residual": (0.0, 0.0)}, {"residual": (-3e38, 3e38)},
    {"total": 1e-30}, {"total": 1e30}])
@pytest.mark.parametrize("mid", [48, 128, 160])
def test_block_ranges(mid, kwargs):
    have, want, _ = blocks(2, 10, 11, 64, mid, 96, 32, **kwargs)
    for a, b in zip(have, want):
        assert torch.equal(a, b)


def test_short_forms_are_found():
    """They hold for nearly all ranges; without them the launch computes the definition, which
    test_block_ranges also covers (ranges of 0 and of the largest floats have none)."""
    flags = [blocks(1, 4, 5, 16, 16, 32, 16, seed=i, spread=0.4 + 0.07 * i,
                    residual=(-2.0 - 0.3 * i, 2.2))[2] for i in range(12)]
    for bit in range(4):
        assert sum(f >> bit & 1 for f in flags) >= 8, (bit, flags)
    assert blocks(1, 4, 5, 16, 16, 32, 16, residual=(0.0, 0.0))[2] & 8 == 0


def stage(c, mid, out, count, sizes):
    """`count` blocks, the first with a projection; every second without the last one's first
    layer behind it"""
    shapes = {}

    def layer(x, name, i, o, k=1):
        shapes[name + "_weight"], shapes[name + "_bias"] = (o, i, k, k), (o,)
        return conv(x, name, o, k)

    x = relu(layer(S.Variable("data"), "stem", c, mid), "stem_relu")
    width, mids = mid, []
    for b in range(count):
        a = layer(x, "a%d" % b, width, mid)
        y = layer(relu(a, "ra%d" % b) if b % 2 == 0 else a, "b%d" % b, mid, mid, 3)
        y = layer(relu(y, "rb%d" % b) if b % 3 != 2 else y, "c%d" % b, mid, out)
        if b == 0:
            x = layer(x, "p", width, out)
        x = relu(S.elemwise_add(*((y, x) if b % 2 == 0 else (x, y)), name="s%d" % b), "rs%d" % b)
        width = out
        mids.append(x)
    return S.Group([conv(x, "last", sizes), mids[1]]), dict(shapes, last_weight=(sizes, out, 1, 1),
                                                            last_bias=(sizes,))


@pytest.mark.parametrize("batch,mid,out,h,w", [(1, 16, 64, 9, 14), (2, 37, 148, 31, 17),
                                               (3, 100, 400, 14, 14), (8, 200, 800, 14, 14)])
def test_plans_take_it(batch, mid, out, h, w):
    sym, shapes = stage(5, mid, out, 4, 20)
    ex = quantized(sym, shapes)
    check(ex, data=torch.randn(batch, 5, h, w, device="cuda"))
    assert sum(key[1] == "block" for key in ex._structure().laid) == 4
