"""Tiles on eight waves that share each stage's reduction, and tiles of 32 columns: at the lines of the rules
that choose them, at their edges and split over work-groups, against float64 products (exact for these lengths)
and, requantized, against the smallest tile pinned."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import mxnet_amd
    return mxnet_amd.capi


def operands(*shapes):
    g = torch.Generator(device="cuda").manual_seed(sum(map(sum, shapes)))
    return [torch.randint(-128, 128, s, dtype=torch.int8, device="cuda", generator=g) for s in shapes]


def ranges():
    return [torch.tensor([v], device="cuda") for v in (-1.0, 1.0, -0.1, 0.1)]


def same(call, pinned, want):
    assert torch.equal(call(want_int32=True)["out32"].double(), want)
    for relu in (False, True):
        kw = dict(want_int32=False, calib=(-2.0, 2.0), relu=relu)
        assert torch.equal(call(**kw)["out8"], call(force=pinned, **kw)["out8"])


# 256 tiles of 64 x 64, a ragged 255, 36, 6 and one; one work-group a tile below 8192, 2 ... 12 from there on
@pytest.mark.parametrize("M,N", [(1024, 1024), (961, 1023), (1090, 79), (300, 385), (121, 153), (33, 17)])
@pytest.mark.parametrize("K", [1536, 1552, 1776, 4096, 8192, 8208, 32784])
def test_fully_connected(capi, M, N, K):
    d, w = operands((M, K), (N, K))
    want = d.double() @ w.double().t().contiguous()
    same(lambda **kw: capi.quantized_fc(d, w, None, *ranges(), **kw), (44, 1, 0), want)
    # pinned, whatever the rule says of the shape
    for cfg, splits in ((33, 1), (33, 3), (34, 1), (34, 4)):
        assert torch.equal(capi.quantized_fc(d, w, None, *ranges(), want_int32=True,
                                             force=(cfg, splits, 0))["out32"].double(), want)


# 128 x 128 tiles: 256 of them, a ragged 176, 133; just below the lengths from which they are split (64 x 64 tiles
# there, split once); and shared by two, three, five and six
@pytest.mark.parametrize("M,N,K", [(2048, 2048, 1536), (2048, 2040, 1552), (1300, 1999, 1664), (2400, 833, 2064),
                                   (699, 2429, 6160), (784, 1387, 6272), (1000, 470, 8208), (450, 1101, 12304),
                                   (699, 2429, 8208), (784, 1387, 8208), (700, 900, 14352), (720, 799, 15696)])
def test_fully_connected_of_larger_tiles(capi, M, N, K):
    d, w = operands((M, K), (N, K))
    same(lambda **kw: capi.quantized_fc(d, w, None, *ranges(), **kw), (44, 1, 0),
         d.double() @ w.double().t().contiguous())


@pytest.mark.parametrize("K", [16, 240, 256, 272, 528, 784])
def test_reductions_of_few_stages(capi, K):
    d, w = operands((130, K), (70, K))
    want = d.double() @ w.double().t().contiguous()
    for cfg in (33, 34):
        assert torch.equal(capi.quantized_fc(d, w, None, *ranges(), want_int32=True,
                                             force=(cfg, 1, 0))["out32"].double(), want)


@pytest.mark.parametrize("M,N,K", [(1000, 500, 1600), (129, 130, 4160)])
def test_float_and_sum_outputs(capi, M, N, K):
    d, w, res = operands((M, K), (N, K), (M, N))
    out = [capi.quantized_fc_f32(d, w, None, *ranges(), calib=(-2.0, 2.0), relu=True, force=f)["outf"]
           for f in ((44, 1), (33, 1), (33, 2), (34, 1), (34, 3))]
    assert all(torch.equal(out[0], o) for o in out[1:])
    for requant in (False, True):
        out = [capi.quantized_fc_sum(d, w, None, res, *ranges(), None, None, *ranges()[:2], (-2.0, 2.0),
                                     (-2.5, 2.5), sum_relu=True, requant=requant, force=f)["out8"]
               for f in ((44, 1, 0), (33, 1, 0), (33, 2, 0), (34, 1, 0), (34, 3, 0))]
        assert all(torch.equal(out[0], o) for o in out[1:])


# 128 x 32 and 64 x 64 tiles of convolutions: rows and columns that leave tiles ragged, windows, strides
@pytest.mark.parametrize("n,h,c,o,k,s", [(16, 30, 64, 32, 7, 1), (16, 30, 64, 19, 7, 1), (9, 47, 64, 27, 5, 1),
                                         (7, 43, 48, 32, 7, 2), (4, 22, 288, 11, 7, 1), (2, 22, 288, 32, 7, 1),
                                         (33, 56, 48, 24, 3, 1), (5, 103, 64, 9, 3, 1), (16, 56, 64, 31, 3, 1),
                                         (16, 46, 128, 65, 3, 2), (1, 41, 272, 98, 7, 1), (3, 10, 960, 161, 3, 1),
                                         (18, 8, 320, 136, 7, 1), (20, 23, 224, 380, 3, 1), (9, 56, 64, 71, 5, 1),
                                         (11, 19, 128, 204, 7, 1), (4, 14, 128, 1000, 7, 1), (4, 48, 352, 51, 3, 1), (1, 5, 1392, 33, 5, 1)])
def test_convolution(capi, n, h, c, o, k, s):
    d, w = operands((n, h, h, c), (o, k, k, c))
    oh = (h + 2 * (k // 2) - k) // s + 1
    columns = torch.nn.functional.unfold(d.permute(0, 3, 1, 2).float(), k, padding=k // 2, stride=s)
    weight = w.permute(0, 3, 1, 2).reshape(o, -1).double()
    want = torch.cat([x.t().double() @ weight.t().contiguous() for x in columns]).reshape(n, oh, oh, o)
    same(lambda **kw: capi.quantized_conv_nhwc(d, w, None, *ranges(), pad=(k // 2, k // 2), stride=(s, s), **kw),
         (25, 1), want)
    for cfg in (40, 41, 42, 43):
        for splits in (1, 2, 5) if n * oh * oh < 20000 else (1,):  # (the partial sums of these fit)
            got = capi.quantized_conv_nhwc(d, w, None, *ranges(), pad=(k // 2, k // 2), stride=(s, s),
                                           want_int32=True, force=(cfg, splits))["out32"]
            assert torch.equal(got.double(), want), (cfg, splits)
