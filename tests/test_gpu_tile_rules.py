"""Fully-connected layers and convolutions at the lines of the tile rules, against float64 products (exact
for these lengths) and, requantized, against the smallest tile pinned."""
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


# two tiles of 64 x 64 a CU (of 256), a few more; lengths around 256, 512, 768, 1024 and 2048
@pytest.mark.parametrize("M,N", [(32768, 64), (32769, 50), (2048, 1024), (2049, 1000), (3000, 1024),
                                 (3000, 970), (130, 200)])
@pytest.mark.parametrize("K", [240, 256, 272, 496, 512, 528, 1040, 2032, 2064])
def test_fully_connected(capi, M, N, K):
    d, w = operands((M, K), (N, K))
    same(lambda **kw: capi.quantized_fc(d, w, None, *ranges(), **kw), (44, 1, 0),
         d.double() @ w.double().t().contiguous())


# one round of 128 x 128 tiles (two to a CU of 256) and a little more, 256 x 256 tiles of one round, a
# little and much more
@pytest.mark.parametrize("M,N", [(8192, 1024), (8193, 1020), (33000, 200), (70000, 100), (131072, 72),
                                 (4352, 4351), (5120, 5120)])
@pytest.mark.parametrize("K", [256, 272, 512, 1040])
def test_fully_connected_of_larger_tiles(capi, M, N, K):
    d, w = operands((M, K), (N, K))
    same(lambda **kw: capi.quantized_fc(d, w, None, *ranges(), **kw), (44, 1, 0),
         d.double() @ w.double().t().contiguous())


@pytest.mark.parametrize("M,K,N", [(8192, 8192, 33), (4096, 8208, 64), (700, 4112, 900)])
def test_long_reductions_of_few_tiles(capi, M, K, N):
    d, w = operands((M, K), (N, K))
    same(lambda **kw: capi.quantized_fc(d, w, None, *ranges(), **kw), (44, 1, 0),
         d.double() @ w.double().t().contiguous())


@pytest.mark.parametrize("n,h,c,o", [(16, 14, 32, 512), (16, 14, 48, 512), (16, 14, 64, 512),
                                     (16, 14, 80, 512), (16, 14, 96, 500), (16, 28, 48, 256),
                                     (16, 28, 48, 270), (16, 28, 64, 270), (32, 28, 64, 64),
                                     (32, 28, 80, 40), (16, 25, 128, 64), (16, 25, 464, 40),
                                     (23, 56, 32, 128), (23, 56, 32, 100), (28, 40, 64, 300),
                                     (20, 31, 80, 300), (24, 40, 128, 276), (23, 40, 288, 640)])
def test_convolution(capi, n, h, c, o):
    d, w = operands((n, h, h, c), (o, 3, 3, c))
    columns = torch.nn.functional.unfold(d.permute(0, 3, 1, 2).float(), 3, padding=1)  # n, c * 9, h * h
    weight = w.permute(0, 3, 1, 2).reshape(o, c * 9).double()
    want = columns.transpose(1, 2).reshape(n * h * h, c * 9).double() @ weight.t().contiguous()
    same(lambda **kw: capi.quantized_conv_nhwc(d, w, None, *ranges(), pad=(1, 1), **kw), (25, 1),
         want.reshape(n, h, h, o))
