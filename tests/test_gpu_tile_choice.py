"""Which tile, and how many work-groups a tile, the entry points choose: at the lines of the rules, with the
workspace that they ask for and without one.  The other tests of these tiles compare values, which a rule that
no longer chose them would leave as they are."""
import ctypes

import pytest
import torch

from mxnet_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def capi():
    import mxnet_amd
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are drawn by the compute units, here for 256")
    return mxnet_amd.capi


def chosen(entry, *args, workspace=0):
    cfg, splits = ctypes.c_int(), ctypes.c_int()
    at = 4096 if workspace else None  # looked at for its alignment alone
    check(entry(*args, at, workspace, ctypes.byref(cfg), ctypes.byref(splits)))
    return cfg.value, splits.value


def partial_sums(tiles, splits, outputs):
    return tiles * splits * outputs * 4


# rows, reduction, columns; configuration and work-groups a tile with the workspace that is asked for, and without
FULLY_CONNECTED = [(1024, 1520, 1024, (59, 1), (59, 1)), (1024, 1536, 1024, (33, 1), (33, 1)),
                   (1024, 4096, 1024, (33, 1), (33, 1)), (12351, 3872, 64, (33, 1), (33, 1)),
                   (1090, 8176, 79, (71, 0), (71, 0)), (1090, 8208, 79, (33, 5), (33, 1)),
                   (4000, 8176, 79, (33, 1), (33, 1)), (4000, 8208, 79, (33, 2), (33, 1)),
                   (121, 8208, 153, (71, 0), (71, 0)), (121, 32752, 153, (71, 0), (71, 0)),
                   (121, 32784, 153, (33, 12), (71, 0)),
                   (720, 14320, 799, (33, 1), (33, 1)), (720, 15680, 799, (34, 6), (33, 1)),
                   (475, 29008, 1145, (34, 7), (33, 1)), (784, 8176, 1387, (59, 1), (59, 1)),
                   (784, 8192, 1387, (34, 3), (59, 1)), (699, 8176, 2429, (59, 1), (59, 1)),
                   (699, 8192, 2429, (34, 2), (59, 1)),
                   (2048, 1520, 2048, (53, 1), (53, 1)), (2048, 1536, 2048, (34, 1), (34, 1))]


@pytest.mark.parametrize("M,K,N,split,whole", FULLY_CONNECTED)
def test_fully_connected(capi, M, K, N, split, whole):
    room = lib.mxq_quantized_fc_workspace(M, N, K, 1)
    assert chosen(lib.mxq_test_fc_plan, M, N, K, 1, 0, 0, workspace=room) == split
    assert chosen(lib.mxq_test_fc_plan, M, N, K, 1, 0, 0) == whole
    if split[1] > 1:
        side = 64 if split[0] == 33 else 128
        tiles = -(-M // side) * -(-N // side)
        sums = partial_sums(tiles, split[1], side * side)
        assert sums < room <= sums + 4 * tiles + 256  # and a counter a tile
        assert chosen(lib.mxq_test_fc_plan, M, N, K, 1, 0, 0, workspace=room - 1) == whole
    else:
        assert room == 0


# images, plane, channels in and out, window, stride; 128 x 32, 64 x 64 and 128 x 128 tiles on eight waves, 128 x 32
# tiles, the window kernel on 128 and 256 pixels and where its rows don't fit
CONVOLUTIONS = [((16, 30, 30, 512, 32, 7, 1), (41, 2), (40, 1)), ((36, 21, 21, 496, 8, 5, 1), (41, 2), (40, 1)),
                ((12, 41, 41, 240, 11, 7, 1), (41, 1), (41, 1)), ((34, 10, 10, 592, 922, 3, 2), (40, 1), (40, 1)),
                ((19, 10, 10, 592, 1145, 7, 2), (43, 7), (40, 1)), ((18, 23, 23, 224, 380, 3, 1), (43, 1), (43, 1)),
                ((1, 5, 5, 1392, 33, 5, 1), (40, 12), (63, 1)), ((31, 74, 74, 80, 10, 7, 1), (42, 1), (42, 1)),
                ((32, 23, 23, 16, 87, 7, 1), (66, 1), (66, 1)), ((61, 40, 40, 16, 24, 3, 1), (66, 1), (66, 1)),
                ((63, 111, 111, 16, 13, 7, 1), (67, 1), (67, 1)), ((15, 66, 66, 16, 75, 5, 1), (67, 1), (67, 1)),
                ((11, 40, 236, 16, 20, 7, 1), (42, 1), (42, 1))]


@pytest.mark.parametrize("layer,split,whole", CONVOLUTIONS)
def test_convolution(capi, layer, split, whole):
    n, h, w, c, o, k, s = layer
    geometry = (n, h, w, c, o, k, k, s, s, k // 2, k // 2, 1, 1)
    room = lib.mxq_quantized_conv_workspace(*geometry, 1)
    assert chosen(lib.mxq_test_conv_plan, *geometry, workspace=room) == split
    assert chosen(lib.mxq_test_conv_plan, *geometry) == whole
    assert (room > 0) == (split[1] > 1)


def operands(*shapes):
    g = torch.Generator(device="cuda").manual_seed(sum(map(sum, shapes)))
    return [torch.randint(-128, 128, s, dtype=torch.int8, device="cuda", generator=g) for s in shapes]


def ranges():
    return [torch.tensor([v], device="cuda") for v in (-1.0, 1.0, -0.1, 0.1)]


# a caller without room for the partial sums of a long reduction: the kernel for few tiles
@pytest.mark.parametrize("M,N", [(121, 153), (33, 17)])
def test_long_reduction_without_a_workspace(capi, M, N):
    d, w = operands((M, 32784), (N, 32784))
    want = d.double() @ w.double().t().contiguous()
    for force in (None, (0, 0, 0)):
        got = capi.quantized_fc(d, w, None, *ranges(), want_int32=True, force=force)["out32"]
        assert torch.equal(got.double(), want)


def test_convolution_without_a_workspace(capi):
    d, w = operands((1, 5, 5, 1392), (33, 5, 5, 1392))
    want = torch.nn.functional.conv2d(d.permute(0, 3, 1, 2).double().cpu(), w.permute(0, 3, 1, 2).double().cpu(),
                                      padding=2).permute(0, 2, 3, 1)
    for force in (None, (0, 0)):
        got = capi.quantized_conv_nhwc(d, w, None, *ranges(), pad=(2, 2), want_int32=True, force=force)["out32"]
        assert torch.equal(got.cpu().double(), want)


def test_rows_past_the_window_kernels_room(capi):
    """236 pixels a row: 128 pixels' rows fit, those of 256 do not, which the rule would take."""
    d, w = operands((11, 40, 236, 16), (20, 7, 7, 16))
    want = torch.nn.functional.conv2d(d.permute(0, 3, 1, 2).double().cpu(), w.permute(0, 3, 1, 2).double().cpu(),
                                      padding=3).permute(0, 2, 3, 1)
    for force in (None, (66, 1)):
        got = capi.quantized_conv_nhwc(d, w, None, *ranges(), pad=(3, 3), want_int32=True, force=force)["out32"]
        assert torch.equal(got.cpu().double(), want)
    with pytest.raises(Exception, match="window kernel"):
        capi.quantized_conv_nhwc(d, w, None, *ranges(), pad=(3, 3), want_int32=True, force=(67, 1))
