"""The transposes of planes to pixels that ask nothing of the plane's size or the channel count:
alone, with channels padded, and with the weights of a convolution in the same launch."""
import numpy as np
import pytest
import torch

import oracle
from tests.data_gen import int8_uniform

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# planes of one column, below, at and above a tile's 64 columns; one piece a row, three, four and more,
# the last with a single channel; channels padded by more than a piece
@pytest.mark.parametrize("N, C, H, W, padded", [
    (1, 1, 1, 1, 16), (3, 16, 1, 1, 16), (2, 7, 3, 3, 16), (2, 47, 9, 7, 48), (3, 33, 5, 13, 48),
    (2, 65, 9, 9, 80), (1, 64, 63, 1, 64), (2, 100, 13, 5, 144), (2, 49, 21, 11, 64),
    (1, 1362, 3, 5, 1376), (2, 128, 15, 15, 128), (5, 16, 29, 29, 32)])
@pytest.mark.parametrize("offset", [0, 1])
def test_planes_to_padded_pixels(N, C, H, W, padded, offset):
    from mxnet_amd._lib import check, lib
    x = int8_uniform((N, C, H, W), seed=C + H)
    held = torch.zeros(x.size + 1, dtype=torch.int8, device="cuda")
    held[offset:offset + x.size] = dev(x).ravel()
    size = N * H * W * padded
    out = torch.full((size + 64,), 0x5A, dtype=torch.int8, device="cuda")
    check(lib.mxq_nchw_to_nhwc_pad_i8(torch.cuda.current_stream().cuda_stream,
                                      held.data_ptr() + offset, out.data_ptr(), N, C, H, W, padded))
    host = out.cpu().numpy()
    want = np.zeros((N, H, W, padded), np.int8)
    want[..., :C] = x.transpose(0, 2, 3, 1)
    np.testing.assert_array_equal(host[:size].reshape(want.shape), want)
    assert (host[size:] == 0x5A).all()


# 3 x 3, 5 x 5, 8 x 8 and 9 x 9 windows (64 and 81 taps), over planes of each kernel that carries them
@pytest.mark.parametrize("N, C, H, O, k", [
    (2, 47, 16, 46, 3), (2, 7, 29, 35, 3), (1, 9, 21, 33, 5), (3, 130, 9, 20, 3), (2, 200, 20, 24, 3),
    (1, 65, 12, 5, 8), (1, 20, 13, 6, 9), (2, 13, 11, 8, 1), (1, 1, 5, 1, 3),
    (2, 32, 12, 37, 3), (1, 16, 16, 70, 5), (1, 48, 8, 3, 9)])  # whole pieces only
def test_data_and_weights_in_one_launch(N, C, H, O, k):
    from mxnet_amd import capi
    d, w, b = (int8_uniform((N, C, H, H), seed=C), int8_uniform((O, C, k, k), seed=O),
               int8_uniform((O,), seed=k))
    r = (-2.0, 2.0, -0.1, 0.1, -1.0, 1.0)
    want, lo, hi = oracle.quantized_conv(d, w, b, *r, (1, 1), (k // 2, k // 2))
    got = capi.quantized_conv_nchw(dev(d), dev(w), dev(b),
                                   *[dev(np.array([v], np.float32)) for v in r],
                                   pad=(k // 2, k // 2))
    np.testing.assert_array_equal(got["out32"].cpu().numpy(), want)


# images that fill a launch's third extent leave no room in it for the weights
@pytest.mark.parametrize("N", [65532, 65533, 65534])
def test_weights_stay_behind_where_images_fill_the_grid(N):
    from mxnet_amd import capi
    d, w, b = (int8_uniform((N, 3, 2, 2), seed=1), int8_uniform((64, 3, 3, 3), seed=2),
               int8_uniform((64,), seed=3))
    r = (-2.0, 2.0, -0.1, 0.1, -1.0, 1.0)
    want = oracle.quantized_conv(d, w, b, *r, (1, 1), (1, 1))[0]
    got = capi.quantized_conv_nchw(dev(d), dev(w), dev(b),
                                   *[dev(np.array([v], np.float32)) for v in r], pad=(1, 1))
    np.testing.assert_array_equal(got["out32"].cpu().numpy(), want)
