"""Outputs whose rows are no multiple of 16 bytes (or of 4 integers), or that begin off a mark:
the tiled kernels write them in whole pieces, the last one of a row in parts.  What lies before and
behind the output stays."""
import numpy as np
import pytest
import torch

import oracle
from tests.data_gen import int8_uniform

pytestmark = pytest.mark.gpu

GUARD = 64  # bytes on either side
RD, RW, RB = 2.0, 0.1, 1.0
CALIB = (-30.0, 28.0)


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def scalars(*values):
    return [dev(np.array([v], np.float32)) for v in values]


class Guarded:
    def __init__(self, shape, dtype, offset):
        self.shape, self.dtype, self.front = shape, dtype, GUARD + offset
        self.nbytes = int(np.prod(shape)) * np.dtype(dtype).itemsize
        self.buf = torch.full((self.front + self.nbytes + GUARD,), 0x5A, dtype=torch.uint8,
                              device="cuda")

    def ptr(self):
        return self.buf.data_ptr() + self.front

    def get(self):
        host = self.buf.cpu().numpy()
        assert (host[:self.front] == 0x5A).all(), "written in front of the output"
        assert (host[self.front + self.nbytes:] == 0x5A).all(), "written behind the output"
        return host[self.front:self.front + self.nbytes].copy().view(self.dtype).reshape(self.shape)


# every tile of the direct-to-LDS kernels; widths that end in each part of a piece
@pytest.mark.parametrize("cfg", [12, 31, 41, 43, 44, 24, 51, 53, 56, 57, 58, 59, 60])
@pytest.mark.parametrize("N, offset", [(395, 0), (135, 4), (30, 1), (257, 0), (64, 8), (9, 3),
                                       (1, 0)])
def test_fc_rows_of_any_width(cfg, N, offset):
    from mxnet_amd._lib import check, lib
    M, K = 131, 128
    d, w, b = (int8_uniform((M, K), seed=N), int8_uniform((N, K), seed=N + 1),
               int8_uniform((N,), seed=2))
    acc, lo, hi = oracle.quantized_fully_connected(d, w, b, -RD, RD, -RW, RW, -RB, RB)
    want8 = oracle.requantize(acc, lo, hi, *CALIB)[0]
    held = [dev(a) for a in (d, w, b)] + scalars(-RD, RD, -RW, RW, -RB, RB)
    out = torch.empty(4, dtype=torch.float32, device="cuda")
    p = [out.data_ptr() + 4 * i for i in range(4)]
    for want32, wants8 in ((False, True), (True, False), (True, True)):
        o8 = Guarded((M, N), np.int8, offset) if wants8 else None
        o32 = Guarded((M, N), np.int32, 4 * (offset % 4)) if want32 else None
        check(lib.mxq_test_quantized_fc(
            torch.cuda.current_stream().cuda_stream, *[t.data_ptr() for t in held[:3]], M, N, K,
            *[t.data_ptr() for t in held[3:]], o32.ptr() if o32 else None, p[0], p[1],
            o8.ptr() if o8 else None, p[2], p[3], 0, *CALIB, None, 0, cfg, 1, 0))
        if o8:
            np.testing.assert_array_equal(o8.get(), want8)
        if o32:
            np.testing.assert_array_equal(o32.get(), acc)


@pytest.mark.parametrize("cfg", [12, 41, 43, 44, 51, 57])
@pytest.mark.parametrize("N, offset, relu", [(395, 0, 1), (30, 1, 0), (9, 0, 1), (64, 4, 0)])
def test_fc_sum_rows_of_any_width(cfg, N, offset, relu):
    from mxnet_amd._lib import check, lib
    M, K = 131, 128
    d, w, b = (int8_uniform((M, K), seed=N), int8_uniform((N, K), seed=N + 1),
               int8_uniform((N,), seed=2))
    res = int8_uniform((M, N), seed=7)
    reach, sums = 20.0, (-40.0, 35.0)
    acc, lo, hi = oracle.quantized_fully_connected(d, w, b, -RD, RD, -RW, RW, -RB, RB)
    q, qlo, qhi = oracle.requantize(acc, lo, hi, *CALIB)
    want = oracle.quantized_elemwise_add(q, res, qlo, qhi, -reach, reach, min_calib_range=sums[0],
                                         max_calib_range=sums[1])[0]
    if relu:
        want = oracle.relu_i8(want)
    held = [dev(a) for a in (d, w, b)] + scalars(-RD, RD, -RW, RW, -RB, RB)
    r = Guarded((M, N), np.int8, offset)
    r.buf[r.front:r.front + r.nbytes] = dev(res.view(np.uint8).ravel())
    rs = scalars(-reach, reach)
    out = torch.empty(4, dtype=torch.float32, device="cuda")
    p = [out.data_ptr() + 4 * i for i in range(4)]
    o = Guarded((M, N), np.int8, offset)
    check(lib.mxq_test_quantized_fc_sum(
        torch.cuda.current_stream().cuda_stream, *[t.data_ptr() for t in held[:3]], M, N, K,
        *[t.data_ptr() for t in held[3:]], r.ptr(), *[t.data_ptr() for t in rs], o.ptr(), *p,
        *CALIB, *sums, relu, None, 0, cfg, 1, 0))
    np.testing.assert_array_equal(o.get(), want)


@pytest.mark.parametrize("cfg", [11, 22, 23, 24, 25, 31, 33, 36, 37, 38, 39])
@pytest.mark.parametrize("O, H", [(57, 6), (30, 7), (131, 8)])
def test_conv_rows_and_planes_of_any_channel_count(cfg, O, H):
    from mxnet_amd import capi
    N, C = 3, 16
    d, w, b = (int8_uniform((N, C, H, H), seed=O), int8_uniform((O, C, 3, 3), seed=1),
               int8_uniform((O,), seed=2))
    acc, lo, hi = oracle.quantized_conv(d, w, b, -RD, RD, -RW, RW, -RB, RB, (1, 1), (1, 1))
    want8 = oracle.requantize(acc, lo, hi, *CALIB)[0]
    s = scalars(-RD, RD, -RW, RW, -RB, RB)
    got = capi.quantized_conv_nhwc(dev(d.transpose(0, 2, 3, 1)), dev(w.transpose(0, 2, 3, 1)),
                                   dev(b), *s, pad=(1, 1), want_int32=False, calib=CALIB,
                                   relu=False, force=(cfg, 1))
    np.testing.assert_array_equal(got["out8"].cpu().numpy().transpose(0, 3, 1, 2), want8)
    planes = capi.quantized_conv_nchw(dev(d), dev(w), dev(b), *s, pad=(1, 1))
    np.testing.assert_array_equal(planes["out32"].cpu().numpy(), acc)


# tiles whose stages are too small to turn a 32-bit tile round: stored as they lie
@pytest.mark.parametrize("O", [112, 113, 114, 115])
@pytest.mark.parametrize("H", [33, 40])
def test_conv_planes_from_small_tiles(O, H):
    from mxnet_amd import capi
    d, w, b = (int8_uniform((8, 3, H, H), seed=O), int8_uniform((O, 3, 3, 3), seed=1),
               int8_uniform((O,), seed=2))
    acc = oracle.quantized_conv(d, w, b, -RD, RD, -RW, RW, -RB, RB, (2, 2), (1, 1))[0]
    planes = capi.quantized_conv_nchw(dev(d), dev(w), dev(b), *scalars(-RD, RD, -RW, RW, -RB, RB),
                                      stride=(2, 2), pad=(1, 1))
    np.testing.assert_array_equal(planes["out32"].cpu().numpy(), acc)


# reductions below 64 bytes on either side of the tiles from which the rows are padded first
@pytest.mark.parametrize("M, K, N", [(1569, 13, 1024), (1537, 13, 1024), (1536, 13, 1024),
                                     (3000, 1, 600), (2048, 63, 1001), (50000, 11, 14)])
def test_fc_short_rows_of_many_tiles(M, K, N):
    from mxnet_amd import capi
    d, w, b = (int8_uniform((M, K), seed=N), int8_uniform((N, K), seed=N + 1),
               int8_uniform((N,), seed=2))
    acc, lo, hi = oracle.quantized_fully_connected(d, w, b, -RD, RD, -RW, RW, -RB, RB)
    want8 = oracle.requantize(acc, lo, hi, *CALIB)[0]
    got = capi.quantized_fc(dev(d), dev(w), dev(b), *scalars(-RD, RD, -RW, RW, -RB, RB),
                            want_int32=True, calib=CALIB)
    np.testing.assert_array_equal(got["out32"].cpu().numpy(), acc)
    np.testing.assert_array_equal(got["out8"].cpu().numpy(), want8)


# convolutions on either side of the lines between the tiles of 64 and 128 pixels
@pytest.mark.parametrize("M_side, C, O, k, N", [
    (16, 64, 57, 3, 127), (16, 64, 57, 3, 129), (16, 128, 30, 3, 130), (16, 128, 30, 3, 16),
    (12, 176, 132, 5, 40), (16, 512, 20, 3, 20), (32, 512, 33, 3, 33), (7, 208, 9, 9, 3),
    (64, 16, 41, 3, 33), (64, 16, 24, 3, 32)])
def test_conv_of_few_channels_out(M_side, C, O, k, N):
    from mxnet_amd import capi
    d, w, b = (int8_uniform((N, C, M_side, M_side), seed=O), int8_uniform((O, C, k, k), seed=1),
               int8_uniform((O,), seed=2))
    r = (-RD, RD, -RW, RW, -RB, RB)
    x, y, z = (dev(a) for a in (d.transpose(0, 2, 3, 1), w.transpose(0, 2, 3, 1), b))
    got = capi.quantized_conv_nhwc(x, y, z, *scalars(*r), pad=(k // 2, k // 2), want_int32=True,
                                   calib=CALIB)
    want = capi.quantized_conv_nhwc(x, y, z, *scalars(*r), pad=(k // 2, k // 2), want_int32=True,
                                    force=(25, 1))
    assert torch.equal(got["out32"], want["out32"])
    acc = got["out32"].cpu().numpy()
    some = [0, N - 1]
    few, lo, hi = oracle.quantized_conv(d[some], w, b, *r, (1, 1), (k // 2, k // 2))
    np.testing.assert_array_equal(acc[some].transpose(0, 3, 1, 2), few)
    # the bytes of all images, with int32 rows beside them and alone
    want8 = oracle.requantize(acc, lo, hi, *CALIB)[0]
    alone = capi.quantized_conv_nhwc(x, y, z, *scalars(*r), pad=(k // 2, k // 2), want_int32=False,
                                     calib=CALIB)
    for out in (got, alone):
        np.testing.assert_array_equal(out["out8"].cpu().numpy(), want8)


# more than six tiles a CU over weights, or data, of fewer than the 16 bytes that a padding copy reads at
# once, and of 16 exactly
@pytest.mark.parametrize("M, K, N", [(50000, 3, 4), (50000, 1, 8), (50000, 13, 1), (50000, 15, 1),
                                     (50000, 2, 8), (50000, 3, 6), (1, 3, 60000), (5, 3, 60000),
                                     (6, 3, 60000)])
def test_fc_operands_of_a_few_bytes(M, K, N):
    from mxnet_amd import capi
    d, w, b = (int8_uniform((M, K), seed=N), int8_uniform((N, K), seed=N + 1),
               int8_uniform((N,), seed=2))
    acc, lo, hi = oracle.quantized_fully_connected(d, w, b, -RD, RD, -RW, RW, -RB, RB)
    want8 = oracle.requantize(acc, lo, hi, *CALIB)[0]
    got = capi.quantized_fc(dev(d), dev(w), dev(b), *scalars(-RD, RD, -RW, RW, -RB, RB),
                            want_int32=True, calib=CALIB)
    np.testing.assert_array_equal(got["out32"].cpu().numpy(), acc)
    np.testing.assert_array_equal(got["out8"].cpu().numpy(), want8)


@pytest.mark.parametrize("O", [3, 4, 5, 6])
def test_conv_1x1_of_an_image_to_a_few_channels(O):
    from mxnet_amd import capi
    d, w, b = (int8_uniform((1, 3, 224, 224), seed=O), int8_uniform((O, 3, 1, 1), seed=1),
               int8_uniform((O,), seed=2))
    r = (-RD, RD, -RW, RW, -RB, RB)
    want = oracle.quantized_conv(d, w, b, *r, (1, 1), (0, 0))[0]
    got = capi.quantized_conv_nhwc(dev(d.transpose(0, 2, 3, 1)), dev(w.transpose(0, 2, 3, 1)),
                                   dev(b), *scalars(*r), want_int32=True)
    np.testing.assert_array_equal(got["out32"].cpu().numpy().transpose(0, 3, 1, 2), want)
