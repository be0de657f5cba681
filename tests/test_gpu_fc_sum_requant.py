"""The residual sum that is calibrated behind the operator, fused into the layer: against the
operators one after the other, to the last bit, on every kernel the chooser takes for it, ragged
widths, the corner values of both operands and ranges whose scales overflow."""
import pytest
import torch

from mxnet_amd import capi, contrib

pytestmark = pytest.mark.gpu


def scalar(v):
    return torch.tensor([v], dtype=torch.float32, device="cuda")


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("m,k,n", [
    (1, 16, 16), (33, 64, 48), (49, 2048, 512), (257, 250, 37),   # small, long, unaligned
    (32768, 64, 256), (32801, 128, 128),                          # the short-K streaming kernel
    (12544, 256, 1024), (50176, 128, 512), (3136, 512, 2048),     # 256- and 128-wide tiles
    (300, 96, 20)])                                               # output rows off 16 bytes
@pytest.mark.parametrize("ranges", [(3.0, 2.0, 4.0), (1e-3, 500.0, 0.7), (1e-30, 1e-30, 1e30)])
def test_fused_sum_is_the_operators(m, k, n, relu, ranges):
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    draw = lambda *s: torch.randint(-128, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight, bias, res = draw(m, k), draw(n, k), draw(n), draw(m, n)
    res[0, :2] = -128
    layer, residual, total = ranges
    args = [scalar(v) for v in (-1.0, 1.0, -2.0, 2.0, -0.5, 0.5)]
    res_range = scalar(-residual), scalar(residual)
    reach = layer * k ** 0.5
    got = capi.quantized_fc_sum(data, weight, bias, res, *args, *res_range, (-reach, reach),
                                (-total, 0.9 * total), sum_relu=relu, requant=True)
    q = capi.quantized_fc(data, weight, bias, *args, want_int32=False, calib=(-reach, reach))
    acc, lo, hi = contrib.quantized_elemwise_add(q["out8"], res, q["rmin"], q["rmax"], *res_range)
    want, lo, hi = contrib.requantize(acc, lo, hi, min_calib_range=-total,
                                      max_calib_range=0.9 * total)
    if relu:
        want, lo, hi = contrib.quantized_act(want, lo, hi)
    assert torch.equal(got["out8"], want)
    assert torch.equal(got["rmin"], lo) and torch.equal(got["rmax"], hi)
