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


@pytest.mark.parametrize("m,k,n", [
    (1, 64, 16), (33, 64, 256), (49, 2048, 512), (32768, 64, 256), (32801, 128, 128),
    (49185, 32, 64), (12289, 64, 512), (24577, 128, 128), (131073, 64, 256), (12544, 256, 1024),
    (50176, 128, 512), (3136, 512, 2048), (300, 96, 20)])
@pytest.mark.parametrize("ranges", [
    (3.0, 2.0, 4.0), (1.37, 5.21, 3.3), (4.0, 4.0, 4.0),      # the last: exact ties in number
    (1e-3, 500.0, 0.7), (1e-30, 1e-30, 1e30), (0.0, 1.0, 1.0)])
def test_short_form_is_the_sum(m, k, n, ranges):
    """With what sum_requant_pairs found, or did not find, the launch gives the same bits: every
    pair of int8 operands occurs in the larger shapes."""
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    draw = lambda *s: torch.randint(-128, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight, bias, res = draw(m, k), draw(n, k), draw(n), draw(m, n)
    layer, residual, total = ranges
    args = [scalar(v) for v in (-1.0, 1.0, -2.0, 2.0, -0.5, 0.5)]
    reach = layer * k ** 0.5
    call = lambda pairs: capi.quantized_fc_sum(
        data, weight, bias, res, *args, scalar(-residual), scalar(residual), (-reach, reach),
        (-total, 0.9 * total), sum_relu=True, requant=True, pairs=pairs)["out8"]
    pairs = capi.sum_requant_pairs((-reach, reach), (-residual, residual),
                                   (-total, 0.9 * total))
    want = call(None)
    assert torch.equal(call(pairs), want)


@pytest.mark.parametrize("m,k,n", [(33, 64, 64), (130, 96, 132), (65, 128, 37), (40, 256, 128)])
@pytest.mark.parametrize("force", [(1, 1, 0), (3, 1, 0), (4, 1, 0), (43, 1, 0), (44, 1, 0),
                                   (55, 1, 0), (71, 4, 0), (71, -8, 0)])
def test_short_form_on_every_kind_of_kernel(m, k, n, force):
    """Register-staged, direct-to-LDS and few-tiles kernels, rows on and off the 4- and 16-byte
    marks."""
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    draw = lambda *s: torch.randint(-128, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight, bias, res = draw(m, k), draw(n, k), draw(n), draw(m, n)
    args = [scalar(v) for v in (-1.0, 1.0, -2.0, 2.0, -0.5, 0.5, -2.0, 2.0)]
    reach = 3.0 * k ** 0.5
    pairs = capi.sum_requant_pairs((-reach, reach), (-2.0, 2.0), (-4.0, 4.0))
    assert int(pairs[2]) == 1
    got, want = (capi.quantized_fc_sum(data, weight, bias, res, *args, (-reach, reach),
                                       (-4.0, 4.0), sum_relu=True, requant=True, force=force,
                                       pairs=p)["out8"] for p in (pairs, None))
    assert torch.equal(got, want)


def test_short_form_is_found_for_most_ranges():
    g = torch.Generator().manual_seed(0)
    found = [capi.sum_requant_pairs(*((-v, v) for v in (0.5 + 4 * torch.rand(3, generator=g))
                                      .tolist()))[2] for _ in range(64)]
    assert sum(int(f) for f in found) >= 48
    assert int(capi.sum_requant_pairs((-1.0, 1.0), (0.0, 0.0), (0.0, 0.0))[2]) == 0


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("m,k,n", [
    (12289, 64, 512), (24577, 128, 128), (3073, 32, 1024), (49153, 32, 64), (6145, 128, 1024)])
def test_streamed_layer_is_the_operators(m, k, n, relu):
    """The short-K streaming kernel at one row more than it is chosen from, both strip widths,
    several strips of columns: against the int32 output and a requantize of its own."""
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    draw = lambda *s: torch.randint(-128, 128, s, device="cuda", generator=g, dtype=torch.int8)
    data, weight, bias = draw(m, k), draw(n, k), draw(n)
    args = [scalar(v) for v in (-1.0, 1.0, -2.0, 2.0, -0.5, 0.5)]
    calib = -2.0 * k ** 0.5, 1.9 * k ** 0.5
    got = capi.quantized_fc(data, weight, bias, *args, want_int32=False, calib=calib, relu=relu)
    acc = capi.quantized_fc(data, weight, bias, *args)
    want, lo, hi = contrib.requantize(acc["out32"], acc["omin"], acc["omax"],
                                      min_calib_range=calib[0], max_calib_range=calib[1])
    if relu:
        want, lo, hi = contrib.quantized_act(want, lo, hi)
    assert torch.equal(got["out8"], want)
