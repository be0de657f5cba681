"""What the margin of the entropy bounds rests on: a logarithm of at most two last places on every normal
number, and quotients that are the division's."""
import pytest
import torch

from mxnet_amd._lib import check, lib

pytestmark = pytest.mark.gpu


def functions(a, b=None, exact=None, near=None, logs=None):
    ptr = lambda t: None if t is None else t.data_ptr()
    check(lib.mxq_test_entropy_functions(torch.cuda.current_stream().cuda_stream, ptr(a), ptr(b), a.numel(),
                                         ptr(exact), ptr(near), ptr(logs)))


def test_logarithm_of_every_normal_number():
    chunk, worst = 1 << 26, 0.0
    logs = torch.empty(chunk, device="cuda")
    for first in range(0x00800000, 0x7f800000, chunk):
        bits = torch.arange(first, min(first + chunk, 0x7f800000), dtype=torch.int32, device="cuda")
        x = bits.view(torch.float32)
        functions(x, logs=logs)
        want = x.double().log()
        off = (logs[:x.numel()].double() - want).abs_() / want.abs()
        off[want == 0] = logs[:x.numel()][want == 0].double().abs()
        worst = max(worst, off.max().item())
    assert worst <= 4 * 2.0 ** -24, worst * 2.0 ** 24


def inverse(b, bits):
    """Of odd numbers, modulo 2 ** bits."""
    x = b.clone()
    for _ in range(5):
        x = x * (2 - b * x) & (1 << bits) - 1
    return x


def check_quotients(a, b):
    a, b = a.float(), b.float()
    exact, near = torch.empty_like(a), torch.empty_like(a)
    functions(a, b, exact, near)
    want = (a.double() / b.double()).float()  # (53 bits are enough for the rounding to 24)
    assert torch.equal(exact, want)
    assert (near.view(torch.int32) - want.view(torch.int32)).abs().max().item() <= 1


@pytest.mark.parametrize("n", [n for n in range(-7, 8) if n])
def test_quotients_next_to_a_midpoint(n):
    """b = B 2^-23 and a midpoint M of 25 bits, n / b from it in units of 2^-48 (a quotient below one) or 2^-47:
    a 2^23 = (B M + n) / 2^25 or 2^24.  B may hold as many factors of two as n does."""
    for bits, least in ((25, 1), (24, 1 << 23)):
        for k in range(3):
            if n % (1 << k):
                continue
            odd = torch.arange((1 << 23 - k) | 1, 1 << 24 - k, 2, dtype=torch.int64, device="cuda")
            first = inverse(odd, bits - k) * (-n >> k) & (1 << bits - k) - 1
            for more in range(0, 1 << 25, 1 << bits - k):
                m, b = first + more, odd << k
                a = b * m + n >> bits
                ok = (m > 1 << 24) & (m < 1 << 25) & (m % 2 == 1) & (a >= least) & (a < 1 << 24)
                assert (((a << bits) - b * m)[ok] == n).all()
                if bits == 25:
                    ok &= a < b
                if ok.any():
                    check_quotients(a[ok], b[ok])


@pytest.mark.parametrize("scale", [1.0, 2.0 ** -60, 2.0 ** 31])
def test_quotients_of_any_numbers(scale):
    g = torch.Generator(device="cuda").manual_seed(int(scale) + 3)
    for _ in range(4):
        a, b = ((torch.rand(1 << 24, device="cuda", generator=g, dtype=torch.float64) + 1e-6).float() for _ in "ab")
        check_quotients(a * scale, b * scale ** 0.5)
