"""The steps that plans put in the place of layers: that they are taken where a graph has them, and
that the pass is the walked one's with each, also after its parameters have changed."""
import pytest
import torch

from mxnet_amd import _frontend, _plan
from mxnet_amd import symbol as S
from tests.test_gpu_plan import check, conv, quantized, relu, residual_net

pytestmark = pytest.mark.gpu


@pytest.fixture
def kinds(monkeypatch):
    """The kinds of the steps of the plans made since."""
    seen, make = [], _frontend.plan

    def plan(size, held, steps, outputs):
        seen.append([s[0] for s in steps])
        return make(size, held, steps, outputs)

    monkeypatch.setattr(_frontend, "plan", plan)
    return seen


def conv3_net(c, o, after):
    """Layers of 3 x 3 over many channels, on their own: the second is no block's (nothing is added
    to it), the third has a column tile that is short."""
    shapes = {"a_weight": (c, 5, 1, 1), "a_bias": (c,), "b_weight": (o, c, 3, 3), "b_bias": (o,),
              "c_weight": (after, o, 1, 1), "c_bias": (after,)}
    x = relu(conv(S.Variable("data"), "a", c), "ra")
    x = relu(conv(x, "b", o, 3), "rb")
    return conv(x, "c", after), shapes


@pytest.mark.parametrize("batch,c,o,h,w", [(64, 512, 512, 7, 7), (32, 256, 112, 14, 13),
                                           (30, 500, 256, 9, 11)])
def test_3x3_over_many_channels(kinds, batch, c, o, h, w):
    sym, shapes = conv3_net(c, o, 20)
    ex = quantized(sym, shapes)
    x = torch.randn(batch, 5, h, w, device="cuda")
    check(ex, data=x)
    assert len(kinds) == 1 and kinds[0].count(_plan._CONV3) == 1
    laid = [key for key in ex._structure().laid if key[1] == "conv3x3"]
    assert len(laid) == 1
    weight = ex.params["b_weight_quantize"]
    weight.copy_(weight.flip(0).roll(1, 2))           # in place: laid out anew
    check(ex, data=x)
    ex.params["b_weight_quantize"] = -weight          # another tensor
    ex.params["b_weight_quantize_max"] = ex.params["b_weight_quantize_max"] * 2
    check(ex, data=x)
    ex.params["b_bias_quantize"] = ex.params["b_bias_quantize"].flip(0)
    check(ex, data=x)
    assert all(k.count(_plan._CONV3) == 1 for k in kinds)
    # few pixels take the general way, beside the same executor's other plans
    check(ex, data=x[:1])
    assert kinds[-1].count(_plan._CONV3) == 0
    check(ex, data=x)


@pytest.mark.parametrize("batch,c,mid,out,size", [(2, 3, 64, 256, 64), (1, 1, 32, 64, 44),
                                                  (5, 4, 48, 192, 58)])
def test_stem_pair_and_blocks(kinds, batch, c, mid, out, size):
    sym, shapes = residual_net(c, mid, out, 1, 10)
    ex = quantized(sym, shapes)
    x = torch.randn(batch, c, size, size, device="cuda")
    check(ex, data=x)
    for name in ("stem", "a0", "p"):
        weight = ex.params[name + "_weight_quantize"]
        weight.copy_(weight.flip(0))
        check(ex, data=x)
        ex.params[name + "_weight_quantize_max"] = ex.params[name + "_weight_quantize_max"] * 1.5
        check(ex, data=x)
    assert len(kinds) > 1
    for k in kinds:
        assert (k.count(_plan._CONV_POOL), k.count(_plan._PAIR), k.count(_plan._BLOCK)) == (1, 1, 2)
