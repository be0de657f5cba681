"""Plans of quantized graphs against the same graphs walked operator by operator: every output
the same to the last bit, for channel counts off the padding, odd planes, every fused chain and
the layers that stay registered operators between them."""
import pytest
import torch

from mxnet_amd import _lib, contrib
from mxnet_amd import quantization as Q
from mxnet_amd import symbol as S
from mxnet_amd.executor import Executor

pytestmark = pytest.mark.gpu


class KnownRanges(Q.CalibrationCollector):
    def post_collect(self):
        return {name: (-3.0, 3.0) for name in self.include_layers}


def quantized(sym, shapes, seed=0, skip=()):
    """(executor of the int8 graph, every requantize but those of `skip` calibrated)"""
    g = torch.Generator(device="cuda").manual_seed(seed)
    params = {n: torch.randn(s, device="cuda", generator=g) * (0.4 if n.endswith("bias") else 0.15)
              for n, s in shapes.items()}
    qsym, _, _, known, _ = Q.quantize_graph(sym, params, {}, calib_mode="custom",
                                            LayerOutputCollector=KnownRanges())
    known.include_layers = [n for n in known.include_layers if not n.startswith(tuple(skip) or "-")]
    qsym, qarg, _ = Q.calib_graph(qsym, params, {}, known, calib_mode="custom")
    return Executor(qsym, qarg)


def walked(ex, **feed):
    """The same forward pass operator by operator: a hook sees every tensor."""
    other = Executor(ex.symbol, ex.params)
    other.register_op_hook(lambda *a: None)
    return other.forward(**feed)


def check(ex, plan=True, **feed):
    want = walked(ex, **feed)
    for _ in range(2):
        got = ex.forward(**feed)
        assert len(got) == len(want)
        for a, b in zip(got, want):
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b)
    assert (next(iter(ex._plans.values())) is not None) == plan


def conv(x, name, o, k=1, s=1, p=None, **kw):
    return S.Convolution(x, kernel=(k, k), stride=(s, s), pad=((k // 2 if p is None else p),) * 2,
                         num_filter=o, name=name, **kw)


def relu(x, name):
    return S.Activation(x, act_type="relu", name=name)


def residual_net(c, mid, out, stride, classes, stem_k=7):
    shapes = {}

    def layer(x, name, i, o, k=1, s=1):
        shapes[name + "_weight"], shapes[name + "_bias"] = (o, i, k, k), (o,)
        return conv(x, name, o, k, s)

    x = relu(layer(S.Variable("data"), "stem", c, mid, stem_k, 2), "stem_relu")
    x = S.Pooling(x, kernel=(3, 3), stride=(2, 2), pad=(1, 1), pool_type="max", name="pool1")
    width = mid
    for b in range(2):
        y = relu(layer(x, "a%d" % b, width, mid, 1, stride if b == 0 else 1), "ra%d" % b)
        y = relu(layer(y, "b%d" % b, mid, mid, 3), "rb%d" % b)
        y = layer(y, "c%d" % b, mid, out)
        if b == 0:
            x = layer(x, "p", width, out, 1, stride)
        x = relu(S.elemwise_add(y, x, name="sum%d" % b), "rs%d" % b)
        width = out
    x = S.Flatten(S.Pooling(x, kernel=(2, 2), global_pool=True, pool_type="avg", name="gap"),
                  name="flat")
    shapes["fc_weight"], shapes["fc_bias"] = (classes, out), (classes,)
    return S.FullyConnected(x, num_hidden=classes, name="fc"), shapes


@pytest.mark.parametrize("batch,c,mid,out,stride,size", [
    (1, 3, 16, 64, 2, 32), (2, 3, 37, 148, 1, 45), (3, 1, 19, 33, 2, 31), (5, 4, 64, 256, 1, 56),
    (2, 5, 16, 48, 1, 33), (64, 3, 64, 256, 1, 64)])
def test_residual_network(batch, c, mid, out, stride, size):
    sym, shapes = residual_net(c, mid, out, stride, 10 + mid)
    x = torch.randn(batch, c, size, size, device="cuda")
    check(quantized(sym, shapes), data=x)


@pytest.mark.parametrize("pool_type,kernel,stride,pad,convention,count", [
    ("max", 2, 2, 0, "valid", True), ("avg", 3, 2, 1, "full", True), ("avg", 3, 1, 1, "valid", False),
    ("max", 3, 2, 1, "full", True), ("avg", 5, 3, 2, "valid", True), ("avg", 4, 4, 0, "valid", True)])
def test_pooling_between_convolutions(pool_type, kernel, stride, pad, convention, count):
    x = conv(S.Variable("data"), "c1", 24, 3)
    x = S.Pooling(x, kernel=(kernel,) * 2, stride=(stride,) * 2, pad=(pad,) * 2,
                  pool_type=pool_type, pooling_convention=convention, count_include_pad=count,
                  name="pool")
    sym = conv(x, "c2", 17, 3)
    ex = quantized(sym, {"c1_weight": (24, 6, 3, 3), "c1_bias": (24,),
                         "c2_weight": (17, 24, 3, 3), "c2_bias": (17,)})
    check(ex, data=torch.randn(2, 6, 19, 19, device="cuda"))


def test_sums_that_no_convolution_takes():
    """A 3 x 3 convolution's sum, a sum without relu, one operand used again, and a sum whose
    operands are the same tensor."""
    x = conv(S.Variable("data"), "c1", 20, 3)
    y = conv(x, "c2", 20, 3)
    s1 = S.elemwise_add(y, x, name="s1")
    s2 = S.elemwise_add(conv(s1, "c3", 20), s1, name="s2")
    s3 = relu(S.elemwise_add(s2, s2, name="s3"), "r3")
    sym = S.Group([conv(s3, "c4", 8), conv(s2, "c5", 9, 3, 2)])
    shapes = {}
    for n, (o, k) in {"c1": (20, 3), "c2": (20, 3), "c3": (20, 1), "c4": (8, 1),
                      "c5": (9, 3)}.items():
        shapes[n + "_weight"], shapes[n + "_bias"] = (o, 20 if n != "c1" else 7, k, k), (o,)
    check(quantized(sym, shapes), data=torch.randn(3, 7, 14, 14, device="cuda"))


def test_uncalibrated_layers_and_operators_without_an_nhwc_form():
    x = conv(S.Variable("data"), "c1", 24, 3, no_bias=True)
    y = conv(x, "c2", 24, 3)  # its requantize stays uncalibrated: registered operators
    z = S.Concat(relu(conv(x, "c3", 10), "r"), y, name="cat")
    z = conv(z, "c4", 12)
    sym = S.FullyConnected(S.transpose(z, axes=(0, 2, 3, 1), name="t"), num_hidden=6, name="fc")
    shapes = {"c1_weight": (24, 3, 3, 3), "c2_weight": (24, 24, 3, 3), "c2_bias": (24,),
              "c3_weight": (10, 24, 1, 1), "c3_bias": (10,), "c4_weight": (12, 34, 1, 1),
              "c4_bias": (12,), "fc_weight": (6, 12 * 9 * 9), "fc_bias": (6,)}
    check(quantized(sym, shapes, skip=("c2",)), data=torch.randn(2, 3, 9, 9, device="cuda"))


@pytest.mark.parametrize("flatten,shape", [(True, (9, 40)), (False, (3, 5, 40)), (False, (1, 48))])
def test_fully_connected_network(flatten, shape):
    x = relu(S.FullyConnected(S.Variable("data"), num_hidden=50, flatten=flatten, name="f1"), "r")
    x = S.FullyConnected(x, num_hidden=33, flatten=flatten, no_bias=True, name="f2")
    sym = S.FullyConnected(x, num_hidden=7, flatten=flatten, name="f3")
    shapes = {"f1_weight": (50, shape[-1]), "f1_bias": (50,), "f2_weight": (33, 50),
              "f3_weight": (7, 33), "f3_bias": (7,)}
    check(quantized(sym, shapes), data=torch.randn(*shape, device="cuda"))


def test_parameters_that_change():
    sym, shapes = residual_net(3, 16, 32, 1, 11)
    ex = quantized(sym, shapes)
    x = torch.randn(2, 3, 40, 40, device="cuda")
    check(ex, data=x)
    w = ex.params["b0_weight_quantize"]
    w.copy_(-w)                                              # in place
    check(ex, data=x)
    ex.params["a1_weight_quantize"] = torch.zeros_like(ex.params["a1_weight_quantize"])
    ex.params["fc_weight_quantize_max"] = ex.params["fc_weight_quantize_max"] * 2
    check(ex, data=x)


def test_shapes_and_streams_take_turns():
    sym, shapes = residual_net(3, 16, 32, 1, 11)
    ex = quantized(sym, shapes)
    xs = [torch.randn(b, 3, 40, 40, device="cuda") for b in (1, 3, 2, 1, 3)]
    want = [walked(ex, data=x)[0] for x in xs]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for _ in range(3):
        got = []
        for i, x in enumerate(xs):
            with torch.cuda.stream(side if i % 2 else torch.cuda.current_stream()):
                got.append(ex.forward(data=x)[0])
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert len(ex._plans) == 3


def test_replayed_plan():
    """A captured forward pass: the graph's replays give what eager passes give."""
    sym, shapes = residual_net(3, 16, 32, 1, 11)
    ex = quantized(sym, shapes)
    x = torch.randn(2, 3, 40, 40, device="cuda")
    ex.forward(data=x)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ex.forward(data=x)[0]
    for seed in range(4):
        x.copy_(torch.randn(x.shape, device="cuda", generator=torch.Generator(
            device="cuda").manual_seed(seed)))
        want = walked(ex, data=x)[0]
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_graphs_that_are_walked():
    data = S.Variable("data")
    sym = S.softmax(S.FullyConnected(data, num_hidden=7, name="f"), name="s")
    check(quantized(sym, {"f_weight": (7, 16), "f_bias": (7,)}), plan=False,
          data=torch.randn(4, 16, device="cuda"))


@pytest.mark.parametrize("n,c,h,w,stride,pad,convention", [
    (1, 16, 1, 1, 1, 1, "valid"), (2, 48, 7, 9, 2, 1, "valid"), (3, 16, 8, 5, 3, 2, "valid"),
    (1, 64, 33, 20, 1, 0, "valid"), (2, 32, 10, 11, 2, 1, "full"), (1, 16, 4, 4, 3, 1, "full")])
def test_nhwc_max_over_3x3_windows(n, c, h, w, stride, pad, convention):
    """The NHWC kernel of the plans against the NCHW operator, -128 and the image's borders among
    the windows' contents."""
    g = torch.Generator(device="cuda").manual_seed(h * w)
    x = torch.randint(-128, -100, (n, c, h, w), device="cuda", generator=g, dtype=torch.int8)
    lo, hi = (torch.tensor([v], dtype=torch.float32, device="cuda") for v in (-1.0, 1.0))
    want = contrib.quantized_pooling(x, lo, hi, kernel=(3, 3), stride=(stride,) * 2,
                                     pad=(pad,) * 2, pool_type="max",
                                     pooling_convention=convention)[0]
    oh, ow = want.shape[2:]
    nhwc = x.permute(0, 2, 3, 1).contiguous()
    out = torch.empty((n, oh, ow, c), dtype=torch.int8, device="cuda")
    _lib.check(_lib.lib.mxq_quantized_pooling_nhwc(
        torch.cuda.current_stream().cuda_stream, nhwc.data_ptr(), n, h, w, c, 3, 3, stride, stride,
        pad, pad, oh, ow, 0, 1, out.data_ptr()))
    assert torch.equal(out.permute(0, 3, 1, 2), want)
