"""The calls whose speed matters to a program that runs int8 networks on this package.

A case is a dict of plain values; `prepare` makes what such a program holds before the call
(inputs, int8 weights with their ranges, an executor), `run` makes one pass through the public
entry points.  The kinds:

  fc_layers    mxnet_amd.contrib: quantize_v2 -> quantized_fully_connected -> requantize ->
               dequantize for one or more layers, each on its own activations
  fc_fused     mxnet_amd.capi.quantized_fc with the calibrated requantize (and relu) fused
  casts        mxnet_amd.contrib: the cast operators on flat tensors
  conv_layers  mxnet_amd.contrib on NCHW: quantized_conv -> requantize -> quantized_act
  conv_fused   mxnet_amd.capi.quantized_conv_nhwc with relu and requantize fused
  network      mxnet_amd.executor.Executor.forward of a residual network quantized by
               mxnet_amd.quantization (stem, bottleneck stages, pooling, classifier)
  tensor_ops   mxnet_amd.contrib: the operators between the layers, NCHW int8
  calibrate    mxnet_amd.quantization.quantize_model: the offline direction, a float network
               and calibration batches in, thresholds and int8 parameters out
"""
import math

import torch

from mxnet_amd import capi, contrib
from mxnet_amd import quantization as Q
from mxnet_amd import symbol as S
from mxnet_amd.executor import Executor

# ResNet-50 v1 bottleneck convolutions as plane x in x out x kernel x stride
RESNET50_CONVS = ("56x64x64x1x1,56x64x64x3x1,56x64x256x1x1,56x256x64x1x1,56x256x128x1x2,"
                  "28x128x128x3x1,28x128x512x1x1,28x512x128x1x1,56x256x512x1x2,28x512x256x1x2,"
                  "14x256x256x3x1,14x256x1024x1x1,14x1024x256x1x1,28x512x1024x1x2,"
                  "14x1024x512x1x2,7x512x512x3x1,7x512x2048x1x1,7x2048x512x1x1,14x1024x2048x1x2")
# stages of its body as blocks x bottleneck width x output width x stride
RESNET50_STAGES = "3x64x256x1,4x128x512x2,6x256x1024x2,3x512x2048x2"
BERT_BASE_FCS = "768x2304,768x768,768x3072,3072x768"
CASTS = ("quantize", "quantize_uncal", "quantize_uint8_uncal", "requantize", "requantize_uncal",
         "dequantize")
TENSOR_OPS = ("add", "add_int8", "mul_int8", "act", "maxpool", "avgpool", "concat", "to_nhwc",
              "bn_relu", "flatten", "embedding")


def listed():
    return [
        # one layer of a small batch: the shortest call sequence a float caller makes
        {"name": "fc_layer_128x1024", "kind": "fc_layers", "rows": 128, "layers": "1024x1024",
         "calibrated": True, "bias": True, "outliers": False},
        # the same without calibration (ranges reduced on the device) at sizes of no power of 2
        {"name": "fc_layer_ragged", "kind": "fc_layers", "rows": 77, "layers": "1001x510",
         "calibrated": False, "bias": True, "outliers": True},
        # the FC layers of one BERT-base encoder block at 32 x 128 tokens
        {"name": "bert_base_fcs", "kind": "fc_layers", "rows": 4096, "layers": BERT_BASE_FCS,
         "calibrated": True, "bias": True, "outliers": True},
        # the square layers int8 rates are quoted on
        {"name": "fc_4096", "kind": "fc_fused", "rows": 4096, "inner": 4096, "hidden": 4096,
         "relu": False, "bias": True},
        {"name": "fc_8192", "kind": "fc_fused", "rows": 8192, "inner": 8192, "hidden": 8192,
         "relu": False, "bias": True},
        # large flat tensors: what the cast operators cost a network without fused layers
        {"name": "casts_64m", "kind": "casts", "n": 1 << 26,
         "ops": "quantize,quantize_uint8_uncal,requantize,dequantize"},
        # the bottleneck convolutions at batch 64, operator by operator
        {"name": "conv_operators_b64", "kind": "conv_layers", "batch": 64,
         "layers": RESNET50_CONVS, "calibrated": True, "bias": True},
        # the same layers for a caller that keeps its tensors NHWC and fuses the epilogue
        {"name": "conv_fused_b64", "kind": "conv_fused", "batch": 64, "layers": RESNET50_CONVS,
         "relu": True, "bias": True},
        # a whole quantized ResNet-50: throughput (batch 64) and latency (one image)
        {"name": "resnet50_b64", "kind": "network", "batch": 64, "size": 224,
         "stages": RESNET50_STAGES, "classes": 1000},
        {"name": "resnet50_b1", "kind": "network", "batch": 1, "size": 224,
         "stages": RESNET50_STAGES, "classes": 1000},
        # the operators between the layers, on the largest activation of that network
        {"name": "tensor_ops_b64", "kind": "tensor_ops", "batch": 64, "channels": 256,
         "size": 56, "ops": "add,act,maxpool,concat,to_nhwc,bn_relu,embedding"},
        # quantizing a trained feed-forward block, default calibration
        {"name": "calibrate_ffn", "kind": "calibrate", "rows": 256, "features": 768,
         "hidden": 3072, "batches": 2, "mode": "entropy"},
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of [lo, hi]; one in three rounded to 16."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if rng.random() < 1 / 3 and v >= 16:
        v = v // 16 * 16
    return max(lo, min(hi, v))


def _conv_list(rng, count):
    layers = []
    for _ in range(count):
        k = rng.choice((1, 1, 3, 3, 5, 7))
        s = rng.choice((1, 1, 1, 2))
        size = _log(rng, 7, 112)
        c = _log(rng, 3, 2048 if size < 16 else 512 if size < 57 else 128)
        o = _log(rng, 8, 2048 if size < 16 else 512 if size < 57 else 128)
        layers.append("%dx%dx%dx%dx%d" % (size, c, o, k, s))
    return ",".join(layers)


def draw(rng):
    while True:
        kind = rng.choice(("fc_layers", "fc_layers", "fc_fused", "casts", "conv_layers",
                           "conv_layers", "conv_fused", "network", "tensor_ops", "calibrate"))
        if kind == "fc_layers":
            layers = ",".join("%dx%d" % (_log(rng, 16, 4096), _log(rng, 8, 4096))
                              for _ in range(rng.choice((1, 1, 2, 4))))
            case = {"kind": kind, "rows": _log(rng, 1, 4096), "layers": layers,
                    "calibrated": rng.random() < 0.7, "bias": rng.random() < 0.8,
                    "outliers": rng.random() < 0.5}
        elif kind == "fc_fused":
            case = {"kind": kind, "rows": _log(rng, 1, 8192), "inner": _log(rng, 64, 8192),
                    "hidden": _log(rng, 16, 8192), "relu": rng.random() < 0.5,
                    "bias": rng.random() < 0.8}
        elif kind == "casts":
            case = {"kind": kind, "n": _log(rng, 1, 1 << 26),
                    "ops": ",".join(rng.sample(CASTS, rng.choice((1, 2, 4))))}
        elif kind == "conv_layers":
            case = {"kind": kind, "batch": _log(rng, 1, 64),
                    "layers": _conv_list(rng, rng.choice((1, 1, 2, 4))),
                    "calibrated": rng.random() < 0.8, "bias": rng.random() < 0.8}
        elif kind == "conv_fused":
            case = {"kind": kind, "batch": _log(rng, 1, 64),
                    "layers": _conv_list(rng, rng.choice((1, 1, 2, 4))),
                    "relu": rng.random() < 0.7, "bias": rng.random() < 0.8}
        elif kind == "network":
            stages, width = [], _log(rng, 16, 64)
            for i in range(rng.choice((1, 2, 3, 4))):
                stages.append("%dx%dx%dx%d" % (rng.choice((1, 2, 3)), width, 4 * width,
                                               1 if i == 0 else 2))
                width *= 2
            case = {"kind": kind, "batch": _log(rng, 1, 64), "size": _log(rng, 32, 224),
                    "stages": ",".join(stages), "classes": _log(rng, 10, 1000)}
        elif kind == "tensor_ops":
            case = {"kind": kind, "batch": _log(rng, 1, 64), "channels": _log(rng, 3, 512),
                    "size": _log(rng, 7, 112),
                    "ops": ",".join(rng.sample(TENSOR_OPS, rng.choice((1, 2, 4))))}
        else:
            case = {"kind": kind, "rows": _log(rng, 8, 256), "features": _log(rng, 32, 768),
                    "hidden": _log(rng, 64, 3072), "batches": rng.choice((1, 2, 3)),
                    "mode": rng.choice(("naive", "entropy"))}
        w = work(case)
        # no draw costs more than the largest listed cases
        if w["bytes"] <= 0.7e9 and w["flops"] <= 5.2e11 or kind == "fc_fused":
            return case


# ---- inputs --------------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _scalar(v):
    return torch.tensor([float(v)], dtype=torch.float32, device="cuda")


def _int8(g, *shape):
    return torch.randint(-127, 128, shape, device="cuda", generator=g, dtype=torch.int8)


def _activations(g, shape, outliers):
    """U(-1,1), or N(0,1) with 0.1% of the values at +-20 (transformer activations)."""
    if not outliers:
        return torch.rand(shape, device="cuda", generator=g) * 2 - 1
    x = torch.randn(shape, device="cuda", generator=g)
    far = torch.rand(shape, device="cuda", generator=g) < 0.001
    return torch.where(far, 20.0 * x.sign(), x)


def _own_range(w):
    """A float parameter over its own range, as the parameter conversion does it."""
    return capi.quantize(w, w.min().reshape(1), w.max().reshape(1), "int8")


def _weight(g, shape, fan_in, std=None):
    return _own_range(torch.randn(shape, device="cuda", generator=g)
                      * (std if std is not None else math.sqrt(2.0 / fan_in)))


def _bias(g, n, wanted):
    if not wanted:
        return None, None, None
    return _own_range(torch.randn(n, device="cuda", generator=g) * 0.1)


def _fcs(text):
    return [tuple(int(v) for v in layer.split("x")) for layer in text.split(",")]


def _convs(text):
    """(plane, in, out, kernel, stride, pad, out plane) of every layer."""
    rows = []
    for layer in text.split(","):
        size, c, o, k, s = (int(v) for v in layer.split("x"))
        rows.append((size, c, o, k, s, k // 2, (size + 2 * (k // 2) - k) // s + 1))
    return rows


# ---- the quantized residual network ----------------------------------------------------------


def _network_convs(case):
    """Every convolution as (name, plane, in, out, kernel, stride, out plane), and the
    classifier's input width."""
    size = (case["size"] + 6 - 7) // 2 + 1
    rows = [("stem", case["size"], 3, 64, 7, 2, size)]
    size = (size + 2 - 3) // 2 + 1
    width = 64
    for i, stage in enumerate(case["stages"].split(",")):
        blocks, mid, out, stride = (int(v) for v in stage.split("x"))
        for j in range(blocks):
            s = stride if j == 0 else 1
            after = (size - 1) // s + 1
            tag = "s%db%d" % (i, j)
            rows.append((tag + "a", size, width, mid, 1, s, after))
            rows.append((tag + "b", after, mid, mid, 3, 1, after))
            rows.append((tag + "c", after, mid, out, 1, 1, after))
            if j == 0:
                rows.append((tag + "p", size, width, out, 1, s, after))
            size, width = after, out
    return rows, width


class _KnownRanges(Q.CalibrationCollector):
    """Thresholds a program has from an earlier calibration."""

    def __init__(self, ranges):
        super().__init__()
        self.min_max_dict = ranges


def _network(case, g):
    """The float network with batch norm folded into the convolutions, its parameters and the
    range of every tensor that gets calibrated (4.5 standard deviations, propagated)."""
    params, ranges = {}, {}
    convs = {row[0]: row for row in _network_convs(case)[0]}

    def conv(x, m2, name, gain=1.0):
        _, _, c, o, k, s, _ = convs[name]
        std = gain * math.sqrt(2.0 / (c * k * k))
        params[name + "_weight"] = torch.randn((o, c, k, k), device="cuda", generator=g) * std
        sigma = std * math.sqrt(c * k * k * m2)
        params[name + "_bias"] = torch.randn(o, device="cuda", generator=g) * (0.1 * sigma)
        ranges[name + "_output"] = (-4.5 * sigma, 4.5 * sigma)
        y = S.Convolution(x, kernel=(k, k), stride=(s, s), pad=(k // 2, k // 2), num_filter=o,
                          name=name)
        return y, sigma * sigma

    def relu(x, m2, name):
        return S.Activation(x, act_type="relu", name=name), m2 / 2

    ranges["stem_data"] = (-4.5, 4.5)
    x, m2 = conv(S.Variable("data"), 1.0, "stem")
    x, m2 = relu(x, m2, "stem_relu")
    x, m2 = S.Pooling(x, kernel=(3, 3), stride=(2, 2), pad=(1, 1), pool_type="max",
                      name="stem_pool"), 3 * m2
    for i, stage in enumerate(case["stages"].split(",")):
        for j in range(int(stage.split("x")[0])):
            tag = "s%db%d" % (i, j)
            y, n2 = conv(x, m2, tag + "a")
            y, n2 = relu(y, n2, tag + "a_relu")
            y, n2 = conv(y, n2, tag + "b")
            y, n2 = relu(y, n2, tag + "b_relu")
            y, n2 = conv(y, n2, tag + "c", gain=0.5)
            if j == 0:
                x, m2 = conv(x, m2, tag + "p")
            total = n2 + m2
            ranges[tag + "_sum_output"] = (-4.5 * math.sqrt(total), 4.5 * math.sqrt(total))
            x = S.elemwise_add(y, x, name=tag + "_sum")
            x, m2 = S.Activation(x, act_type="relu", name=tag + "_relu"), 0.75 * total
    x = S.Pooling(x, kernel=(7, 7), global_pool=True, pool_type="avg", name="pool")
    x = S.Flatten(x, name="flat")
    width = _network_convs(case)[1]
    params["fc_weight"] = torch.randn((case["classes"], width), device="cuda",
                                      generator=g) * math.sqrt(1.0 / width)
    params["fc_bias"] = torch.randn(case["classes"], device="cuda", generator=g) * 0.1
    ranges["fc_output"] = (-4.5 * math.sqrt(m2), 4.5 * math.sqrt(m2))
    return S.FullyConnected(x, num_hidden=case["classes"], name="fc"), params, ranges


def _quantized_network(case, g):
    sym, params, ranges = _network(case, g)
    known = _KnownRanges(ranges)
    qsym, _, _, known, _ = Q.quantize_graph(sym, params, {}, calib_mode="custom",
                                            LayerOutputCollector=known)
    qsym, qarg, _ = Q.calib_graph(qsym, params, {}, known, calib_mode="custom")
    return Executor(qsym, qarg)


# ---- prepare / run -----------------------------------------------------------------------------


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    state = dict(case)
    if kind == "fc_layers":
        state["rows_of"] = []
        for (inner, hidden) in _fcs(case["layers"]):
            x = _activations(g, (case["rows"], inner), case["outliers"])
            w = _weight(g, (hidden, inner), inner, std=0.02)
            b = _bias(g, hidden, case["bias"])
            limit = 20.0 if case["outliers"] else 1.0
            reach = 4.5 * 0.02 * math.sqrt(inner * (1.4 if case["outliers"] else 1 / 3))
            state["rows_of"].append((hidden, x, w, b, limit, reach))
    elif kind == "fc_fused":
        m, k, n = case["rows"], case["inner"], case["hidden"]
        x = _activations(g, (m, k), False)
        state["data"] = capi.quantize_v2(x, "int8", min_calib_range=-1.0, max_calib_range=1.0)
        state["weight"] = _weight(g, (n, k), k, std=0.02)
        state["bias_q"] = _bias(g, n, case["bias"])
        reach = 4.5 * 0.02 * math.sqrt(k / 3.0)
        state["calib"] = (-reach, reach)
    elif kind == "casts":
        n = case["n"]
        x = torch.randn(n, device="cuda", generator=g)
        if n > 1000:  # 0.01% outliers
            x[torch.randint(0, n, (n // 10000 + 1,), device="cuda", generator=g)] = 50.0
        state["x"] = x
        state["acc"] = torch.randint(-2 ** 28, 2 ** 28, (n,), device="cuda", generator=g,
                                     dtype=torch.int32)
        state["q"] = _int8(g, n)
        state["range"] = (_scalar(-3.0), _scalar(3.0))
    elif kind in ("conv_layers", "conv_fused"):
        state["rows_of"] = []
        for (size, c, o, k, s, pad, _) in _convs(case["layers"]):
            shape = (c, size, size) if kind == "conv_layers" else (size, size, c)
            x = torch.randn((case["batch"],) + shape, device="cuda", generator=g)
            d = capi.quantize_v2(x, "int8", min_calib_range=-4.5, max_calib_range=4.5)
            wshape = (c, k, k) if kind == "conv_layers" else (k, k, c)
            w = _weight(g, (o,) + wshape, c * k * k)
            b = _bias(g, o, case["bias"])
            state["rows_of"].append(((k, s, pad, o), d, w, b, 4.5 * math.sqrt(2.0)))
    elif kind == "network":
        state["executor"] = _quantized_network(case, g)
        state["data"] = torch.randn((case["batch"], 3, case["size"], case["size"]),
                                    device="cuda", generator=g)
    elif kind == "tensor_ops":
        b, c, h = case["batch"], case["channels"], case["size"]
        state["a"], state["b"] = _int8(g, b, c, h, h), _int8(g, b, c, h, h)
        state["range"] = (_scalar(-3.0), _scalar(3.0))
        state["wide"] = (_scalar(-4.0), _scalar(4.0))
        state["bn"] = [torch.rand(c, device="cuda", generator=g) + 0.5,
                       torch.randn(c, device="cuda", generator=g),
                       torch.randn(c, device="cuda", generator=g),
                       torch.rand(c, device="cuda", generator=g) + 0.5]
        state["table"] = _int8(g, 30522, c)
        state["ids"] = torch.randint(0, 30522, (b, h), device="cuda", generator=g,
                                     dtype=torch.int32)
    else:
        x = S.FullyConnected(S.Variable("data"), num_hidden=case["hidden"], flatten=False,
                             name="fc1")
        x = S.Activation(x, act_type="relu", name="relu1")
        state["sym"] = S.FullyConnected(x, num_hidden=case["features"], flatten=False, name="fc2")
        state["arg"] = {
            name: torch.randn(shape, device="cuda", generator=g) * 0.02 for name, shape in (
                ("fc1_weight", (case["hidden"], case["features"])),
                ("fc1_bias", (case["hidden"],)),
                ("fc2_weight", (case["features"], case["hidden"])),
                ("fc2_bias", (case["features"],)))}
        state["batches_of"] = [_activations(g, (case["rows"], case["features"]), True)
                               for _ in range(case["batches"])]
    return state


def _run_fc_layers(state):
    outs = []
    for (hidden, x, (w, wlo, whi), (b, blo, bhi), limit, reach) in state["rows_of"]:
        first = {"min_calib_range": -limit, "max_calib_range": limit}
        second = {"min_calib_range": -reach, "max_calib_range": reach}
        if not state["calibrated"]:
            first = second = {}
        q, lo, hi = contrib.quantize_v2(x, out_type="int8", **first)
        acc, lo, hi = contrib.quantized_fully_connected(
            q, w, b, lo, hi, wlo, whi, blo, bhi, num_hidden=hidden, no_bias=b is None,
            flatten=False)
        q, lo, hi = contrib.requantize(acc, lo, hi, **second)
        outs.append((q, contrib.dequantize(q, lo, hi)))
    return outs


def _run_casts(state):
    outs = []
    for op in state["ops"].split(","):
        if op == "quantize":
            outs.append(contrib.quantize_v2(state["x"], out_type="int8", min_calib_range=-50.0,
                                            max_calib_range=50.0))
        elif op == "quantize_uncal":
            outs.append(contrib.quantize_v2(state["x"], out_type="int8"))
        elif op == "quantize_uint8_uncal":
            outs.append(contrib.quantize_v2(state["x"], out_type="uint8"))
        elif op == "requantize":
            outs.append(contrib.requantize(state["acc"], *state["range"], min_calib_range=-0.3,
                                           max_calib_range=0.3))
        elif op == "requantize_uncal":
            outs.append(contrib.requantize(state["acc"], *state["range"]))
        else:
            outs.append(contrib.dequantize(state["q"], *state["range"]))
    return outs


def _run_conv_layers(state):
    outs = []
    for ((k, s, pad, o), (d, lo, hi), (w, wlo, whi), (b, blo, bhi), reach) in state["rows_of"]:
        acc, lo, hi = contrib.quantized_conv(
            d, w, b, lo, hi, wlo, whi, blo, bhi, kernel=(k, k), stride=(s, s), pad=(pad, pad),
            num_filter=o, no_bias=b is None)
        ranges = {"min_calib_range": -reach, "max_calib_range": reach}
        q, lo, hi = contrib.requantize(acc, lo, hi, **(ranges if state["calibrated"] else {}))
        outs.append(contrib.quantized_act(q, lo, hi, act_type="relu"))
    return outs


def _run_conv_fused(state):
    outs = []
    for ((k, s, pad, _), (d, lo, hi), (w, wlo, whi), (b, blo, bhi), reach) in state["rows_of"]:
        r = capi.quantized_conv_nhwc(d, w, b, lo, hi, wlo, whi, blo, bhi, stride=(s, s),
                                     pad=(pad, pad), want_int32=False, calib=(-reach, reach),
                                     relu=state["relu"])
        outs.append((r["out8"], r["rmin"], r["rmax"]))
    return outs


def _run_tensor_ops(state):
    a, b, (lo, hi), (wlo, whi) = state["a"], state["b"], state["range"], state["wide"]
    outs = []
    for op in state["ops"].split(","):
        if op == "add":
            outs.append(contrib.quantized_elemwise_add(a, b, lo, hi, wlo, whi))
        elif op == "add_int8":
            outs.append(contrib.quantized_elemwise_add(a, b, lo, hi, wlo, whi,
                                                       min_calib_range=-5.0, max_calib_range=5.0))
        elif op == "mul_int8":
            outs.append(contrib.quantized_elemwise_mul(a, b, lo, hi, wlo, whi,
                                                       min_calib_range=-12.0,
                                                       max_calib_range=12.0))
        elif op == "act":
            outs.append(contrib.quantized_act(a, lo, hi))
        elif op == "maxpool":
            outs.append(contrib.quantized_pooling(a, lo, hi, kernel=(3, 3), stride=(2, 2),
                                                  pad=(1, 1), pool_type="max"))
        elif op == "avgpool":
            outs.append(contrib.quantized_pooling(a, lo, hi, kernel=(7, 7), global_pool=True,
                                                  pool_type="avg"))
        elif op == "concat":
            outs.append(contrib.quantized_concat(a, b, lo, hi, wlo, whi, dim=1))
        elif op == "to_nhwc":
            outs.append(contrib.quantized_transpose(a, lo, hi, axes=(0, 2, 3, 1)))
        elif op == "bn_relu":
            outs.append(contrib.quantized_batch_norm(a, *state["bn"], lo, hi, fix_gamma=False,
                                                     min_calib_range=-6.0, max_calib_range=6.0,
                                                     relu=True))
        elif op == "flatten":
            outs.append(contrib.quantized_flatten(a, lo, hi))
        else:
            outs.append(contrib.quantized_embedding(state["ids"], state["table"], lo, hi,
                                                    input_dim=30522,
                                                    output_dim=state["channels"]))
    return outs


def _run_calibrate(state):
    qsym, qarg, _ = Q.quantize_model(state["sym"], state["arg"], {}, calib_mode=state["mode"],
                                     calib_data=state["batches_of"], quantize_mode="full")
    found = {}
    for name, attrs in qsym.attr_dict().items():
        if "min_calib_range" in attrs:
            found[name] = (float(attrs["min_calib_range"]), float(attrs["max_calib_range"]))
    return found, {name: qarg[name] for name in qarg}


def run(state):
    kind = state["kind"]
    if kind == "fc_layers":
        return _run_fc_layers(state)
    if kind == "fc_fused":
        r = capi.quantized_fc(*state["data"][:1], state["weight"][0], state["bias_q"][0],
                              *state["data"][1:], *state["weight"][1:], *state["bias_q"][1:],
                              want_int32=False, calib=state["calib"], relu=state["relu"])
        return r["out8"], r["rmin"], r["rmax"]
    if kind == "casts":
        return _run_casts(state)
    if kind == "conv_layers":
        return _run_conv_layers(state)
    if kind == "conv_fused":
        return _run_conv_fused(state)
    if kind == "network":
        return state["executor"].forward(data=state["data"])
    if kind == "tensor_ops":
        return _run_tensor_ops(state)
    return _run_calibrate(state)


# ---- what a pass cannot do without --------------------------------------------------------------


def work(case):
    """Bytes: what each call of the pass takes and hands back, read or written once (operator
    calls hand back their int32 results; fused calls and the executor owe the caller none, there
    an int8 activation is written by its layer and read by the next).  Operations: two per
    multiply-accumulate of the layers."""
    kind = case["kind"]
    nbytes = flops = 0.0
    if kind == "fc_layers":
        m = case["rows"]
        for (k, n) in _fcs(case["layers"]):
            # float in, int8 out; int8 operands, int32 out; int32 in, int8 out; int8 in, float out
            nbytes += 5.0 * m * k + m * k + n * k + 4.0 * m * n + 5.0 * m * n + 5.0 * m * n
            flops += 2.0 * m * k * n
    elif kind == "fc_fused":
        m, k, n = case["rows"], case["inner"], case["hidden"]
        nbytes, flops = float(m * k + n * k + m * n), 2.0 * m * k * n
    elif kind == "casts":
        nbytes = 5.0 * case["n"] * len(case["ops"].split(","))
    elif kind in ("conv_layers", "conv_fused"):
        for (size, c, o, k, s, pad, after) in _convs(case["layers"]):
            out = float(case["batch"]) * o * after * after
            nbytes += float(case["batch"]) * c * size * size + o * c * k * k
            # fused: int8 out; operators: int32 out and in, int8 out, in and out
            nbytes += out if kind == "conv_fused" else 11.0 * out
            flops += 2.0 * out * c * k * k
    elif kind == "network":
        convs, width = _network_convs(case)
        nbytes = 4.0 * case["batch"] * 3 * case["size"] ** 2 + 4.0 * case["batch"] * case["classes"]
        nbytes += width * case["classes"]
        flops = 2.0 * case["batch"] * width * case["classes"]
        for (name, size, c, o, k, s, after) in convs:
            # an int8 activation is written once and read by the next layer
            nbytes += o * c * k * k + 2.0 * case["batch"] * o * after * after
            flops += 2.0 * case["batch"] * o * after * after * c * k * k
    elif kind == "tensor_ops":
        n = float(case["batch"]) * case["channels"] * case["size"] ** 2
        per = {"add": 6.0, "add_int8": 3.0, "mul_int8": 3.0, "act": 2.0, "maxpool": 1.25,
               "avgpool": 1.0, "concat": 4.0, "to_nhwc": 2.0, "bn_relu": 2.0, "flatten": 2.0,
               "embedding": 2.0 / case["size"]}
        nbytes = sum(per[op] * n for op in case["ops"].split(","))
    else:
        m, k, h = case["rows"] * case["batches"], case["features"], case["hidden"]
        # calibrated tensors: the input, both layers' outputs; weights in float, out in int8
        nbytes = 4.0 * m * (2 * k + 2 * h) + 5.0 * 2 * k * h
        flops = 4.0 * m * k * h
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Integer results are exact.  Float results are one rounding of an integer times a scale
    (or a reduction's own operand), so they stay within a few units of the last place; the
    thresholds of a calibration follow a float32 network."""
    if case["kind"] == "calibrate":
        return {"rel": 1e-5}
    return {"rel": 1e-6}
