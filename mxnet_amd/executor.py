"""A minimal symbol executor for calibration runs and end-to-end checks.

It walks a symbol in depth-first post-order and evaluates each node on the GPU: the
`_contrib_*` operators through the C++ operator host (FCompute<gpu> of this package),
the float operators of the surrounding network through torch.  The reference runs
symbols through CachedOp / the graph executor (src/imperative/cached_op.cc), which is
outside this package; this is only the harness the calibration collectors hook into,
the way `SymbolBlock.register_op_hook(collector.collect, monitor_all=True)` does in
`_collect_layer_statistics` (python/mxnet/contrib/quantization.py:364-380): the callback
sees every operator output as `<node>_<output name>` and, with monitor_all, every
operator input as `<node>_<argument name>`; operators without registered names get
the decimal output index and `input<i>` (src/common/utils.cc:53-107).

Without a hook, a graph of quantized operators runs as a plan (_plan.py): one native call per
forward pass, the same outputs.  A pass under stream capture is walked.
"""
import threading

import torch

from . import _frontend, _plan
from . import operator as _operator

# Input shape combinations an executor keeps a plan for, the ones used last.  A plan by itself is
# small (1 KiB of device memory for a quantized ResNet-50); the laid-out weights are the graph's, for
# all of its plans: 11 MB packed, and what its launches of several layers (7 MB at batch 64, 1 on one
# image) and of 3 x 3 layers over many channels (7 MB at batch 64) read, made of those and beside them.
_MAX_PLANS = 64


def _tuple(text, n=2, default=None):
    if text is None:
        return default
    t = text.strip().strip("()[]")
    vals = tuple(int(x) for x in t.split(",") if x.strip())
    return vals if vals else default


def _bool(text, default=False):
    if text is None:
        return default
    return text.strip().lower() in ("true", "1")


def _convolution(a, data, weight, bias=None):
    kernel = _tuple(a.get("kernel"))
    return torch.nn.functional.conv2d(data, weight, bias, stride=_tuple(a.get("stride"), default=(1, 1)),
                                      padding=_tuple(a.get("pad"), default=(0, 0)),
                                      dilation=_tuple(a.get("dilate"), default=(1, 1)),
                                      groups=int(a.get("num_group", "1")))


def _fully_connected(a, data, weight, bias=None):
    if _bool(a.get("flatten"), True):
        data = data.reshape(data.shape[0], -1)
    return torch.nn.functional.linear(data, weight, bias)


def _activation(a, data):
    return {"relu": torch.relu, "sigmoid": torch.sigmoid, "tanh": torch.tanh,
            "softrelu": torch.nn.functional.softplus,
            "softsign": torch.nn.functional.softsign}[a["act_type"]](data)


def _pooling(a, data):
    pool_type = a.get("pool_type", "max")
    if _bool(a.get("global_pool")):
        return data.amax(dim=(2, 3), keepdim=True) if pool_type == "max" else \
            data.mean(dim=(2, 3), keepdim=True)
    kernel = _tuple(a.get("kernel"))
    stride = _tuple(a.get("stride"), default=(1, 1))
    pad = _tuple(a.get("pad"), default=(0, 0))
    ceil = a.get("pooling_convention", "valid") == "full"
    if pool_type == "max":
        return torch.nn.functional.max_pool2d(data, kernel, stride, pad, ceil_mode=ceil)
    if pool_type == "avg":
        return torch.nn.functional.avg_pool2d(
            data, kernel, stride, pad, ceil_mode=ceil,
            count_include_pad=_bool(a.get("count_include_pad"), True))
    raise NotImplementedError("Pooling pool_type=%s" % pool_type)


def _batch_norm(a, data, gamma, beta, mean, var):
    if _bool(a.get("fix_gamma"), True):
        gamma = torch.ones_like(gamma)
    eps = float(a.get("eps", "0.001"))
    shape = [1, -1] + [1] * (data.dim() - 2)
    return (data - mean.reshape(shape)) / torch.sqrt(var.reshape(shape) + eps) * \
        gamma.reshape(shape) + beta.reshape(shape)


def _shape_attr(value):
    text = str(value).strip()
    if text in ("", "None", "()", "[]"):
        return ()
    return tuple(int(v) for v in text.strip("()[] ").split(",") if v.strip())


def _reshape(a, x):
    """`Reshape` for the plain target shapes (positive extents, 0 = keep, one -1); the
    other special values are resolved by the operator host for the quantized twin only."""
    shape = list(_shape_attr(a.get("shape", "()")))
    if any(v < -1 for v in shape) or _bool(a.get("reverse"), False):
        raise NotImplementedError("Reshape special values -2/-3/-4 in the float executor")
    shape = [x.shape[i] if v == 0 else v for i, v in enumerate(shape)]
    return x.reshape(shape)


def _transpose(a, x):
    axes = _shape_attr(a.get("axes", "()"))
    return x.permute(*(axes if axes else reversed(range(x.dim())))).contiguous()


def _embedding(a, idx, weight):
    j = idx.to(torch.int64).clamp(0, weight.shape[0] - 1)
    return weight[j]


_FLOAT_OPS = {
    "Convolution": _convolution,
    "FullyConnected": _fully_connected,
    "Activation": _activation,
    "Pooling": _pooling,
    "BatchNorm": _batch_norm,
    "Flatten": lambda a, x: x.reshape(x.shape[0], -1),
    "flatten": lambda a, x: x.reshape(x.shape[0], -1),
    "softmax": lambda a, x: torch.softmax(x, dim=int(a.get("axis", "-1"))),
    "SoftmaxOutput": lambda a, x, label=None: torch.softmax(x, dim=1),
    "Dropout": lambda a, x: x,
    "elemwise_add": lambda a, x, y: x + y,
    "_plus": lambda a, x, y: x + y,
    "elemwise_mul": lambda a, x, y: x * y,
    "Embedding": _embedding,
    "Reshape": _reshape,
    "reshape": _reshape,
    "transpose": _transpose,
    "Concat": lambda a, *xs: torch.cat(xs, dim=int(a.get("dim", "1"))),
    "concat": lambda a, *xs: torch.cat(xs, dim=int(a.get("dim", "1"))),
}


_UNKNOWN = object()


class _Graph:
    """What an executor knows of one symbol.  Its operator nodes live as long as it does: plans
    refer to them."""

    def __init__(self, symbol):
        self.symbol = symbol
        self.nodes, self.heads = symbol.nodes(), symbol.heads()
        self.inputs = tuple(dict.fromkeys(name for op, name, _, _ in self.nodes if op == "null"))
        self.made = {}       # position -> operator.Node
        self.plans = {}      # feed names, shapes and types -> (plan, parameters it read) or None
        self.laid = {}       # layout -> (parameters it read, tensor, its stream), for every plan
        self.lock = threading.Lock()      # guards `plans`
        self.building = threading.Lock()  # one thread at a time lays out parameters

    def op_node(self, i, op, name, attrs):
        node = self.made.get(i)
        if node is None:  # threads that meet here go on with the same one
            node = self.made.setdefault(i, _operator.Node(op, name, **attrs))
        return node

    def known(self, key, params):
        """The plan kept for `key`, None where such a pass is walked, _UNKNOWN without either."""
        with self.lock:
            entry = self.plans.pop(key, _UNKNOWN)
            if entry is not _UNKNOWN:
                self.plans[key] = entry  # the last used at the end
        if entry is None or entry is _UNKNOWN:
            return entry
        return entry[0] if _frontend.same_params(params, entry[1]) else _UNKNOWN

    def keep(self, key, entry, params):
        """Keeps the plan for `key`; those of other parameters than `params` go, as do those whose
        last use is longest ago."""
        with self.lock:
            plans = {k: e for k, e in self.plans.items()
                     if k != key and (e is None or _frontend.same_params(params, e[1]))}
            for old in list(plans)[:max(0, len(plans) + 1 - _MAX_PLANS)]:
                del plans[old]
            plans[key] = entry
            self.plans = plans


class Executor:
    """`Executor(symbol, params).forward(data=...)` -> list of outputs (torch tensors on
    the GPU).  `params` maps variable names to tensors.  Passes may run from several threads.

    `ex.params` may change between passes: entries replaced, tensors written in place or given
    other memory (`p.data = w`).  Writes that torch's version counter does not see, through
    `p.data.copy_(w)`, a DLPack or storage alias or a raw pointer, need `ex.drop_plans()` behind
    them: a plan computes with weights that it laid out before."""

    def __init__(self, symbol, params, device="cuda"):
        self.symbol = symbol
        self.device = device
        self.params = {k: (v if isinstance(v, torch.Tensor) else torch.as_tensor(v)).to(device)
                       for k, v in params.items()}
        self.monitor = None
        self.monitor_all = False
        self._graph = None

    def register_op_hook(self, callback, monitor_all=False):
        """callback(name, op_name, array) as in Block.register_op_hook."""
        self.monitor = callback
        self.monitor_all = monitor_all

    def drop_plans(self):
        """The next pass of every shape lays out the parameters anew."""
        self._graph = None

    @property
    def _plans(self):
        return self._structure().plans

    def _structure(self):
        graph = self._graph
        if graph is None or graph.symbol is not self.symbol:
            graph = self._graph = _Graph(self.symbol)
        return graph

    def _planned(self, graph, feed):
        """The outputs for these inputs, None where the graph has to be walked.  A plan holds
        parameters in its own layout, so it lives as long as `params` holds the tensors it read,
        over the same memory and unwritten."""
        if torch.cuda.is_current_stream_capturing():
            # A replay would read the plan's own copies of the parameters, which go when the plan
            # is dropped and miss what is written to the parameters afterwards.  Walked, the
            # captured launches read `params` themselves; temporaries are the graph's.
            return None
        key = tuple((name, v.shape, v.dtype, v.device) for name, v in feed.items())
        plan = graph.known(key, self.params)
        if plan is _UNKNOWN:
            plan = self._plan_for(graph, key, feed)
        if plan is None:
            return None
        try:
            return _frontend.run_plan(plan, *feed.values())
        except _operator.MXNetError:
            # A launch refused its sizes (before anything of it ran).  The operators have other
            # limits: the walk does it or reports it.
            graph.keep(key, None, self.params)
            return None

    def _plan_for(self, graph, key, feed):
        with graph.building:
            plan = graph.known(key, self.params)
            if plan is not _UNKNOWN:
                return plan
            stream = torch.cuda.current_stream()
            params = dict(self.params)
            try:
                entry = _plan.build(params, graph, feed, stream.cuda_stream)
            except _operator.MXNetError:
                entry = None  # the walk reports it
            # what was laid out may be read on any stream from here on, or be given back
            stream.synchronize()
            if entry is not None:
                graph.laid.update(entry[2])
                entry = entry[:2]
            graph.keep(key, entry, params)
            return entry and entry[0]

    def forward(self, **feed):
        graph = self._structure()
        # what the graph has no variable for is left alone
        feed = {name: (v if isinstance(v, torch.Tensor) else torch.as_tensor(v)).to(self.device)
                for name, v in ((n, feed[n]) for n in graph.inputs if n in feed)}
        if self.monitor is None and feed and all(v.is_cuda for v in feed.values()):
            tensors = {name: v.contiguous() for name, v in feed.items()}
            outputs = self._planned(graph, tensors)
            if outputs is not None:
                return outputs
        values = []
        for i, (op, name, attrs, inputs) in enumerate(graph.nodes):
            if op == "null":
                if name in feed:
                    v = feed[name]
                elif name in self.params:
                    v = self.params[name]
                else:
                    raise KeyError("no value for variable %r" % name)
                values.append([v])
                continue
            args = [values[j][k] for j, k in inputs]
            if op.startswith("_contrib_") or op.startswith("_npx_"):
                node = graph.op_node(i, op, name, attrs)
                out = node(*[a.contiguous() for a in args])
                outs = list(out) if isinstance(out, (tuple, list)) else [out]
                in_names, out_names = node.list_inputs(), node.list_outputs()
            else:
                fn = _FLOAT_OPS.get(op)
                if fn is None:
                    raise NotImplementedError("the harness executor has no float operator %r" % op)
                out = fn(attrs, *args)
                outs = list(out) if isinstance(out, (tuple, list)) else [out]
                try:
                    probe = graph.op_node(i, op, name, attrs)
                    in_names, out_names = probe.list_inputs(), probe.list_outputs()
                except _operator.MXNetError:
                    in_names, out_names = [], []
            values.append(outs)
            if self.monitor is not None:
                if self.monitor_all:
                    for k, arr in enumerate(args):
                        arg = in_names[k] if k < len(in_names) else "input%d" % k
                        self.monitor("%s_%s" % (name, arg), op, arr)
                for k, arr in enumerate(outs):
                    out_name = out_names[k] if k < len(out_names) else str(k)
                    self.monitor("%s_%s" % (name, out_name), op, arr)
        return [values[j][k] for j, k in graph.heads]
