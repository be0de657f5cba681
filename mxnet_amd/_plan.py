"""Plans of quantized graphs: the launches of one forward pass for given input shapes.

Run operator by operator, a quantized ResNet-50 is 194 calls whose int32 tensors cross memory
twice between a convolution and its requantize, and twice more around every residual sum.  A plan
keeps the graph's results and drops that traffic:

  * convolution -> requantize (-> relu), fully connected -> requantize (-> relu, -> dequantize)
    and convolution -> requantize -> sum (-> requantize) (-> relu) become one launch each (the
    fused epilogues of include/mxq.h, bit-identical to the operators one after the other);
  * the tail of a residual block (3 x 3 convolution, 1 x 1 convolution, sum, the next block's first
    1 x 1 convolution) becomes one launch where its ranges stay (fuse_blocks);
  * activations between convolutions and pooling stay NHWC with the channels padded to a multiple
    of 16; weights are laid out once, when the plan is made;
  * every range that a calibrated operator hands on is a constant of the plan;
  * everything else of the graph runs as the registered operator it is, on NCHW tensors.

`build` returns None for a graph it does not cover (a float operator between the quantized ones, a
head that is a range, parameters off the device): executor.py then walks the graph node by node.
"""
import struct

import numpy as np
import torch

from . import _frontend, _lib

_ALIGN = 256
_FLAG_OF = {torch.float32: 0, torch.float64: 1, torch.float16: 2, torch.uint8: 3, torch.int32: 4,
            torch.int8: 5, torch.int64: 6, torch.bool: 7, torch.bfloat16: 12}
_SIZE_OF = {0: 4, 1: 8, 2: 2, 3: 1, 4: 4, 5: 1, 6: 8, 7: 1, 12: 2}
_FLOAT32, _INT32, _INT8 = 0, 4, 5
(_NODE, _CONV, _FC, _FC_F32, _FC_SUM, _FC_SUM_RQ, _QUANT_NHWC, _TO_NHWC, _FROM_NHWC, _POOL, _RELU,
 _ADD, _REQUANTIZE, _BLOCK, _PAIR, _CONV_POOL, _CONV3) = range(17)
_NULL, _ARENA, _HELD, _FEED, _OUTPUT = range(5)


class _Unsupported(Exception):
    pass


def _pad16(c):
    return (c + 15) // 16 * 16


def _pair(text, default):
    vals = tuple(int(x) for x in (text or "").strip("()[] ").split(",") if x.strip())
    return vals if vals else default


def _flag(text, default=False):
    return default if text is None else text.strip().lower() in ("true", "1")


_bits = struct.Struct("<d").pack  # a float as part of a key: NaN is itself and the zeros differ


class _Buffer:
    """Bytes that a step writes and later steps read: part of the arena, or an output."""

    def __init__(self, nbytes):
        self.nbytes = nbytes
        self.first = self.last = None
        self.place = None  # (base, index, offset)


class _Place:
    """An operand outside the arena: (base, index, offset) known at once."""

    def __init__(self, base, index, offset=0):
        self.place = (base, index, offset)


class _Value:
    """A tensor of the graph: its logical shape and type, and where it lies.  `channels` is 0 for
    the operator's own contiguous layout; else the memory is [N, H, W, channels] (or, of a
    flattened tensor, rows of `channels` bytes).  `s2d` = (off_h, off_w, rows, columns) marks the
    space-to-depth form of an image."""

    def __init__(self, flag, shape, at, channels=0, s2d=None):
        self.flag, self.shape, self.at, self.channels, self.s2d = flag, shape, at, channels, s2d


class _Builder:
    def __init__(self, given, graph, feeds):
        self.given, self.graph, self.nodes, self.heads = given, graph, graph.nodes, graph.heads
        self.held, self.steps, self.buffers, self.constants = [], [], [], []
        self.values = {}   # (node, output) -> _Value; range outputs -> an operand
        self.params = {}   # name -> as_read() of a parameter the plan has read
        self.name_of = {}  # id of a parameter -> its name
        self.param_at = {}  # name -> where the plan holds it
        self.made = {}     # what laid() made for this plan and later ones
        self.origin = {}   # index of a held tensor -> its key in the graph's layouts, its names
        self.plain = {}    # id of an NHWC value -> its NCHW form
        self.absorbed = {}  # node -> True: part of an earlier step
        self.deferred = {}  # sum node -> (conv node, its requantize node)
        self.feeds = {name: i for i, name in enumerate(feeds)}
        self.feed_tensors = feeds
        self.table = _Place(_HELD, None)
        self.scratch = None
        self.users = {}
        for i, (op, _, _, inputs) in enumerate(self.nodes):
            for slot, (j, k) in enumerate(inputs):
                self.users.setdefault((j, k), []).append((i, slot))
        self.head_set = set(self.heads)

    # ---- operands -----------------------------------------------------------------------
    def hold(self, tensor, key=None, names=()):
        self.held.append(tensor)
        if key is not None:
            self.origin[len(self.held) - 1] = key, names
        return _Place(_HELD, len(self.held) - 1)

    def hold_param(self, tensor):
        name = self.name_of[id(tensor)]
        if name not in self.param_at:
            self.param_at[name] = self.hold(tensor, ("param", name), (name,))
        return self.param_at[name]

    def laid(self, key, names, make):
        """Holds the tensor that `make()` lays out from parameters `names`.  It does not depend on
        the shapes of the feeds beyond what `key` says: plans of one graph share it while the
        parameters stay as they were read."""
        key = (self.device,) + key
        entry = self.made.get(key) or self.graph.laid.get(key)
        if entry is None or not _frontend.same_params(self.given, entry[0]):
            entry = self.made[key] = tuple(self.params[n] for n in names), make(), self.stream
        elif entry[2] != self.stream:
            entry[1].record_stream(torch.cuda.current_stream())
        return self.hold(entry[1], key, names)

    def buffer(self, nbytes):
        b = _Buffer(max(int(nbytes), 1))
        self.buffers.append(b)
        return b

    def constant(self, value):
        """Operand of one float32 of the plan's constant table."""
        self.constants.append(float(value))
        place = _Place(_HELD, None, 4 * (len(self.constants) - 1))
        place.in_table = True
        return place

    def constant_range(self, lo, hi):
        return [self.constant(lo), self.constant(hi)]

    def scratch_range(self):
        """Four floats that the launches write their own ranges to: nothing reads them, the
        graph's ranges are the table's constants."""
        if self.scratch is None:
            self.scratch = self.hold(torch.empty(4, dtype=torch.float32, device=self.device))
        return self.scratch

    def emit(self, kind, ints, floats, refs, node=None, blobs=None):
        at = len(self.steps)
        for r in refs:
            if isinstance(r, _Buffer):
                r.first = at if r.first is None else r.first
                r.last = at
        self.steps.append((kind, ints, floats, refs, node, blobs))

    def param(self, i):
        """The device tensor of a variable node that is a parameter; None for anything else."""
        op, name, _, _ = self.nodes[i]
        if op != "null" or name in self.feeds:
            return None
        t = self.given.get(name)
        if t is None:
            return None
        if not (t.is_cuda and t.is_contiguous()) or t.is_inference():
            raise _Unsupported("parameter %s" % name)
        if name not in self.params:  # as it was before anything of it is laid out
            self.params[name] = _frontend.as_read(name, t)
            self.name_of[id(t)] = name
        return t

    def value(self, ref):
        return self.values[ref]

    def sole_user(self, i, count=3):
        """The node that takes all `count` outputs of node i, if nothing else takes any."""
        found = set()
        for k in range(count):
            if (i, k) in self.head_set:
                return None
            found.update(u for u, _ in self.users.get((i, k), []))
        return found.pop() if len(found) == 1 else None

    # ---- layouts --------------------------------------------------------------------------
    def as_plain(self, v):
        """The value in the operator's own layout."""
        if v.channels == 0:
            return v
        if v.s2d is not None:
            raise _Unsupported("space-to-depth image outside a convolution")
        if v.shape[1] == v.channels and (len(v.shape) == 2 or v.shape[2] * v.shape[3] == 1):
            return _Value(v.flag, v.shape, v.at)
        if id(v) not in self.plain:
            n, c = v.shape[:2]
            h, w = (v.shape[2], v.shape[3]) if len(v.shape) == 4 else (1, 1)
            out = self.buffer(n * c * h * w)
            self.emit(_FROM_NHWC, (n, c, h, w, v.channels), (), [v.at, out])
            self.plain[id(v)] = _Value(v.flag, v.shape, out)
            self.plain[id(v)].source = v  # keeps id(v) taken
        return self.plain[id(v)]

    def as_nhwc(self, v):
        if v.s2d is not None:
            raise _Unsupported("space-to-depth image outside its convolution")
        if v.channels != 0:
            return v
        if v.flag != _INT8 or len(v.shape) != 4:
            raise _Unsupported("NHWC form of this tensor")
        n, c, h, w = v.shape
        channels = _pad16(c)
        out = self.buffer(n * h * w * channels)
        self.emit(_TO_NHWC, (n, c, h, w, channels), (), [v.at, out])
        return _Value(v.flag, v.shape, out, channels)

    # ---- parameters -------------------------------------------------------------------------
    def pack(self, weight, o, c, kh, kw, o_padded, channels, s2d=False):
        okh, okw = ((kh + 1) // 2, (kw + 1) // 2) if s2d else (kh, kw)

        def make():
            out = torch.empty(o_padded * okh * okw * channels, dtype=torch.int8,
                              device=self.device)
            _lib.check(_lib.lib.mxq_pack_weight(self.stream, weight.data_ptr(), out.data_ptr(), o,
                                                c, kh, kw, o_padded, channels, int(s2d)))
            return out

        name = self.name_of[id(weight)]
        return self.laid(("packed", name, o, c, kh, kw, o_padded, channels, s2d), (name,), make)

    def operands(self, inputs, no_bias):
        """(data, weight, bias, [six ranges]) of a convolution or fully-connected node."""
        ni = 2 if no_bias else 3
        weight = self.param(inputs[1][0])
        bias = None if no_bias else self.param(inputs[2][0])
        if weight is None or (bias is None and not no_bias):
            raise _Unsupported("computed weights")
        ranges = [self.values[r] for r in inputs[ni:]]
        if no_bias:
            ranges += [None, None]
        return self.value(inputs[0]), weight, bias, ranges

    def bias_of(self, bias, o, o_padded):
        if bias is None:
            return None
        if o == o_padded:
            return self.hold_param(bias)
        return self.pack(bias, o, 1, 1, 1, o_padded, 1)

    # ---- what follows a layer ------------------------------------------------------------------
    def calibration(self, i):
        """(lo, hi) of node i's calibrated range, None without one."""
        attrs = self.nodes[i][2]
        lo, hi = attrs.get("min_calib_range", "None"), attrs.get("max_calib_range", "None")
        if "None" in (lo.strip(), hi.strip()):
            return None
        return _frontend.float_of(lo), _frontend.float_of(hi)

    def requantize_behind(self, i):
        """The calibrated int8 requantize that alone consumes node i."""
        j = self.sole_user(i)
        if j is None or self.nodes[j][0] != "_contrib_requantize" or self.calibration(j) is None:
            return None
        if self.described(j)[0][0] != _INT8 or [r for r in self.nodes[j][3]] != [
                (i, 0), (i, 1), (i, 2)]:
            return None
        return j

    def relu_behind(self, i):
        j = self.sole_user(i)
        if j is None or self.nodes[j][0] != "_contrib_quantized_act":
            return None
        return j if self.nodes[j][3] == [(i, 0), (i, 1), (i, 2)] else None

    def finish(self, i, value, ranges):
        """Node i's outputs: the tensor and its range operands."""
        self.values[(i, 0)] = value
        self.values[(i, 1)], self.values[(i, 2)] = ranges

    def symmetric(self, lo, hi):
        r = max(abs(np.float32(lo)), abs(np.float32(hi)))
        return self.constant_range(-r, r)

    # ---- nodes ----------------------------------------------------------------------------------
    def node_of(self, i):
        op, name, attrs, _ = self.nodes[i]
        return self.graph.op_node(i, op, name, attrs)

    def described(self, i):
        """[(type flag, shape)] of node i's outputs, inferred from the graph's own shapes."""
        if i not in self.outs:
            given = tuple(self.meta[r] for r in self.nodes[i][3])
            self.outs[i], self.temps[i] = _frontend.describe(self.node_of(i)._call, given)
        return self.outs[i]

    def infer(self):
        """Shapes and types of every tensor of the graph."""
        self.meta, self.outs, self.temps = {}, {}, {}
        for i, (op, name, _, inputs) in enumerate(self.nodes):
            if op == "null":
                t = self.feed_tensors.get(name, self.given.get(name))
                if t is None or t.dtype not in _FLAG_OF:
                    raise _Unsupported("no value for %s" % name)
                self.meta[(i, 0)] = (_FLAG_OF[t.dtype], tuple(t.shape))
            elif op.startswith("_contrib_") or op.startswith("_npx_"):
                for k, m in enumerate(self.described(i)):
                    self.meta[(i, k)] = (m[0], tuple(m[1]))
            else:
                raise _Unsupported("float operator %s" % op)

    def build(self, stream):
        self.stream = stream
        device = {t.device for t in self.feed_tensors.values()}
        if len(device) != 1 or not all(t.is_cuda for t in self.feed_tensors.values()):
            raise _Unsupported("feeds off the device")
        self.device = device.pop()
        if any(t.numel() == 0 for t in self.feed_tensors.values()):
            raise _Unsupported("empty feeds")
        self.infer()
        for i, (op, name, attrs, inputs) in enumerate(self.nodes):
            if i in self.absorbed:
                continue
            if op == "null":
                flag, shape = self.meta[(i, 0)]
                if name in self.feeds:
                    self.values[(i, 0)] = _Value(flag, shape, _Place(_FEED, self.feeds[name]))
                else:
                    self.variable(i, flag, shape)
                continue
            handler = _HANDLERS.get(op)
            if handler is None or not handler(self, i, attrs, inputs):
                self.generic(i, inputs)
        return self.assemble()

    def variable(self, i, flag, shape):
        at = self.hold_param(self.param(i))
        # one-element float parameters are ranges: consumers take the bare operand
        self.values[(i, 0)] = _Value(flag, shape, at)

    def generic(self, i, inputs):
        """The registered operator on tensors in its own layout."""
        refs, blobs = [], []
        for r in inputs:
            v = self.values[r]
            if isinstance(v, _Value):
                v = self.as_plain(v)
                refs.append(v.at)
            else:
                refs.append(v)
            blobs.append(self.meta[r])
        outs = self.described(i)
        for k, (flag, shape) in enumerate(outs):
            out = self.buffer(int(np.prod(shape, dtype=np.int64)) * _SIZE_OF[flag])
            refs.append(out)
            blobs.append((flag, tuple(shape)))
            self.values[(i, k)] = _Value(flag, tuple(shape), out)
        temp = self.temps[i]
        refs.append(self.buffer(temp) if temp else None)
        node = self.node_of(i)
        self.emit(_NODE, (temp,), (), refs, node, (len(inputs), tuple(blobs)))

    def quantize(self, i, attrs, inputs):
        """quantize_v2 of an image that only convolutions read: straight into their layout."""
        calib = self.calibration(i)
        x = self.values[inputs[0]]
        outs = self.described(i)
        if (calib is None or x.flag != _FLOAT32 or outs[0][0] != _INT8 or len(x.shape) != 4 or
                x.channels or any((i, k) in self.head_set for k in range(3))):
            return False
        users = {u for k in range(3) for u, _ in self.users.get((i, k), [])}
        if not users or not all(self.nodes[u][0] == "_contrib_quantized_conv" and
                                self.nodes[u][3][0] == (i, 0) and self.fusable_conv(u)
                                for u in users):
            return False
        n, c, h, w = x.shape
        s2d = self.s2d_of(users.pop(), c, h, w) if len(users) == 1 else None
        channels = _pad16(c if s2d is None else 4 * c)
        off_h, off_w, oh, ow = (0, 0, h, w) if s2d is None else s2d
        out = self.buffer(n * oh * ow * channels)
        self.emit(_QUANT_NHWC, (n, c, h, w, channels, int(s2d is not None), off_h, off_w, oh, ow),
                  calib, [x.at, out, self.scratch_range()])
        self.finish(i, _Value(_INT8, x.shape, out, channels, s2d), self.symmetric(*calib))
        return True

    def conv_geometry(self, i):
        attrs = self.nodes[i][2]
        return (_pair(attrs.get("kernel"), (1, 1)), _pair(attrs.get("stride"), (1, 1)),
                _pair(attrs.get("pad"), (0, 0)), _pair(attrs.get("dilate"), (1, 1)))

    def s2d_of(self, i, c, h, w):
        """(off_h, off_w, rows, columns) where the convolution runs on the space-to-depth form of its
        image: a stride-2 stem over at most 4 channels, 4 * C real channels out of 16 instead of C.
        Where the last window reaches one pixel past an odd extent, the form has another row (or
        column) of zeros for it: such stems too are two launches then (a network of four blocks
        on 10 images of 185 x 185 82.5 us in three launches over 16 padded channels, 68 so)."""
        (kh, kw), stride, (ph, pw), dilate = self.conv_geometry(i)
        if c > 4 or stride != (2, 2) or dilate != (1, 1) or kh < 2 or kw < 2:
            return None
        off_h, off_w = ph & 1, pw & 1
        oh, ow = self.described(i)[0][1][2:]
        # what a 1-strided convolution over ceil(k / 2) taps needs for as many outputs
        rows, columns = (o + (k + 1) // 2 - 1 - (p - off) for off, p, k, o in
                         ((off_h, ph, kh, oh), (off_w, pw, kw, ow)))
        fits = (0 <= rows - (h + off_h + 1) // 2 <= 1 and
                0 <= columns - (w + off_w + 1) // 2 <= 1)
        return (off_h, off_w, rows, columns) if fits else None

    def fusable_conv(self, i):
        inputs = self.nodes[i][3]
        variables = [self.nodes[j][0] == "null" and self.nodes[j][1] not in self.feeds
                     for j, _ in inputs[1:2 if len(inputs) == 6 else 3]]
        return all(variables) and self.requantize_behind(i) is not None

    def conv(self, i, attrs, inputs):
        if not self.fusable_conv(i):
            return False
        j = self.requantize_behind(i)
        if self.defer_to_sum(i, j):
            return True
        return self.emit_conv(i, j, self.relu_behind(j))

    def is_dense(self, i):
        return self.conv_geometry(i) == ((1, 1), (1, 1), (0, 0), (1, 1))

    def defer_to_sum(self, i, j):
        """Leaves a 1 x 1 convolution whose requantized output goes into a sum alone to the sum's
        launch."""
        if not self.is_dense(i):
            return False
        k = self.sole_user(j)
        if (k is None or self.nodes[k][0] != "_contrib_quantized_elemwise_add" or
                k in self.deferred):
            return False
        inputs = self.nodes[k][3]
        if self.summand(k, j) is None or [f for f, _ in (self.meta[r] for r in inputs[:2])] != [
                _INT8, _INT8]:
            return False
        if self.calibration(k) is None and self.requantize_behind(k) is None:
            return False
        self.deferred[k] = (i, j)
        self.absorbed[j] = True
        return True

    def summand(self, k, j):
        """0 or 1 where node j's tensor and range are that operand of sum k and nothing else of it
        is node j's, None otherwise."""
        inputs = self.nodes[k][3]
        for slot in (0, 1):
            rest = [inputs[1 - slot]] + inputs[4 - 2 * slot:6 - 2 * slot]
            if ([inputs[slot]] + inputs[2 + 2 * slot:4 + 2 * slot] == [(j, 0), (j, 1), (j, 2)] and
                    all(node != j for node, _ in rest)):
                return slot
        return None

    def emit_conv(self, i, j, relu):
        """Convolution i with its requantize j and relu, if any, as one launch."""
        inputs = self.nodes[i][3]
        x, weight, bias, ranges = self.operands(inputs, len(inputs) == 6)
        (kh, kw), (sh, sw), (ph, pw), (dh, dw) = self.conv_geometry(i)
        (o, c) = weight.shape[:2]
        n, oh, ow = (self.described(i)[0][1][d] for d in (0, 2, 3))
        o_padded = _pad16(o)
        h, w = x.shape[2:]
        if x.s2d is not None:
            off_h, off_w, h, w = x.s2d
            packed = self.pack(weight, o, c, kh, kw, o_padded, x.channels, s2d=True)
            kh, kw = (kh + 1) // 2, (kw + 1) // 2
            ph, pw, sh, sw = (ph - off_h) // 2, (pw - off_w) // 2, 1, 1
        else:
            x = self.as_nhwc(x)
            packed = self.dense_weight(weight, o, c, kh, kw, o_padded, x.channels)
        geo = (n, h, w, x.channels, o_padded, kh, kw, sh, sw, ph, pw, dh, dw)
        ws = int(_lib.lib.mxq_quantized_conv_workspace(*geo, 1))
        out = self.buffer(n * oh * ow * o_padded)
        calib = self.calibration(j)
        self.emit(_CONV, geo + (int(relu is not None), ws), calib,
                  [x.at, packed, self.bias_of(bias, o, o_padded)] + [self.bare(r) for r in ranges] +
                  [self.scratch_range(), out, self.buffer(ws) if ws else None])
        self.close(j, relu, _Value(_INT8, (n, o, oh, ow), out, o_padded), self.symmetric(*calib))
        return True

    def rows(self, m):
        """m, where a launch can count that many rows (it takes an int)."""
        if m >= 1 << 31:
            raise _Unsupported("%d rows" % m)
        return m

    def dense_weight(self, weight, o, c, kh, kw, o_padded, channels):
        if kh == kw == 1 and c == channels and o == o_padded:
            return self.hold_param(weight)
        return self.pack(weight, o, c, kh, kw, o_padded, channels)

    def close(self, j, relu, value, ranges):
        """Results of a fused chain that ends at node j, or at its relu."""
        self.absorbed[j] = True
        if relu is not None:
            self.absorbed[relu] = True
            j = relu
        self.finish(j, value, ranges)

    def bare(self, r):
        return r.at if isinstance(r, _Value) else r

    def add(self, i, attrs, inputs):
        if [f for f, _ in (self.meta[r] for r in inputs[:2])] != [_INT8, _INT8]:
            return False
        calib = self.calibration(i)
        j = None
        if calib is None:
            j = self.requantize_behind(i)
            if j is None:
                return False
        if i in self.deferred:
            return self.sum_into_conv(i, j, calib)
        lhs, rhs = self.values[inputs[0]], self.values[inputs[1]]
        if lhs.channels == 0 or rhs.channels == 0 or lhs.s2d or rhs.s2d:
            return False
        # two NHWC tensors of one shape: the sum does not care for the layout
        n = lhs.shape[0] * int(np.prod(lhs.shape[2:], dtype=np.int64)) * lhs.channels
        ranges = [self.bare(self.values[r]) for r in inputs[2:]]
        sum_range = self.buffer(8)
        out = self.buffer(n if j is None else 4 * n)
        self.emit(_ADD, (n, _INT8 if j is None else _INT32, int(calib is not None)),
                  calib or (0.0, 0.0), [lhs.at, rhs.at, out] + ranges + [sum_range])
        if j is None:
            self.finish(i, _Value(_INT8, lhs.shape, out, lhs.channels),
                        self.constant_range(*calib))
            return True
        calib = self.calibration(j)
        narrow = self.buffer(n)
        high = _Offset(sum_range, 4)
        self.emit(_REQUANTIZE, (n,), calib, [out, narrow, sum_range, high, self.scratch_range()])
        self.absorbed[j] = True
        self.finish(j, _Value(_INT8, lhs.shape, narrow, lhs.channels), self.symmetric(*calib))
        return True

    def sum_into_conv(self, i, j, calib):
        """Sum i (and the requantize j behind it) in the epilogue of the convolution left to it."""
        conv, requantize = self.deferred[i]
        inputs = self.nodes[i][3]
        slot = self.summand(i, requantize)
        residual = self.as_nhwc(self.values[inputs[1 - slot]])
        residual_range = [self.bare(self.values[r]) for r in inputs[4 - 2 * slot:6 - 2 * slot]]
        conv_inputs = self.nodes[conv][3]
        x, weight, bias, ranges = self.operands(conv_inputs, len(conv_inputs) == 6)
        x = self.as_nhwc(x)
        o, c = weight.shape[:2]
        o_padded = _pad16(o)
        n, _, h, w = x.shape
        m = self.rows(n * h * w)
        ws = int(_lib.lib.mxq_quantized_fc_workspace(m, o_padded, x.channels, 1))
        out = self.buffer(m * o_padded)
        last = i if j is None else j
        relu = self.relu_behind(last)
        layer = self.calibration(requantize)
        total = calib if j is None else self.calibration(j)
        self.emit(_FC_SUM if j is None else _FC_SUM_RQ,
                  (m, o_padded, x.channels, int(relu is not None), ws), layer + total,
                  [x.at, self.dense_weight(weight, o, c, 1, 1, o_padded, x.channels),
                   self.bias_of(bias, o, o_padded)] + [self.bare(r) for r in ranges] +
                  [self.scratch_range(), out, self.buffer(ws) if ws else None, residual.at] +
                  residual_range +
                  ([] if j is None else [self.pairs(layer, residual_range, total, relu)]))
        self.close(last, relu, _Value(_INT8, (n, o, h, w), out, o_padded),
                   self.constant_range(*total) if j is None else self.symmetric(*total))
        return True

    def pairs(self, layer, residual, total, relu):
        """What mxq_sum_requant_pairs finds for a sum with a relu behind it whose ranges are the
        plan's constants, once the step turns out to be one of the plan; None for any other."""
        if relu is None or not all(getattr(r, "in_table", False) for r in residual):
            return None
        ranges = (*layer, *(self.constants[r.place[2] // 4] for r in residual), *total)

        def make():
            found = torch.empty(3, dtype=torch.int32, device=self.device)
            _lib.check(_lib.lib.mxq_sum_requant_pairs(self.stream, *ranges, found.data_ptr()))
            return found

        return _Later(lambda: self.laid(("pairs",) + tuple(map(_bits, ranges)), (), make).place)

    def act(self, i, attrs, inputs):
        x = self.values[inputs[0]]
        if x.flag != _INT8 or x.channels == 0 or x.s2d:
            return False
        n = x.shape[0] * int(np.prod(x.shape[2:], dtype=np.int64)) * x.channels
        out = self.buffer(n)
        ranges = [self.values[r] for r in inputs[1:]]
        self.emit(_RELU, (n,), (), [x.at, out] + [self.bare(r) for r in ranges] +
                  [self.scratch_range()])
        self.finish(i, _Value(_INT8, x.shape, out, x.channels), ranges)
        return True

    def pooling(self, i, attrs, inputs):
        x = self.values[inputs[0]]
        if x.flag != _INT8 or x.channels == 0 or len(x.shape) != 4 or x.s2d:
            return False
        n, c, h, w = x.shape
        oh, ow = self.described(i)[0][1][2:]
        pool_type = attrs.get("pool_type", "max").strip()
        if pool_type not in ("max", "avg"):
            return False
        if _flag(attrs.get("global_pool")):
            kernel, stride, pad = (h, w), (1, 1), (0, 0)
        else:
            kernel = _pair(attrs.get("kernel"), None)
            stride, pad = _pair(attrs.get("stride"), (1, 1)), _pair(attrs.get("pad"), (0, 0))
        count_pad = attrs.get("count_include_pad", "None").strip()
        count_pad = True if count_pad == "None" else _flag(count_pad)
        out = self.buffer(n * oh * ow * x.channels)
        self.emit(_POOL, (n, h, w, x.channels) + kernel + stride + pad +
                  (oh, ow, int(pool_type == "avg"), int(count_pad)), (), [x.at, out])
        self.finish(i, _Value(_INT8, (n, c, oh, ow), out, x.channels),
                    [self.values[r] for r in inputs[1:]])
        return True

    def flatten(self, i, attrs, inputs):
        """The same bytes under another shape."""
        x = self.values[inputs[0]]
        if (i, 0) in self.head_set or not isinstance(x.at, _Buffer):
            return False
        flag, shape = self.described(i)[0]
        shape = tuple(shape)
        if x.channels and len(x.shape) == 4 and x.shape[2] * x.shape[3] == 1 and not x.s2d:
            value = _Value(flag, shape, x.at, x.channels)
        else:
            value = _Value(flag, shape, self.as_plain(x).at)
        self.finish(i, value, [self.values[r] for r in inputs[1:]])
        return True

    def fully_connected(self, i, attrs, inputs):
        j = self.requantize_behind(i)
        if j is None or self.nodes[inputs[1][0]][0] != "null" or \
                self.nodes[inputs[1][0]][1] in self.feeds:
            return False
        no_bias = len(inputs) == 6
        if not no_bias and (self.nodes[inputs[2][0]][0] != "null" or
                            self.nodes[inputs[2][0]][1] in self.feeds):
            return False
        x, weight, bias, ranges = self.operands(inputs, no_bias)
        o, k = weight.shape
        shape = tuple(self.described(i)[0][1])
        if x.channels and len(x.shape) == 2 and x.shape[1] == k:
            m, packed, k = x.shape[0], self.dense_weight(weight, o, k, 1, 1, o, x.channels), \
                x.channels
        else:
            x = self.as_plain(x)
            m, packed = int(np.prod(shape[:-1], dtype=np.int64)), self.hold_param(weight)
        self.rows(m)
        calib = self.calibration(j)
        relu = self.relu_behind(j)
        deq = self.sole_user(relu if relu is not None else j)
        if deq is not None and (self.nodes[deq][0] != "_contrib_dequantize" or
                                self.nodes[deq][3] != [(relu if relu is not None else j, s)
                                                       for s in range(3)]):
            deq = None
        ws = int(_lib.lib.mxq_quantized_fc_workspace(m, o, k, int(deq is None)))
        out = self.buffer(m * o * (1 if deq is None else 4))
        self.emit(_FC if deq is None else _FC_F32, (m, o, k, int(relu is not None), ws), calib,
                  [x.at, packed, None if bias is None else self.hold_param(bias)] +
                  [self.bare(r) for r in ranges] +
                  [self.scratch_range(), out, self.buffer(ws) if ws else None])
        if deq is None:
            self.close(j, relu, _Value(_INT8, shape, out), self.symmetric(*calib))
            return True
        self.absorbed[j] = self.absorbed[deq] = True
        if relu is not None:
            self.absorbed[relu] = True
        self.values[(deq, 0)] = _Value(_FLOAT32, shape, out)
        return True

    # ---- the finished plan --------------------------------------------------------------------
    def assemble(self):
        outputs = []
        for r in self.heads:
            v = self.values.get(r)
            if not isinstance(v, _Value):
                raise _Unsupported("a head that is no tensor of the plan")
            v = self.as_plain(v)
            if not isinstance(v.at, _Buffer) or v.at.place is not None:
                raise _Unsupported("a head that is an input, or the same as another head")
            v.at.place = (_OUTPUT, len(outputs), 0)
            outputs.append((v.flag, v.shape))
        self.fuse()
        # offsets: first fit over the buffers alive at the same steps
        taken, size = [], 0
        for b in sorted((b for b in self.buffers if b.place is None and b.first is not None),
                        key=lambda b: (b.first, -b.nbytes)):
            need = (b.nbytes + _ALIGN - 1) // _ALIGN * _ALIGN
            taken = [t for t in taken if t[2] >= b.first]
            offset = 0
            for lo, hi, _ in sorted(taken):
                if offset + need <= lo:
                    break
                offset = max(offset, hi)
            taken.append((offset, offset + need, b.last))
            size = max(size, offset + need)
            b.place = (_ARENA, 0, offset)
        table = torch.tensor(self.constants or [0.0], dtype=torch.float32).to(self.device)
        self.held.append(table)
        self.table_index = len(self.held) - 1

        def place(r):
            if r is None:
                return (_NULL, 0, 0)
            if isinstance(r, _Offset):
                base, at, offset = r.buffer.place
                return (base, at, offset + r.offset)
            if isinstance(r, _Later):
                return r.find()
            if getattr(r, "in_table", False):
                return (_HELD, self.table_index, r.place[2])
            return r.place

        steps = []
        for kind, ints, floats, refs, node, blobs in self.steps:
            places = [place(r) for r in refs]
            if kind == _BLOCK:
                layers, blobs = blobs, None
                layers = [(columns, calib, [place(r) for r in refs])
                          for columns, calib, refs in layers]
                places[1] = self.block_weights(ints, layers)
                places[3:6] = [self.prepared(*layer) if layer[2] else (_NULL, 0, 0)
                               for layer in layers]
                places[2] = self.block_forms(floats, layers, places[3:6])
            if kind == _PAIR:
                layers, blobs = blobs, None
                places[5:7] = [self.prepared(columns, calib, [place(r) for r in refs], True)
                               for columns, calib, refs in layers]
            if kind == _CONV3:
                (columns, calib, refs), blobs = blobs, None
                places[1] = self.conv3x3_weights(ints, place(refs[1]))
                places[2] = self.prepared(columns, calib, [place(r) for r in refs], True)
            if kind == _CONV_POOL:
                (columns, calib, refs), blobs = blobs, None
                places[2] = self.prepared(columns, calib, [place(r) for r in refs])
            if kind in (_CONV, _FC, _FC_F32, _FC_SUM, _FC_SUM_RQ):
                places.append(self.prepared(ints[4 if kind == _CONV else 1], floats, places))
            step = (kind, tuple(int(v) for v in ints), tuple(float(v) for v in floats),
                    tuple(places))
            steps.append(step if node is None else step + (node._call, blobs))
        plan = _frontend.plan(size, self.held, steps, [(f, tuple(s)) for f, s in outputs])
        return plan, tuple(self.params.values()), self.made

    def fuse(self):
        """Steps that go out together as one; the buffers' lifetimes follow."""
        users = {}  # id of a buffer -> the steps that read or write it
        for at, step in enumerate(self.steps):
            for r in step[3]:
                b = r.buffer if type(r) is _Offset else r
                if type(b) is _Buffer:
                    users.setdefault(id(b), []).append(at)
        gone = set()
        self.fuse_stem(users, gone)
        self.fuse_blocks(users, gone)
        self.pair_convs(gone)
        self.single_convs(gone)
        self.steps = [s for at, s in enumerate(self.steps) if at not in gone]
        for b in self.buffers:
            b.first = b.last = None
        for at, step in enumerate(self.steps):
            for r in step[3]:
                b = r.buffer if type(r) is _Offset else r
                if type(b) is _Buffer:
                    b.first = at if b.first is None else b.first
                    b.last = at

    def fuse_stem(self, users, gone):
        """A 4 x 4 convolution over 16 channels that only a 3 x 3 maximum reads, and that, as one
        step."""
        for at, (kind, geo, _, refs, _, _) in enumerate(self.steps):
            if kind != _POOL or geo[4:10] != (3, 3, 2, 2, 1, 1) or geo[12]:
                continue
            mid = refs[0]
            if not isinstance(mid, _Buffer) or mid.place is not None or len(users[id(mid)]) != 2:
                continue
            first = users[id(mid)][0]
            kind, conv, calib, layer, _, _ = self.steps[first]
            if (kind != _CONV or layer[10] is not mid or conv[7:9] != (1, 1) or
                    conv[11:13] != (1, 1) or geo[3] != conv[4] or not self.stays(layer) or
                    not _lib.lib.mxq_quantized_conv_pool_fits(*conv[:7], *conv[9:11], *geo[10:12])):
                continue
            self.steps[at] = (_CONV_POOL, conv[:7] + conv[9:11] + geo[10:12] + (conv[13],), (),
                              [layer[0], layer[1], None, refs[1]], None, (conv[4], calib, layer))
            gone.add(first)

    def fuse_blocks(self, users, gone):
        """The tail of a residual block as one step: a 3 x 3 convolution that only the sum's 1 x 1
        convolution reads, that convolution with the sum, and a 1 x 1 convolution that reads the
        sum."""
        for at, (kind, ints, floats, refs, _, _) in enumerate(self.steps):
            if kind != _FC_SUM_RQ or not ints[3] or not self.stays(refs):
                continue
            mid = refs[0]
            first = users[id(mid)][0] if isinstance(mid, _Buffer) else at
            if len(users.get(id(mid), ())) != 2 or first >= at or mid.place is not None:
                continue
            kind, geo, calib, conv, _, _ = self.steps[first]
            n, h, w, c, c_mid = geo[:5]
            if (kind != _CONV or conv[10] is not mid or geo[5:13] != (3, 3, 1, 1, 1, 1, 1, 1) or
                    not self.stays(conv) or c_mid != ints[2] or n * h * w != ints[0]):
                continue
            layers = [(c_mid, calib, conv), (ints[1], floats, refs)]
            shape, relu, out, third = (n, h, w, c, c_mid, ints[1]), 0, None, None
            for j in users[id(refs[10])]:
                kind, geo, calib, after, _, _ = self.steps[j]
                if (j > at and kind == _CONV and j not in gone and after[0] is refs[10] and
                        geo[:4] == (n, h, w, ints[1]) and self.stays(after) and
                        geo[5:13] == (1, 1, 1, 1, 0, 0, 1, 1) and
                        _lib.lib.mxq_quantized_block_fits(*shape, geo[4])):
                    layers.append((geo[4], calib, after))
                    relu, out, third = geo[13], after[10], j
                    break
            if third is None:
                if not _lib.lib.mxq_quantized_block_fits(*shape, 0):
                    continue
                layers.append((0, (), ()))
            gone.update((first, third))
            self.steps[at] = (_BLOCK, shape + (layers[2][0], self.steps[first][1][13], relu),
                              floats, [conv[0], None, None, None, None, None, refs[12],
                                       refs[10], out], None, layers)

    def pair_convs(self, gone):
        """Two 1 x 1 convolutions of the same tensor as one step, at the place of the first."""
        first = {}  # id of the tensor -> a convolution of it that has no partner yet
        for j, (kind, geo2, calib2, refs2, _, _) in enumerate(self.steps):
            if (kind != _CONV or j in gone or geo2[5:7] != (1, 1) or geo2[9:11] != (0, 0) or
                    not self.stays(refs2)):
                continue
            at = first.setdefault(id(refs2[0]), j)
            _, geo, calib, refs, _, _ = self.steps[at]
            if (at == j or geo2[:4] + geo2[5:13] != geo[:4] + geo[5:13] or
                    not _lib.lib.mxq_quantized_conv_pair_fits(*geo[:5], geo2[4], *geo[7:9])):
                first[id(refs2[0])] = j
                continue
            self.steps[at] = (_PAIR, geo[:5] + (geo2[4],) + geo[7:9] + (geo[13], geo2[13]),
                              tuple(calib) + tuple(calib2),
                              [refs[0], refs[1], refs2[1], refs[10], refs2[10], None, None], None,
                              [(geo[4], calib, refs), (geo2[4], calib2, refs2)])
            gone.add(j)
            del first[id(refs2[0])]

    def single_convs(self, gone):
        """3 x 3 convolutions that are left on their own and have a kernel for that."""
        for at, (kind, geo, calib, refs, _, _) in enumerate(self.steps):
            if (kind == _CONV and at not in gone and geo[5:13] == (3, 3, 1, 1, 1, 1, 1, 1) and
                    self.stays(refs) and _lib.lib.mxq_quantized_conv3x3_fits(*geo[:5])):
                self.steps[at] = (_CONV3, geo[:5] + (geo[13],), (), [refs[0], None, None, refs[10]],
                                  None, (geo[4], calib, refs))

    def conv3x3_weights(self, ints, at):
        what, names = self.origin[at[1]]

        def make():
            out = torch.empty(int(_lib.lib.mxq_quantized_conv3x3_weights(*ints[3:5])),
                              dtype=torch.int8, device=self.device)
            _lib.check(_lib.lib.mxq_pack_conv3x3_weights(
                self.stream, self.held[at[1]].data_ptr(), int(ints[3]), int(ints[4]),
                out.data_ptr()))
            return out

        return self.laid(("conv3x3", what), names, make).place

    @staticmethod
    def stays(refs):
        """Whether a layer's bias and six ranges are constants of the plan."""
        return all(r is None or (isinstance(r, _Place) and r.place[0] == _HELD)
                   for r in refs[2:9] + refs[13:15])

    def block_weights(self, ints, layers):
        """[where the weights of a _BLOCK step lie]"""
        places = [refs[1] if refs else None for _, _, refs in layers]
        names = sum((self.origin[p[1]][1] for p in places if p), ())

        def make():
            out = torch.empty(int(_lib.lib.mxq_quantized_block_weights(*ints[3:7])),
                              dtype=torch.int8, device=self.device)
            _lib.check(_lib.lib.mxq_pack_block_weights(
                self.stream, *[self.held[p[1]].data_ptr() if p else None for p in places],
                *ints[3:7], out.data_ptr()))
            return out

        key = ("block",) + tuple(self.origin[p[1]][0] if p else None for p in places)
        return self.laid(key, names, make).place

    def block_forms(self, floats, layers, prepared):
        """Where what mxq_prepare_block makes of a _BLOCK step's scales and sum lies."""
        residual = layers[1][2][13:15]
        key, names = self.constants_key(residual)
        for _, calib, refs in layers:  # whatever the bias is, its scale is one of the ranges
            more, read = self.constants_key(refs[3:9])
            key += [len(more), refs[2:3] != [(_NULL, 0, 0)]] + more + [_bits(f) for f in calib]
            names += read

        def make():
            out = torch.empty(int(_lib.lib.mxq_quantized_block_forms()), dtype=torch.int8,
                              device=self.device)
            _lib.check(_lib.lib.mxq_prepare_block(
                self.stream, *[None if base == _NULL else self.held[i].data_ptr()
                               for base, i, _ in prepared],
                *[self.held[i].data_ptr() + offset for _, i, offset in residual],
                *[float(f) for f in floats], out.data_ptr()))
            return out

        return self.laid(("forms",) + tuple(key), tuple(names), make).place

    def constants_key(self, places):
        """Operands that stay as part of a layout's key, and the parameters among them."""
        key, names = [], []
        for base, i, offset in places:
            if base == _NULL:
                key.append(None)
            elif i == self.table_index:
                key.append(_bits(self.constants[offset // 4]))
            else:
                what, read = self.origin[i]
                key += [what, offset]
                names += read
        return key, names

    def prepared(self, columns, calib, places, forms=False):
        """What mxq_prepare_layer makes of a layer's bias and six ranges, if they stay; with the
        short forms that mxq_prepare_forms finds."""
        given = places[2:9]
        if any(base not in (_HELD, _NULL) for base, _, _ in given):
            return (_NULL, 0, 0)
        key, names = self.constants_key(given)
        key = ["prepared", forms, int(columns), _bits(calib[0]), _bits(calib[1])] + key

        def make():
            at = [None if base == _NULL else self.held[i].data_ptr() + offset
                  for base, i, offset in given]
            out = torch.empty(64 + 4 * columns, dtype=torch.int8, device=self.device)
            _lib.check(_lib.lib.mxq_prepare_layer(self.stream, at[0], int(columns), *at[1:],
                                                  float(calib[0]), float(calib[1]),
                                                  out.data_ptr()))
            if forms:
                _lib.check(_lib.lib.mxq_prepare_forms(self.stream, out.data_ptr()))
            return out

        return self.laid(tuple(key), tuple(names), make).place


class _Later:
    """An operand that is laid out when its step is assembled."""

    def __init__(self, find):
        self.find = find


class _Offset:
    """Bytes inside a buffer."""

    def __init__(self, buffer, offset):
        self.buffer, self.offset = buffer, offset


_HANDLERS = {
    "_contrib_quantize_v2": _Builder.quantize,
    "_contrib_quantized_conv": _Builder.conv,
    "_contrib_quantized_elemwise_add": _Builder.add,
    "_contrib_quantized_act": _Builder.act,
    "_contrib_quantized_pooling": _Builder.pooling,
    "_contrib_quantized_flatten": _Builder.flatten,
    "_contrib_quantized_fully_connected": _Builder.fully_connected,
}


def build(params, graph, feeds, stream):
    """(plan, parameters it read, what it laid out of them) of an executor's graph for tensors
    `feeds`, or None.  Works on `stream`, which the caller waits for before the plan runs elsewhere
    and before the graph hands the layouts to another plan."""
    try:
        return _Builder(params, graph, feeds).build(stream)
    except _Unsupported:
        return None
