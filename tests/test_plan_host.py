"""The host side of plans and of the imperative call path, without a GPU."""
import threading

import pytest
import torch

from mxnet_amd import _frontend, _lib, contrib, operator
from mxnet_amd import symbol as S
from mxnet_amd.executor import Executor, _Graph


def replaced(params):
    params["w"] = params["w"].clone()


def written(params):
    params["w"].add_(1)


def written_through_a_view(params):
    params["w"][1:].zero_()


def written_in_inference_mode(params):
    with torch.inference_mode():
        params["w"].add_(1)


def other_memory(params):
    params["w"].data = params["w"].clone()


def other_extents(params):
    params["w"].data = params["w"].reshape(6, 4)


def other_strides(params):
    params["w"].data = params["w"].t()


def other_type(params):
    params["w"].data = params["w"].view(torch.uint8)


def removed(params):
    del params["w"]


@pytest.mark.parametrize("change", [replaced, written, written_through_a_view,
                                    written_in_inference_mode, other_memory, other_extents,
                                    other_strides, other_type, removed])
def test_changed_parameters_are_noticed(change):
    params = {"w": torch.arange(24, dtype=torch.int8).reshape(4, 6), "b": torch.zeros(3)}
    read = tuple(_frontend.as_read(name, t) for name, t in params.items())
    assert _frontend.same_params(params, read)
    change(params)
    assert not _frontend.same_params(params, read)


@pytest.mark.parametrize("invoke", [operator.invoke, contrib.invoke])
def test_name_is_the_nodes_name(invoke):
    """`name` is no attribute of the operator: the call gets as far as its tensors."""
    x = torch.zeros(4)
    with pytest.raises(operator.MXNetError, match="device tensors"):
        invoke("_contrib_quantize_v2", x, name="q", out_type="int8")
    with pytest.raises(operator.MXNetError, match="device tensors"):
        invoke("_contrib_quantize_v2", x, name=None)
    with pytest.raises(AttributeError, match="encode"):
        invoke("_contrib_quantize_v2", x, name=3)
    with pytest.raises(operator.MXNetError, match="(?s)Cannot find argument 'nam'.*name=.q2."):
        invoke("_contrib_quantize_v2", x, nam="q", name="q2")


def float_layer():
    sym = S.FullyConnected(S.Variable("data"), num_hidden=3, name="f")
    w, b = torch.arange(12.0).reshape(3, 4), torch.ones(3)
    x = torch.tensor([[1.0, -2.0, 3.0, 0.5]])
    return Executor(sym, {"f_weight": w, "f_bias": b}, device="cpu"), x, x @ w.t() + b


def test_float_graph_on_the_host():
    ex, x, want = float_layer()
    assert torch.equal(ex.forward(data=x)[0], want)
    assert torch.equal(ex.forward(data=x.numpy())[0], want)


def test_inputs_that_the_graph_has_no_variable_for():
    ex, x, want = float_layer()
    assert torch.equal(ex.forward(label=None, data=x, more=object())[0], want)


def test_threads_share_a_graphs_nodes():
    """Plans refer to a node by its handle: whichever thread makes it, there is one, and a symbol
    put in the executor's hands later does not take it away from a pass that goes on."""
    sym = S.Variable("data")
    for i in range(40):
        sym = S.FullyConnected(sym, num_hidden=3, name="f%d" % i)
    for _ in range(5):
        graph, seen, start = _Graph(sym), [], threading.Barrier(8)

        def walk():
            start.wait()
            seen.append([graph.op_node(i, op, name, attrs)
                         for i, (op, name, attrs, _) in enumerate(graph.nodes) if op != "null"])

        threads = [threading.Thread(target=walk) for _ in range(8)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert len(seen) == 8 and all(a is b for nodes in seen for a, b in zip(nodes, seen[0]))
    ex, x, want = float_layer()
    before = ex._structure()
    ex.symbol = S.Activation(ex.symbol, act_type="relu", name="r")
    assert torch.equal(ex.forward(data=-x)[0], torch.relu(ex.params["f_bias"] + 1 - want))
    assert ex._structure() is not before and before.symbol is not ex.symbol


# image columns (padded by 7 on either side), channels, pooled columns
@pytest.mark.parametrize("w,o,pw,fits", [(2 ** 22 - 12, 1008, 2 ** 21, True),
                                         (2 ** 22 - 13, 1024, 2 ** 21 - 1, True),
                                         (2 ** 22 - 12, 1024, 2 ** 21, False),
                                         (2 ** 23, 1024, 2 ** 22, False)])
def test_stem_offsets_of_a_pooled_row(w, o, pw, fits):
    """A lane stores at an offset of 32 bits in its pooled row, and one that has nothing to store at
    2^31, which the row must not reach."""
    assert _lib.lib.mxq_quantized_conv_pool_fits(1, 1, w, 16, o, 4, 4, 2, 7, 1, pw) == fits


@pytest.mark.parametrize("n,fits", [(2 ** 26 - 5, True), (2 ** 26 - 4, False), (2 ** 27, False)])
def test_stem_lanes_of_a_launch(n, fits):
    """A wave for each image of one strip: a launch has less than 2^32 lanes."""
    assert _lib.lib.mxq_quantized_conv_pool_fits(n, 1, 1, 16, 16, 4, 4, 2, 2, 1, 1) == fits


@pytest.mark.parametrize("pad,fits", [(2 ** 30, True), (2 ** 30 + 1, False), (2 ** 31 - 1, False)])
def test_stem_extent_of_a_padded_image(pad, fits):
    """The convolution's extents are ints: 1 + 2 * pad - 3 of them."""
    args = [1, 1, 1, 16, 16, 4, 4, 2, 2, 1, 1]
    for axis in (7, 8):
        assert _lib.lib.mxq_quantized_conv_pool_fits(*args[:axis], pad, *args[axis + 1:]) == fits
