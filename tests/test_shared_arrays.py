"""Arrays that all calls of a compiled graph share: a graph whose calls may overlap (no GPU: launch lists only)."""
import numpy as np
import pytest

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper
from dace_onnx_amd.sdfg import I64Array, KernelCall, Ptr, Stream
from dace_onnx_amd.transformation import packing
from dace_onnx_amd.transformation.partial_sums import split_products

SHAPE = [1, 512, 7, 7]   # parts pay here


def _conv_graph(before=(), after=(), source="x", result="y", outputs=(("y", SHAPE), ), input_shape=SHAPE):
    rng = np.random.default_rng(2)
    info = lambda n, s: helper.make_tensor_value_info(n, TensorProto.FLOAT, s)   # noqa: E731
    nodes = [*before, helper.make_node("Conv", [source, "w"], [result], kernel_shape=[3, 3], pads=[1] * 4), *after]
    weights = [numpy_helper.from_array(rng.standard_normal((512, 512, 3, 3), dtype=np.float32), "w"), numpy_helper.from_array(np.array(SHAPE, np.int64), "image"),
               numpy_helper.from_array(np.array([512, 49], np.int64), "rows")]
    graph = helper.make_graph(nodes, "g", [info("x", input_shape)], [info(*o) for o in outputs], initializer=weights)
    return helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)])


def _functions_and_transients(model):
    model = donnx.ONNXModel("shared", model)
    model.expand()
    packing.convolutions_in_parts(model)
    return [n.function for s in model.sdfg.nodes() for n in s.nodes() if isinstance(n, KernelCall)], [d for d in model.sdfg.arrays.values() if d.transient]


node = helper.make_node


@pytest.mark.parametrize("graph", [
    lambda: _conv_graph(),
    lambda: _conv_graph(after=[node("Add", ["c", "x"], ["s"]), node("Relu", ["s"], ["y"])], result="c"),
    lambda: _conv_graph(before=[node("Reshape", ["x", "image"], ["i"])], after=[node("Reshape", ["c", "rows"], ["y"])], source="i", result="c",
                        outputs=[("y", [512, 49])], input_shape=[512, 49]),
])
def test_a_convolution_between_arrays_of_the_caller_keeps_none_of_its_own(graph):
    functions, transients = _functions_and_transients(graph())
    assert len(functions) == 1 and functions[0] in ("mi355x_conv2d_f32", "mi355x_conv2d_res_f32")
    assert not any(np.prod(d.shape) > np.prod(SHAPE) for d in transients)


@pytest.mark.parametrize("graph", [
    lambda: _conv_graph(after=[node("Exp", ["c"], ["y"])], result="c"),
    lambda: _conv_graph(before=[node("Exp", ["x"], ["e"])], source="e"),
    lambda: _conv_graph(after=[node("GlobalAveragePool", ["c"], ["y"])], result="c", outputs=[("y", [1, 512, 1, 1])]),
])
def test_one_that_reads_or_writes_an_array_of_the_graph_is_computed_in_parts(graph):
    functions, _ = _functions_and_transients(graph())
    assert "mi355x_conv2d_parts_f32" in functions


def test_the_launch_is_told_how_many_parts_its_array_holds():
    """However many pay where it is launched: the kernel writes as many as there is room for."""
    model = donnx.ONNXModel("parts", _conv_graph(before=[node("Exp", ["x"], ["e"])], source="e"))
    model.expand()
    packing.convolutions_in_parts(model)
    (call, sums), = [(n, model.sdfg.arrays[e.data.data]) for s in model.sdfg.nodes() for n in s.nodes() if isinstance(n, KernelCall) for e in s.out_edges(n)
                     if e.src_conn == "_parts"]
    place = [a.connector if isinstance(a, Ptr) else None for a in call.args].index("_parts")
    assert call.args[place + 1] == sums.shape[0] > 1
    values = [_lib.i64_array(a.values) if isinstance(a, I64Array) else 0 if isinstance(a, Stream) else 16 if isinstance(a, Ptr) else a for a in call.args]
    values[place + 1] = 0
    with pytest.raises(_lib.MI355XError, match="0 parts"):
        _lib.check(_lib.library().mi355x_conv2d_parts_f32(*values), "mi355x_conv2d_parts_f32")


def test_a_graph_with_an_array_of_that_name_already():
    """"c_parts" of the caller's, beside the product and the convolution whose results are "c"."""
    functions, _ = _functions_and_transients(_conv_graph(before=[node("Exp", ["x"], ["c_parts"])], source="c_parts", after=[node("Abs", ["c"], ["y"])], result="c"))
    assert "mi355x_conv2d_parts_f32" in functions
    weights = [numpy_helper.from_array(np.ones(s, np.float32), n) for n, s in (("w", (3072, 768)), ("g", (768, )))]
    infos = [helper.make_tensor_value_info(n, TensorProto.FLOAT, s) for n, s in (("x", [16, 3072]), ("y", [16, 768]))]
    nodes = [node("Exp", ["x"], ["c_parts"]), node("MatMul", ["c_parts", "w"], ["c"]), node("LayerNormalization", ["c", "g"], ["y"], axis=-1)]
    graph = helper.make_graph(nodes, "g", infos[:1], infos[1:], initializer=weights)
    model = donnx.ONNXModel("named", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 17)]))
    model.expand()
    assert split_products(model) == 1
