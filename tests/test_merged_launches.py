"""Pairs of launches become one where fusion was asked for, and nowhere else (no GPU: launch lists only)."""
import numpy as np
import pytest
import torch
import torch.nn as nn

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper
from dace_onnx_amd.pytorch.module import DaceModule
from dace_onnx_amd.sdfg import KernelCall


def _model(**options):
    info = lambda n, *s: helper.make_tensor_value_info(n, TensorProto.FLOAT, list(s))   # noqa: E731
    nodes = [helper.make_node("Gemm", ["x", "w", "b"], ["y"], transB=1), helper.make_node("Softmax", ["y"], ["p"], axis=1), helper.make_node("Softmax", ["z"], ["q"], axis=1),
             helper.make_node("ReduceMax", ["z"], ["m"], axes=[1], keepdims=0)]
    weights = [numpy_helper.from_array(np.ones(s, np.float32), n) for n, s in (("w", (10, 64)), ("b", (10, )))]
    graph = helper.make_graph(nodes, "g", [info("x", 5, 64), info("z", 5, 33)], [info("p", 5, 10), info("q", 5, 33), info("m", 5)], initializer=weights)
    return donnx.ONNXModel("merged", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)]), **options)


def _module(**options):
    return DaceModule(nn.Sequential(nn.Linear(64, 10), nn.Softmax(dim=1)).eval(), dummy_inputs=(torch.zeros(5, 64), ), **options).dace_model


def _functions(model, expand):
    expand(model)
    model.expand()   # as its first call does
    model._merge_launches()
    return sorted(n.function for s in model.sdfg.nodes() for n in s.nodes() if isinstance(n, KernelCall))


APART = ["mi355x_gemm_f32", "mi355x_reduce_f32", "mi355x_softmax_f32", "mi355x_softmax_f32"]


@pytest.mark.parametrize("make, expand", [(lambda: _model(auto_optimize=False), lambda m: None), (lambda: _model(fuse=False), lambda m: None),
                                          (_model, lambda m: m.expand_onnx_nodes()), (lambda: _model(fuse=False), lambda m: m.auto_optimize()),
                                          (lambda: _module(auto_optimize=False), lambda m: None)])
def test_launches_stay_apart_without_fusion(make, expand):
    functions = _functions(make(), expand)
    assert functions == APART or functions == ["mi355x_gemm_f32", "mi355x_softmax_f32"]


@pytest.mark.parametrize("make, expand", [(_model, lambda m: None), (_model, lambda m: m.expand()), (_model, lambda m: m.auto_optimize()), (_module, lambda m: None)])
def test_launches_are_merged_with_fusion(make, expand):
    assert _functions(make(), expand) in (["mi355x_gemm_softmax_f32", "mi355x_softmax_max_f32"], ["mi355x_gemm_softmax_f32"])
