"""The launch list for other buffers of the caller, against one resolved from the plan (no GPU: nothing is launched)."""
import ctypes

import numpy as np
import pytest
import torch

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper
from dace_onnx_amd.testing.graphs import bert_encoder_layer_model
from oracle import pure_ops


def _chain_model():
    """Reshape of the input, element-wise nodes with a per-column operand, Reshape into the output."""
    nodes = [helper.make_node("Reshape", ["x", "s1"], ["a"], name="n0"), helper.make_node("Mul", ["a", "w"], ["b"], name="n1"),
             helper.make_node("Sub", ["b", "a"], ["c"], name="n2"), helper.make_node("Erf", ["c"], ["d"], name="n3"),
             helper.make_node("Mul", ["d", "b"], ["e"], name="n4"), helper.make_node("Reshape", ["e", "s2"], ["y"], name="n5")]
    weights = [numpy_helper.from_array(v, n) for n, v in (("s1", np.array([6, 8], np.int64)), ("s2", np.array([3, 16], np.int64)),
                                                          ("w", np.arange(8, dtype=np.float32)))]
    info = lambda n, shape: helper.make_tensor_value_info(n, TensorProto.FLOAT, shape)   # noqa: E731
    return helper.make_model(helper.make_graph(nodes, "chain", [info("x", [2, 24])], [info("y", [3, 16])], initializer=weights),
                             opset_imports=[helper.make_opsetid("", 13)])


def _plain(args):
    return [list(a) if isinstance(a, ctypes.Array) else a for a in args]


@pytest.mark.parametrize("graph", ["encoder", "chain"])
@pytest.mark.parametrize("fuse", [True, False])
def test_rebinding_equals_binding(graph, fuse):
    if graph == "encoder":
        weights = pure_ops.bert_layer_weights(np.random.default_rng(3), hidden=128, ffn=256)
        onnx = bert_encoder_layer_model(weights, 2, 32, 4)
    else:
        onnx = _chain_model()
    model = donnx.ONNXModel(f"rebinding_{graph}_{fuse}", onnx, fuse=fuse)
    compiled = model.expand().compile()
    compiled.device = torch.device("cpu")
    buffers = lambda: {k: torch.empty(compiled.sdfg.arrays[k].shape, dtype=compiled._torch_types[k]) for k in compiled._external}   # noqa: E731
    first, second = buffers(), buffers()
    launches, compiled._patches = compiled._bind(first)
    assert compiled._patches is not None and len(compiled._patches) == len(launches) == compiled.num_launches
    before = [_plain(item[3]) for item in launches]
    again = compiled._rebind(launches, {k: t.data_ptr() for k, t in second.items()})
    expected, _ = compiled._bind(second)
    assert [_plain(item[3]) for item in again] == [_plain(item[3]) for item in expected] != before
    assert [_plain(item[3]) for item in launches] == before   # another thread may be walking it
    assert [(i[0], i[1], i[2], i[4], i[6]) for i in again] == [(i[0], i[1], i[2], i[4], i[6]) for i in expected]


def test_recordings_are_not_destroyed_during_a_capture(monkeypatch):
    """A dropped model's recording goes when garbage is collected; not while the caller captures a stream."""
    import gc
    import weakref
    from dace_onnx_amd.sdfg import _Recording
    capturing = []
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: bool(capturing))
    graph = np.zeros(1)   # like a graph no object that the collector tracks itself: only its holder is
    alive, holder = weakref.ref(graph), {"recording": _Recording(graph)}
    holder["itself"] = holder   # as a model and its compiled graph are
    del graph, holder
    capturing.append(1)
    gc.collect()
    assert alive() is not None
    capturing.clear()
    second = _Recording(np.zeros(2))
    assert alive() is None
    alive = weakref.ref(second.graph)
    del second
    assert alive() is None


@pytest.mark.parametrize("after", ["a collection", "a call", "a replay"])
def test_a_recording_that_was_put_aside_is_given_back_after_the_capture(monkeypatch, after):
    """Also where no other recording is ever made or dropped."""
    import gc
    import weakref
    from dace_onnx_amd.sdfg import _Program, _Recording
    capturing = [1]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: bool(capturing))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: type("Stream", (), {"cuda_stream": 0})())
    monkeypatch.setattr(_Program, "run", lambda *a: None)
    compiled = donnx.ONNXModel("given_back", _chain_model()).expand().compile()
    compiled.device = torch.device("cpu")

    def use():
        if after == "a collection":
            gc.collect()
        elif after == "a call":
            compiled(**{k: np.zeros(d.shape, d.dtype.np_dtype) for k, d in compiled.sdfg.arrays.items() if not d.transient})
        else:
            compiled._graph = type("Kept", (), {"graph": type("Graph", (), {"replay": lambda self: None})()})()
            compiled.replay()

    graph = np.zeros(1)
    alive, recording = weakref.ref(graph), _Recording(graph)
    del graph, recording
    use()
    assert alive() is not None
    capturing.clear()
    use()
    assert alive() is None
