"""Packed copies of constant operands: which tensors they are made of and when they are used (no GPU: packing launches are recorded, not issued)."""
import contextlib
import copy

import numpy as np
import pytest
import torch
import torch.nn as nn

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper
from dace_onnx_amd.pytorch.module import DaceModule
from dace_onnx_amd.sdfg import _Program
from dace_onnx_amd.testing.graphs import bert_encoder_layer_model
from dace_onnx_amd.transformation import packing
from oracle import pure_ops


class _Library:
    """The library with the packing launches recorded instead of issued."""

    def __init__(self, lib, launches):
        self._lib, self._launches = lib, launches

    def __getattr__(self, name):
        if name not in ("mi355x_pack_f32", "mi355x_pack_conv_f32"):
            return getattr(self._lib, name)
        return lambda *args: self._launches.append((name, *args)) or 0


@pytest.fixture
def pack_launches(monkeypatch):
    launches = []
    library = _Library(_lib.library(), launches)
    monkeypatch.setattr(packing._lib, "library", lambda: library)
    monkeypatch.setattr(packing._lib, "current_stream", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: type("Stream", (), {"synchronize": lambda self: None, "cuda_stream": 0})())
    return launches


def _encoder():
    weights = pure_ops.bert_layer_weights(np.random.default_rng(0))
    return donnx.ONNXModel("encoder", bert_encoder_layer_model(weights, 8, 128, 12))


@pytest.mark.parametrize("construction", [True, False])
def test_models_made_or_first_called_under_inference_mode_are_packed(pack_launches, construction):
    """Their weights, or the copies that fusion derives from them, are tensors without a version counter."""
    with torch.inference_mode() if construction else contextlib.nullcontext():
        model = _encoder()
    with torch.inference_mode():
        model.expand()
        copies = packing.pack_constant_operands(model)
    assert len(copies) == len(pack_launches) == 4 and all(c.weight.is_inference() for c in copies)
    assert all(c.current() for c in copies)


@pytest.fixture
def program_runs(monkeypatch):
    """Calls of compiled graphs, recorded instead of issued."""
    runs = []
    monkeypatch.setattr(_Program, "run", lambda program, addresses, stream: runs.append(list(addresses)))
    return runs


def _ready(model):
    """``model`` as its first call finds it, in host memory."""
    model.expand()
    model._packed = packing.pack_constant_operands(model)
    model._compiled = model.sdfg.compile()
    model._compiled.device = torch.device("cpu")
    return model


def _operands(model):
    """(packed copy or None, weight) of each launch by a packed copy, as addresses."""
    return [tuple(item[3][1:3]) for item in model._compiled._launch_list if item[2] == "mi355x_gemm_packed_f32"]


def _packed_by(model):
    return [(c.packed.data_ptr(), c.weight.data_ptr()) for c in model._packed]


X = torch.zeros(8, 128, 768)


def test_a_weight_that_was_written_or_replaced_is_read_itself(pack_launches, program_runs):
    model = _ready(_encoder())
    assert len(model._packed) == 4
    model(X)
    assert sorted(_operands(model)) == sorted(_packed_by(model))
    first, second = model._packed[:2]
    first.weight[0] += 1
    model.weights[second.weight_name] = second.weight.clone()
    model(X)
    expected = {(0, first.weight.data_ptr()), (0, model.weights[second.weight_name].data_ptr())} | set(_packed_by(model)[2:])
    assert {(p or 0, w) for p, w in _operands(model)} == expected
    model.weights[second.weight_name] = second.weight
    model(X)
    assert _packed_by(model)[1] in _operands(model)
    assert len(pack_launches) == 4 and len(program_runs) == 3


@pytest.mark.parametrize("replace", [lambda w: w.double(), lambda w: w[:8].contiguous(), lambda w: w.t().contiguous().t(), lambda w: w.numpy()[:4]])
def test_no_launch_reads_a_replaced_weight_that_the_call_refuses(pack_launches, program_runs, replace):
    model = _ready(_encoder())
    name = model._packed[0].weight_name
    model.weights[name] = replace(model.weights[name])
    with pytest.raises(TypeError):
        model(X)
    assert len(pack_launches) == 4 and not program_runs


def test_recordings_keep_the_weights_they_were_made_with(pack_launches, program_runs, monkeypatch):
    """A weight written in place takes effect at the next replay, one that is replaced does not, whether packed or not."""
    model = _ready(_encoder())
    model.use_hip_graph = True
    replays = []
    monkeypatch.setattr(model._compiled, "capture_graph", lambda with_packed: None)
    monkeypatch.setattr(model._compiled, "replay", lambda: replays.append(1))
    model(X)
    model(X)
    assert (len(program_runs), len(replays)) == (1, 1) and sorted(_operands(model)) == sorted(_packed_by(model))
    first, second = model._packed[:2]
    first.weight[0] += 1
    model.weights[second.weight_name] = second.weight + 1
    bias = next(n for n, w in model.weights.items() if w.dim() == 1 and w.dtype is torch.float32)
    kept, model.weights[bias] = model.weights[bias], torch.ones_like(model.weights[bias])
    model(X)
    assert (len(program_runs), len(replays)) == (2, 1)
    assert {(p or 0, w) for p, w in _operands(model)} == {(0, w) for _, w in _packed_by(model)[:2]} | set(_packed_by(model)[2:])
    assert model.weights[bias].data_ptr() not in program_runs[-1] and kept.data_ptr() in program_runs[-1] + program_runs[0]
    model(X)
    assert (len(program_runs), len(replays)) == (2, 2) and len(pack_launches) == 4


def _head(**options):
    """A dense layer whose odd width leaves fusion nothing to derive: the product is by the initializer itself."""
    rng = np.random.default_rng(0)
    weight = numpy_helper.from_array(rng.standard_normal((768, 3001), dtype=np.float32), "w")
    info = lambda n, shape: helper.make_tensor_value_info(n, TensorProto.FLOAT, shape)   # noqa: E731
    graph = helper.make_graph([helper.make_node("MatMul", ["x", "w"], ["y"])], "head", [info("x", [1024, 768])], [info("y", [1024, 3001])], initializer=[weight])
    return donnx.ONNXModel("head", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 13)]), **options)


HEAD_X = torch.zeros(1024, 768)


@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("read", [lambda w: w["w"], lambda w: w.get("w"), lambda w: w.setdefault("w"), lambda w: dict(w)["w"], lambda w: {**w}["w"],
                                  lambda w: list(w.values())[0], lambda w: [t for n, t in w.items() if n == "w"][0], lambda w: w.copy()["w"], lambda w: (w | {})["w"],
                                  lambda w: ({} | w)["w"], lambda w: copy.copy(w)["w"], lambda w: w.pop("w")])
def test_a_weight_that_was_handed_out_is_read_itself(pack_launches, program_runs, read, first):
    """Whoever holds it can write it in ways that torch does not count."""
    model = _head()
    handed = read(model.weights) if first else None
    if first and "w" not in model.weights:
        model.weights["w"] = handed
    _ready(model)
    model(HEAD_X)
    assert len(model._packed) == 1 and not model._packed[0].derived
    packed = model._packed[0].packed
    if first:
        assert packed is None and not pack_launches
    else:
        assert _operands(model) == [(packed.data_ptr(), model._packed[0].weight.data_ptr())]
        handed = read(model.weights)
        if "w" not in model.weights:
            model.weights["w"] = handed
        model(HEAD_X)
    assert _operands(model) == [(0 if not first else None, handed.data_ptr())]
    compiled = model._compiled   # called without the model
    compiled(x=HEAD_X, y=torch.zeros(1024, 3001), **model.clean_weights)
    assert _operands(model)[0][0] in (0, None) and "_packed = nullptr" in compiled.program_source("head")[0]


def test_names_and_sizes_hand_nothing_out(pack_launches):
    model = _head()
    assert list(model.weights) == ["w"] == list(model.weights.keys()) and "w" in model.weights and len(model.weights) == 1
    assert len(packing.pack_constant_operands(model) if model.expand() else ()) == len(pack_launches) == 1


def test_parameters_of_a_module_are_packed_on_request(pack_launches, program_runs, monkeypatch):
    linear = nn.Linear(768, 1024)
    model = _ready(DaceModule(nn.Sequential(linear, nn.ReLU()), dummy_inputs=(HEAD_X, )).dace_model)
    model(HEAD_X)
    assert not pack_launches and _operands(model) == [(None, linear.weight.data_ptr())]
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    model.pack_weights()
    model(HEAD_X)
    assert len(pack_launches) == 1 and _operands(model) == _packed_by(model)
    with torch.no_grad():
        linear.weight.mul_(2)   # (torch counts this)
    model(HEAD_X)
    assert _operands(model) == [(0, linear.weight.data_ptr())]
    model.pack_weights()
    model(HEAD_X)
    assert len(pack_launches) == 2 and _operands(model) == _packed_by(model)


def test_weights_packed_on_request_are_those_that_the_call_takes(pack_launches, program_runs, monkeypatch):
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    model = _ready(_head())
    weight = model.weights["w"]
    for replaced in (weight.double(), weight[:8], weight.t().contiguous().t(), weight.numpy()):
        model.weights["w"] = replaced
        model.pack_weights()
    assert len(pack_launches) == 1 and not model._packed[0].current()


def test_a_recording_is_made_again_when_a_weight_is_handed_out(pack_launches, program_runs, monkeypatch):
    model = _ready(_head(use_hip_graph=True))
    replays = []
    monkeypatch.setattr(model._compiled, "capture_graph", lambda with_packed: None)
    monkeypatch.setattr(model._compiled, "replay", lambda: replays.append(1))
    model(HEAD_X)
    model(HEAD_X)
    assert _operands(model) == _packed_by(model) and (len(program_runs), len(replays)) == (1, 1)
    handed = model.weights["w"]
    model(HEAD_X)
    model(HEAD_X)
    assert _operands(model) == [(0, handed.data_ptr())] and (len(program_runs), len(replays)) == (2, 2)


def test_a_callers_recording_reads_the_weights_themselves(pack_launches, program_runs, monkeypatch):
    """Its replays follow weights that are written after it, which nobody is asked about then."""
    model, recorded = _ready(_head()), []
    model(HEAD_X)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: None)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "graph", lambda g: contextlib.nullcontext())
    monkeypatch.setattr(model._compiled, "_run", recorded.extend)
    model._compiled.capture_graph()
    assert [item[3][1] for item in recorded] == [0] and _operands(model) == _packed_by(model)
    monkeypatch.setattr(model, "_capturing", lambda: True)
    model(HEAD_X)
    assert _operands(model) == [(0, model._packed[0].weight.data_ptr())]


@pytest.mark.parametrize("build", [_encoder, _head])
def test_a_first_call_under_stream_capture_packs_nothing_and_waits_for_nothing(pack_launches, monkeypatch, build):
    """A packing launch would be recorded instead of run, and a wait ends the capture: the launches read the weights themselves."""
    model = build()
    model.expand()
    weights = list(dict.items(model.weights))
    monkeypatch.setattr(model, "_capturing", lambda: True)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: pytest.fail("waits for a stream that is being captured"))
    copies = packing.pack_constant_operands(model)
    assert copies and not pack_launches and not any(c.current() for c in copies)
    assert [(n, id(t)) for n, t in dict.items(model.weights)] == [(n, id(t)) for n, t in weights]


def test_names_of_arrays_are_kept_once():
    from dace_onnx_amd.onnx.onnx_importer import clean_onnx_name
    assert not hasattr(clean_onnx_name.__wrapped__, "cache_info")
    names = [f"{i}.a/b:c-d" for i in range(5000)]   # more than one large graph has
    cleaned = [clean_onnx_name(n) for n in names]
    misses = clean_onnx_name.cache_info().misses
    assert [clean_onnx_name(n) for n in names] == cleaned and clean_onnx_name.cache_info().misses == misses
    assert cleaned[7] == "ONNX_7DOTaSLASHbCOLONcDASHd"


@pytest.mark.parametrize("M, N, K, kc", [(1, 20149, 832, True), (5, 20736, 2432, True), (8, 4576, 2080, True), (16, 768, 3072, True), (20, 7232, 2368, False),
                                         (25, 3776, 1568, True), (13, 4650, 800, False), (1245, 96, 1056, True)])
def test_products_that_the_weights_bytes_bound_are_not_packed(M, N, K, kc):
    """A packed copy has half as many bytes again: these took 1.07 to 1.39 times as long by it, with weights from beyond the L2."""
    assert _lib.library().mi355x_gemm_packed_pays(1, M, N, K, int(kc)) == 0


@pytest.mark.parametrize("M, N, K", [(128, 768, 3072), (128, 2304, 768), (865, 3072, 768), (1024, 768, 768), (8192, 768, 3072), (28, 13792, 1280)])
def test_products_of_more_rows_are_packed(M, N, K):
    assert _lib.library().mi355x_gemm_packed_pays(1, M, N, K, 1) == 1
