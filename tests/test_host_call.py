"""Models without csrc/host_call.cpp, or with one built against another torch: calls take the general way (no GPU: plans only)."""
import shutil

import numpy as np
import pytest
import torch

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib, sdfg
from dace_onnx_amd.onnx.proto import TensorProto, helper


@pytest.fixture
def loader():
    sdfg._host_call.cache_clear()
    yield sdfg._host_call
    sdfg._host_call.cache_clear()


def test_the_built_module_is_for_this_torch(loader):
    assert loader().built_against.split() == [torch.__version__, torch.version.git_version]


@pytest.mark.parametrize("fault", ["missing", "no module", "another torch"])
def test_without_the_module_there_is_no_plan(loader, tmp_path, monkeypatch, caplog, fault):
    info = helper.make_tensor_value_info
    graph = helper.make_graph([helper.make_node("Relu", ["x"], ["y"])], "g", [info("x", TensorProto.FLOAT, [4])], [info("y", TensorProto.FLOAT, [4])])
    compiled = donnx.ONNXModel("no_plan", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)])).expand().compile()
    compiled.device, compiled._program = torch.device("cuda:0"), object()   # as after a first call
    name = loader().__spec__.origin.rsplit("/", 1)[1]
    if fault == "no module":
        (tmp_path / name).write_bytes(np.arange(64, dtype=np.uint8).tobytes())
    elif fault == "another torch":
        shutil.copy(loader().__spec__.origin, tmp_path / name)
        monkeypatch.setattr(torch.version, "git_version", "0" * 40)
    loader.cache_clear()
    monkeypatch.setattr(_lib, "LIBRARY_PATH", str(tmp_path / "libmi355x_onnx.so"))
    for _ in range(2):
        assert compiled.host_plan({"x": 0}, {"y": 0}, {}, {}) is None
    assert len([r for r in caplog.records if "general way" in r.message]) == 1
