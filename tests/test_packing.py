"""Packed copies of constant operands: which tensors they are made of and when they are used (no GPU: packing launches are recorded, not issued)."""
import contextlib

import numpy as np
import pytest
import torch

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
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
    monkeypatch.setattr(torch.cuda, "current_stream", lambda *a: type("Stream", (), {"synchronize": lambda self: None})())
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
    for copy in copies:   # nothing to do again, in the mode or out of it
        copy.refresh()
    assert len(pack_launches) == 4
