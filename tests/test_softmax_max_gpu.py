"""Softmax over rows of any length and address, and with the largest value of each row in the same launch."""
import numpy as np
import pytest
import torch

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
from dace_onnx_amd.onnx.proto import TensorProto, helper

pytestmark = pytest.mark.gpu
COLUMNS = [1, 3, 4, 63, 64, 65, 128, 129, 197, 256, 257, 512, 513, 516, 1024, 1027, 1028, 2048, 2051, 2053, 4099, 4100, 8195, 8197, 16387, 16389, 30522, 32768, 32769]


def call(name, *args):
    _lib.check(getattr(_lib.library(), name)(*args, torch.cuda.current_stream().cuda_stream), name)


def _check(x, y, log=False):
    wide = x.double()
    expected = torch.log_softmax(wide, 1) if log else torch.softmax(wide, 1)
    below = wide.amax(1, keepdim=True) - wide
    # the exponent's rounding is the distance from the maximum times 2^-24 (twice: the product with log2 e), a thread sums at most 64
    # values in a row and a dozen partial sums; the rest are single roundings
    relative = (2 * below + 64 + 16) * 2.0**-24
    if log:
        bound = (below + 8) * 2.0**-23 + (64 + 16) * 2.0**-24
    else:
        bound = expected * relative + 2.0**-126
    assert bool(((y.double() - expected).abs() <= bound).all())


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("cols", COLUMNS)
def test_rows_of_any_length(cols, offset):
    rows = 5 if cols > 2000 else 9
    rng = np.random.default_rng(cols)
    flat = torch.from_numpy(rng.standard_normal(rows * cols + offset, dtype=np.float32) * np.float32(3)).cuda()
    x = flat[offset:].reshape(rows, cols)
    out, largest = torch.full((rows * cols + offset + 8, ), -7.0, device="cuda"), torch.full((rows + 1, ), -7.0, device="cuda")
    y = out[offset:offset + rows * cols].reshape(rows, cols)
    for function in ("softmax", "log_softmax"):
        call(f"mi355x_{function}_f32", x.data_ptr(), y.data_ptr(), rows, cols, 1)
        _check(x, y, log=function == "log_softmax")
    call("mi355x_softmax_max_f32", x.data_ptr(), y.data_ptr(), largest.data_ptr(), rows, cols)
    _check(x, y)
    assert torch.equal(largest[:rows], x.amax(1))
    assert bool((out[:offset] == -7).all()) and bool((out[offset + rows * cols:] == -7).all()) and float(largest[rows]) == -7


@pytest.mark.parametrize("cols", [4, 61, 128, 300, 515, 1001, 2052, 9001, 40000])
def test_largest_values_as_reduce_max_gives_them(cols):
    x = torch.from_numpy(np.random.default_rng(cols).standard_normal((6, cols), dtype=np.float32)).cuda()
    x[1, cols // 2], x[2, 0], x[3, cols - 1], x[4] = float("nan"), float("inf"), float("-inf"), float("-inf")
    x[5, 0], x[5, cols - 1] = float("inf"), float("nan")
    y, apart, largest, reduced = torch.empty_like(x), torch.empty_like(x), torch.empty(6, device="cuda"), torch.empty(6, device="cuda")
    call("mi355x_softmax_max_f32", x.data_ptr(), y.data_ptr(), largest.data_ptr(), 6, cols)
    call("mi355x_softmax_f32", x.data_ptr(), apart.data_ptr(), 6, cols, 1)
    call("mi355x_reduce_f32", _lib.REDUCE_MAX, x.data_ptr(), reduced.data_ptr(), 6, cols, 1)
    assert torch.equal(largest.nan_to_num(nan=-3), reduced.nan_to_num(nan=-3)) and torch.equal(largest.isnan(), reduced.isnan())
    assert torch.equal(y.isnan(), apart.isnan()) and torch.allclose(y.nan_to_num(), apart.nan_to_num(), rtol=1e-6, atol=0)


@pytest.mark.parametrize("axis, keepdims, launches", [(-1, 0, 1), (2, 1, 1), (1, 0, 2)])
def test_softmax_and_reduce_max_of_one_input_in_a_graph(axis, keepdims, launches):
    shape = [3, 7, 45]
    info = lambda n, s: helper.make_tensor_value_info(n, TensorProto.FLOAT, s)   # noqa: E731
    reduced = [d if i != axis % 3 else 1 for i, d in enumerate(shape) if i != axis % 3 or keepdims]
    nodes = [helper.make_node("Softmax", ["x"], ["p"], axis=2), helper.make_node("ReduceMax", ["x"], ["m"], axes=[axis], keepdims=keepdims)]
    graph = helper.make_graph(nodes, "g", [info("x", shape)], [info("p", shape), info("m", reduced)])
    proto = helper.make_model(graph, opset_imports=[helper.make_opsetid("", 13)])
    x = torch.from_numpy(np.random.default_rng(0).standard_normal(shape, dtype=np.float32)).cuda()
    for fuse in (True, False):
        model = donnx.ONNXModel(f"scores_{fuse}", proto, fuse=fuse)
        p, m = model(x)
        assert model.compile_and_init().num_launches == (launches if fuse else 2)
        _check(x.reshape(-1, 45), p.reshape(-1, 45))
        assert torch.equal(m, x.amax(axis, keepdim=bool(keepdims)))
