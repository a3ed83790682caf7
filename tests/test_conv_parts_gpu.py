"""Convolutions in parts of their channels and the launch that adds them up, against float64."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper

pytestmark = pytest.mark.gpu


def call(name, *args):
    _lib.check(getattr(_lib.library(), name)(*args, torch.cuda.current_stream().cuda_stream), name)


def normal(seed, *shapes):
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).cuda() for s in shapes]


def conv(x, w, bias, residual, stride, epilogue, mean, packed=True, count=4):
    (N, C, H, Wd), M, i64 = x.shape, w.shape[0], _lib.i64_array
    OH, OW = (H - 1) // stride + 1, (Wd - 1) // stride + 1
    geometry = (N, C, H, Wd, M, 3, 3, i64([1] * 4), i64([stride] * 2), i64([1, 1]))
    copy = torch.empty(-(-M // 32) * -(-C // 16) * 9 * 768, dtype=torch.int32, device="cuda") if packed else None
    if packed:
        call("mi355x_pack_conv_f32", w.data_ptr(), copy.data_ptr(), M, C, 3, 3)
    outputs = N * M * OH * OW
    parts = torch.full((count * outputs + 64, ), -7.0, device="cuda")
    y = torch.full((N * M * (1 if mean else OH * OW) + 64, ), -7.0, device="cuda")
    call("mi355x_conv2d_parts_f32", x.data_ptr(), w.data_ptr(), _lib.ptr(copy), _lib.ptr(bias), _lib.ptr(residual), parts.data_ptr(), count, y.data_ptr(), *geometry, epilogue, int(mean))
    assert bool((y[-64:] == -7).all()) and bool((parts[-64:] == -7).all()) and bool((parts[(count - 1) * outputs:-64] != -7).any()) == (packed or (mean and count == 1))
    return y[:-64].reshape((N, M) if mean else (N, M, OH, OW))


def wide_conv(x, w, bias, residual, stride, epilogue):
    N, C, H, Wd = x.shape
    M, OH, OW = w.shape[0], (H - 1) // stride + 1, (Wd - 1) // stride + 1
    columns = F.unfold(x.double(), 3, padding=1, stride=stride)

    def total(f, relu):
        v = torch.stack([f(w.double()).reshape(M, -1) @ f(c) for c in columns]).reshape(N, M, OH, OW)
        v = v + f(bias.double()).reshape(1, -1, 1, 1) if epilogue & _lib.EPI_BIAS else v
        v = v.relu() if epilogue & _lib.EPI_RELU else v
        v = v + f(residual.double()) if epilogue & _lib.EPI_RESIDUAL else v
        return v.relu() if epilogue & _lib.EPI_RELU_AFTER else v
    # one rounding (2^-23, truncation included) for each step of at least two products of a sum, eight for the parts, biases and residuals
    return total(lambda v: v, True), total(torch.abs, False) * (9 * C // 2 + 8) * 2.0**-23


@pytest.mark.parametrize("mean", [False, True])
@pytest.mark.parametrize("epilogue", [0, _lib.EPI_BIAS | _lib.EPI_RELU, _lib.EPI_BIAS | _lib.EPI_RESIDUAL | _lib.EPI_RELU_AFTER])
@pytest.mark.parametrize("N, C, H, Wd, M, stride", [(1, 512, 7, 7, 512, 1), (1, 128, 1, 1, 33, 1), (2, 256, 9, 13, 70, 2), (3, 256, 8, 8, 64, 1), (1, 512, 17, 5, 1, 1), (1, 256, 16, 16, 40, 1)])
def test_convolution_in_parts(N, C, H, Wd, M, stride, epilogue, mean):
    x, w, bias = normal(C + M, (N, C, H, Wd), (M, C, 3, 3), (M, ))
    residual, = normal(1, (N, M, (H - 1) // stride + 1, (Wd - 1) // stride + 1))
    expected, bound = wide_conv(x, w, bias, residual, stride, epilogue)
    if mean:
        expected, bound = expected.mean((2, 3)), bound.mean((2, 3)) * 1.1
    for packed, count in ((C >= 256, 4), (C >= 256, 2), (False, 2)):   # (no more parts than there is room for, whatever would pay)
        got = conv(x, w, bias, residual, stride, epilogue, mean, packed, count)
        assert bool(((got.double() - expected).abs() <= bound + 1e-30).all())


@pytest.mark.parametrize("mean", [False, True])
def test_parts_keep_infinities_nan_and_the_largest_values(mean):
    x, w = normal(7, (2, 256, 7, 7), (64, 256, 3, 3))
    w *= 1e-2
    x[0, 3, 2, 2], x[0, 200, 6, 6], x[1, 130, 0, 0], x[1, 255, 6, 0] = float("inf"), float("nan"), float("-inf"), 3e37
    got, apart = (conv(x, w, None, None, 1, 0, mean, packed) for packed in (True, False))
    assert torch.equal(got.isnan(), apart.isnan()) and torch.equal(got[got.isinf()], apart[apart.isinf()]) and bool(got.isnan().any())
    finite = apart.isfinite()
    assert torch.equal(finite, got.isfinite()) and torch.allclose(got[finite], apart[finite], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("pooled", [True, False])
def test_end_of_a_classifier_in_a_graph(pooled):
    rng = np.random.default_rng(2)
    w = (rng.standard_normal((512, 512, 3, 3)) * np.sqrt(2 / 4608)).astype(np.float32)
    b = rng.standard_normal(512).astype(np.float32)
    info = lambda n, s: helper.make_tensor_value_info(n, TensorProto.FLOAT, s)   # noqa: E731
    nodes = [helper.make_node("Conv", ["x", "w", "b"], ["c"], kernel_shape=[3, 3], pads=[1] * 4), helper.make_node("Add", ["c", "x"], ["s"]), helper.make_node("Relu", ["s"], ["r"])]
    nodes += [helper.make_node("GlobalAveragePool", ["r"], ["y"])] if pooled else [helper.make_node("Exp", ["r"], ["y"])]
    graph = helper.make_graph(nodes, "end", [info("x", [1, 512, 7, 7])], [info("y", [1, 512, 1, 1] if pooled else [1, 512, 7, 7])],
                              initializer=[numpy_helper.from_array(w, "w"), numpy_helper.from_array(b, "b")])
    model = donnx.ONNXModel("end", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)]))
    x, = normal(3, (1, 512, 7, 7))
    got = model(x)
    names = [n.function for n, _ in model.compile_and_init().bound_launches()]
    assert names[0] == "mi355x_conv2d_parts_f32" and len(names) == (1 if pooled else 2)
    epilogue = _lib.EPI_BIAS | _lib.EPI_RESIDUAL | _lib.EPI_RELU_AFTER
    expected, bound = wide_conv(x, torch.from_numpy(w).cuda(), torch.from_numpy(b).cuda(), x, 1, epilogue)
    finish = (lambda v: v.mean((2, 3), keepdim=True)) if pooled else torch.exp
    close = lambda y: bool(((y.double() - finish(expected)).abs() <= (finish(bound) * 1.1 if pooled else 2 * bound * finish(expected) + 2e-6 * finish(expected))).all())   # noqa: E731
    assert close(got) and torch.equal(model(x), got)
    replayed = donnx.ONNXModel("end_replayed", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)]), use_hip_graph=True)
    for _ in range(3):
        assert torch.equal(replayed(x), got)
        torch.cuda.synchronize()
    list(model.weights.values())   # handed out: the launches read the weights themselves
    assert close(model(x))
