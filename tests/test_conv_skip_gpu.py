"""The end of a residual block and the 1 x 1 convolution of its other branch in one launch, against float64."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper

pytestmark = pytest.mark.gpu
FORMS = range(1, 10)


def call(name, *args):
    _lib.check(getattr(_lib.library(), name)(*args, torch.cuda.current_stream().cuda_stream), name)


def pack(w):
    M, C, KH, KW = w.shape
    packed = torch.empty(-(-M // 32) * -(-C // 16) * KH * KW * 768, dtype=torch.int32, device="cuda")
    call("mi355x_pack_conv_f32", w.data_ptr(), packed.data_ptr(), M, C, KH, KW)
    return packed


def block(x, w, b, x2, w2, b2, strides2, relu, packed=True):
    N, C, H, Wd = x.shape
    M, C2, i64 = w.shape[0], x2.shape[1], _lib.i64_array
    geometry = (N, C, H, Wd, M, 3, 3, i64([1] * 4), i64([1, 1]), i64([1, 1]), C2, *x2.shape[2:], i64(strides2))
    copies = (pack(w), pack(w2)) if packed else (None, None)
    scratch, y = torch.full((N, M, H, Wd), -7.0, device="cuda"), torch.full((N * M * H * Wd + 64, ), -7.0, device="cuda")
    assert not packed or _lib.library().mi355x_conv2d_skip_pays(*geometry)
    call("mi355x_conv2d_skip_f32", x.data_ptr(), w.data_ptr(), _lib.ptr(copies[0]), _lib.ptr(b), x2.data_ptr(), w2.data_ptr(), _lib.ptr(copies[1]), _lib.ptr(b2),
         scratch.data_ptr(), y.data_ptr(), *geometry, (_lib.EPI_BIAS if b is not None else 0) | (_lib.EPI_RELU_AFTER if relu else 0))
    assert bool((y[-64:] == -7).all()) and bool((scratch == -7).all()) == packed
    return y[:-64].reshape(N, M, H, Wd)


def wide_block(x, w, b, x2, w2, b2, strides2, relu):
    """In float64, and a bound of the error."""
    N, _, H, Wd = x.shape
    M = w.shape[0]
    at = x2.double()[:, :, ::strides2[0], ::strides2[1]].reshape(N, x2.shape[1], -1)
    columns = F.unfold(x.double(), 3, padding=1)

    def total(f):
        sums = torch.stack([f(w.double()).reshape(M, -1) @ f(c) for c in columns]) + torch.stack([f(w2.double()).reshape(M, -1) @ f(c) for c in at])
        return sums + sum(f(v.double()).reshape(1, -1, 1) for v in (b, b2) if v is not None)
    terms = 9 * x.shape[1] + x2.shape[1]
    # one rounding (2^-23, truncation included) for each step of at least two products of a sum, and eight for the sums of the groups, the products left out, biases
    return (total(lambda v: v).relu() if relu else total(lambda v: v)).reshape(N, M, H, Wd), (total(torch.abs) * (terms // 2 + 8) * 2.0**-23).reshape(N, M, H, Wd)


def normal(seed, *shapes):
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).cuda() for s in shapes]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("N, C, H, Wd, M, C2, strides2, relu, bias", [(1, 8, 3, 3, 1, 8, (1, 1), False, False), (2, 24, 7, 9, 33, 40, (2, 2), True, True),
                                                                      (1, 64, 14, 14, 64, 32, (2, 2), True, True), (3, 16, 11, 5, 70, 136, (2, 3), False, True),
                                                                      (1, 128, 7, 7, 96, 264, (2, 2), True, False)])
def test_block(tuning, form, N, C, H, Wd, M, C2, strides2, relu, bias):
    tuning(MI355X_CONV_PACKED=form)
    x, w, b, x2, w2, b2 = normal(C, (N, C, H, Wd), (M, C, 3, 3), (M, ), (N, C2, (H - 1) * strides2[0] + 1, (Wd - 1) * strides2[1] + strides2[1]), (M, C2, 1, 1), (M, ))
    b, b2 = (b, b2) if bias else (None, None)
    expected, bound = wide_block(x, w, b, x2, w2, b2, strides2, relu)
    assert bool(((block(x, w, b, x2, w2, b2, strides2, relu).double() - expected).abs() <= bound).all())
    assert bool(((block(x, w, b, x2, w2, b2, strides2, relu, packed=False).double() - expected).abs() <= 2 * bound + 1e-30).all())


@pytest.mark.parametrize("form", FORMS)
def test_block_keeps_infinities_nan_and_the_largest_values(tuning, form):
    tuning(MI355X_CONV_PACKED=form)
    x, w, x2, w2 = normal(7, (2, 40, 9, 10), (36, 40, 3, 3), (2, 24, 17, 19), (36, 24, 1, 1))
    x[0, 3, 4, 4], x2[0, 11, 0, 2], x2[1, 23, 8, 8], x2[1, 2, 16, 0] = float("inf"), float("nan"), float("-inf"), 3e38
    x2[1, 7, 3, 3] = float("nan")   # between the positions that are sampled
    w2 *= 1e-3
    got, apart = (block(x, w, None, x2, w2, None, (2, 2), False, packed) for packed in (True, False))
    assert torch.equal(got.isnan(), apart.isnan()) and torch.equal(got[got.isinf()], apart[apart.isinf()]) and bool(got.isnan().any())
    finite = apart.isfinite()
    assert torch.equal(finite, got.isfinite()) and torch.allclose(got[finite], apart[finite], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("batch, size, launches", [(1, 28, 3), (8, 56, 2), (13, 50, 2)])
def test_residual_block_in_a_graph(batch, size, launches):
    rng = np.random.default_rng(2)
    w = lambda *s: (rng.standard_normal(s) * np.sqrt(2 / np.prod(s[1:]))).astype(np.float32)   # noqa: E731
    info = lambda n, s: helper.make_tensor_value_info(n, TensorProto.FLOAT, s)   # noqa: E731
    arrays = {"w1": w(128, 64, 3, 3), "w2": w(128, 128, 3, 3), "w3": w(128, 64, 1, 1), "b1": w(128, 1)[:, 0], "b2": w(128, 1)[:, 0], "b3": w(128, 1)[:, 0]}
    nodes = [helper.make_node("Conv", ["x", "w1", "b1"], ["c1"], kernel_shape=[3, 3], pads=[1] * 4, strides=[2, 2]), helper.make_node("Relu", ["c1"], ["r1"]),
             helper.make_node("Conv", ["r1", "w2", "b2"], ["c2"], kernel_shape=[3, 3], pads=[1] * 4, strides=[1, 1]),
             helper.make_node("Conv", ["x", "w3", "b3"], ["c3"], kernel_shape=[1, 1], pads=[0] * 4, strides=[2, 2]),
             helper.make_node("Add", ["c2", "c3"], ["s"]), helper.make_node("Relu", ["s"], ["y"])]
    graph = helper.make_graph(nodes, "block", [info("x", [batch, 64, size, size])], [info("y", [batch, 128, size // 2, size // 2])],
                              initializer=[numpy_helper.from_array(v, k) for k, v in arrays.items()])
    model = donnx.ONNXModel("block", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)]))
    x, = normal(3, (batch, 64, size, size))
    got = model(x)
    names = [n.function for n, _ in model.compile_and_init().bound_launches()]
    assert len(names) == launches and ("mi355x_conv2d_skip_f32" in names) == (launches == 2)
    assert torch.equal(model(x), got)
    g = {k: torch.from_numpy(v).cuda() for k, v in arrays.items()}
    columns = F.unfold(x.double(), 3, padding=1, stride=2)
    inner = (torch.stack([g["w1"].double().reshape(128, -1) @ c for c in columns]) + g["b1"].double().reshape(1, -1, 1)).relu().reshape(batch, 128, size // 2, size // 2)
    expected, bound = wide_block(inner, g["w2"], g["b2"], x, g["w3"], g["b3"], (2, 2), True)
    close = lambda y: bool(((y.double() - expected).abs() <= 4 * bound).all())   # noqa: E731  (the inner layer's error among them)
    assert close(got)
    list(model.weights.values())   # handed out: the launches read the weights themselves
    assert close(model(x))
