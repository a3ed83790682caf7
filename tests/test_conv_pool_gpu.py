"""The stem of an image classifier, convolution, Relu and pooling in one launch, against float64."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper

pytestmark = pytest.mark.gpu
FORMS = range(1, 8)


def call(name, *args):
    _lib.check(getattr(_lib.library(), name)(*args, torch.cuda.current_stream().cuda_stream), name)


def stem(x, w, bias, pads, pool_pads, relu, packed=True):
    N, C, H, Wd = x.shape
    M = w.shape[0]
    i64 = _lib.i64_array
    geometry = (N, C, H, Wd, M, 7, 7, i64(pads), i64([2, 2]), i64([1, 1]))
    pooling = (3, 3, i64(pool_pads), i64([2, 2]), i64([1, 1]))
    size = _lib.library().mi355x_conv2d_pool_packed_pays(*geometry, *pooling)
    OH, OW = ((e + pads[i] + pads[i + 2] - 7) // 2 + 1 for i, e in enumerate((H, Wd)))
    PH, PW = ((e + pool_pads[i] + pool_pads[i + 2] - 3) // 2 + 1 for i, e in enumerate((OH, OW)))
    copy = torch.empty(size // 4, dtype=torch.int32, device="cuda") if packed else None
    if packed:
        assert size
        call("mi355x_pack_conv_pool_f32", w.data_ptr(), copy.data_ptr(), M, C, 7, 7)
    scratch, y = torch.full((N, M, OH, OW), -7.0, device="cuda"), torch.full((N * M * PH * PW + 64, ), -7.0, device="cuda")
    call("mi355x_conv2d_pool_packed_f32", x.data_ptr(), w.data_ptr(), _lib.ptr(copy), _lib.ptr(bias), scratch.data_ptr(), y.data_ptr(), *geometry,
         (_lib.EPI_BIAS if bias is not None else 0) | (_lib.EPI_RELU if relu else 0), *pooling)
    assert bool((y[-64:] == -7).all()) and bool((scratch == -7).all()) == packed
    return y[:-64].reshape(N, M, PH, PW)


def wide_stem(x, w, bias, pads, pool_pads, relu):
    """In float64, and a bound of the error: of a maximum the largest of its window."""
    M = w.shape[0]
    padded = F.pad(x.double(), (pads[1], pads[3], pads[0], pads[2]))
    OH, OW = ((e - 7) // 2 + 1 for e in padded.shape[2:])
    columns, rows = F.unfold(padded, 7, stride=2), w.double().reshape(M, -1)
    sums, magnitude = (torch.stack([r @ c for c in cols]).reshape(-1, M, OH, OW) for r, cols in ((rows, columns), (rows.abs(), columns.abs())))
    if bias is not None:
        sums, magnitude = sums + bias.double().reshape(1, -1, 1, 1), magnitude + bias.double().abs().reshape(1, -1, 1, 1)
    if relu:
        sums = sums.relu()
    pool = lambda v, fill: F.pad(v, (pool_pads[1], pool_pads[3], pool_pads[0], pool_pads[2]), value=fill).unfold(2, 3, 2).unfold(3, 3, 2).amax((4, 5))   # noqa: E731
    # one rounding (2^-23, truncation included) for each of the eleven steps, three of 2^-24 for the products left out and the sets of sums
    return pool(sums, float("-inf")), pool(magnitude, 0.0) * (11 + 8) * 2.0**-23


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("N, H, Wd, M, pads, pool_pads, relu, bias", [(1, 7, 7, 1, [0] * 4, [1] * 4, False, False), (2, 97, 111, 33, [3] * 4, [1] * 4, True, True),
                                                                      (1, 64, 70, 64, [3] * 4, [1] * 4, True, True), (3, 35, 29, 70, [2, 0, 5, 6], [0, 1, 2, 0], False, True),
                                                                      (1, 129, 33, 130, [6, 3, 0, 1], [2, 2, 2, 2], True, False), (1, 36, 130, 64, [3] * 4, [0] * 4, True, True)])
def test_stem(tuning, form, N, H, Wd, M, pads, pool_pads, relu, bias):
    tuning(MI355X_CONV_POOL=form)
    rng = np.random.default_rng(H + Wd)
    normal = lambda *s: torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).cuda()   # noqa: E731
    x, w, b = normal(N, 3, H, Wd), normal(M, 3, 7, 7), normal(M) if bias else None
    expected, bound = wide_stem(x, w, b, pads, pool_pads, relu)
    got = stem(x, w, b, pads, pool_pads, relu)
    assert bool(((got.double() - expected).abs() <= bound).all())
    apart = stem(x, w, b, pads, pool_pads, relu, packed=False)
    assert bool(((apart.double() - expected).abs() <= bound * 147 / 19 + 1e-30).all())


@pytest.mark.parametrize("form", FORMS)
def test_stem_keeps_infinities_nan_and_the_largest_values(tuning, form):
    """As the two launches do: NaN wins a maximum, -inf is a value like any other, padding none."""
    tuning(MI355X_CONV_POOL=form)
    rng = np.random.default_rng(1)
    x = torch.from_numpy(rng.standard_normal((2, 3, 61, 67), dtype=np.float32)).cuda()
    w = torch.from_numpy(np.abs(rng.standard_normal((40, 3, 7, 7), dtype=np.float32)) * 1e-2 + 1e-3).cuda()
    x[0, 0, 5, 9], x[0, 2, 40, 44], x[1, 1, 20, 20], x[1, 0, 50, 8] = float("nan"), float("inf"), float("-inf"), 3e38
    got, apart = (stem(x, w, None, [3] * 4, [1] * 4, False, packed) for packed in (True, False))
    assert bool(got.isnan().any()) and bool(got.isposinf().any())
    assert torch.equal(got.isnan(), apart.isnan()) and torch.equal(got[got.isinf()], apart[apart.isinf()])
    finite = apart.isfinite()
    assert torch.equal(finite, got.isfinite()) and torch.allclose(got[finite], apart[finite], rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("relu", [True, False])
def test_stem_in_a_graph(relu):
    rng = np.random.default_rng(2)
    normal = lambda *s: rng.standard_normal(s, dtype=np.float32)   # noqa: E731
    info = lambda n, s: helper.make_tensor_value_info(n, TensorProto.FLOAT, s)   # noqa: E731
    nodes = [helper.make_node("Conv", ["x", "w", "b"], ["c"], kernel_shape=[7, 7], pads=[3] * 4, strides=[2, 2])] + ([helper.make_node("Relu", ["c"], ["r"])] if relu else []) \
        + [helper.make_node("MaxPool", ["r" if relu else "c"], ["y"], kernel_shape=[3, 3], pads=[1] * 4, strides=[2, 2])]
    weights = [numpy_helper.from_array(normal(64, 3, 7, 7), "w"), numpy_helper.from_array(normal(64), "b")]
    graph = helper.make_graph(nodes, "stem", [info("x", [2, 3, 96, 100])], [info("y", [2, 64, 24, 25])], initializer=weights)
    model = donnx.ONNXModel("stem", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 12)]))
    x = torch.from_numpy(normal(2, 3, 96, 100)).cuda()
    got = model(x)
    assert [n.function for n, _ in model.compile_and_init().bound_launches()] == ["mi355x_conv2d_pool_packed_f32"]
    assert torch.equal(model(x), got)
    expected, bound = wide_stem(x, model.weights["w"], model.weights["b"], [3] * 4, [1] * 4, relu)   # (hands the weights out)
    assert bool(((got.double() - expected).abs() <= bound).all())
    assert bool(((model(x).double() - expected).abs() <= bound * 147 / 19).all())
