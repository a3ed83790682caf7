"""The kernels that multiply by packed constants, at the edges of their tiles and values, against float64."""
import numpy as np
import pytest
import torch
import torch.nn as nn

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
from dace_onnx_amd.onnx.proto import TensorProto, helper, numpy_helper
from dace_onnx_amd.pytorch.module import DaceModule
from dace_onnx_amd.testing.graphs import bert_encoder_layer_model
from dace_onnx_amd.testing.profiling import graph_time_us
from oracle import pure_ops

pytestmark = pytest.mark.gpu
FORMS = range(1, 11)


def call(name, *args):
    _lib.check(getattr(_lib.library(), name)(*args, torch.cuda.current_stream().cuda_stream), name)


def gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def pack(w, rows, k, s_row, s_k):
    packed = torch.empty(-(-rows // 32), k // 32, 2, 3, 64, 4, dtype=torch.int32, device="cuda")
    call("mi355x_pack_f32", w.data_ptr(), packed.data_ptr(), rows, k, s_row, s_k)
    return packed


def packed_gemm(a, b, kc, bias=None, res=None, epi=0, alpha=1.0, batch=1, c_gap=0):
    """C = a @ b; ``b`` is [N, K] if ``kc`` else [K, N]; rows of C ``c_gap`` apart, which stays as it was."""
    M, K = a.shape[-2:]
    N = b.shape[0] if kc else b.shape[1]
    assert _lib.library().mi355x_gemm_packed_pays(batch, M, N, K, int(kc)) == 1   # (a form that does not take it would leave it to the kernels before)
    c = torch.full((batch, M, N + c_gap), -7.0, device="cuda")
    i64 = _lib.i64_array
    call("mi355x_gemm_packed_f32", a.data_ptr(), pack(b, N, K, *((K, 1) if kc else (1, N))).data_ptr(), b.data_ptr(), c.data_ptr(), _lib.ptr(bias),
         _lib.ptr(res), 1, batch, M, N, K, i64([0, M * K, K, 1]), i64([0, 0] + ([1, K] if kc else [N, 1])), i64([0, M * (N + c_gap), N + c_gap]),
         i64([0, M * N, N]), alpha, epi)
    assert bool((c[..., N:] == -7).all())
    return c[..., :N]


def test_a_packed_operand_holds_every_bit():
    w = gpu(np.random.default_rng(0).standard_normal((45, 96), dtype=np.float32) * np.float32(2.0)**np.arange(-140, 100, 2.5, dtype=np.float32))
    parts = pack(w, 45, 96, 96, 1).cpu().view(torch.bfloat16).reshape(2, 3, 2, 3, 2, 32, 2, 4).double().sum(3)   # block, step, s, h, row, a, e
    rows = parts.permute(0, 4, 1, 5, 2, 3, 6).reshape(64, 96) / 65536
    assert torch.equal(rows[:45], w.cpu().double()) and not rows[45:].any()


@pytest.mark.parametrize("kc", [True, False])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("batch, M, N, K, epi", [(1, 1, 1, 32, 0), (1, 31, 33, 64, 1), (1, 64, 64, 96, 9), (2, 129, 127, 160, 13), (1, 257, 130, 32, 3),
                                                 (1, 255, 258, 768, 9), (3, 96, 515, 1056, 8)])
def test_gemm_by_a_packed_constant(tuning, form, kc, batch, M, N, K, epi):
    """A sum of K products: at most one rounding (2^-23, truncation included) for each of the K / 16 steps, and three of 2^-24 for the
    products left out and the sets of sums."""
    tuning(MI355X_GEMM_PACKED=form)
    rng = np.random.default_rng(M + N + K)
    a = gpu(rng.standard_normal((batch, M, K), dtype=np.float32))
    b = gpu(rng.standard_normal((N, K) if kc else (K, N), dtype=np.float32))
    bias, res = gpu(rng.standard_normal(N, dtype=np.float32)), gpu(rng.standard_normal((batch, M, N), dtype=np.float32))
    got = packed_gemm(a, b, kc, bias, res, epi, 0.5, batch, c_gap=3)
    wide = b.double().t() if kc else b.double()
    expected = 0.5 * (a.double() @ wide) + (bias.double() if epi & 1 else 0)
    if epi & 2:
        expected = expected.relu()
    if epi & 4:
        expected = torch.nn.functional.gelu(expected)
    if epi & 8:
        expected = expected + res.double()
    bound = (a.double().abs() @ wide.abs() + 1) * (K // 16 + 8) * 2.0**-23
    assert bool(((expected - got.double()).abs() <= 1.2 * bound).all())   # 1.13 is Gelu's steepest slope


@pytest.mark.parametrize("form", FORMS)
def test_gemm_by_a_packed_constant_keeps_infinities_nan_and_the_largest_values(tuning, form):
    tuning(MI355X_GEMM_PACKED=form)
    a = torch.randn(1, 300, 96, device="cuda")
    b = torch.rand(200, 96, device="cuda") + 0.5
    a[0, 3, 5], a[0, 70, 95], a[0, 130, 0], a[0, 131, 1:3] = float("inf"), -float("inf"), float("nan"), torch.tensor([float("inf"), -float("inf")])
    a[0, 200], a[0, 200, 7], a[0, 290, 9] = 0, 3.4e38, 3.3999e38   # rounds up to infinity in bf16
    b[:, 7] = 0.75
    b[11, 9], b[150, 9], b[150, 60] = 0, 0.5, float("inf")   # (0.5: no product of its own overflows next to the infinite one)
    expected = a[0].double() @ b.double().t()
    single = expected.float()
    fine = torch.isfinite(single)
    for kc in (True, False):
        got = packed_gemm(a, b if kc else b.t().contiguous(), kc)[0]
        assert torch.equal(torch.isnan(single), torch.isnan(got)) and torch.equal(torch.isinf(single), torch.isinf(got))
        assert torch.equal(single[~fine].nan_to_num(nan=0), got[~fine].nan_to_num(nan=0))
        assert bool(((expected - got.double()).abs()[fine] <= 1e-5 * (a[0].double().abs().nan_to_num(0, 0) @ b.double().abs().nan_to_num(0, 0, 0).t())[fine]).all())


@pytest.mark.parametrize("M, N, K", [(128, 768, 3072), (1024, 768, 3072), (1024, 2304, 768)])
def test_a_row_that_is_not_finite_takes_a_bounded_time(M, N, K):
    """Blocks with such a row are summed again by the fp32 MFMA, at a sixth of the rate: 1.6 to 2.6 times the launch (10 to 12 times where its loads
    come one at a time)."""
    a, b = torch.randn(M, K, device="cuda"), torch.randn(N, K, device="cuda")
    c, packed, i64 = torch.empty(M, N, device="cuda"), pack(b, N, K, K, 1), _lib.i64_array
    launch = lambda: _lib.library().mi355x_gemm_packed_f32(a.data_ptr(), packed.data_ptr(), b.data_ptr(), c.data_ptr(), None, None, 1, 1, M, N, K,   # noqa: E731
                                                           i64([0, M * K, K, 1]), i64([0, 0, 1, K]), i64([0, M * N, N]), None, 1.0, 0, _lib.current_stream())
    before = graph_time_us(launch, reps=20)
    a[M // 2, 5] = float("nan")
    assert graph_time_us(launch, reps=20) < 5 * before
    torch.cuda.synchronize()
    assert bool(torch.isnan(c[M // 2]).all()) and int(torch.isnan(c).sum()) == N


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("low, high", [(-100, 90), (-120, 100), (-148, 105), (-60, -58), (90, -3)])
def test_gemm_by_a_packed_constant_keeps_small_values(tuning, form, low, high):
    """Values down to the smallest subnormal against values that bring the sums back to ordinary size: exact products, so the bound is
    that of ordinary ones."""
    tuning(MI355X_GEMM_PACKED=form)
    rng = np.random.default_rng(form)
    a, b = (gpu(np.ldexp(rng.uniform(1, 2, s) * rng.choice([-1, 1], s), e).astype(np.float32)) for s, e in (((1, 70, 96), low), ((70, 96), high)))
    got = packed_gemm(a, b, True)[0]
    expected, size = a[0].double() @ b.double().t(), a[0].double().abs() @ b.double().abs().t()
    assert bool(((expected - got.double()).abs() <= size * 14 * 2.0**-23 + 2.0**-149).all())


def test_a_packed_copy_follows_its_weight():
    """Parameters written in place after the first call: the next call multiplies by the new ones (and not by the packed copy)."""
    linear = nn.Linear(768, 1024).cuda()
    x = torch.randn(512, 768, device="cuda")
    model = DaceModule(nn.Sequential(linear, nn.ReLU()), dummy_inputs=(x, ))
    for _ in range(2):
        with torch.no_grad():
            linear.weight.mul_(0.5)
            linear.weight[3] += 1
        got, expected = model(x), torch.relu(x.double() @ linear.weight.double().t() + linear.bias.double()).detach()
        assert float((got.double() - expected).norm() / expected.norm()) < 1e-6
    assert [n.function for n, _ in model.dace_model.compile_and_init().bound_launches()] == ["mi355x_gemm_packed_f32"]


def encoder(**options):
    weights = pure_ops.bert_layer_weights(np.random.default_rng(0))
    torch.manual_seed(0)
    return donnx.ONNXModel("encoder", bert_encoder_layer_model(weights, 8, 128, 12), **options), torch.randn(8, 128, 768, device="cuda")


@pytest.mark.parametrize("where", ["cpu", "numpy", "cuda"])
def test_a_replaced_weight_is_multiplied_by_wherever_it_lies(where):
    model, x = encoder()
    before = model(x)
    packed = {c.weight_name: c for c in model._packed}
    assert len(packed) == 4
    for name, copy in packed.items():   # twice the weights of every product, elsewhere
        moved = copy.weight * 2
        model.weights[name] = moved.cpu().numpy() if where == "numpy" else moved.to(where)
    replaced = model(x)
    for name, copy in packed.items():   # the same in place, with the launches that read the weights themselves
        model.weights[name] = copy.weight.mul_(2)
    assert torch.equal(replaced, model(x)) and not torch.allclose(replaced, before)


def test_a_replay_follows_weights_that_are_written():
    model, x = encoder(use_hip_graph=True)
    eager, _ = encoder()
    for _ in range(3):
        assert torch.equal(model(x), eager(x))
    for m in (model, eager):
        for copy in m._packed[1:3]:
            copy.weight.mul_(0.5)
    for _ in range(3):   # (a replay every time but the first)
        assert torch.equal(model(x), eager(x))
    model.weights[model._packed[3].weight_name] = model._packed[3].weight * 3
    for _ in range(3):
        got, expected = model(x), eager(x)
        assert torch.allclose(got, expected, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("construction", [True, False])
def test_a_model_made_or_first_called_under_inference_mode(construction):
    expected, x = encoder()
    expected = expected(x)
    if construction:
        with torch.inference_mode():
            model, _ = encoder()
    else:
        model, _ = encoder()
    with torch.inference_mode():
        first = model(x)
    assert torch.equal(first, expected) and torch.equal(model(x), expected) and model._packed


def head(**options):
    rng = np.random.default_rng(0)
    weight = numpy_helper.from_array(rng.standard_normal((768, 3001), dtype=np.float32), "w")
    info = lambda n, shape: helper.make_tensor_value_info(n, TensorProto.FLOAT, shape)   # noqa: E731
    graph = helper.make_graph([helper.make_node("MatMul", ["x", "w"], ["y"])], "head", [info("x", [1024, 768])], [info("y", [1024, 3001])], initializer=[weight])
    return donnx.ONNXModel("head", helper.make_model(graph, opset_imports=[helper.make_opsetid("", 13)]), **options), torch.randn(1024, 768, device="cuda")


def close(got, x, w):
    expected = x.double() @ w.double()
    return float((got.double() - expected).norm() / expected.norm()) < 1e-6


@pytest.mark.parametrize("replayed", [False, True])
def test_writes_that_torch_does_not_count_take_effect_at_the_next_call(replayed):
    model, x = head(use_hip_graph=replayed)
    for _ in range(3):
        model(x)
    assert model._packed[0].current()
    weight = model.weights["w"]
    for _ in range(3):
        weight.data.mul_(0.5)
        assert close(model(x), x, weight)
        model.weights["w"].data[3] += 1
        assert close(model(x), x, weight)
    model.pack_weights()
    for _ in range(3):
        assert model._packed[0].current() and close(model(x), x, weight)
    weight.data.mul_(0.5)
    model.pack_weights()
    for _ in range(2):
        assert close(model(x), x, weight)


def test_writes_to_parameters_that_torch_does_not_count_take_effect_at_the_next_call():
    linear, conv = nn.Linear(768, 1024).cuda(), nn.Conv2d(64, 64, 3, padding=1).cuda()
    x, image = torch.randn(512, 768, device="cuda"), torch.randn(32, 64, 28, 28, device="cuda")
    dense, convolution = DaceModule(linear, dummy_inputs=(x, )), DaceModule(conv, dummy_inputs=(image, ))
    dense(x), convolution(image)
    for _ in range(2):
        linear.weight.data.mul_(0.5)
        conv.weight.data.mul_(0.5)
        with torch.no_grad():
            assert close(dense(x) - linear.bias, x, linear.weight.t())
            expected = torch.nn.functional.conv2d(image.cpu().double(), conv.weight.cpu().double(), conv.bias.cpu().double(), padding=1)
            assert float((convolution(image).cpu().double() - expected).norm() / expected.norm()) < 1e-6


def test_a_callers_recordings_follow_weights_that_are_written_after_them():
    model, x = head()
    model(x)
    weight = model._packed[0].weight
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = model(x)
    assert model._packed[0].current()
    for _ in range(3):
        weight.data.mul_(0.5)
        graph.replay()
        assert close(recorded, x, weight)
    y = model(x)
    compiled = model.compile_and_init()
    compiled.capture_graph()   # of the call above
    for _ in range(3):
        weight.data.mul_(0.5)
        compiled.replay()
        assert close(y, x, weight)


def test_a_first_call_under_stream_capture():
    model, x = head()
    graph, weight = torch.cuda.CUDAGraph(), dict.get(model.weights, "w")
    with torch.cuda.graph(graph):
        y = model(x)
    for _ in range(3):
        y.zero_()
        graph.replay()
        assert close(y, x, weight)
    assert close(model(x), x, weight)


@pytest.mark.parametrize("kc", [True, False])
@pytest.mark.parametrize("batch, M, N, K, epi", [(1, 1, 1, 32, 0), (1, 127, 193, 64, 1), (2, 129, 191, 160, 13), (1, 300, 400, 768, 9), (3, 96, 577, 1056, 8)])
def test_gemm_by_twelve_waves(tuning, kc, batch, M, N, K, epi):
    """128 x 192 tiles, whose rows eight of the twelve waves load."""
    test_gemm_by_a_packed_constant(tuning, 11, kc, batch, M, N, K, epi)


def test_gemm_by_twelve_waves_keeps_infinities_nan_and_the_largest_values(tuning):
    test_gemm_by_a_packed_constant_keeps_infinities_nan_and_the_largest_values(tuning, 11)
