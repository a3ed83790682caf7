"""A dense layer of few classes and the probabilities of its rows in one launch, against float64."""
import numpy as np
import pytest
import torch
import torch.nn as nn

from dace_onnx_amd import _lib
from dace_onnx_amd.pytorch.module import DaceModule

pytestmark = pytest.mark.gpu


def normal(seed, *shapes):
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(rng.standard_normal(s, dtype=np.float32)).cuda() for s in shapes]


def dense_softmax(a, b, kc, bias, epilogue, alpha=1.0):
    M, K = a.shape
    N = b.shape[0] if kc else b.shape[1]
    scratch, y = torch.full((M, N), -7.0, device="cuda"), torch.full((M + 1, N), -7.0, device="cuda")
    _lib.check(_lib.library().mi355x_gemm_softmax_f32(a.data_ptr(), b.data_ptr(), _lib.ptr(bias), scratch.data_ptr(), y.data_ptr(), M, N, K, a.stride(0), *(b.stride()[::-1] if kc else b.stride()),
                                                      alpha, epilogue, torch.cuda.current_stream().cuda_stream), "gemm_softmax")
    assert bool((y[M] == -7).all())
    return y[:M], bool((scratch == -7).all())


@pytest.mark.parametrize("M, N, K, kc, one", [(1, 1, 4, True, True), (5, 10, 300, True, True), (16, 16, 17, True, True), (17, 15, 257, True, True), (4096, 3, 33, True, True),
                                              (4097, 3, 33, True, False), (9, 17, 64, True, False), (9, 12, 64, False, False), (6, 5, 3, True, False)])
def test_probabilities(M, N, K, kc, one):
    a, b, bias = normal(M + N + K, (M, K), (N, K) if kc else (K, N), (N, ))
    for epilogue in (0, _lib.EPI_BIAS, _lib.EPI_BIAS | _lib.EPI_RELU):
        got, in_one = dense_softmax(a, b, kc, bias, epilogue, 0.25)
        assert in_one == one
        wide = b.double().t() if kc else b.double()
        x, magnitude = 0.25 * (a.double() @ wide), 0.25 * (a.double().abs() @ wide.abs()) + bias.double().abs()
        x = x + bias.double() if epilogue else x
        x = x.relu() if epilogue & _lib.EPI_RELU else x
        p = torch.softmax(x, 1)
        # an error e of the logits moves a probability by at most 2 e of itself; a rounding for each of K products, then of the exponentials and their sum
        e = magnitude.amax(1, keepdim=True) * (K + 8) * 2.0**-24 + (x.amax(1, keepdim=True) - x) * 2.0**-23
        assert bool(((got.double() - p).abs() <= p * (2.1 * e + 24 * 2.0**-24) + 2.0**-126).all())


def test_rows_that_are_not_finite():
    """As the two launches give them."""
    a, b = normal(3, (20, 32), (7, 32))
    b.abs_()
    a[2, 3], a[9, 0], a[17, 5] = float("nan"), float("inf"), float("-inf")
    got, apart = dense_softmax(a, b, True, None, 0)[0], dense_softmax(a, b.t().contiguous(), False, None, 0)[0]
    assert torch.equal(got.isnan(), apart.isnan()) and torch.allclose(got.nan_to_num(), apart.nan_to_num(), rtol=1e-5, atol=1e-30)


@pytest.mark.parametrize("classes, launches", [(10, 2), (17, 3)])
def test_classifier_of_a_module(classes, launches):
    x, = normal(0, (5, 64))
    torch.manual_seed(0)
    net = nn.Sequential(nn.Linear(64, 30), nn.ReLU(), nn.Linear(30, classes), nn.Softmax(dim=1)).cuda().eval()
    module = DaceModule(net, dummy_inputs=(x, ), sdfg_name="classifier")
    with torch.no_grad():
        for _ in range(2):
            assert torch.allclose(module(x), net(x), rtol=1e-5, atol=1e-6)
        assert module.dace_model.compile_and_init().num_launches == launches
        net[2].weight.mul_(-1)   # read where it lies
        assert torch.allclose(module(x), net(x), rtol=1e-5, atol=1e-6)
