"""Products computed in parts of K and added up by the normalization that follows, against float64."""
import numpy as np
import pytest
import torch

import dace_onnx_amd.onnx as donnx
from dace_onnx_amd import _lib
from dace_onnx_amd.testing.graphs import bert_encoder_layer_model
from oracle import pure_ops

pytestmark = pytest.mark.gpu


def call(name, *args):
    _lib.check(getattr(_lib.library(), name)(*args, torch.cuda.current_stream().cuda_stream), name)


def normal(rng, *shape):
    return torch.from_numpy(rng.standard_normal(shape, dtype=np.float32)).cuda()


def parts_of(a, b, kc, packed, parts, alpha=1.0):
    M, K = a.shape
    N = b.shape[0] if kc else b.shape[1]
    strides = (1, K) if kc else (N, 1)
    copy = torch.empty(-(-N // 32), K // 32, 2, 3, 64, 4, dtype=torch.int32, device="cuda") if packed else None
    if packed:
        call("mi355x_pack_f32", b.data_ptr(), copy.data_ptr(), N, K, strides[1], strides[0])
    sums = torch.full((parts + 1, M, N), -7.0, device="cuda")
    call("mi355x_gemm_parts_f32", a.data_ptr(), b.data_ptr(), _lib.ptr(copy), sums.data_ptr(), parts, M, N, K, K, *strides, alpha)
    assert bool((sums[parts] == -7).all())
    return sums[:parts]


def wide_parts(a, b, kc, parts):
    """The parts in float64, and the sums of their absolute values."""
    w = b.double().t() if kc else b.double()
    shares = [(x, y) for x, y in zip(a.double().chunk(parts, 1), w.chunk(parts, 0))]
    return torch.stack([x @ y for x, y in shares]), torch.stack([x.abs() @ y.abs() for x, y in shares])


@pytest.mark.parametrize("kc", [True, False])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("M, N, K, parts", [(1, 4, 512, 2), (16, 768, 3072, 8), (17, 252, 768, 3), (33, 256, 1536, 6), (129, 1020, 512, 2), (865, 768, 768, 3), (300, 1024, 4096, 4)])
def test_parts_of_a_product(tuning, kc, packed, M, N, K, parts):
    rng = np.random.default_rng(M + N + K)
    a, b = normal(rng, M, K), normal(rng, N, K) if kc else normal(rng, K, N)
    if packed:
        tuning(MI355X_GEMM_PACKED=4)   # (64 x 128 tiles; what the rule picks at these sizes is in the graphs below)
    got = parts_of(a, b, kc, packed, parts, 0.5).double()
    wide, magnitude = wide_parts(a, b, kc, parts)
    # one rounding (2^-23, truncation included) for each step of at least four k of a sum, three of 2^-24 more for the split form
    assert bool(((got - 0.5 * wide).abs() <= 0.5 * magnitude * (K // parts // 4 + 8) * 2.0**-23).all())


def test_parts_keep_infinities_nan_and_the_largest_values(tuning):
    tuning(MI355X_GEMM_PACKED=5)
    rng = np.random.default_rng(5)
    a, b = normal(rng, 70, 512), normal(rng, 96, 512)
    a[3, 100], a[40, 300], a[69, 511], b[64, 260] = float("inf"), float("nan"), 3e38, 0.0
    b[:, 511] *= 1e-3
    got = parts_of(a, b, True, True, 2).double()
    wide, magnitude = wide_parts(a, b, True, 2)
    finite = wide.isfinite()
    assert torch.equal(got.isnan(), wide.isnan()) and torch.equal(got[wide.isinf()], wide[wide.isinf()])
    assert bool(((got - wide).abs() <= magnitude * (256 // 2 + 8) * 2.0**-23)[finite].all())


@pytest.mark.parametrize("bias, residual, beta", [(True, True, True), (False, True, False), (True, False, True), (False, False, False)])
@pytest.mark.parametrize("rows, cols, parts", [(1, 4, 2), (16, 768, 8), (5, 252, 3), (17, 256, 4), (9, 260, 6), (1023, 512, 2), (1025, 772, 3), (1027, 1024, 8)])
def test_normalization_of_parts(rows, cols, parts, bias, residual, beta):
    rng = np.random.default_rng(rows + cols)
    p, c, r, g, b = normal(rng, parts, rows, cols), normal(rng, cols + 1), normal(rng, rows, cols + 5), normal(rng, cols + 1), normal(rng, cols + 1)
    c, g, b = c[1:], g[1:], b[1:]   # at odd addresses, as weights may be
    y = torch.full((rows + 1, cols), -7.0, device="cuda")
    call("mi355x_layernorm_parts_f32", p.data_ptr(), parts, c.data_ptr() if bias else None, r.data_ptr() if residual else None, cols + 5, g.data_ptr(),
         b.data_ptr() if beta else None, y.data_ptr(), rows, cols, 1e-5)
    terms = [v.double() for v in p] + ([c.double().expand(rows, cols)] if bias else []) + ([r[:, :cols].double()] if residual else [])
    x, magnitude = sum(terms), sum(t.abs() for t in terms)
    centred = x - x.mean(1, keepdim=True)
    std = (centred.square().mean(1, keepdim=True) + 1e-5).sqrt()
    expected = centred / std * g.double() + (b.double() if beta else 0)
    # a sum of up to ten terms, then a mean and a variance of cols values: an error e of every value moves the result by at most
    # (2 + |x|) e / std, and each of the few operations after by 2^-24
    e = magnitude.amax(1, keepdim=True) * (len(terms) + 12) * 2.0**-24
    bound = g.double().abs() * (e / std) * (2 + (centred / std).abs()) + 8 * 2.0**-24 * (expected.abs() + 1)
    assert bool(((expected - y[:rows].double()).abs() <= bound).all()) and bool((y[rows] == -7).all())


@pytest.mark.parametrize("bsz, seq, parts", [(1, 16, 2), (1, 128, 2), (5, 173, 2), (16, 512, 0)])
def test_encoder_layers_with_and_without_parts(bsz, seq, parts):
    """The projections before both normalizations, eager, recorded, and with a weight that is read itself after it was handed out."""
    weights = pure_ops.bert_layer_weights(np.random.default_rng(0))
    x = torch.from_numpy(np.random.default_rng(1).standard_normal((bsz, seq, 768), dtype=np.float32)).cuda()
    model = donnx.ONNXModel("encoder", bert_encoder_layer_model(weights, bsz, seq, 12))
    got = model(x)
    names = [n.function for n, _ in model.compile_and_init().bound_launches()]
    assert len(names) == 7 and (names.count("mi355x_layernorm_parts_f32") == 0) == (parts == 0)
    expected = torch.from_numpy(pure_ops.bert_layer(x.cpu().numpy(), weights, heads=12)).cuda()
    close = lambda y: float((y - expected).abs().max() / expected.abs().max()) < 1e-5   # noqa: E731
    assert close(got)
    replayed = donnx.ONNXModel("encoder_replayed", bert_encoder_layer_model(weights, bsz, seq, 12), use_hip_graph=True)
    for _ in range(3):
        assert torch.equal(replayed(x), got)
        torch.cuda.synchronize()
    for name in list(model.weights):
        model.weights[name]   # handed out: launches read it itself
    assert close(model(x))
