"""Attention on the bf16 matrix unit, at the edges of its blocks and values: against float64, and against the fp32 kernel where sums are not finite."""
import pytest
import torch

from dace_onnx_amd import _lib
from dace_onnx_amd.testing.profiling import graph_time_us

pytestmark = pytest.mark.gpu


def attention(q, k, v, mask=None, scale=0.125):
    (b0, b1, sq, _), sk = q.shape, k.shape[2]
    rows = sq + 1
    out = torch.full((b0, b1, rows, 64), -7.0, device="cuda")   # one row more than is written
    strides = lambda t: _lib.i64_array([t.stride(0), t.stride(1), t.stride(2)])   # noqa: E731
    args = [q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr()]
    geometry = [b0, b1, sq, sk, 64, strides(q), strides(k), strides(v), strides(out)]
    if mask is None:
        name, args = "mi355x_attention_f32", args + geometry
    else:
        broadcast = _lib.i64_array([st if e > 1 else 0 for st, e in zip(mask.stride()[:3], mask.shape)])
        name, args = "mi355x_attention_masked_f32", args + [mask.data_ptr()] + geometry + [broadcast]
    _lib.check(getattr(_lib.library(), name)(*args, scale, torch.cuda.current_stream().cuda_stream), name)
    assert bool((out[:, :, sq:] == -7).all())
    return out[:, :, :sq]


def inputs(b0, b1, sq, sk, seed=0):
    torch.manual_seed(sq + sk + seed)
    return [torch.randn(b0, n, b1, 64, device="cuda").transpose(1, 2) for n in (sq, sk, sk)]   # heads side by side in a row


@pytest.mark.parametrize("sq, sk", [(1, 1), (127, 63), (128, 64), (129, 65), (33, 130), (257, 200)])
@pytest.mark.parametrize("shape", [None, "keys", "rows", "all"])
def test_split_attention(tuning, sq, sk, shape):
    """Scores of up to 8 in magnitude: 2^-24 of that, a few times, in the exponent of every probability; sums of up to 200 of them."""
    tuning(MI355X_ATTN_SPLIT=1)
    b0, b1 = 2, 3
    q, k, v = inputs(b0, b1, sq, sk)
    extents = {"keys": (b0, 1, 1, sk), "rows": (1, 1, sq, sk), "all": (b0, b1, sq, sk)}.get(shape)
    mask = None
    if extents:
        memory = torch.where(torch.rand(b0 * b1 * sq * sk + 1, device="cuda") < 0.3, -10000.0, 0.0)[1:]   # (not 16-byte aligned)
        mask = memory[:extents[0] * extents[1] * extents[2] * sk].view(extents)
        mask[..., sk // 2] = 0
    scores = 0.125 * (q.double() @ k.double().transpose(-1, -2).contiguous())
    expected = torch.softmax(scores + mask.double() if extents else scores, -1) @ v.double()
    got = attention(q, k, v, mask)
    assert bool(((expected - got.double()).abs() <= 2.0**-19 * v.abs().max()).all())
    assert float((expected - got.double()).norm() / expected.norm()) < 1e-6


@pytest.mark.parametrize("fill", [-float("inf"), torch.finfo(torch.float32).min, -10000.0])
@pytest.mark.parametrize("sk", [64, 150])
def test_split_attention_over_masked_blocks_and_rows(tuning, sk, fill):
    """A first block without a valid key and a row without one: as the fp32 kernel, NaN in the same places."""
    q, k, v = inputs(2, 3, 70, sk)
    mask = torch.zeros(2, 1, 70, sk, device="cuda")
    mask[0, :, :40, :sk - 3], mask[1, :, 5] = fill, fill
    results = []
    for form in (0, 1):
        tuning(MI355X_ATTN_SPLIT=form)
        results.append(attention(q, k, v, mask))
    assert torch.equal(torch.isnan(results[0]), torch.isnan(results[1])) and bool(torch.isnan(results[0]).any()) == (fill == -float("inf"))
    masked_row = torch.zeros(2, 1, 70, 1, dtype=torch.bool, device="cuda")
    masked_row[1, :, 5] = fill == -10000.0   # the scores there have lost all but 2^-11
    difference = (results[0] - results[1]).abs().nan_to_num(0)
    assert float(difference.masked_fill(masked_row, 0).max()) < 1e-5 and float(difference.max()) < 5e-3


@pytest.mark.parametrize("masked", [False, True])
def test_split_attention_keeps_infinities_nan_and_the_largest_values(tuning, masked):
    mask = torch.zeros(1, 1, 1, 100, device="cuda") if masked else None
    for place, value in ((0, float("inf")), (0, float("nan")), (1, -float("inf")), (1, float("nan")), (2, float("inf")), (2, float("nan")), (2, 3.0e38), (0, 1.0e36)):
        tensors = inputs(2, 2, 150, 100, seed=place)
        tensors[place][1, 0, 70, 9] = value
        results = []
        for form in (0, 1):
            tuning(MI355X_ATTN_SPLIT=form)
            results.append(attention(*tensors, mask))
        assert torch.equal(torch.isnan(results[0]), torch.isnan(results[1])) and torch.equal(torch.isinf(results[0]), torch.isinf(results[1]))
        fine = torch.isfinite(results[0])
        assert bool(((results[0] - results[1]).abs()[fine] <= 1e-5 * results[0].abs()[fine].clamp(min=1)).all())


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("scale", [0.125, -0.125])
def test_split_attention_of_scores_that_only_the_split_form_cannot_hold(tuning, masked, scale):
    """A score of 0 whose largest product is -1.5 x 2^96, past what sums of scaled values hold: the fp32 kernel's result, not a masked key."""
    tuning(MI355X_ATTN_SPLIT=1)
    q, k, v = inputs(2, 2, 150, 100)
    mask = torch.zeros(1, 1, 1, 100, device="cuda") if masked else None
    q[1, 0, 70, 0], q[1, 0, 70, 16:49:16] = 1.5 * 2.0**49, 2.0**48
    k[..., 0::16], k[1, 0, 9] = 0, 0
    k[1, 0, 9, 0], k[1, 0, 9, 16:49:16] = -2.0**47, 2.0**47
    expected = torch.softmax(scale * (q.double() @ k.double().transpose(-1, -2).contiguous()), -1) @ v.double()
    got = attention(q, k, v, mask, scale)
    assert float((expected[1, 0, 70] - got[1, 0, 70].double()).norm() / expected[1, 0, 70].norm()) < 1e-6
    assert float((expected - got.double()).norm() / expected.norm()) < 1e-6


def test_sentences_without_a_valid_key_take_no_longer():
    """Their rows are 0 / 0: nothing to compute again (twice the time and more where the fp32 kernel runs after)."""
    q, k, v = inputs(32, 12, 64, 64)
    mask, out = torch.zeros(32, 1, 1, 64, device="cuda"), torch.empty_like(q)
    strides = lambda t: _lib.i64_array(t.stride()[:3])   # noqa: E731
    launch = lambda: _lib.library().mi355x_attention_masked_f32(q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), mask.data_ptr(), 32, 12, 64, 64, 64,   # noqa: E731
                                                                strides(q), strides(k), strides(v), strides(out), _lib.i64_array([64, 0, 0]), 0.125, _lib.current_stream())
    before = graph_time_us(launch)
    mask[::2] = -float("inf")
    assert graph_time_us(launch) < 1.5 * before
    torch.cuda.synchronize()
    assert bool(torch.isnan(out[::2]).all()) and bool(torch.isfinite(out[1::2]).all())


@pytest.mark.parametrize("waves", [1, 2, 4, 8])
@pytest.mark.parametrize("sq, sk", [(1, 1), (16, 16), (17, 15), (33, 130), (5, 129), (64, 300)])
@pytest.mark.parametrize("shape", [None, "keys", "rows", "all"])
def test_attention_of_few_rows(tuning, waves, sq, sk, shape):
    """Chunks of 16 keys shared by the waves, fewer and more of them than waves, ragged ones: bounds as for the split form."""
    tuning(MI355X_ATTN_FEW=waves)
    b0, b1 = 2, 3
    q, k, v = inputs(b0, b1, sq, sk)
    extents = {"keys": (b0, 1, 1, sk), "rows": (1, 1, sq, sk), "all": (b0, b1, sq, sk)}.get(shape)
    mask = None
    if extents:
        memory = torch.where(torch.rand(b0 * b1 * sq * sk + 1, device="cuda") < 0.3, -10000.0, 0.0)[1:]   # (not 16-byte aligned)
        mask = memory[:extents[0] * extents[1] * extents[2] * sk].view(extents)
        mask[..., sk // 2] = 0
    scores = 0.125 * (q.double() @ k.double().transpose(-1, -2).contiguous())
    expected = torch.softmax(scores + mask.double() if extents else scores, -1) @ v.double()
    got = attention(q, k, v, mask)
    assert bool(((expected - got.double()).abs() <= 2.0**-19 * v.abs().max()).all())
    assert float((expected - got.double()).norm() / expected.norm()) < 1e-6


@pytest.mark.parametrize("waves", [1, 4, 8])
@pytest.mark.parametrize("masked", [False, True])
def test_attention_of_few_rows_keeps_infinities_nan_and_the_largest_values(tuning, waves, masked):
    """Against the fp32 kernel; a mask of -inf over whole chunks and over a whole row among the values."""
    mask = torch.zeros(1, 1, 20, 100, device="cuda") if masked else None
    if masked:
        mask[..., :40], mask[:, :, 7] = -float("inf"), -float("inf")
    for place, value in ((0, float("inf")), (0, float("nan")), (1, -float("inf")), (1, float("nan")), (2, float("inf")), (2, float("nan")), (2, 3.0e38), (0, 1.0e36)):
        tensors = inputs(2, 2, 20, 100, seed=place)
        tensors[place][1, 0, 13 if place == 0 else 70, 9] = value
        results = []
        for form in (dict(MI355X_ATTN_SPLIT=0), dict(MI355X_ATTN_FEW=waves)):
            tuning(MI355X_ATTN_SPLIT=None, MI355X_ATTN_FEW=None)
            tuning(**form)
            results.append(attention(*tensors, mask))
        assert torch.equal(torch.isnan(results[0]), torch.isnan(results[1])) and torch.equal(torch.isinf(results[0]), torch.isinf(results[1]))
        fine = torch.isfinite(results[0])
        assert bool(((results[0] - results[1]).abs()[fine] <= 1e-5 * results[0].abs()[fine].clamp(min=1)).all())


@pytest.mark.parametrize("form", [dict(MI355X_ATTN_FEW=1), dict(MI355X_ATTN_FEW=2), dict(MI355X_ATTN_FEW=4), dict(MI355X_ATTN_FEW=8), dict(MI355X_ATTN_SPLIT=1),
                                  dict(MI355X_ATTN_SPLIT=0), {}], ids=str)
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("sk", [1, 15, 16, 33, 100, 128, 130, 200])
def test_an_infinite_value_of_the_last_key(tuning, form, masked, sk):
    """Keys beyond the last have no probability, and no value that could turn it into NaN: against float64."""
    tuning(**form)
    q, k, v = inputs(2, 2, 20, sk)
    v[1, 0, sk - 1, 9], v[0, 1, sk - 1, 63] = float("inf"), -float("inf")
    mask = torch.zeros(1, 1, 20, sk, device="cuda") if masked else None
    expected = torch.softmax(0.125 * (q.double() @ k.double().transpose(-1, -2).contiguous()), -1) @ v.double()
    got = attention(q, k, v, mask).double()
    fine = torch.isfinite(expected)
    assert torch.equal(got[~fine], expected[~fine]) and bool(((got - expected).abs()[fine] <= 2.0**-19 * v[v.isfinite()].abs().max()).all())
