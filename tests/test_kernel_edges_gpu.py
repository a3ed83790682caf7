"""Kernels at the edges of their tiles and of the rules that pick them, through the C ABI, against float64.

Tolerances: sums and exponentials of a row are fp32 with at most a few dozen additions per thread and then a tree, so
1e-6 of the largest value is a handful of roundings (2^-24 each); maxima are exact.
"""
import numpy as np
import pytest
import torch

from dace_onnx_amd import _lib

pytestmark = pytest.mark.gpu


def call(name, *args):
    _lib.check(getattr(_lib.library(), name)(*args, torch.cuda.current_stream().cuda_stream), name)


def gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def worst(expected, got):
    """Largest difference over the largest magnitude."""
    return float((expected - got.double()).abs().max() / expected.abs().max())


@pytest.mark.parametrize("rows", [1, 5])
@pytest.mark.parametrize("cols", [1, 63, 65, 129, 255, 257, 511, 513, 2047, 2049, 8191, 8193, 30522, 32767, 32768, 32769])
def test_softmax_of_rows_without_alignment(rows, cols):
    x = gpu(np.random.default_rng(cols).standard_normal(rows * cols + 1, dtype=np.float32) * 3)
    for offset in (0, 1):   # rows that start at odd multiples of four bytes too
        view = x[offset:offset + rows * cols].view(rows, cols)
        for name, reference in (("mi355x_softmax_f32", torch.softmax), ("mi355x_log_softmax_f32", torch.log_softmax)):
            y = torch.full((rows, cols), np.nan, device="cuda")
            call(name, view.data_ptr(), y.data_ptr(), rows, cols, 1)
            assert worst(reference(view.double(), 1), y) < 1e-6 if cols > 1 else bool((reference(view, 1) == y).all())


def test_softmax_of_odd_rows_keeps_nan_and_infinities_in_their_row():
    x = torch.randn(6, 197, device="cuda")
    x[1, 7], x[2, 196], x[3, :100] = float("nan"), float("inf"), -float("inf")
    x[4, :] = -float("inf")
    y = torch.empty_like(x)
    call("mi355x_softmax_f32", x.data_ptr(), y.data_ptr(), 6, 197, 1)
    assert torch.allclose(torch.softmax(x, 1), y, rtol=2e-6, atol=1e-9, equal_nan=True)


@pytest.mark.parametrize("kind, reference", [(0, lambda x: x.mean(1)), (1, lambda x: x.sum(1)), (2, lambda x: x.amax(1)), (3, lambda x: x.amin(1))])
@pytest.mark.parametrize("rows, cols", [(4096, 1), (4099, 63), (4097, 64), (4098, 65), (5000, 197), (4111, 256), (4096, 257), (4095, 197)])
def test_reductions_of_many_short_rows(kind, reference, rows, cols):
    x = gpu(np.random.default_rng(rows).standard_normal((rows, cols), dtype=np.float32))
    x[3, cols // 2] = float("nan")
    y = torch.empty(rows, device="cuda")
    call("mi355x_reduce_f32", kind, x.data_ptr(), y.data_ptr(), rows, cols, 1)
    assert torch.isnan(y).nonzero().flatten().tolist() == [3]
    x[3], y[3] = 0, 0
    assert worst(reference(x.double()), y) < (1e-6 if kind < 2 else 1e-12)
