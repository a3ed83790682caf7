"""The convolution by packed filters, at the edges of its tiles, patches and values, against float64."""
import os
import re

import numpy as np
import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

from dace_onnx_amd import _lib
from dace_onnx_amd.pytorch.module import DaceModule
from dace_onnx_amd.testing.profiling import graph_time_us

pytestmark = pytest.mark.gpu
FORMS = range(1, 10)
PIXEL_FORMS, POINT_FORMS = (1, 4, 9), (4, 7, 8, 9)


def call(name, *args):
    _lib.check(getattr(_lib.library(), name)(*args, torch.cuda.current_stream().cuda_stream), name)


def gpu(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def words(C, KH, M):
    steps = 14 if C <= 4 else KH * KH
    return -(-M // 32) * (1 if C <= 4 else -(-C // 16)) * steps * 768


def packed_conv(x, w, bias=None, res=None, pads=(0, 0, 0, 0), strides=(1, 1), dilations=(1, 1), epi=0):
    (N, C, H, W), (M, _, KH, KW) = x.shape, w.shape
    geometry = [N, C, H, W, M, KH, KW, _lib.i64_array(pads), _lib.i64_array(strides), _lib.i64_array(dilations)]
    if os.environ.get("MI355X_CONV_PACKED") != "0":   # a form that does not take the layer would leave it to the kernels before
        assert _lib.library().mi355x_conv2d_packed_pays(*geometry, 1) == 4 * words(C, KH, M)
    packed = torch.empty(words(C, KH, M), dtype=torch.int32, device="cuda")
    call("mi355x_pack_conv_f32", w.data_ptr(), packed.data_ptr(), M, C, KH, KW)
    oh, ow = ((e + pads[i] + pads[i + 2] - (k - 1) * dilations[i] - 1) // strides[i] + 1 for i, (e, k) in enumerate(((H, KH), (W, KW))))
    guard = 64
    y = torch.full((N * M * oh * ow + guard, ), -7.0, device="cuda")
    call("mi355x_conv2d_packed_f32", x.data_ptr(), packed.data_ptr(), w.data_ptr(), _lib.ptr(bias), _lib.ptr(res), y.data_ptr(), *geometry, epi)
    assert bool((y[-guard:] == -7).all())
    return y[:-guard].reshape(N, M, oh, ow)


def exact_conv(x, w, pads=(0, 0, 0, 0), strides=(1, 1), dilations=(1, 1)):
    """In float64, as products of unfolded images."""
    x = F.pad(x.double(), (pads[1], pads[3], pads[0], pads[2]))
    KH, KW = w.shape[2:]
    oh, ow = ((e - (k - 1) * d - 1) // s + 1 for e, k, d, s in zip(x.shape[2:], (KH, KW), dilations, strides))
    flat = w.double().reshape(w.shape[0], -1)
    return torch.stack([flat @ F.unfold(image[None], (KH, KW), dilation=dilations, stride=strides)[0] for image in x]).reshape(len(x), len(w), oh, ow)


# N, C, H, W, M, kernel, pads, strides, dilations, epilogue: one position; images that end inside a tile; odd extents and half a group of
# channels; a stride and a dilation per axis (with patches for every form, and one that three of them do not hold); strips (48 and 64 columns) and none (47: patches of up to
# 150 KB of LDS); the residual block's end; few channels
LAYERS = [(1, 8, 3, 3, 1, 3, (0, 0, 0, 0), (1, 1), (1, 1), 0), (5, 16, 7, 7, 33, 3, (1, 1, 1, 1), (1, 1), (1, 1), 25),
          (2, 40, 13, 11, 70, 3, (1, 0, 2, 1), (1, 1), (1, 1), 3), (3, 24, 19, 17, 64, 3, (2, 1, 0, 3), (2, 1), (1, 2), 1),
          (2, 48, 9, 48, 96, 3, (1, 1, 1, 1), (1, 1), (1, 1), 9), (1, 136, 30, 64, 40, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1),
          (1, 128, 9, 47, 33, 3, (1, 1, 1, 1), (1, 1), (1, 1), 1), (1, 64, 15, 17, 130, 3, (1, 1, 1, 1), (2, 2), (1, 1), 0), (2, 8, 5, 6, 31, 1, (0, 0, 0, 0), (1, 1), (1, 1), 1),
          (3, 72, 14, 15, 65, 1, (0, 1, 1, 0), (2, 3), (1, 1), 25), (1, 320, 20, 33, 128, 1, (0, 0, 0, 0), (1, 1), (1, 1), 3),
          (2, 3, 40, 33, 33, 7, (3, 3, 3, 3), (2, 2), (1, 1), 3), (1, 4, 21, 64, 70, 7, (0, 2, 5, 1), (1, 1), (1, 1), 9), (3, 1, 9, 8, 5, 7, (3, 3, 3, 3), (1, 2), (1, 1), 0),
          (4, 2, 17, 48, 31, 7, (0, 1, 1, 0), (1, 1), (1, 1), 25), (2, 24, 9, 8, 64, 3, (2, 1, 0, 3), (2, 1), (1, 2), 1),
          (2, 24, 11, 7, 64, 3, (2, 2, 2, 2), (1, 1), (2, 2), 9), (1, 320, 9, 13, 70, 1, (0, 0, 0, 0), (1, 1), (1, 1), 3)]


def forms_of(N, C, H, W, M, kernel, pads, strides, dilations, epi):
    """The forms there are for such filters, but those that do not hold the layer's patch."""
    too_large = {(3, 24, 19, 17): (1, 2, 6), (1, 320, 20, 33): (8, )}.get((N, C, H, W), ())
    return [f for f in (PIXEL_FORMS if C <= 4 else POINT_FORMS if kernel == 1 else FORMS) if f not in too_large]


@pytest.mark.parametrize("N, C, H, W, M, kernel, pads, strides, dilations, epi, form", [(*layer, form) for layer in LAYERS for form in forms_of(*layer)])
def test_convolution_by_packed_filters(tuning, form, N, C, H, W, M, kernel, pads, strides, dilations, epi):
    """A sum of K products: at most one rounding (2^-23, truncation included) for each of the MFMA steps, of which few channels take up to
    K / 4, and three of 2^-24 for the products left out and the sets of sums."""
    tuning(MI355X_CONV_PACKED=form)
    rng = np.random.default_rng(N + C + H + M)
    x, w, bias = (gpu(rng.standard_normal(s, dtype=np.float32)) for s in ((N, C, H, W), (M, C, kernel, kernel), (M, )))
    wide = exact_conv(x, w, pads, strides, dilations)
    size = exact_conv(x.abs(), w.abs(), pads, strides, dilations) + 1
    res = gpu(rng.standard_normal(tuple(wide.shape), dtype=np.float32))
    got = packed_conv(x, w, bias, res, pads, strides, dilations, epi)
    expected = wide + (bias.double()[:, None, None] if epi & 1 else 0)
    expected = expected.relu() if epi & 2 else expected
    expected = expected + (res.double() if epi & 8 else 0)
    expected = expected.relu() if epi & 16 else expected
    steps = C * kernel * kernel // (4 if C <= 4 else 16)
    assert bool(((expected - got.double()).abs() <= (size + res.abs() * bool(epi & 8)) * (steps + 9) * 2.0**-23).all())


@pytest.mark.parametrize("form, C, kernel", [(f, 24, 3) for f in FORMS] + [(f, 24, 1) for f in POINT_FORMS] + [(f, 3, 7) for f in PIXEL_FORMS])
def test_convolution_by_packed_filters_keeps_infinities_nan_and_the_largest_values(tuning, form, C, kernel):
    tuning(MI355X_CONV_PACKED=form)
    torch.manual_seed(form)
    x, w = torch.randn(2, C, 12, 21, device="cuda"), torch.rand(40, C, kernel, kernel, device="cuda") + 0.5
    x[0, 1, 2, 3], x[0, 2, 9, 9], x[1, 0, 6, 6], x[1, 2, 0, 20], x[1, 1, 11, 0] = float("inf"), -float("inf"), float("nan"), 3.3999e38, -3.0e38
    w[:, 2] = 0.25   # (the largest value stays below infinity)
    w[7, 0, 0, 0] = float("inf")
    pads = [kernel // 2] * 4
    got = packed_conv(x, w, pads=pads)
    tuning(MI355X_CONV_PACKED=0)
    single = packed_conv(x, w, pads=pads)
    fine = torch.isfinite(single)
    assert torch.equal(torch.isnan(single), torch.isnan(got)) and torch.equal(single[~fine].nan_to_num(nan=0), got[~fine].nan_to_num(nan=0))
    size = exact_conv(x.abs().nan_to_num(0, 0), w.abs().nan_to_num(0, 0), pads)   # both are sums of C kernel^2 products
    assert bool(((single.double() - got.double()).abs()[fine] <= 2 * (C * kernel * kernel + 3) * 2.0**-24 * size[fine]).all())


@pytest.mark.parametrize("N, C, H, M", [(32, 128, 28, 128), (32, 512, 7, 512), (1, 512, 7, 512)])
def test_a_pixel_that_is_not_finite_takes_a_bounded_time(N, C, H, M):
    """Tiles with such a pixel are summed again by the fp32 MFMA: 3.2 to 3.8 times the launch (14 to 35 times where their loads come one at a time)."""
    x, w = torch.randn(N, C, H, H, device="cuda"), torch.randn(M, C, 3, 3, device="cuda")
    y, packed, i64 = torch.empty(N, M, H, H, device="cuda"), torch.empty(words(C, 3, M), dtype=torch.int32, device="cuda"), _lib.i64_array
    call("mi355x_pack_conv_f32", w.data_ptr(), packed.data_ptr(), M, C, 3, 3)
    launch = lambda: _lib.library().mi355x_conv2d_packed_f32(x.data_ptr(), packed.data_ptr(), w.data_ptr(), None, None, y.data_ptr(), N, C, H, H, M, 3, 3,   # noqa: E731
                                                             i64([1] * 4), i64([1, 1]), i64([1, 1]), 0, _lib.current_stream())
    before = graph_time_us(launch, reps=20)
    x[N // 2, 0, H // 2, H // 2] = float("nan")
    assert graph_time_us(launch, reps=20) < 8 * before
    torch.cuda.synchronize()
    assert int(torch.isnan(y).sum()) == 9 * M


@pytest.mark.parametrize("low, high", [(-100, 90), (-148, 105), (90, -3)])
@pytest.mark.parametrize("form, C, kernel", [(1, 32, 3), (7, 32, 3), (9, 32, 1), (4, 3, 7)])
def test_convolution_by_packed_filters_keeps_small_values(tuning, form, C, kernel, low, high):
    """Values down to the smallest subnormal against values that bring the sums back to ordinary size: the bound is that of ordinary ones."""
    tuning(MI355X_CONV_PACKED=form)
    rng = np.random.default_rng(form)
    x, w = (gpu(np.ldexp(rng.uniform(1, 2, s) * rng.choice([-1, 1], s), e).astype(np.float32)) for s, e in (((1, C, 12, 12), low), ((35, C, kernel, kernel), high)))
    got, expected, size = packed_conv(x, w), exact_conv(x, w), exact_conv(x.abs(), w.abs())
    assert bool(((expected - got.double()).abs() <= size * (C * kernel * kernel // 4 + 9) * 2.0**-23 + 2.0**-149).all())


@pytest.mark.parametrize("N, C, H, W, M, kernel, pads, strides, dilations, epi, form",
                         [(*layer, form) for layer in LAYERS if layer[1] > 4 and layer[5] == 3 and layer[:4] != (3, 24, 19, 17) for form in (10, 11)])
def test_tiles_of_128_filters(tuning, form, N, C, H, W, M, kernel, pads, strides, dilations, epi):
    """The edges above (one patch does not fit), and values that are not finite."""
    test_convolution_by_packed_filters(tuning, form, N, C, H, W, M, kernel, pads, strides, dilations, epi)
    test_convolution_by_packed_filters_keeps_infinities_nan_and_the_largest_values(tuning, form, 24, 3)


@pytest.mark.parametrize("low, high", [(-100, 90), (-148, 105), (90, -3)])
@pytest.mark.parametrize("form", [10, 11])
def test_tiles_of_128_filters_keep_small_values(tuning, form, low, high):
    test_convolution_by_packed_filters_keeps_small_values(tuning, form, 32, 3, low, high)


@pytest.mark.parametrize("N, C, H, M", [(32, 64, 56, 120), (30, 128, 28, 256), (17, 64, 49, 250), (16, 64, 49, 128)])
def test_layers_that_take_tiles_of_128_filters(tuning, N, C, H, M):
    """By the rule (the kernel's fourth template argument counts blocks of 32 filters), with no more error than by tiles of 64: as many groups of waves
    share the channels, or more, and the sums of one group are the same. 1.6e-7 of the norm leaves a tenth over the largest seen."""
    torch.manual_seed(N)
    x, w = torch.randn(N, C, H, H, device="cuda"), torch.randn(M, C, 3, 3, device="cuda")
    layer = dict(pads=(1, 1, 1, 1), strides=(2, 2))
    packed_conv(x, w, **layer)
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as profile:
        got = packed_conv(x, w, **layer)
        torch.cuda.synchronize()
    kernels = [re.search(r"conv2d_f32_packed_kernel<.*?>, \w+, \d+, (\d+),", e.name) for e in profile.events()]
    assert [k.group(1) for k in kernels if k] == ["4"]
    tuning(MI355X_CONV_PACKED=10)
    wide_tiles = packed_conv(x, w, **layer)
    tuning(MI355X_CONV_PACKED=9)
    tiles = packed_conv(x, w, **layer)
    assert torch.equal(wide_tiles, tiles)
    expected = exact_conv(x, w, (1, 1, 1, 1), (2, 2))
    error, before = (float((y.double() - expected).norm() / expected.norm()) for y in (got, tiles))
    assert error <= before and error < 1.6e-7


def test_a_packed_convolution_follows_its_filters():
    """A block of a residual network: filters written in place after the first call; the next call multiplies by the new ones."""
    conv = nn.Conv2d(64, 64, 3, padding=1).cuda()
    x = torch.randn(32, 64, 56, 56, device="cuda")
    model = DaceModule(nn.Sequential(conv, nn.ReLU()), dummy_inputs=(x, ))
    for _ in range(2):
        with torch.no_grad():
            conv.weight.mul_(0.5)
            conv.weight[3] += 1
        got = model(x)
        expected = (exact_conv(x, conv.weight.detach(), (1, 1, 1, 1)) + conv.bias.detach().double()[:, None, None]).relu()
        assert float((got.double() - expected).norm() / expected.norm()) < 1e-6
    assert [n.function for n, _ in model.dace_model.compile_and_init().bound_launches()] == ["mi355x_conv2d_packed_f32"]
