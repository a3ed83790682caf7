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


@pytest.mark.parametrize("rows, cols", [((1 << 24) + 5, 513), ((1 << 26) + 9, 3)])
def test_softmax_of_more_rows_than_a_grid_holds(rows, cols):
    """2^32 threads and more are several launches; rows on both sides of the seam."""
    x, y = torch.empty(rows, cols, device="cuda"), torch.empty(rows, cols, device="cuda")
    seam = [0, 1, (1 << 24) - 2, (1 << 24) - 1, 1 << 24, rows - 2, rows - 1] + [r for r in ((1 << 26) - 5, (1 << 26) - 4, 1 << 26) if r < rows]
    x[seam] = torch.randn(len(seam), cols, device="cuda")
    y[seam] = float("nan")
    call("mi355x_softmax_f32", x.data_ptr(), y.data_ptr(), rows, cols, 1)
    assert worst(torch.softmax(x[seam].double(), 1), y[seam]) < 1e-6


def test_gemm_of_more_small_products_than_a_grid_of_the_few_tile_kernel_holds():
    """2^22 workgroups of 1024 threads are too many for a launch: another kernel takes them."""
    batch, N, K = (1 << 22) + 3, 4, 160
    a, b = torch.empty(batch, 1, K, device="cuda"), torch.randn(N, K, device="cuda")
    ends = [0, 1, 1 << 22, batch - 1]
    a[ends] = torch.randn(len(ends), 1, K, device="cuda")
    got = split_gemm(a, b, True, batch=batch)[ends]
    assert worst(a[ends].double() @ b.double().t(), got) < 2e-6   # K / 16 + 24 roundings of 2^-24 at most


@pytest.mark.parametrize("kind, reference", [(0, lambda x: x.mean(1)), (1, lambda x: x.sum(1)), (2, lambda x: x.amax(1)), (3, lambda x: x.amin(1))])
@pytest.mark.parametrize("rows, cols", [(4096, 1), (4099, 63), (4097, 64), (4098, 65), (5000, 197), (4111, 256), (4096, 257), (4095, 197),
                                        (12287, 33), (12288, 33), (12291, 64), (16383, 65), (16385, 79), (18431, 256), (18433, 200)])
def test_reductions_of_many_short_rows(kind, reference, rows, cols):
    x = gpu(np.random.default_rng(rows).standard_normal((rows, cols), dtype=np.float32))
    x[3, cols // 2] = float("nan")
    y = torch.empty(rows, device="cuda")
    call("mi355x_reduce_f32", kind, x.data_ptr(), y.data_ptr(), rows, cols, 1)
    assert torch.isnan(y).nonzero().flatten().tolist() == [3]
    x[3], y[3] = 0, 0
    assert worst(reference(x.double()), y) < (1e-6 if kind < 2 else 1e-12)


def split_gemm(a, b, kc, bias=None, res=None, epi=0, alpha=1.0, batch=1):
    """C = a @ b through mi355x_gemm_f32; ``b`` is [N, K] if ``kc`` else [K, N]; a batch shares b."""
    M, K = a.shape[-2:]
    N = b.shape[0] if kc else b.shape[1]
    c = torch.full((batch, M, N), np.nan, device="cuda")
    i64 = _lib.i64_array
    call("mi355x_gemm_f32", a.data_ptr(), b.data_ptr(), c.data_ptr(), bias.data_ptr() if bias is not None else None,
         res.data_ptr() if res is not None else None, 1, batch, M, N, K, i64([0, M * K, K, 1]), i64([0, 0] + ([1, K] if kc else [N, 1])),
         i64([0, M * N, N]), i64([0, M * N, N]), alpha, epi)
    return c


@pytest.mark.parametrize("kc", [True, False])
@pytest.mark.parametrize("rows", [64, 128, 256])
@pytest.mark.parametrize("batch, M, N, K, epi", [(1, 1, 1, 32, 0), (1, 63, 65, 64, 1), (1, 64, 64, 96, 9), (2, 129, 127, 160, 13), (1, 257, 130, 32, 3),
                                                 (1, 255, 258, 768, 9), (3, 512, 128, 1056, 8)])
def test_gemm_of_values_split_in_three(tuning, rows, kc, batch, M, N, K, epi):
    """Every form of the bf16 kernel at the edges of its tiles. A sum of K products: at most one rounding (2^-23, truncation
    included) for each of the K / 32 steps, and three of 2^-24 for the products left out and the two sets of sums."""
    tuning(MI355X_GEMM_SPLIT=rows)
    rng = np.random.default_rng(M + N + K)
    a = gpu(rng.standard_normal((batch, M, K), dtype=np.float32))
    b = gpu(rng.standard_normal((N, K) if kc else (K, N), dtype=np.float32))
    bias, res = gpu(rng.standard_normal(N, dtype=np.float32)), gpu(rng.standard_normal((batch, M, N), dtype=np.float32))
    got = split_gemm(a, b, kc, bias, res, epi, 0.5, batch)
    wide = b.double().t() if kc else b.double()
    expected = 0.5 * (a.double() @ wide) + (bias.double() if epi & 1 else 0)
    if epi & 2:
        expected = expected.relu()
    if epi & 4:
        expected = torch.nn.functional.gelu(expected)
    if epi & 8:
        expected = expected + res.double()
    bound = (a.double().abs() @ wide.abs() + 1) * (K // 32 + 8) * 2.0**-23
    assert bool(((expected - got.double()).abs() <= 1.2 * bound).all())   # 1.13 is Gelu's steepest slope


@pytest.mark.parametrize("kc", [True, False])
@pytest.mark.parametrize("rows", [64, 128, 256])
def test_split_gemm_keeps_infinities_nan_and_the_largest_values(tuning, rows, kc):
    tuning(MI355X_GEMM_SPLIT=rows)
    a = torch.randn(1, 300, 96, device="cuda")
    b = torch.rand(200, 96, device="cuda") + 0.5
    a[0, 3, 5], a[0, 70, 95], a[0, 130, 0], a[0, 131, 1:3] = float("inf"), -float("inf"), float("nan"), torch.tensor([float("inf"), -float("inf")])
    a[0, 200], a[0, 200, 7], a[0, 290, 9] = 0, 3.4e38, 3.3999e38   # rounds up to infinity in bf16
    b[:, 7] = 0.75
    b[11, 9], b[150, 9], b[150, 60] = 0, 0.5, float("inf")   # (0.5: no product of its own overflows next to the infinite one)
    expected = a[0].double() @ b.double().t()
    got = split_gemm(a, b if kc else b.t().contiguous(), kc)[0]
    single = expected.float()
    assert torch.equal(torch.isnan(single), torch.isnan(got)) and torch.equal(torch.isinf(single), torch.isinf(got))
    fine = torch.isfinite(single)
    assert torch.equal(single[~fine].nan_to_num(nan=0), got[~fine].nan_to_num(nan=0))
    assert bool(((expected - got.double()).abs()[fine] <= 1e-5 * (a[0].double().abs().nan_to_num(0, 0) @ b.double().abs().nan_to_num(0, 0, 0).t())[fine]).all())


@pytest.mark.parametrize("kc", [True, False])
@pytest.mark.parametrize("rows", [64, 128, 256])
def test_split_gemm_keeps_small_values(tuning, rows, kc):
    """Values down to the smallest subnormal against values that bring the sums back to ordinary size, on either side, and sums
    close to the smallest normal number. Where the values are ordinary floats nothing may be lost to their size: the bound is that
    of the split itself. A subnormal is exact as well, so its products are."""
    tuning(MI355X_GEMM_SPLIT=rows)
    M, N, K = 130, 140, 96
    rng = np.random.default_rng(rows)
    for low, high in ((-100, 90), (-105, 95), (-112, 100), (-120, 100), (-126, 105), (-134, 105), (-148, 105), (-60, -58), (-3, 90)):
        small, large = (torch.from_numpy(np.ldexp(rng.uniform(1, 2, s) * rng.choice([-1, 1], s), e).astype(np.float32)) for s, e in (((M, K), low), ((N, K), high)))
        small[::2, ::3] = torch.from_numpy(rng.uniform(1, 2, small[::2, ::3].shape).astype(np.float32)) * 2.0**min(low + 20, 0)   # two sizes in a row
        for a, b in ((small, large), (torch.cat([large, large])[:M], torch.cat([small, small])[:N])):
            a, b = a.cuda().contiguous(), b.cuda().contiguous()
            got = split_gemm(a[None], b if kc else b.t().contiguous(), kc)[0]
            expected = a.double() @ b.double().t().contiguous()
            bound = (a.double().abs() @ b.double().abs().t().contiguous()) * (K // 32 + 8) * 2.0**-23 + 2.0**-149
            assert bool(((expected - got.double()).abs() <= bound).all()), (low, high)


@pytest.mark.parametrize("form, kc", [(11, True), (12, True), (22, True), (14, False), (24, False)])
@pytest.mark.parametrize("batch, M, N, K, epi", [(1, 1, 4, 4, 0), (1, 1, 5, 5, 1), (1, 15, 17, 15, 9), (2, 16, 16, 16, 0), (1, 17, 33, 18, 3), (3, 31, 63, 255, 13),
                                                 (1, 33, 65, 257, 9), (1, 5, 10, 300, 1), (1, 40, 130, 1503, 8), (2, 7, 66, 3072, 9), (1, 64, 127, 4099, 0)])
def test_gemm_straight_from_memory(tuning, form, kc, batch, M, N, K, epi):
    """Every form at the edges of its tiles and of its waves' shares of K, from addresses that are only 4-byte aligned, between values
    that would show; and an infinity stays in its row. Sums of K / 16 products by each wave, then sixteen: a rounding of 2^-24 each."""
    tuning(MI355X_GEMM_DIRECT=form)
    rng = np.random.default_rng(M + N + K)
    held = [torch.full((n + 9,), np.nan, device="cuda") for n in (batch * M * K, N * K, N, batch * M * N)]
    a, b, bias, res = (h[5:-4] for h in held)
    for view in (a, b, bias, res):
        view.copy_(gpu(rng.standard_normal(view.numel(), dtype=np.float32)))
    a, b, res = a.view(batch, M, K), b.view(N, K) if kc else b.view(K, N), res.view(batch, M, N)
    got = split_gemm(a, b, kc, bias, res, epi, 0.5, batch)
    wide = b.double().t().contiguous() if kc else b.double()
    expected = 0.5 * (a.double() @ wide) + (bias.double() if epi & 1 else 0)
    if epi & 2:
        expected = expected.relu()
    if epi & 4:
        expected = torch.nn.functional.gelu(expected)
    if epi & 8:
        expected = expected + res.double()
    bound = (a.double().abs() @ wide.abs() + 1) * (K // 16 + 24) * 2.0**-24
    assert bool(((expected - got.double()).abs() <= 1.2 * bound).all())   # 1.13 is Gelu's steepest slope
    a[0, M - 1, K - 1] = float("inf")
    got = split_gemm(a, b, kc, batch=batch)
    assert bool(torch.isfinite(got).flatten()[:(M - 1) * N].all()) and bool(torch.isinf(got[0, M - 1]).all())


@pytest.mark.parametrize("variable, form", [("MI355X_GEMM_DIRECT", f) for f in (11, 12, 22, 14, 24)] + [("MI355X_GEMM_SPLIT", f) for f in (64, 128, 256)])
@pytest.mark.parametrize("kc", [True, False])
@pytest.mark.parametrize("M, N, K", [(37, 70, 64), (130, 131, 96), (1, 5, 160)])
def test_gemm_forms_take_any_strides(tuning, variable, form, kc, M, N, K):
    """Rows further apart than their length in every operand, two batch levels in either order and broadcast, a residual laid out
    otherwise than the result; nothing between the rows of the result is written. The bound is that of the kernels through LDS."""
    rng = np.random.default_rng(M + N + K + form)
    B0, B1 = 2, 3
    for order, share_a, share_b in (((0, 1), False, False), ((1, 0), True, False), ((0, 1), False, True)):
        def laid_out(rows, cols, gap, shared):
            pitch = cols + gap
            strides = [0, 0] if shared else [rows * pitch * (B1 if order == (0, 1) else 1), rows * pitch * (1 if order == (0, 1) else B0)]
            memory = torch.full(((1 if shared else B0 * B1) * rows * pitch,), np.nan, device="cuda")
            view = torch.as_strided(memory, (B0, B1, rows, cols), (*strides, pitch, 1))
            torch.as_strided(memory, (memory.numel() // (rows * pitch), rows, cols), (rows * pitch, pitch, 1)).copy_(
                gpu(rng.standard_normal((memory.numel() // (rows * pitch), rows, cols), dtype=np.float32)))
            return memory, view, [*strides, pitch]
        (_, a, sa), (_, b, sb) = laid_out(M, K, 4, share_a), laid_out(N if kc else K, K if kc else N, 8, share_b)
        (cm, c, sc), (_, r, sr) = laid_out(M, N, 5, False), laid_out(M, N, 3, False)
        bias, before = gpu(rng.standard_normal(N, dtype=np.float32)), cm.clone()
        i64, results = _lib.i64_array, []
        for forced in (form, 0):
            tuning(**{"MI355X_GEMM_DIRECT": 0, "MI355X_GEMM_SPLIT": 0, variable: forced})
            cm.copy_(before)
            call("mi355x_gemm_f32", a.data_ptr(), b.data_ptr(), c.data_ptr(), bias.data_ptr(), r.data_ptr(), B0, B1, M, N, K, i64([*sa, 1]),
                 i64([*sb[:2], *([1, sb[2]] if kc else [sb[2], 1])]), i64(sc), i64(sr), 0.5, _lib.EPI_BIAS | _lib.EPI_RESIDUAL)
            results.append(c.clone())
            assert torch.equal(torch.isnan(cm), torch.isnan(before))
        wide = b.double().transpose(-1, -2).contiguous() if kc else b.double().contiguous()
        expected = 0.5 * (a.double().contiguous() @ wide) + bias.double() + r.double()
        bound = (a.double().abs().contiguous() @ wide.abs() + 2) * (K // 4 + 8) * 2.0**-24
        for got in results:
            assert bool(((expected - got.double()).abs() <= bound).all())


@pytest.mark.parametrize("batch, M, N, K, kc, form", [(48, 1338, 457, 47, False, 24), (96, 275, 1303, 120, False, 24), (96, 14, 2720, 64, True, 12),
                                                        (200, 168, 382, 144, False, 24), (200, 1461, 43, 148, False, 24)])
def test_gemm_of_many_rounds_of_workgroups_is_not_one_of_few_tiles(tuning, batch, M, N, K, kc, form):
    """Which kernel ran shows in the order of the sums: the bits are those of the kernels through LDS, not of the few-tile form."""
    a, b = torch.randn(batch, M, K, device="cuda"), torch.randn(*((N, K) if kc else (K, N)), device="cuda")
    results = []
    for forced in (None, 0, form):
        tuning(MI355X_GEMM_DIRECT=forced)
        results.append(split_gemm(a, b, kc, batch=batch))
    assert torch.equal(results[0], results[1]) and not torch.equal(results[1], results[2])


@pytest.mark.parametrize("batch, M, N, K", [(12, 675, 160, 1472), (1, 1237, 1536, 2592), (8, 1024, 256, 2816)])
def test_gemm_of_two_tiles_to_a_cu_stays_on_the_fp32_unit(tuning, batch, M, N, K):
    a, b = torch.randn(batch, M, K, device="cuda"), torch.randn(N, K, device="cuda")
    results = []
    for forced in (None, 0, 64):
        tuning(MI355X_GEMM_SPLIT=forced)
        results.append(split_gemm(a, b, True, batch=batch))
    assert torch.equal(results[0], results[1]) and not torch.equal(results[1], results[2])


def test_gemm_picks_the_same_result_whatever_kernel(tuning):
    """Sizes on both sides of the rules that pick the bf16 kernel, against the kernels it takes over from."""
    for M, N, K, kc in ((512, 3072, 512, False), (2048, 3072, 512, False), (1024, 3072, 768, True), (4096, 1024, 768, True), (2048, 1001, 256, True),
                        (64, 1002, 768, False), (64, 1002, 96, False), (64, 1002, 100, False), (3000, 2000, 776, True),
                        (16, 768, 3072, True), (128, 768, 768, True), (5, 300, 784, True), (33, 1000, 1503, True), (3, 1001, 512, False)):
        a, b = torch.randn(1, M, K, device="cuda"), torch.randn(*((N, K) if kc else (K, N)), device="cuda")
        tuning(MI355X_GEMM_SPLIT=None, MI355X_GEMM_DIRECT=None)
        chosen = split_gemm(a, b, kc)
        tuning(MI355X_GEMM_SPLIT=0, MI355X_GEMM_DIRECT=0)
        assert worst(split_gemm(a, b, kc).double(), chosen) < 5e-6   # two roundings of 2^-24 sqrt(K) each, five sigma


@pytest.mark.parametrize("sk", [1, 3, 127, 128, 129, 173, 300])
@pytest.mark.parametrize("fill", [-10000.0, float(np.finfo(np.float32).min), -float("inf")])
def test_masked_attention(sk, fill):
    """The mask per key, per query row and per head; whole blocks and whole rows masked; a mask at an odd address."""
    b0, b1, sq = 2, 3, 70
    q, k, v = (torch.randn(b0, b1, n, 64, device="cuda") for n in (sq, sk, sk))
    strides = lambda t: _lib.i64_array([t.stride(0), t.stride(1), t.stride(2)])   # noqa: E731
    for shape in ((b0, 1, 1, sk), (1, 1, sq, sk), (b0, b1, sq, sk), (1, 1, 1, sk)):
        buffer = torch.where(torch.rand(int(np.prod(shape)) + 1, device="cuda") < 0.3, fill, 0.0)
        mask = buffer[1:].view(shape)
        mask[..., :max(0, sk - 3)] = mask[..., :max(0, sk - 3)] if sk < 200 else fill   # a first block without one valid key
        mask[0, 0, 0] = fill                                                            # a row without one (all of them if it is broadcast)
        wide = mask.expand(b0, b1, sq, sk)
        out = torch.full((b0, b1, sq, 64), np.nan, device="cuda")
        call("mi355x_attention_masked_f32", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), mask.data_ptr(), b0, b1, sq, sk, 64,
             strides(q), strides(k), strides(v), strides(out),
             _lib.i64_array([st if e > 1 else 0 for st, e in zip(mask.stride()[:3], shape)]), 0.125)
        # the scores in fp32 as the nodes compute them: a mask of the type's lowest value absorbs them there
        scores = (0.125 * (q.double() @ k.double().transpose(-1, -2).contiguous())).float() + wide
        expected = torch.softmax(scores.double(), -1) @ v.double()
        nan = torch.isnan(expected)
        assert torch.equal(nan, torch.isnan(out))
        # fp32 scores of up to 10 in magnitude: 2^-21 relative on a probability; -10000 leaves 2^-11 of rounding in a row of masked keys only
        error = (expected - out.double()).abs().nan_to_num(0).amax(-1)
        masked = (wide == fill).all(-1)
        assert float(error[~masked].max() if bool((~masked).any()) else 0) < 2e-5
        assert float(error.max()) < (2e-5 if fill != -10000.0 else 5e-3)


@pytest.mark.parametrize("b0, b1, sq, sk", [(2, 12, 69, 300), (1, 12, 64, 512)])
@pytest.mark.parametrize("scale", [1.0, 8.0])
def test_masked_attention_is_as_exact_as_the_launches_it_replaces(tuning, b0, b1, sq, sk, scale):
    """2-norm of the error against float64, the mean over thousands of rows: two percent is many times its spread."""
    tuning(MI355X_GEMM_DIRECT=0)
    torch.manual_seed(sk)
    q, k, v = (torch.randn(b0, b1, n, 64, device="cuda") for n in (sq, sk, sk))
    q *= scale
    mask = torch.where(torch.rand(b0, 1, 1, sk, device="cuda") < 0.2, -10000.0, 0.0)
    i64, full = _lib.i64_array, mask.expand(b0, b1, sq, sk).contiguous()
    strides = lambda t: i64([t.stride(0), t.stride(1), t.stride(2)])   # noqa: E731
    out, three, scores, probabilities = torch.empty_like(q), torch.empty_like(q), torch.empty_like(full), torch.empty_like(full)
    call("mi355x_attention_masked_f32", q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), mask.data_ptr(), b0, b1, sq, sk, 64,
         strides(q), strides(k), strides(v), strides(out), i64([sk, 0, 0]), 0.125)
    call("mi355x_gemm_f32", q.data_ptr(), k.data_ptr(), scores.data_ptr(), None, full.data_ptr(), 1, b0 * b1, sq, sk, 64, i64([0, sq * 64, 64, 1]),
         i64([0, sk * 64, 1, 64]), i64([0, sq * sk, sk]), i64([0, sq * sk, sk]), 0.125, _lib.EPI_RESIDUAL)
    call("mi355x_softmax_f32", scores.data_ptr(), probabilities.data_ptr(), b0 * b1 * sq, sk, 1)
    call("mi355x_gemm_f32", probabilities.data_ptr(), v.data_ptr(), three.data_ptr(), None, None, 1, b0 * b1, sq, 64, sk, i64([0, sq * sk, sk, 1]),
         i64([0, sk * 64, 64, 1]), i64([0, sq * 64, 64]), None, 1.0, 0)
    expected = torch.softmax(0.125 * (q.double() @ k.double().transpose(-1, -2).contiguous()) + full.double(), -1) @ v.double()
    error = [float((x.double() - expected).norm() / expected.norm()) for x in (out, three)]
    assert error[0] <= 1.02 * error[1]


@pytest.mark.parametrize("tile", [0, 64, 128])
@pytest.mark.parametrize("M, N, K", [(1, 1, 1), (3, 7, 5), (2, 9, 8), (5, 1, 3), (5, 1, 4), (1, 3, 300), (63, 65, 127), (64, 64, 112), (65, 129, 129),
                                     (130, 66, 33), (128, 128, 144), (129, 127, 257), (200, 130, 385), (129, 3, 20), (129, 130, 1), (1, 2, 70), (16, 1, 4),
                                     (129, 129, 70), (130, 132, 80), (257, 100, 784)])
def test_matmul_integer_of_any_extent_and_address(tuning, tile, M, N, K):
    """Whole vectors from any address, clamped at the end of a matrix: both operands end where their allocation's view ends, the
    bytes around them are not theirs, and the result is exact."""
    tuning(MI355X_MMI_TILE=tile)
    rng = np.random.default_rng(M * N + K)
    for a_unsigned, b_unsigned, shift in ((0, 0, 0), (1, 0, 1), (0, 1, 2), (1, 1, 3)):
        a_low, b_low = (0 if a_unsigned else -128), (0 if b_unsigned else -128)
        a, b = rng.integers(a_low, a_low + 256, (M, K)), rng.integers(b_low, b_low + 256, (K, N))
        za, zb = rng.integers(a_low, a_low + 256, M if shift % 2 else 1), rng.integers(b_low, b_low + 256, N if shift % 2 == 0 else 1)
        held = [np.full(shift + v.size + 5, 77, np.uint8) for v in (a, b)]
        for memory, v in zip(held, (a, b)):
            memory[shift:shift + v.size] = v.astype(np.int64).astype(np.uint8).reshape(-1)
        ga, gb, gza, gzb = gpu(held[0]), gpu(held[1]), gpu(za.astype(np.int64) & 255).to(torch.uint8), gpu(zb.astype(np.int64) & 255).to(torch.uint8)
        y = torch.full((M, N), -1, dtype=torch.int32, device="cuda")
        call("mi355x_matmul_integer", ga.data_ptr() + shift, gb.data_ptr() + shift, gza.data_ptr(), gzb.data_ptr(), y.data_ptr(), M, N, K,
             a_unsigned, b_unsigned, za.size, zb.size)
        assert np.array_equal((a - za[:, None]) @ (b - zb[None, :]), y.cpu().numpy())


@pytest.mark.parametrize("M, N, K", [(2, (1 << 24) - 1, 3), (2, (1 << 24) + 5, 3), (3, 2, (1 << 24) + 70)])
def test_matmul_integer_of_rows_past_32_bit_offsets(M, N, K):
    rng = np.random.default_rng(K)
    a, b = rng.integers(-128, 128, (M, K), dtype=np.int8), rng.integers(-128, 128, (K, N), dtype=np.int8)
    ga, gb, y = gpu(a), gpu(b), torch.full((M, N), -1, dtype=torch.int32, device="cuda")
    call("mi355x_matmul_integer", ga.data_ptr(), gb.data_ptr(), None, None, y.data_ptr(), M, N, K, 0, 0, 1, 1)
    a, b = a.astype(np.float64), b.astype(np.float64)   # sums below 2^14 K, exact
    assert np.array_equal((a @ b).astype(np.int64).astype(np.int32), y.cpu().numpy())


@pytest.mark.parametrize("form", [None, 11, 21, 22])
@pytest.mark.parametrize("N, C, H, W, M, kernel, stride, pads, dilation", [(1, 32, 1, 1, 1, 1, 1, (0, 0, 0, 0), 1), (1, 32, 3, 3, 17, 3, 1, (1, 1, 1, 1), 1),
                                                                           (2, 64, 5, 7, 33, 3, 2, (0, 2, 1, 0), 1), (1, 96, 9, 4, 16, 3, 1, (2, 1, 2, 3), 2),
                                                                           (3, 544, 3, 3, 15, 3, 1, (1, 1, 1, 1), 1), (2, 32, 11, 6, 40, 1, 2, (0, 0, 0, 0), 1),
                                                                           (1, 1056, 5, 5, 65, 1, 1, (1, 0, 0, 1), 1), (1, 512, 7, 7, 512, 3, 1, (1, 1, 1, 1), 1)])
def test_convolution_of_few_tiles(tuning, form, N, C, H, W, M, kernel, stride, pads, dilation):
    """Every form at the edges of its tiles and of its waves' shares of the channels, all steps of the epilogue, between values that
    would show. Sums of K / 16 products by each wave, then sixteen: a rounding of 2^-24 each."""
    tuning(MI355X_CONV_DIRECT=form)
    rng = np.random.default_rng(N + C + M)
    top, left, bottom, right = pads
    rows, cols = ((e + a + b - dilation * (kernel - 1) - 1) // stride + 1 for e, a, b in ((H, top, bottom), (W, left, right)))
    held = [torch.full((n + 12,), np.nan, device="cuda") for n in (N * C * H * W, M * C * kernel * kernel, M, N * M * rows * cols)]
    x, w, bias, res = (h[4:-8] for h in held)
    for view in (x, w, bias, res):
        view.copy_(gpu(rng.standard_normal(view.numel(), dtype=np.float32)))
    wide = torch.nn.functional.pad(x.view(N, C, H, W).double(), (left, right, top, bottom))
    columns = torch.nn.functional.unfold(wide, kernel, dilation=dilation, stride=stride)
    flat = w.view(M, -1).double()
    product = torch.stack([flat @ c for c in columns]).view(N, M, rows, cols)
    bound = torch.stack([flat.abs() @ c.abs() for c in columns]).view(N, M, rows, cols)
    for epi in (0, 1 + 2, 1 + 8 + 16):   # bias and relu; bias, residual and relu after it
        y = torch.full((N, M, rows, cols), np.nan, device="cuda")
        call("mi355x_conv2d_res_f32", x.data_ptr(), w.data_ptr(), bias.data_ptr(), res.data_ptr(), y.data_ptr(), N, C, H, W, M, kernel, kernel,
             _lib.i64_array(pads), _lib.i64_array([stride] * 2), _lib.i64_array([dilation] * 2), epi)
        expected = product + (bias.double().view(1, M, 1, 1) if epi & 1 else 0) + (res.double().view(N, M, rows, cols) if epi & 8 else 0)
        if epi:
            expected = expected.relu()
        assert bool(((expected - y.double()).abs() <= (bound + 8) * (C * kernel * kernel // 16 + 24) * 2.0**-24).all())


@pytest.mark.parametrize("N, C, H, M, kernel, stride, form", [(3, 32, 20, 512, 3, 1, 22), (5, 512, 33, 100, 1, 1, 22), (3, 1024, 33, 200, 1, 1, 22),
                                                              (4, 1024, 56, 100, 1, 2, 22)])
def test_convolution_of_more_rounds_is_not_one_of_few_tiles(tuning, N, C, H, M, kernel, stride, form):
    """Which kernel ran shows in the order of the sums: the bits are those of the kernel through LDS, not of the few-tile form."""
    x, w = torch.randn(N, C, H, H, device="cuda"), torch.randn(M, C, kernel, kernel, device="cuda")
    size = (H - 1) // stride + 1
    results = []
    for forced in (None, 0, form):
        tuning(MI355X_CONV_DIRECT=forced)
        results.append(torch.full((N, M, size, size), np.nan, device="cuda"))
        call("mi355x_conv2d_f32", x.data_ptr(), w.data_ptr(), None, results[-1].data_ptr(), N, C, H, H, M, kernel, kernel,
             _lib.i64_array([kernel // 2] * 4), _lib.i64_array([stride] * 2), _lib.i64_array([1, 1]), 0)
    assert torch.equal(results[0], results[1]) and not torch.equal(results[1], results[2])
