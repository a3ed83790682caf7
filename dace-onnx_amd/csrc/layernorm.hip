// ONNX LayerNormalization over the last axis, fp32, one pass over HBM.
//
// The reference reaches this op only as the exporter's nine-node chain
// ReduceMean, Sub, Pow, ReduceMean, Add(eps), Sqrt, Div, Mul(gamma), Add(beta)
// (daceml/onnx/op_implementations/pure_implementations.py:97-109,82-84,59-74,
// 77-79,41-56,92-94), each with a materialised intermediate. Here a row stays
// in registers: mean, then the biased variance of the centred values (the same
// two-step order as the chain, not E[x^2]-E[x]^2), then the affine output.
//
// Kernels:
//   layernorm_rows_reg<NV>  cols % 4 == 0, cols <= 256*NV: one wave per row,
//       NV float4 per lane (768 columns = 3 loads of 16 bytes per lane), DPP +
//       readlane reductions, no LDS.
//   layernorm_rows_loop     any cols: one wave per row, three sweeps.
//   layernorm_parts_reg<NV, PARTS>  the first, over partial sums of the product before it.
#include "common.h"

#include <type_traits>

namespace mi355x {

template <int NV>
__global__ __launch_bounds__(256) void layernorm_rows_reg(const float* __restrict__ X,
                                                          const float* __restrict__ gamma,
                                                          const float* __restrict__ beta,
                                                          float* __restrict__ Y, int64_t rows,
                                                          int cols, float eps) {
    const int lane = threadIdx.x % WAVE;
    const int64_t row = (int64_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
    if (row >= rows) return;  // wave-uniform
    const int cols4 = cols >> 2;
    const f32x4* src = reinterpret_cast<const f32x4*>(X + row * cols);

    f32x4 v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c4 = lane + j * WAVE;
        v[j] = (c4 < cols4) ? __builtin_nontemporal_load(src + c4) : f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // gamma / beta are shared by every row: ordinary (cached) loads
    f32x4 g[NV], b[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c4 = lane + j * WAVE;
        g[j] = (c4 < cols4) ? reinterpret_cast<const f32x4*>(gamma)[c4] : f32x4{0.f, 0.f, 0.f, 0.f};
        b[j] = (beta != nullptr && c4 < cols4) ? reinterpret_cast<const f32x4*>(beta)[c4]
                                               : f32x4{0.f, 0.f, 0.f, 0.f};
    }

    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) s += (v[j].x + v[j].y) + (v[j].z + v[j].w);
    const float inv_n = 1.0f / (float)cols;
    const float mean = wave_sum(s) * inv_n;

    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c4 = lane + j * WAVE;
        if (c4 < cols4) {
            v[j] -= mean;
            q += (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w);
        }
    }
    const float var = wave_sum(q) * inv_n;
    const float inv_std = 1.0f / sqrtf(var + eps);

    f32x4* dst = reinterpret_cast<f32x4*>(Y + row * cols);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c4 = lane + j * WAVE;
        if (c4 < cols4) {
            f32x4 o = (v[j] * inv_std) * g[j] + b[j];
            __builtin_nontemporal_store(o, dst + c4);
        }
    }
}

// The same over the sums of a product that was computed in parts (mi355x_gemm_parts_f32): x = sum_s P[s] + bias + residual, in that order. One wave
// per row, all of a row's loads in flight at once; values at any 4-byte boundary. Bound by the launch and one trip to memory for few rows (16 x 768 in
// eight parts 3.2 us, layernorm_rows_reg 2.2), so up to 1024 rows a workgroup is one wave; by the bytes for many (2048 x 768 in four parts 5.3 us).
template <int NV, int PARTS>
__global__ __launch_bounds__(256) void layernorm_parts_reg(const float* __restrict__ P, const float* __restrict__ bias,
                                                           const float* __restrict__ residual, int64_t r_sm,
                                                           const float* __restrict__ gamma, const float* __restrict__ beta,
                                                           float* __restrict__ Y, int64_t rows, int cols, float eps) {
    typedef f32x4 unaligned __attribute__((aligned(4)));
    const int lane = threadIdx.x % WAVE;
    const int64_t row = (int64_t)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (row >= rows) return;  // wave-uniform
    const int cols4 = cols >> 2;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 v[PARTS][NV], r[NV], c[NV], g[NV], b[NV];
#pragma unroll
    for (int s = 0; s < PARTS; ++s) {
        const f32x4* src = reinterpret_cast<const f32x4*>(P + (s * rows + row) * cols);
#pragma unroll
        for (int j = 0; j < NV; ++j) v[s][j] = lane + j * WAVE < cols4 ? src[lane + j * WAVE] : zero;
    }
    auto vectors = [&](f32x4 (&to)[NV], const float* from) {
#pragma unroll
        for (int j = 0; j < NV; ++j) to[j] = from != nullptr && lane + j * WAVE < cols4 ? f32x4(reinterpret_cast<const unaligned*>(from)[lane + j * WAVE]) : zero;
    };
    vectors(r, residual ? residual + row * r_sm : nullptr);
    vectors(c, bias);
    vectors(g, gamma);
    vectors(b, beta);

    float sum = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
#pragma unroll
        for (int s = 1; s < PARTS; ++s) v[0][j] += v[s][j];
        if (bias != nullptr) v[0][j] += c[j];
        if (residual != nullptr) v[0][j] += r[j];
        sum += (v[0][j].x + v[0][j].y) + (v[0][j].z + v[0][j].w);
    }
    const float inv_n = 1.0f / (float)cols;
    const float mean = wave_sum(sum) * inv_n;
    float q = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (lane + j * WAVE < cols4) {
            v[0][j] -= mean;
            q += (v[0][j].x * v[0][j].x + v[0][j].y * v[0][j].y) + (v[0][j].z * v[0][j].z + v[0][j].w * v[0][j].w);
        }
    const float inv_std = 1.0f / sqrtf(wave_sum(q) * inv_n + eps);
    unaligned* dst = reinterpret_cast<unaligned*>(Y + row * cols);
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (lane + j * WAVE < cols4) dst[lane + j * WAVE] = (v[0][j] * inv_std) * g[j] + b[j];
}

__global__ __launch_bounds__(256) void layernorm_rows_loop(const float* __restrict__ X,
                                                           const float* __restrict__ gamma,
                                                           const float* __restrict__ beta,
                                                           float* __restrict__ Y, int64_t rows,
                                                           int64_t cols, float eps) {
    const int lane = threadIdx.x % WAVE;
    const int64_t row = (int64_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE;
    if (row >= rows) return;
    const float* x = X + row * cols;
    float* y = Y + row * cols;
    float s = 0.0f;
    for (int64_t c = lane; c < cols; c += WAVE) s += x[c];
    const float mean = wave_sum(s) / (float)cols;
    float q = 0.0f;
    for (int64_t c = lane; c < cols; c += WAVE) {
        const float d = x[c] - mean;
        q += d * d;
    }
    const float var = wave_sum(q) / (float)cols;
    const float inv_std = 1.0f / sqrtf(var + eps);
    for (int64_t c = lane; c < cols; c += WAVE) {
        const float bb = beta ? beta[c] : 0.0f;
        y[c] = ((x[c] - mean) * inv_std) * gamma[c] + bb;
    }
}

}  // namespace mi355x

extern "C" int mi355x_layernorm_f32(const float* X, const float* gamma, const float* beta,
                                    float* Y, int64_t rows, int64_t cols, float eps,
                                    void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(rows >= 0 && cols >= 0, "layernorm: negative extent (rows=%lld cols=%lld)",
                   (long long)rows, (long long)cols);
    if (rows == 0 || cols == 0) return MI355X_OK;
    MI355X_REQUIRE(X && Y && gamma, "layernorm: null pointer (X, Y and gamma are required)");
    MI355X_REQUIRE(grid_fits(ceil_div(rows, 256 / WAVE), 256), "layernorm: too many rows");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const dim3 grid((unsigned)ceil_div(rows, 256 / WAVE)), block(256);
    auto aligned = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
    const bool vec_ok = (cols % 4 == 0) && aligned(X) && aligned(Y) && aligned(gamma) &&
                        (beta == nullptr || aligned(beta));
    const int c = (int)cols;
    if (vec_ok && cols <= 256) hipLaunchKernelGGL(layernorm_rows_reg<1>, grid, block, 0, st, X, gamma, beta, Y, rows, c, eps);
    else if (vec_ok && cols <= 512) hipLaunchKernelGGL(layernorm_rows_reg<2>, grid, block, 0, st, X, gamma, beta, Y, rows, c, eps);
    else if (vec_ok && cols <= 768) hipLaunchKernelGGL(layernorm_rows_reg<3>, grid, block, 0, st, X, gamma, beta, Y, rows, c, eps);
    else if (vec_ok && cols <= 1024) hipLaunchKernelGGL(layernorm_rows_reg<4>, grid, block, 0, st, X, gamma, beta, Y, rows, c, eps);
    else if (vec_ok && cols <= 2048) hipLaunchKernelGGL(layernorm_rows_reg<8>, grid, block, 0, st, X, gamma, beta, Y, rows, c, eps);
    else if (vec_ok && cols <= 4096) hipLaunchKernelGGL(layernorm_rows_reg<16>, grid, block, 0, st, X, gamma, beta, Y, rows, c, eps);
    else hipLaunchKernelGGL(layernorm_rows_loop, grid, block, 0, st, X, gamma, beta, Y, rows, cols, eps);
    return check_launch("layernorm_rows");
}

extern "C" int mi355x_layernorm_parts_f32(const float* P, int64_t parts, const float* bias, const float* residual, int64_t r_row_stride,
                                          const float* gamma, const float* beta, float* Y, int64_t rows, int64_t cols, float eps, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(rows >= 0 && cols >= 0 && cols % 4 == 0 && cols <= 1024 && (parts == 2 || parts == 3 || parts == 4 || parts == 6 || parts == 8),
                   "layernorm_parts: %lld parts of %lld x %lld", (long long)parts, (long long)rows, (long long)cols);
    if (rows == 0 || cols == 0) return MI355X_OK;
    MI355X_REQUIRE(P && Y && gamma && (reinterpret_cast<uintptr_t>(P) & 15) == 0, "layernorm_parts: null or unaligned pointer");
    const unsigned waves = rows <= 1024 ? 1 : 4;
    MI355X_REQUIRE(grid_fits(ceil_div(rows, (int64_t)waves), waves * WAVE), "layernorm_parts: too many rows");
    const dim3 grid((unsigned)ceil_div(rows, (int64_t)waves)), block(waves * WAVE);
    auto launch = [&](auto nv, auto n) {
        hipLaunchKernelGGL((layernorm_parts_reg<decltype(nv)::value, decltype(n)::value>), grid, block, 0, static_cast<hipStream_t>(stream), P, bias, residual,
                           r_row_stride, gamma, beta, Y, rows, (int)cols, eps);
    };
    auto with_parts = [&](auto nv) {
        if (parts == 2) launch(nv, std::integral_constant<int, 2>{});
        else if (parts == 3) launch(nv, std::integral_constant<int, 3>{});
        else if (parts == 4) launch(nv, std::integral_constant<int, 4>{});
        else if (parts == 6) launch(nv, std::integral_constant<int, 6>{});
        else launch(nv, std::integral_constant<int, 8>{});
    };
    if (cols <= 256) with_parts(std::integral_constant<int, 1>{});
    else if (cols <= 512) with_parts(std::integral_constant<int, 2>{});
    else if (cols <= 768) with_parts(std::integral_constant<int, 3>{});
    else with_parts(std::integral_constant<int, 4>{});
    return check_launch("layernorm_parts_reg");
}
