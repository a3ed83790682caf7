// ONNX Softmax and LogSoftmax, fp32, one pass over HBM.
//
// The reference expansion (daceml/onnx/op_implementations/pure_implementations.py:346-366)
// runs max, subtract, exp, sum and divide as five maps with three full-size
// temporaries. Here a row lives in registers between the read and the write,
// so HBM traffic is the algorithmic minimum: one read and one write per element.
// LogSoftmax (PureLogSoftmax, :594-616: (x - max) - log(sum(exp(x - max)))) is the same
// kernels with a different last step (template parameter LOG).
//
// Kernels:
//   softmax_rows_reg<L, NV, UNR>  last axis, cols % 4 == 0, cols <= L*4*NV.
//       A row is owned by L lanes (16, 32 or 64) holding NV float4 each, so a
//       128-column row is one 16-byte load per lane of a half wave and the two
//       reductions are DPP row operations, no LDS. Each group handles UNR rows
//       with all loads issued before the first reduction to keep HBM requests
//       in flight.
//   softmax_rows_any<THREADS, NV>  last axis, any cols <= THREADS*NV, no alignment asked
//       of a row: the row in the registers of one wave (THREADS = 64) or of one workgroup,
//       NV single floats per thread.
//   softmax_rows_loop   last axis, longer rows: one workgroup of 1024 per row, three
//       sweeps (max, sum, write).
//   softmax_strided     axis is not last: one thread per (outer, inner) column,
//       lanes adjacent along `inner` so every access is coalesced.
#include "common.h"

namespace mi355x {

template <int L>
__device__ __forceinline__ float group_sum(float v) {
    if constexpr (L == 16) return row16_sum(v);
    else if constexpr (L == 32) return half32_sum(v);
    else return wave_sum(v);
}
template <int L>
__device__ __forceinline__ float group_max(float v) {
    if constexpr (L == 16) return row16_max(v);
    else if constexpr (L == 32) return half32_max(v);
    else return wave_max(v);
}

template <int L, int NV, int UNR, bool LOG>
__global__ __launch_bounds__(256) void softmax_rows_reg(const float* __restrict__ X,
                                                        float* __restrict__ Y,
                                                        int64_t rows, int cols) {
    constexpr int GROUPS_PER_BLOCK = 256 / L;
    const int lane = threadIdx.x % L;
    const int group = threadIdx.x / L;
    const int64_t row0 = ((int64_t)blockIdx.x * GROUPS_PER_BLOCK + group) * UNR;
    const int cols4 = cols >> 2;

    f32x4 v[UNR][NV];
#pragma unroll
    for (int u = 0; u < UNR; ++u) {
        const int64_t row = row0 + u;
        const f32x4* src = reinterpret_cast<const f32x4*>(X + row * cols);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c4 = lane + j * L;
            if (row < rows && c4 < cols4) {
                v[u][j] = __builtin_nontemporal_load(src + c4);
            } else {
                v[u][j] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
            }
        }
    }

#pragma unroll
    for (int u = 0; u < UNR; ++u) {
        const int64_t row = row0 + u;
        float m = -INFINITY;
#pragma unroll
        for (int j = 0; j < NV; ++j)
            m = fmaxf(m, fmaxf(fmaxf(v[u][j].x, v[u][j].y), fmaxf(v[u][j].z, v[u][j].w)));
        m = group_max<L>(m);
        constexpr float LOG2E = 1.4426950408889634f;
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            // padded lanes hold -inf: exp(-inf - m) == 0 contributes nothing
            if constexpr (LOG) {
                v[u][j] = v[u][j] - m;   // kept for the result; the exponentials only feed the sum
                s += (expf(v[u][j].x) + expf(v[u][j].y)) + (expf(v[u][j].z) + expf(v[u][j].w));
            } else {
                // exp(x - m) as 2^((x - m) log2 e): one v_exp_f32 per element instead of the library routine.
                // The argument t is <= 0 (no overflow); its rounding error |t| 2^-24 shows as a relative error of
                // the result below 1.3e-6 for every element that is at least 2^-30 of the row maximum.
                v[u][j].x = __builtin_amdgcn_exp2f((v[u][j].x - m) * LOG2E);
                v[u][j].y = __builtin_amdgcn_exp2f((v[u][j].y - m) * LOG2E);
                v[u][j].z = __builtin_amdgcn_exp2f((v[u][j].z - m) * LOG2E);
                v[u][j].w = __builtin_amdgcn_exp2f((v[u][j].w - m) * LOG2E);
                s += (v[u][j].x + v[u][j].y) + (v[u][j].z + v[u][j].w);
            }
        }
        s = group_sum<L>(s);
        const float inv = 1.0f / s, log_s = LOG ? logf(s) : 0.0f;
        f32x4* dst = reinterpret_cast<f32x4*>(Y + row * cols);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c4 = lane + j * L;
            if (row < rows && c4 < cols4) {
                f32x4 o = LOG ? v[u][j] - log_s : v[u][j] * inv;
                __builtin_nontemporal_store(o, dst + c4);
            }
        }
    }
}

// Reduction over a workgroup of THREADS (the wave itself where THREADS is 64): `part` holds one value per wave.
template <int THREADS, bool MAX>
__device__ __forceinline__ float block_reduce(float v, float* part) {
    v = MAX ? wave_max(v) : wave_sum(v);
    if constexpr (THREADS == WAVE) return v;
    constexpr int WAVES = THREADS / WAVE;
    __syncthreads();   // the previous reduction's values have been read
    if (threadIdx.x % WAVE == 0) part[threadIdx.x / WAVE] = v;
    __syncthreads();
    v = part[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v = MAX ? fmaxf(v, part[w]) : v + part[w];
    return v;
}

// Bound by HBM: one read and one write. Rows of any length start at any multiple of four bytes, so lanes take single
// floats (a wave's load is 256 contiguous bytes, at most one cache line more than an aligned one). All of a row's
// loads are issued before the first reduction; a row stays with one wave up to 512 columns (no barrier, eight loads in
// flight per lane) and takes as many waves as keep the loads per thread at 32 or fewer above that. Against three
// sweeps by one wave per row: LogSoftmax [1024, 30522] 442 -> 58 us (4.3 TB/s), Softmax [18912, 197] 12.7 -> 8.3 us.
template <int THREADS, int NV, bool LOG>
__global__ __launch_bounds__(THREADS == WAVE ? 256 : THREADS) void softmax_rows_any(const float* __restrict__ X, float* __restrict__ Y,
                                                                                    int64_t rows, int cols) {
    constexpr int ROWS = THREADS == WAVE ? 4 : 1;   // rows per workgroup
    __shared__ float part[THREADS / WAVE];
    const int t = threadIdx.x % THREADS;
    const int64_t row = (int64_t)blockIdx.x * ROWS + threadIdx.x / THREADS;
    if (row >= rows) return;  // a whole wave, and only where no barrier follows (ROWS > 1)
    const float* x = X + row * cols;
    float* y = Y + row * cols;
    float v[NV];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = t + j * THREADS < cols ? __builtin_nontemporal_load(x + t + j * THREADS) : -INFINITY;
#pragma unroll
    for (int j = 0; j < NV; ++j) m = fmaxf(m, v[j]);
    m = block_reduce<THREADS, true>(m, part);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {   // columns beyond the row hold -inf: exp(-inf - m) adds nothing
        v[j] -= m;
        const float e = expf(v[j]);
        s += e;
        if constexpr (!LOG) v[j] = e;
    }
    s = block_reduce<THREADS, false>(s, part);
    const float inv = 1.0f / s, log_s = LOG ? logf(s) : 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (t + j * THREADS < cols) __builtin_nontemporal_store(LOG ? v[j] - log_s : v[j] * inv, y + t + j * THREADS);
}

template <bool LOG>
__global__ __launch_bounds__(1024) void softmax_rows_loop(const float* __restrict__ X, float* __restrict__ Y, int64_t cols) {
    __shared__ float part[1024 / WAVE];
    const float* x = X + (int64_t)blockIdx.x * cols;
    float* y = Y + (int64_t)blockIdx.x * cols;
    float m = -INFINITY;
    for (int64_t c = threadIdx.x; c < cols; c += 1024) m = fmaxf(m, x[c]);
    m = block_reduce<1024, true>(m, part);
    float s = 0.0f;
    for (int64_t c = threadIdx.x; c < cols; c += 1024) s += expf(x[c] - m);
    s = block_reduce<1024, false>(s, part);
    const float inv = 1.0f / s, log_s = LOG ? logf(s) : 0.0f;
    for (int64_t c = threadIdx.x; c < cols; c += 1024) y[c] = LOG ? (x[c] - m) - log_s : expf(x[c] - m) * inv;
}

template <bool LOG>
__global__ __launch_bounds__(256) void softmax_strided(const float* __restrict__ X,
                                                       float* __restrict__ Y,
                                                       int64_t outer, int64_t axis_len,
                                                       int64_t inner) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= outer * inner) return;
    const int64_t o = idx / inner, i = idx % inner;
    const float* x = X + o * axis_len * inner + i;
    float* y = Y + o * axis_len * inner + i;
    float m = -INFINITY;
    for (int64_t a = 0; a < axis_len; ++a) m = fmaxf(m, x[a * inner]);
    // eight running sums (independent chains for the loads), kept in double: a thread adds up a whole
    // column by itself, and in float the rounding error of the denominator would grow with axis_len
    // (3e-6 relative at 4100 elements); the kernel waits on strided loads, the wider adds are free
    double s[8] = {0., 0., 0., 0., 0., 0., 0., 0.};
    int64_t a = 0;
    for (; a + 8 <= axis_len; a += 8) {
#pragma unroll
        for (int u = 0; u < 8; ++u) s[u] += (double)expf(x[(a + u) * inner] - m);
    }
    for (int u = 0; a < axis_len; ++a, ++u) s[u] += (double)expf(x[a * inner] - m);
    const double total = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
    const float inv = (float)(1.0 / total), log_s = LOG ? (float)log(total) : 0.0f;
    for (a = 0; a < axis_len; ++a) y[a * inner] = LOG ? (x[a * inner] - m) - log_s : expf(x[a * inner] - m) * inv;
}

template <int L, int NV, int UNR, bool LOG>
static void launch_reg(const float* X, float* Y, int64_t rows, int cols, hipStream_t st) {
    constexpr int rows_per_block = (256 / L) * UNR;
    constexpr int64_t MOST = MAX_GRID_THREADS / 256 * rows_per_block;   // rows of one launch
    for (int64_t row = 0; row < rows; row += MOST) {
        const int64_t n = rows - row < MOST ? rows - row : MOST;
        hipLaunchKernelGGL((softmax_rows_reg<L, NV, UNR, LOG>), dim3((unsigned)ceil_div(n, (int64_t)rows_per_block)), dim3(256), 0, st,
                           X + row * cols, Y + row * cols, n, cols);
    }
}

template <int THREADS, int NV, bool LOG>
static void launch_any(const float* X, float* Y, int64_t rows, int64_t cols, hipStream_t st) {
    constexpr int ROWS = THREADS == WAVE ? 4 : 1;
    constexpr int64_t MOST = MAX_GRID_THREADS / (THREADS * ROWS) * ROWS;   // rows of one launch
    for (int64_t row = 0; row < rows; row += MOST) {
        const int64_t n = rows - row < MOST ? rows - row : MOST;
        hipLaunchKernelGGL((softmax_rows_any<THREADS, NV, LOG>), dim3((unsigned)ceil_div(n, (int64_t)ROWS)), dim3(THREADS * ROWS), 0, st,
                           X + row * cols, Y + row * cols, n, (int)cols);
    }
}

// Rows per lane group. Inputs of a few MB are one round trip to memory per CU and finish sooner the more
// workgroups share it (12288 rows of 128: 3.1 us with 2 rows per group, 3.6 us with 3, 4.4 us with 6, against
// 2.8 us for a plain copy of the same bytes and 1.8 us for an empty kernel); inputs that stream for many
// rounds run faster with three rows of loads in flight per lane.
template <int L, int NV, bool LOG>
static void launch_reg_unr(const float* X, float* Y, int64_t rows, int cols, hipStream_t st) {
    constexpr int groups = 256 / L;
    const bool streams = rows * (int64_t)cols * 4 >= ((int64_t)64 << 20);
    if (NV <= 2 && streams)
        launch_reg<L, NV, (NV <= 2 ? 3 : 1), LOG>(X, Y, rows, cols, st);
    else if (NV <= 2 && rows >= (int64_t)groups * 2 * 512)
        launch_reg<L, NV, (NV <= 2 ? 2 : 1), LOG>(X, Y, rows, cols, st);
    else
        launch_reg<L, NV, 1, LOG>(X, Y, rows, cols, st);
}

template <bool LOG>
static int softmax_dispatch(const float* X, float* Y, int64_t outer, int64_t axis_len, int64_t inner, void* stream) {
    MI355X_REQUIRE(outer >= 0 && axis_len >= 0 && inner >= 0,
                   "softmax: negative extent (outer=%lld axis_len=%lld inner=%lld)",
                   (long long)outer, (long long)axis_len, (long long)inner);
    if (outer == 0 || axis_len == 0 || inner == 0) return MI355X_OK;
    MI355X_REQUIRE(X != nullptr && Y != nullptr, "softmax: null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);

    if (inner == 1) {
        const int64_t rows = outer, cols = axis_len;
        MI355X_REQUIRE(rows < ((int64_t)1 << 31), "softmax: too many rows (%lld)", (long long)rows);
        const bool vec_ok = (cols % 4 == 0) && ((reinterpret_cast<uintptr_t>(X) & 15) == 0) &&
                            ((reinterpret_cast<uintptr_t>(Y) & 15) == 0);
        if (vec_ok && cols <= 64) launch_reg_unr<16, 1, LOG>(X, Y, rows, (int)cols, st);
        else if (vec_ok && cols <= 128) launch_reg_unr<32, 1, LOG>(X, Y, rows, (int)cols, st);
        else if (vec_ok && cols <= 256) launch_reg_unr<64, 1, LOG>(X, Y, rows, (int)cols, st);
        else if (vec_ok && cols <= 512) launch_reg_unr<64, 2, LOG>(X, Y, rows, (int)cols, st);
        else if (vec_ok && cols <= 1024) launch_reg_unr<64, 4, LOG>(X, Y, rows, (int)cols, st);
        else if (vec_ok && cols <= 2048) launch_reg_unr<64, 8, LOG>(X, Y, rows, (int)cols, st);
        else if (cols <= 64) launch_any<64, 1, LOG>(X, Y, rows, cols, st);
        else if (cols <= 128) launch_any<64, 2, LOG>(X, Y, rows, cols, st);
        else if (cols <= 256) launch_any<64, 4, LOG>(X, Y, rows, cols, st);
        else if (cols <= 512) launch_any<64, 8, LOG>(X, Y, rows, cols, st);
        else if (cols <= 2048) launch_any<256, 8, LOG>(X, Y, rows, cols, st);
        else if (cols <= 8192) launch_any<512, 16, LOG>(X, Y, rows, cols, st);
        else if (cols <= 32768) launch_any<1024, 32, LOG>(X, Y, rows, cols, st);
        else if (!grid_fits(rows, 1024)) return set_error(MI355X_ERR_INVALID_ARGUMENT, "softmax: too many rows (%lld)", (long long)rows);
        else hipLaunchKernelGGL(softmax_rows_loop<LOG>, dim3((unsigned)rows), dim3(1024), 0, st, X, Y, cols);
        return check_launch("softmax_rows");
    }
    const int64_t n = outer * inner;
    MI355X_REQUIRE(grid_fits(ceil_div(n, 256), 256), "softmax: grid too large");
    hipLaunchKernelGGL(softmax_strided<LOG>, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, st, X, Y,
                       outer, axis_len, inner);
    return check_launch("softmax_strided");
}

}  // namespace mi355x

extern "C" int mi355x_softmax_f32(const float* X, float* Y, int64_t outer, int64_t axis_len,
                                  int64_t inner, void* stream) {
    return mi355x::softmax_dispatch<false>(X, Y, outer, axis_len, inner, stream);
}

extern "C" int mi355x_log_softmax_f32(const float* X, float* Y, int64_t outer, int64_t axis_len,
                                      int64_t inner, void* stream) {
    return mi355x::softmax_dispatch<true>(X, Y, outer, axis_len, inner, stream);
}
