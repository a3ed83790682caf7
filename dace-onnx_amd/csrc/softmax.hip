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
//   softmax_rows_any<THREADS, NV>  last axis, any cols, cols / 4 <= THREADS*NV, no alignment asked
//       of a row: the row in the registers of one wave (THREADS = 64) or of one workgroup,
//       NV vectors of four floats per thread and the last cols % 4 one by one.
//   softmax_rows_short<NV>  last axis, cols <= 64*NV, no alignment asked of a row: one wave per row, single floats.
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
// Maxima in which NaN wins, as it does in ReduceMax; the probabilities of such a row are NaN either way.
__device__ __forceinline__ float maximum(float a, float b) { return __builtin_elementwise_maximum(a, b); }
__device__ __forceinline__ float maximum(const f32x4& v) { return maximum(maximum(v.x, v.y), maximum(v.z, v.w)); }
template <int L>
__device__ __forceinline__ float group_max(float v) {
    if constexpr (L == 16) return row16_max(v);
    else if constexpr (L == 32) return half32_max(v);
    else return wave_max(v);
}
template <int L>
__device__ __forceinline__ float group_maximum(float v) {
    v = maximum(v, dpp_f32<DPP_QUAD_XOR1>(v));
    v = maximum(v, dpp_f32<DPP_QUAD_XOR2>(v));
    v = maximum(v, dpp_f32<DPP_ROW_HALF_MIRROR>(v));
    v = maximum(v, dpp_f32<DPP_ROW_MIRROR>(v));
    if constexpr (L == 16) return v;
    const float lower = maximum(readlane_f32(v, 0), readlane_f32(v, 16)), upper = maximum(readlane_f32(v, 32), readlane_f32(v, 48));
    if constexpr (L == 32) return threadIdx.x & 32 ? upper : lower;
    return maximum(lower, upper);
}

template <int L, int NV, int UNR, bool LOG, bool MAX>
__global__ __launch_bounds__(256) void softmax_rows_reg(const float* __restrict__ X,
                                                        float* __restrict__ Y,
                                                        float* __restrict__ largest,
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
            m = MAX ? maximum(m, maximum(v[u][j])) : fmaxf(m, fmaxf(fmaxf(v[u][j].x, v[u][j].y), fmaxf(v[u][j].z, v[u][j].w)));
        m = MAX ? group_maximum<L>(m) : group_max<L>(m);
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
        if (MAX && row < rows && lane == 0) largest[row] = m;
    }
}

// Reduction over a workgroup of THREADS (the wave itself where THREADS is 64): `part` holds one value per wave.
template <int THREADS, bool MAX>
__device__ __forceinline__ float block_reduce(float v, float* part) {
    v = MAX ? group_maximum<WAVE>(v) : wave_sum(v);
    if constexpr (THREADS == WAVE) return v;
    constexpr int WAVES = THREADS / WAVE;
    __syncthreads();   // the previous reduction's values have been read
    if (threadIdx.x % WAVE == 0) part[threadIdx.x / WAVE] = v;
    __syncthreads();
    v = part[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) v = MAX ? maximum(v, part[w]) : v + part[w];
    return v;
}

// Bound by HBM: one read and one write. Rows of any length start at any multiple of four bytes; a 16-byte access at such an address
// costs a wave one cache line more. All of a row's loads are issued before the first reduction.
// `largest` (if not null) gets the largest value of each row, which is at hand.
template <int THREADS, int NV, bool LOG>
__global__ __launch_bounds__(THREADS == WAVE ? 256 : THREADS) void softmax_rows_any(const float* __restrict__ X, float* __restrict__ Y, float* __restrict__ largest,
                                                                                    int64_t rows, int cols) {
    typedef f32x4 unaligned __attribute__((aligned(4)));
    constexpr int ROWS = THREADS == WAVE ? 4 : 1;   // rows per workgroup
    __shared__ float part[THREADS / WAVE];
    const int t = threadIdx.x % THREADS;
    const int64_t row = (int64_t)blockIdx.x * ROWS + threadIdx.x / THREADS;
    if (row >= rows) return;  // a whole wave, and only where no barrier follows (ROWS > 1)
    const int cols4 = cols >> 2, last = (cols & ~3) + t;
    const float* x = X + row * cols;
    float* y = Y + row * cols;
    f32x4 v[NV];
#pragma unroll
    for (int j = 0; j < NV; ++j)
        v[j] = t + j * THREADS < cols4 ? f32x4(__builtin_nontemporal_load(reinterpret_cast<const unaligned*>(x) + t + j * THREADS))
                                       : f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
    float rest = last < cols ? __builtin_nontemporal_load(x + last) : -INFINITY;
    float m = rest;
#pragma unroll
    for (int j = 0; j < NV; ++j) m = maximum(m, maximum(v[j]));
    m = block_reduce<THREADS, true>(m, part);
    // columns beyond the row hold -inf: exp(-inf - m) adds nothing
    rest -= m;
    float s = expf(rest);
    if constexpr (!LOG) rest = s;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        v[j] -= m;
        const f32x4 e = {expf(v[j].x), expf(v[j].y), expf(v[j].z), expf(v[j].w)};
        s += (e.x + e.y) + (e.z + e.w);
        if constexpr (!LOG) v[j] = e;
    }
    s = block_reduce<THREADS, false>(s, part);
    const float inv = 1.0f / s, log_s = LOG ? logf(s) : 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (t + j * THREADS < cols4) __builtin_nontemporal_store(unaligned(LOG ? v[j] - log_s : v[j] * inv), reinterpret_cast<unaligned*>(y) + t + j * THREADS);
    if (last < cols) __builtin_nontemporal_store(LOG ? rest - log_s : rest * inv, y + last);
    if (largest && t == 0) largest[row] = m;
}

// Rows of at most 64 NV values with single floats, a row to a wave: a vector of four would leave most lanes idle.
// MAX: with the largest values (plain maxima go with the lane permutation in one instruction: [65536, 33] 12.7 us so, 10.2).
template <int NV, bool LOG, bool MAX>
__global__ __launch_bounds__(256) void softmax_rows_short(const float* __restrict__ X, float* __restrict__ Y, float* __restrict__ largest, int64_t rows, int cols) {
    const int t = threadIdx.x % WAVE;
    const int64_t row = (int64_t)blockIdx.x * 4 + threadIdx.x / WAVE;
    if (row >= rows) return;  // a whole wave
    const float* x = X + row * cols;
    float* y = Y + row * cols;
    float v[NV];
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < NV; ++j) v[j] = t + j * WAVE < cols ? __builtin_nontemporal_load(x + t + j * WAVE) : -INFINITY;
#pragma unroll
    for (int j = 0; j < NV; ++j) m = MAX ? maximum(m, v[j]) : fmaxf(m, v[j]);
    m = MAX ? group_maximum<WAVE>(m) : group_max<WAVE>(m);
    float s = 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        v[j] -= m;
        const float e = expf(v[j]);
        s += e;
        if constexpr (!LOG) v[j] = e;
    }
    s = wave_sum(s);
    const float inv = 1.0f / s, log_s = LOG ? logf(s) : 0.0f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (t + j * WAVE < cols) __builtin_nontemporal_store(LOG ? v[j] - log_s : v[j] * inv, y + t + j * WAVE);
    if (MAX && t == 0) largest[row] = m;
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
static void launch_reg(const float* X, float* Y, float* largest, int64_t rows, int cols, hipStream_t st) {
    constexpr int rows_per_block = (256 / L) * UNR;
    constexpr int64_t MOST = MAX_GRID_THREADS / 256 * rows_per_block;   // rows of one launch
    for (int64_t row = 0; row < rows; row += MOST) {
        const int64_t n = rows - row < MOST ? rows - row : MOST;
        const dim3 grid((unsigned)ceil_div(n, (int64_t)rows_per_block));
        if (!LOG && largest) hipLaunchKernelGGL((softmax_rows_reg<L, NV, UNR, LOG, !LOG>), grid, dim3(256), 0, st, X + row * cols, Y + row * cols, largest + row, n, cols);
        else hipLaunchKernelGGL((softmax_rows_reg<L, NV, UNR, LOG, false>), grid, dim3(256), 0, st, X + row * cols, Y + row * cols, nullptr, n, cols);
    }
}

template <int THREADS, int NV, bool LOG>
static void launch_any(const float* X, float* Y, float* largest, int64_t rows, int64_t cols, hipStream_t st) {
    constexpr int ROWS = THREADS == WAVE ? 4 : 1;
    constexpr int64_t MOST = MAX_GRID_THREADS / (THREADS == WAVE ? 256 : THREADS) * ROWS;   // rows of one launch
    for (int64_t row = 0; row < rows; row += MOST) {
        const int64_t n = rows - row < MOST ? rows - row : MOST;
        hipLaunchKernelGGL((softmax_rows_any<THREADS, NV, LOG>), dim3((unsigned)ceil_div(n, (int64_t)ROWS)), dim3(THREADS == WAVE ? 256 : THREADS), 0, st,
                           X + row * cols, Y + row * cols, largest ? largest + row : nullptr, n, (int)cols);
    }
}

// Rows per lane group. Inputs of a few MB are one round trip to memory per CU and finish sooner the more
// workgroups share it (12288 rows of 128: 3.1 us with 2 rows per group, 3.6 us with 3, 4.4 us with 6, against
// 2.8 us for a plain copy of the same bytes and 1.8 us for an empty kernel); inputs that stream for many
// rounds run faster with three rows of loads in flight per lane.
template <int L, int NV, bool LOG>
static void launch_reg_unr(const float* X, float* Y, float* largest, int64_t rows, int cols, hipStream_t st) {
    constexpr int groups = 256 / L;
    const bool streams = rows * (int64_t)cols * 4 >= ((int64_t)64 << 20);
    if (NV <= 2 && streams)
        launch_reg<L, NV, (NV <= 2 ? 3 : 1), LOG>(X, Y, largest, rows, cols, st);
    else if (NV <= 2 && rows >= (int64_t)groups * 2 * 512)
        launch_reg<L, NV, (NV <= 2 ? 2 : 1), LOG>(X, Y, largest, rows, cols, st);
    else
        launch_reg<L, NV, 1, LOG>(X, Y, largest, rows, cols, st);
}

template <int NV, bool LOG>
static void launch_short(const float* X, float* Y, float* largest, int64_t rows, int64_t cols, hipStream_t st) {
    constexpr int64_t MOST = MAX_GRID_THREADS / 256 * 4;   // rows of one launch
    for (int64_t row = 0; row < rows; row += MOST) {
        const int64_t n = rows - row < MOST ? rows - row : MOST;
        const dim3 grid((unsigned)ceil_div(n, (int64_t)4));
        if (!LOG && largest) hipLaunchKernelGGL((softmax_rows_short<NV, LOG, !LOG>), grid, dim3(256), 0, st, X + row * cols, Y + row * cols, largest + row, n, (int)cols);
        else hipLaunchKernelGGL((softmax_rows_short<NV, LOG, false>), grid, dim3(256), 0, st, X + row * cols, Y + row * cols, nullptr, n, (int)cols);
    }
}

// Rows of up to 32768 values at any address. Single floats and one wave up to 512 ([65536, 33] 10.2 us, with vectors 15.8; [9001, 403] 6.3 and 6.5), vectors
// above: [20000, 517] 25.6 -> 16.2 us, [8000, 2051] 34.7 -> 22.6, LogSoftmax [2048, 12345] 63 -> 38, [1024, 30522] 62.9 -> 48 (5.2 TB/s; 50 with
// 1024 threads for a row). As many waves as leave a thread 16 to 64 values; fewer for a row of 2052 to 4099 ([100, 4093] 3.8 -> 3.3).
template <bool LOG>
static void launch_any_row(const float* X, float* Y, float* largest, int64_t rows, int64_t cols, hipStream_t st) {
    if (cols <= 64) launch_short<1, LOG>(X, Y, largest, rows, cols, st);
    else if (cols <= 128) launch_short<2, LOG>(X, Y, largest, rows, cols, st);
    else if (cols <= 256) launch_short<4, LOG>(X, Y, largest, rows, cols, st);
    else if (cols <= 512) launch_short<8, LOG>(X, Y, largest, rows, cols, st);
    else if (cols < 1028) launch_any<64, 4, LOG>(X, Y, largest, rows, cols, st);
    else if (cols < 2052) launch_any<256, 2, LOG>(X, Y, largest, rows, cols, st);
    else if (cols < 4100) launch_any<256, 4, LOG>(X, Y, largest, rows, cols, st);
    else if (cols < 8196) launch_any<512, 4, LOG>(X, Y, largest, rows, cols, st);
    else if (cols < 16388) launch_any<512, 8, LOG>(X, Y, largest, rows, cols, st);
    else launch_any<512, 16, LOG>(X, Y, largest, rows, cols, st);
}

template <bool LOG>
static int softmax_dispatch(const float* X, float* Y, float* largest, int64_t outer, int64_t axis_len, int64_t inner, void* stream) {
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
        if (vec_ok && cols <= 64) launch_reg_unr<16, 1, LOG>(X, Y, largest, rows, (int)cols, st);
        else if (vec_ok && cols <= 128) launch_reg_unr<32, 1, LOG>(X, Y, largest, rows, (int)cols, st);
        else if (vec_ok && cols <= 256) launch_reg_unr<64, 1, LOG>(X, Y, largest, rows, (int)cols, st);
        else if (vec_ok && cols <= 512) launch_reg_unr<64, 2, LOG>(X, Y, largest, rows, (int)cols, st);
        else if (vec_ok && cols <= 1024) launch_reg_unr<64, 4, LOG>(X, Y, largest, rows, (int)cols, st);
        else if (vec_ok && cols <= 2048) launch_reg_unr<64, 8, LOG>(X, Y, largest, rows, (int)cols, st);
        else if (cols <= 32768) launch_any_row<LOG>(X, Y, largest, rows, cols, st);
        else if (!grid_fits(rows, 1024)) return set_error(MI355X_ERR_INVALID_ARGUMENT, "softmax: too many rows (%lld)", (long long)rows);
        else {
            hipLaunchKernelGGL(softmax_rows_loop<LOG>, dim3((unsigned)rows), dim3(1024), 0, st, X, Y, cols);
            const int status = check_launch("softmax_rows_loop");
            return status == MI355X_OK && largest ? mi355x_reduce_f32(MI355X_REDUCE_MAX, X, largest, rows, cols, 1, stream) : status;
        }
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
    return mi355x::softmax_dispatch<false>(X, Y, nullptr, outer, axis_len, inner, stream);
}

extern "C" int mi355x_log_softmax_f32(const float* X, float* Y, int64_t outer, int64_t axis_len,
                                      int64_t inner, void* stream) {
    return mi355x::softmax_dispatch<true>(X, Y, nullptr, outer, axis_len, inner, stream);
}

extern "C" int mi355x_softmax_max_f32(const float* X, float* Y, float* largest, int64_t rows, int64_t cols, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(rows >= 0 && cols >= 1, "softmax_max: %lld rows of %lld", (long long)rows, (long long)cols);
    MI355X_REQUIRE(rows == 0 || largest, "softmax_max: null pointer");
    return softmax_dispatch<false>(X, Y, largest, rows, cols, 1, stream);
}
