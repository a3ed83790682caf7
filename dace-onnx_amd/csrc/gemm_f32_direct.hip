// fp32 GEMM for outputs of few tiles: operands straight from memory into registers, K split over the sixteen waves of a workgroup.
//
// A product of a few rows (one sentence, a few samples) is bound by the latency of its operand loads: the kernels that stage tiles
// through LDS walk K step by step, a barrier each, on 16 to 64 workgroups. Here a workgroup owns 16 TM x 16 TN outputs, each of its
// waves takes a sixteenth of K with RING chunks of 16 k in flight and no barrier, and the partial sums meet in LDS once, in the
// order of the waves. A lane (li, lq) holds k = 16 c + 4 lq .. + 3 of both operands, so one 16-byte load along k feeds four MFMA
// steps; B contiguous along n is read as 16 bytes along n, four columns of a lane being its columns of the four accumulators.
// Any extent, stride and 4-byte alignment: rows past the end are clamped, the last k-vector is moved back into the row and the
// values it holds twice are zeroed.
#include "common.h"
#include "gemm_tile.h"
#include "gemm_args.h"

namespace mi355x {

constexpr int GD_WAVES = 16;

// B_KC: B contiguous along k, columns n0 + 16 j + li. Otherwise along n, TN = 4: columns n0 + 4 li + j.
// SOFTMAX: N <= 16, the end of a classifier of few classes: the sixteen lanes that hold a row's results make its probabilities of them, and the launch
// that would read them again (2.3 us and 3 of the host's for 5 x 10) is left out.
template <int TM, int TN, bool B_KC, bool SOFTMAX = false>
__global__ __launch_bounds__(WAVE * GD_WAVES) void gemm_f32_direct_kernel(GemmArgs p) {
    static_assert(B_KC || TN == 4, "one 16-byte load along n is four columns");
    static_assert(!SOFTMAX || (TM == 1 && TN == 1 && B_KC), "whole rows in a tile");
    constexpr int TILES = TM * TN;
    constexpr int RING = TILES >= 8 ? 2 : B_KC ? 4 : 3;
    constexpr int NB = B_KC ? TN : 4;
    __shared__ __attribute__((aligned(16))) f32x4 red[GD_WAVES][TILES][WAVE];

    const int tid = threadIdx.x, lane = tid % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int li = lane % 16, lq = lane / 16;
    // consecutive tiles walk down M: the XCD that reads a strip of B uses it for all of its rows
    const uint32_t logical = (uint32_t)xcd_remap(blockIdx.x, p.nwg);
    const uint32_t tiles_m = (uint32_t)p.tiles_m, per_batch = tiles_m * (uint32_t)p.tiles_n;
    const uint32_t b = logical / per_batch, t = logical % per_batch;
    const int64_t b0 = b / (uint32_t)p.batch1, b1 = b % (uint32_t)p.batch1;
    const int m0 = (int)(t % tiles_m) * 16 * TM, n0 = (int)(t / tiles_m) * 16 * TN;
    const int M = (int)p.M, N = (int)p.N, K = (int)p.K;

    // raw buffers of 2^31 - 1 bytes (launch precondition: a matrix spans less): an offset with bit 31 set loads zeros
    const __amdgpu_buffer_rsrc_t a_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.A + b0 * p.a_sb0 + b1 * p.a_sb1), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t b_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.B + b0 * p.b_sb0 + b1 * p.b_sb1), 0, 0x7fffffff, 0x00020000);
    uint32_t a_row[TM], b_row[B_KC ? TN : 1];
#pragma unroll
    for (int i = 0; i < TM; ++i) a_row[i] = 4u * (uint32_t)min(m0 + 16 * i + li, M - 1) * (uint32_t)p.a_sm;
    if constexpr (B_KC) {
#pragma unroll
        for (int j = 0; j < TN; ++j) b_row[j] = 4u * (uint32_t)min(n0 + 16 * j + li, N - 1) * (uint32_t)p.b_sn;
    } else {
        b_row[0] = 4u * (uint32_t)min(n0 + 4 * li, N - 4);
    }
    const uint32_t b_sk = 4u * (uint32_t)p.b_sk;

    // the outputs this thread adds up at the end: rows of tile (ti, tj), one column; its bias and residual values set out now
    const int tile = tid / WAVE;
    const bool sums = tile < TILES;
    const int om = m0 + 16 * (tile / TN) + 4 * lq;
    const int first = n0 + (B_KC ? 16 * (tile % TN) + li : 4 * li);
    const int on = B_KC ? first : min(first, N - 4) + tile % TN;
    const bool stored = sums && on >= first && on < N;   // (a column block moved back repeats columns of the one before it)
    float bias = 0.f, res[4] = {0.f, 0.f, 0.f, 0.f};
    if (stored) {
        if (p.epi & MI355X_EPI_BIAS) bias = p.bias[on];
        if (p.epi & MI355X_EPI_RESIDUAL) {
            const float* R = p.residual + b0 * p.r_sb0 + b1 * p.r_sb1 + on;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (om + r < M) res[r] = R[(int64_t)(om + r) * p.r_sm];
        }
    }

    const int chunks = (K + 15) / 16, per_wave = (chunks + GD_WAVES - 1) / GD_WAVES;
    const int begin = wave * per_wave, end = min(begin + per_wave, chunks);

    f32x4 va[RING][TM], vb[RING][NB];
    auto load = [&](int slot, int c) {
        const int k = 16 * c + 4 * lq;
        const uint32_t kb = (uint32_t)min(k, K - 4);
        const uint32_t outside = k >= K ? 0x80000000u : 0u;
#pragma unroll
        for (int i = 0; i < TM; ++i)
            va[slot][i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, (int)((a_row[i] + 4u * kb) | outside), 0, 0));
#pragma unroll
        for (int j = 0; j < NB; ++j)
            vb[slot][j] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
                b_rsrc, (int)((B_KC ? b_row[j < TN && B_KC ? j : 0] + 4u * kb : b_row[0] + (kb + (uint32_t)j) * b_sk) | outside), 0, 0));
    };

    f32x4 acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int slot, int c) {
        if (16 * c + 16 > K && K % 4 != 0) {   // uniform; the vector that was moved back holds values of the one before it
            const int k = 16 * c + 4 * lq, kb = min(k, K - 4);
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const bool own = kb + s >= k;
#pragma unroll
                for (int i = 0; i < TM; ++i) va[slot][i][s] = own ? va[slot][i][s] : 0.f;
#pragma unroll
                for (int j = 0; j < NB; ++j) {
                    if constexpr (B_KC) vb[slot][j][s] = own ? vb[slot][j][s] : 0.f;
                    else if (j == s && !own) vb[slot][j] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
            }
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[slot][i][s], B_KC ? vb[slot][j][s] : vb[slot][s][j], acc[i][j], 0, 0, 0);
    };

#pragma unroll
    for (int u = 0; u < RING; ++u)
        if (begin + u < end) load(u, begin + u);
    for (int c = begin; c < end; c += RING) {
        static_for<RING>([&](auto u) {
            if (c + u < end) multiply(u, c + u);
            if (c + u + RING < end) load(u, c + u + RING);   // (uniform; a load that is all out of range costs the address unit as much as any)
        });
    }

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) red[wave][i * TN + j][lane] = acc[i][j];
    __syncthreads();
    if (SOFTMAX ? !sums : !stored) return;   // (a whole wave where its lanes go on together)
    f32x4 v = red[0][tile][lane];
#pragma unroll
    for (int w = 1; w < GD_WAVES; ++w) v += red[w][tile][lane];
    if constexpr (SOFTMAX) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float x = stored ? apply_epilogue(v[r] * p.alpha, p.epi, bias) : -INFINITY;
            const float e = expf(x - row16_max(x)), s = row16_sum(e);   // (e of a column that is not there: 0)
            if (stored && om + r < M) p.C[(int64_t)(om + r) * N + on] = e * (1.0f / s);
        }
        return;
    }
    float* C = p.C + b0 * p.c_sb0 + b1 * p.c_sb1 + on;
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (om + r < M) {
            const float o = apply_epilogue(v[r] * p.alpha, p.epi, bias);
            C[(int64_t)(om + r) * p.c_sm] = (p.epi & MI355X_EPI_RESIDUAL) ? o + res[r] : o;
        }
}

// Nanoseconds, from sweeps over M of 1 to 512, N of 256 to 30522 and K of 256 to 3072 with weights that are not in the L2: a launch,
// the first loads and the sum over the waves (`fixed`), then per k while every workgroup has a CU to itself (`alone`). More
// workgroups than CUs run in rounds (one workgroup fills a CU's LDS), each with first loads and a sum of its own (`again`) and `round`
// per k. Without `again` stacks of products over a short K came here and took two or three times as long: 200 x (2666 x 141 x 11) 189
// -> 599 us, 512 x (5 x 1600 x 32) 79 -> 148, 96 x (1849 x 840 x 238) 1179 -> 1415. Beyond eight rounds the fit is up to 15 % low
// where rows are at odd addresses (96 x (512 x 238 x 1347) 531 us as 128 x 64 tiles, 650 here), which the rule then adds. Over 459
// shapes of 1 to 1200 rounds and K of 4 to 4096 it picks no kernel that is more than 4 % behind the one before this file, and is 1.6 %
// behind the best pick on average.
// A CU draws 30 to 40 bytes a nanosecond whatever the form, which is the bound: 16 x 768 x 768 5.7 us (64 x 48 tiles through LDS
// 13.1), 16 x 768 x 3072 13.6 (36.1), 128 x 768 x 768 7.3 (13.7), 128 x 768 x 3072 19.0 (36.2), 256 x 768 x 3072 25.8 (36.4),
// 33 x 1000 x 1503 8.7 (44.6), 16 x 30522 x 768 with B along n 19.2 (31.6); 128 x 2304 x 768 17.1 (13.9) stays where it was.
// (Loads past a wave's share, which a branch now skips, were up to half of the time: 16 x 768 x 768 6.9 us with them. 32 x 16
// tiles equal 16 x 32; 64 x 32 and 32 x 64 tiles are never ahead; both halves of a 128-byte line by one pair of loads changes nothing.)
struct DirectForm { int tm, tn; bool b_kc; double fixed, alone, again, round; };
static const DirectForm kDirectForms[] = {{1, 1, true, 3100, 3.4, 980, 2.4}, {1, 2, true, 3400, 5.0, 1400, 4.5}, {2, 2, true, 3800, 7.1, 2350, 6.8},
                                          {1, 4, false, 3500, 5.8, 1650, 5.6}, {2, 4, false, 4000, 8.0, 3050, 9.1}};

// The fastest form below `best_cost` (which becomes its time), -1 where there is none.
static int choose_direct(const GemmArgs& p, bool b_kc, int force, int cus, double& best_cost) {
    if (force == 0 || p.K < 4 || (!b_kc && p.N < 4)) return -1;
    if (p.a_sm < 0 || p.b_sn < 0 || p.b_sk < 0 || p.M >= ((int64_t)1 << 29) || p.N >= ((int64_t)1 << 29) ||
        (p.M - 1) * p.a_sm + p.K >= ((int64_t)1 << 29) || (p.N - 1) * p.b_sn + (p.K - 1) * p.b_sk + 1 >= ((int64_t)1 << 29)) return -1;
    int best = -1;
    for (int f = 0; f < 5; ++f) {
        const DirectForm& form = kDirectForms[f];
        if (form.b_kc != b_kc) continue;
        const int64_t nwg = p.batch * ceil_div(p.M, (int64_t)16 * form.tm) * ceil_div(p.N, (int64_t)16 * form.tn);
        const int64_t rounds = ceil_div(nwg, (int64_t)cus);
        const double many = rounds > 8 ? 1.15 : 1.0;
        const double cost = form.fixed + (rounds <= 1 ? form.alone * (double)p.K : many * (form.again * (double)(rounds - 1) + form.round * (double)p.K * (double)rounds));
        if (force > 0 ? force == 10 * form.tm + form.tn : cost < best_cost) { best = f; best_cost = cost; }
    }
    return best;
}

double gemm_f32_direct_cost(const GemmArgs& p, bool b_kc, int cus) {
    double cost = 1e300;
    choose_direct(p, b_kc, -1, cus, cost);
    return cost;
}

bool launch_gemm_f32_direct(GemmArgs p, bool b_kc, double other_cost, int cus, hipStream_t stream) {
    double best_cost = 0.95 * other_cost;
    const int best = choose_direct(p, b_kc, tuning().gemm_direct, cus, best_cost);
    if (best < 0) return false;
    p.tiles_m = ceil_div(p.M, (int64_t)16 * kDirectForms[best].tm);
    p.tiles_n = ceil_div(p.N, (int64_t)16 * kDirectForms[best].tn);
    p.nwg = p.batch * p.tiles_m * p.tiles_n;
    if (!grid_fits(p.nwg, WAVE * GD_WAVES)) return false;
    const dim3 grid((unsigned)p.nwg), block(WAVE * GD_WAVES);
    if (best == 0) hipLaunchKernelGGL((gemm_f32_direct_kernel<1, 1, true>), grid, block, 0, stream, p);
    else if (best == 1) hipLaunchKernelGGL((gemm_f32_direct_kernel<1, 2, true>), grid, block, 0, stream, p);
    else if (best == 2) hipLaunchKernelGGL((gemm_f32_direct_kernel<2, 2, true>), grid, block, 0, stream, p);
    else if (best == 3) hipLaunchKernelGGL((gemm_f32_direct_kernel<1, 4, false>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((gemm_f32_direct_kernel<2, 4, false>), grid, block, 0, stream, p);
    return true;
}

}  // namespace mi355x

// Up to 4096 rows: as many workgroups as CUs, which the kernel for few tiles is made for. Against the two launches, 245 products of 1 to 4096 rows, 1 to 16
// classes and a K of 4 to 8192: 0.54 to 0.96 of their time (4096 x 1 x 16 7.4 -> 4.0 us, 5 x 16 x 3072 11.6 -> 10.7, 4096 x 16 x 8192 33.5 -> 32.1).
extern "C" int mi355x_gemm_softmax_pays(int64_t M, int64_t N, int64_t K, int b_kc) { return M > 0 && M <= 4096 && N > 0 && N <= 16 && K >= 4 && b_kc; }

extern "C" int mi355x_gemm_softmax_f32(const float* A, const float* B, const float* bias, float* scratch, float* Y, int64_t M, int64_t N, int64_t K,
                                       int64_t a_row_stride, int64_t b_k_stride, int64_t b_column_stride, float alpha, int epilogue, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(M >= 0 && N >= 0 && K >= 0, "gemm_softmax: negative extent (M=%lld N=%lld K=%lld)", (long long)M, (long long)N, (long long)K);
    MI355X_REQUIRE((epilogue & ~(MI355X_EPI_BIAS | MI355X_EPI_RELU | MI355X_EPI_GELU)) == 0, "gemm_softmax: unknown epilogue bits 0x%x", epilogue);
    MI355X_REQUIRE(!(epilogue & MI355X_EPI_BIAS) || bias, "gemm_softmax: MI355X_EPI_BIAS without bias");
    if (M == 0 || N == 0) return MI355X_OK;
    if (A && B && Y && a_row_stride >= 0 && b_column_stride >= 0 && mi355x_gemm_softmax_pays(M, N, K, b_k_stride == 1) &&
        (M - 1) * a_row_stride + K < ((int64_t)1 << 29) && (N - 1) * b_column_stride + K < ((int64_t)1 << 29)) {
        GemmArgs p = {};
        MI355X_TRACE_INIT(p);
        p.A = A; p.B = B; p.C = Y; p.bias = bias;
        p.batch = p.batch1 = 1; p.M = M; p.N = N; p.K = K;
        p.a_sm = a_row_stride; p.a_sk = 1; p.b_sk = 1; p.b_sn = b_column_stride; p.c_sm = N;
        p.alpha = alpha; p.epi = epilogue;
        p.tiles_m = ceil_div(M, (int64_t)16); p.tiles_n = 1; p.nwg = p.tiles_m;
        hipLaunchKernelGGL((gemm_f32_direct_kernel<1, 1, true, true>), dim3((unsigned)p.nwg), dim3(WAVE * GD_WAVES), 0, static_cast<hipStream_t>(stream), p);
        return check_launch("gemm_f32_direct_kernel");
    }
    const int64_t a[4] = {0, 0, a_row_stride, 1}, b[4] = {0, 0, b_k_stride, b_column_stride}, c[3] = {0, 0, N};
    const int status = mi355x_gemm_f32(A, B, scratch, bias, nullptr, 1, 1, M, N, K, a, b, c, nullptr, alpha, epilogue, stream);
    return status != MI355X_OK ? status : mi355x_softmax_f32(scratch, Y, M, N, 1, stream);
}
