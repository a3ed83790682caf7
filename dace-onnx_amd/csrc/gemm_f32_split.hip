// fp32 GEMM on the bf16 matrix unit: every operand value is split into three bf16 numbers on its way into LDS.
//
// The fp32 MFMA of this part delivers 157 TFLOP/s, the bf16 one 2500. A float has 24 significant bits, a bf16 eight, so
// x = hi + mid + lo (round to nearest, subtract, round again), exactly: values are multiplied by 2^16 before they are split, so that
// the last bit of the smallest float, 2^-149, is the smallest bf16 subnormal, 2^-133 (the MFMA takes subnormals as they are), and
// sums by 2^-32 after. Split as they came, values below 2^-110 lost bits: against values that bring the sums back to ordinary size
// 3.5e-5 (2-norm) at 2^-120 and everything below 2^-136, where 1.6e-7 is left now; the two multiplications of a pair cost
// 1 to 4 %, and 12 % where 64 x 64 tiles come two to a CU (12 x (675 x 160 x 1472): 48.9 -> 54.8 us).
// Of the nine products of two split values the six that reach 2^-24 of the result are
// multiplied, each exact in the fp32 accumulator of the MFMA: hi hi in one set of accumulators, the five small ones in a
// second set, added at the end, so the long sum takes K / 32 roundings where the fp32 MFMA takes K / 4. Against float64 over
// N(0, 1) operands the result is closer than the fp32 kernels': 1.6e-7 against 5.0e-7 (2-norm) at K = 768, 3.4e-7 against
// 7.1e-7 at K = 3072; with one set of accumulators it was 4.2e-7 and 8.7e-7. The three products left out show where a sum has few
// terms: a single product is off by up to 1.0e-7, the rounded product of two floats by 6e-8.
//
// Infinities, NaN, values from 2^112 and sums from 2^96 on make a sum of the split form NaN or infinite whatever the exact
// product is. A wave whose sums are not all finite computes its part of the tile again with the fp32 MFMA, straight from
// global memory: the result of such inputs is that of the fp32 kernels, only slower.
//
// What bounds it: MFMA and LDS traffic of about the same length that hardly overlap. Per 32-k step of a 256 x 128 tile a SIMD issues
// 3072 cycles of MFMA, and the CU 192 fragment reads (8 cycles each) and 72 plane writes (16 cycles each, whatever the width), 2688
// cycles of LDS; the sum of both is the time. Measured on 8192 x 1024 x 3072 (245 us, 211 TFLOP/s): without the reads 205 us,
// without the writes 221 us, without the splitting arithmetic 238 us, without the global loads 240 us.
//
//   * operand tile in LDS: three planes of 16-byte units (eight k of one row) in the order the MFMA reads them. The eight k
//     of a unit are {4 g .. 4 g + 3, 16 + 4 g .. 16 + 4 g + 3}: with that order four neighbouring lanes load 64 contiguous bytes
//     of a row and a unit is still one LDS write (A and B agree on it, and the order of a sum's terms is free).
//   * units of a row are spread over the banks by xor-ing the row with 0, 12, 4, 8 for g = 0..3: reads and writes without
//     conflicts (a rotation by 4 g cost 4 extra cycles per read).
//   * 256 x 128 tiles (eight waves, two LDS stages, the splitting and the LDS traffic placed between the MFMAs) where they
//     fill the chip; 128 x 64 and 64 x 64 tiles with one stage, three and four workgroups to a CU, where they do not: there
//     another workgroup's MFMAs cover the loads, the splitting and the barriers.
//   * B may be contiguous along k (weights [N, K]) or along n (weights as ONNX stores them, any N): in the second case a
//     lane owns a column and loads its eight k one float at a time, neighbouring lanes on neighbouring columns.
#include "common.h"
#include "gemm_tile.h"
#include "gemm_args.h"
#include "split_bf16.h"

#include <algorithm>

namespace mi355x {

constexpr int SP_BK = 32, SP_FRAGMENT = 1024;   // k extent of a tile; bytes of one plane of 16 rows

// byte offset of unit g (0..3) of row r (0..15) inside a fragment
__device__ __forceinline__ int split_unit(int r, int g) {
    return (16 * g + (r ^ (g == 1 ? 12 : g == 2 ? 4 : g == 3 ? 8 : 0))) * 16;
}

// One thread's share of a ROWS x 32 operand tile: global -> registers -> three LDS planes.
template <int ROWS, int THREADS, bool KC>
struct SplitTile {
    static constexpr int PER_T = ROWS * (SP_BK / 8) / THREADS, PLANE = ROWS * SP_BK * 2;
    static constexpr int LOADS = PER_T * (KC ? 2 : 8), WRITES = PER_T * SP_PLANES, VALU = PER_T * 52;   // per thread and tile
    static_assert(ROWS * (SP_BK / 8) % THREADS == 0, "whole units per thread");

    f32x4 v[PER_T][2];
    uint32_t off[PER_T];
    int lds[PER_T];

    __device__ __forceinline__ void init(int tid, int64_t row0, int64_t rows, int64_t s_row, int64_t s_k) {
#pragma unroll
        for (int it = 0; it < PER_T; ++it) {
            const int idx = tid + it * THREADS;
            const int row = KC ? idx / 4 : idx % ROWS, g = KC ? idx % 4 : idx / ROWS;
            int64_t r = row0 + row;
            r = r < rows ? r : rows - 1;   // rows beyond the matrix are computed on its last row and not stored
            off[it] = (uint32_t)(r * s_row + 4 * g * s_k) * 4u;
            lds[it] = (row / 16) * SP_FRAGMENT + split_unit(row % 16, g);
        }
    }
    __device__ __forceinline__ void load(__amdgpu_buffer_rsrc_t rsrc, int it, int kt, uint32_t s_k) {
        const uint32_t base = (uint32_t)kt * (uint32_t)(SP_BK * 4) * (KC ? 1u : s_k);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (KC) {
                v[it][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)(off[it] + 64u * h), (int)base, 0));
            } else {
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    v[it][h][s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        rsrc, (int)off[it], (int)(base + (uint32_t)(16 * h + s) * 4u * s_k), 0));
            }
        }
    }
    __device__ __forceinline__ void store(char* planes, int it) const {
        u32x4 part[SP_PLANES];
        split_unit8(v[it][0], v[it][1], part);
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q) *reinterpret_cast<u32x4*>(planes + q * PLANE + lds[it]) = part[q];
    }
};

// WAVES_M x WAVES_N waves of (16 TM) x (16 TN) outputs each; PER_SIMD: waves a SIMD has to hold.
template <int TM, int TN, int WAVES_M, int WAVES_N, int STAGES, int PER_SIMD, bool B_KC>
__global__ __launch_bounds__(WAVES_M * WAVES_N * WAVE, PER_SIMD) void gemm_f32_split_kernel(GemmArgs p) {
    constexpr int THREADS = WAVES_M * WAVES_N * WAVE, BM = 16 * TM * WAVES_M, BN = 16 * TN * WAVES_N;
    using TileA = SplitTile<BM, THREADS, true>;
    using TileB = SplitTile<BN, THREADS, B_KC>;
    constexpr int B_AT = SP_PLANES * TileA::PLANE, STAGE = SP_PLANES * (TileA::PLANE + TileB::PLANE);
    __shared__ __attribute__((aligned(16))) char lds[STAGES * STAGE];

    const int tid = threadIdx.x, lane = tid % WAVE, wave = tid / WAVE;
    const int li = lane % 16, lq = lane / 16;
    const int wm = wave % WAVES_M, wn = wave / WAVES_M;

    const int64_t logical = xcd_remap(blockIdx.x, p.nwg);
    const uint32_t tiles_per_batch = (uint32_t)(p.tiles_m * p.tiles_n);
    const uint32_t b = (uint32_t)logical / tiles_per_batch, t = (uint32_t)logical % tiles_per_batch;
    const int64_t b0 = b / (uint32_t)p.batch1, b1 = b % (uint32_t)p.batch1;
    int64_t tm, tn;
    tile_coords(t, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
    const int64_t m0 = tm * BM, n0 = tn * BN;

    // operands as raw buffers with 32-bit offsets (launch precondition: a matrix spans less than 2^31 bytes)
    const float* A = p.A + b0 * p.a_sb0 + b1 * p.a_sb1;
    const float* B = p.B + b0 * p.b_sb0 + b1 * p.b_sb1;
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(B), 0, 0x7fffffff, 0x00020000);
    const uint32_t b_sk = (uint32_t)p.b_sk;
    TileA ta;
    TileB tb;
    ta.init(tid, m0, p.M, p.a_sm, 1);
    tb.init(tid, n0, p.N, p.b_sn, p.b_sk);

    f32x4 acc[TM][TN], small[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) acc[i][j] = small[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int last = (int)(p.K / SP_BK) - 1;   // K % 32 == 0 is a launch precondition; look-aheads are clamped to the last tile
    auto multiply = [&](const char* stage) {
        const int at = split_unit(li, lq);
        bf16x8 fa[SP_PLANES][TM], fb[SP_PLANES][TN];
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
                fa[q][i] = *reinterpret_cast<const bf16x8*>(stage + q * TileA::PLANE + (wm * TM + i) * SP_FRAGMENT + at);
#pragma unroll
            for (int j = 0; j < TN; ++j)
                fb[q][j] = *reinterpret_cast<const bf16x8*>(stage + B_AT + q * TileB::PLANE + (wn * TN + j) * SP_FRAGMENT + at);
        }
        // (in the two-stage form the products that need the first planes come first: the later planes are read under them)
        constexpr bool FIRST = STAGES == 2;
        constexpr int QA[6] = {FIRST ? 0 : 2, 0, 1, FIRST ? 1 : 0, FIRST ? 0 : 1, FIRST ? 2 : 0};
        constexpr int QB[6] = {0, FIRST ? 1 : 2, FIRST ? 0 : 1, 1, FIRST ? 2 : 0, 0};
#pragma unroll
        for (int s = 0; s < 6; ++s)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    f32x4& sum = QA[s] + QB[s] > 0 ? small[i][j] : acc[i][j];
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[QA[s]][i], fb[QB[s]][j], sum, 0, 0, 0);
                }
    };
    // registers -> a stage, and the registers filled again with tile kt, unit by unit
    auto store = [&](char* stage, int kt) {
        kt = kt < last ? kt : last;
#pragma unroll
        for (int it = 0; it < TileA::PER_T; ++it) {
            ta.store(stage, it);
            if constexpr (STAGES == 2) ta.load(a_rsrc, it, kt, 1);
        }
#pragma unroll
        for (int it = 0; it < TileB::PER_T; ++it) {
            tb.store(stage + B_AT, it);
            if constexpr (STAGES == 2) tb.load(b_rsrc, it, kt, b_sk);
        }
    };
    auto load = [&](int kt) {
        kt = kt < last ? kt : last;
#pragma unroll
        for (int it = 0; it < TileA::PER_T; ++it) ta.load(a_rsrc, it, kt, 1);
#pragma unroll
        for (int it = 0; it < TileB::PER_T; ++it) tb.load(b_rsrc, it, kt, b_sk);
    };

    load(0);
    store(lds, 1);
    if constexpr (STAGES == 1) {
        for (int kt = 0; kt <= last; ++kt) {
            load(kt + 1);
            __syncthreads();
            multiply(lds);
            __syncthreads();
            store(lds, 0);
        }
    } else {
        for (int kt = 0; kt <= last; ++kt) {
            __syncthreads();   // stage kt is written, and everyone has read the stage that kt + 1 goes to
            store(lds + ((kt + 1) & 1) * STAGE, kt + 2);
            multiply(lds + (kt & 1) * STAGE);
            // issue order: the fragments of the first product, then everything else between the MFMAs
            constexpr int MFMA = 0x008, VALU = 0x002, VMEM_RD = 0x020, DS_RD = 0x100, DS_WR = 0x200;
            constexpr int NM = 6 * TM * TN, NV = TileA::VALU + TileB::VALU, NW = TileA::WRITES + TileB::WRITES;
            constexpr int NL = TileA::LOADS + TileB::LOADS, NRD = 2 * (TM + TN), SPAN = NM * 2 / 3;
            __builtin_amdgcn_sched_group_barrier(DS_RD, TM + TN, 0);
            static_for<NM>([&](auto q_tag) {
                constexpr int q = decltype(q_tag)::value;
                __builtin_amdgcn_sched_group_barrier(MFMA, 1, 0);
                __builtin_amdgcn_sched_group_barrier(VALU, (q + 1) * NV / NM - q * NV / NM, 0);
                if constexpr (q < SPAN) __builtin_amdgcn_sched_group_barrier(DS_RD, (q + 1) * NRD / SPAN - q * NRD / SPAN, 0);
                __builtin_amdgcn_sched_group_barrier(DS_WR, (q + 1) * NW / NM - q * NW / NM, 0);
                __builtin_amdgcn_sched_group_barrier(VMEM_RD, (q + 1) * NL / NM - q * NL / NM, 0);
            });
        }
    }

    float probe = 0.f;   // stays 0 while every sum is finite
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            acc[i][j] = (acc[i][j] + small[i][j]) * SP_UNSCALE;
#pragma unroll
            for (int r = 0; r < 4; ++r) probe = fmaf(acc[i][j][r], 0.f, probe);
        }
    const int64_t wm0 = m0 + 16 * TM * wm, wn0 = n0 + 16 * TN * wn;
    if (__any(probe != 0.f)) {   // (NaN compares unequal)
        const float* ap[TM];
        const float* bp[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int64_t m = wm0 + 16 * i + li;
            ap[i] = A + (m < p.M ? m : p.M - 1) * p.a_sm + lq;
        }
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int64_t n = wn0 + 16 * j + li;
            bp[j] = B + (n < p.N ? n : p.N - 1) * p.b_sn + lq * p.b_sk;
        }
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int64_t k = 0; k < p.K; k += 4) {
            float va[TM], vb[TN];
#pragma unroll
            for (int i = 0; i < TM; ++i) va[i] = ap[i][k];
#pragma unroll
            for (int j = 0; j < TN; ++j) vb[j] = bp[j][k * p.b_sk];
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(va[i], vb[j], acc[i][j], 0, 0, 0);
        }
    }

    // acc[i][j][r] = C[wm0 + 16 i + 4 lq + r][wn0 + 16 j + li]: 64 contiguous bytes of four rows per store, any N and row stride
    float* C = p.C + b0 * p.c_sb0 + b1 * p.c_sb1;
    const float* R = (p.epi & MI355X_EPI_RESIDUAL) ? p.residual + b0 * p.r_sb0 + b1 * p.r_sb1 : nullptr;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int64_t n = wn0 + 16 * j + li;
        if (n >= p.N) continue;
        const float bias = (p.epi & MI355X_EPI_BIAS) ? p.bias[n] : 0.f;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
            const int64_t m = wm0 + 16 * i + 4 * lq;
            float res[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) res[r] = R && m + r < p.M ? R[(m + r) * p.r_sm + n] : 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (m + r < p.M) {
                    const float v = apply_epilogue(acc[i][j][r] * p.alpha, p.epi, bias);
                    C[(m + r) * p.c_sm + n] = R ? v + res[r] : v;
                }
        }
    }
}

// Time per k of each form in nanoseconds, from sweeps over M of 512 to 8192, N of 768 to 3072 and K of 256 to 3072 (and N of
// 1001 to 30522 with B contiguous along n), `n` = tiles per CU. 64 x 64: 26 / 37 / 44 / 56 for up to 1 / 2 / 3 / 4, then 13.7 n
// + 6; 128 x 64: 40 / 48 / 72, then 23 n + 8; 256 x 128: 77 per round. (Over 224 shapes of K = 128 to 3200 the pick is behind the
// kernels it takes over from by more than 2 % in one, 2.4 %, and 1.8 % behind the best form on average. 35 and 38 for the second and
// the first entry, measured before values were scaled: 1237 x 1536 x 2592 96 us here, 89 there. 128 x 128 tiles are never ahead by more than 2 %;
// 128 x 256 tiles equal 256 x 128 and lose 6 % with B contiguous along n.)
struct SplitForm { int bm, bn, resident; };
static const SplitForm kSplitForms[] = {{64, 64, 4}, {128, 64, 3}, {256, 128, 1}};

static double split_cost(int form, int64_t nwg, int cus) {
    const double n = (double)nwg / cus;
    const int64_t up = ceil_div(nwg, (int64_t)cus);
    if (form == 0) return up <= 1 ? 26 : up == 2 ? 37 : up == 3 ? 44 : up == 4 ? 56 : 13.7 * n + 6;
    if (form == 1) return up <= 1 ? 40 : up == 2 ? 48 : up == 3 ? 72 : 23 * n + 8;
    return 77.0 * (double)up;
}

static bool split_takes(const GemmArgs& p) {
    // operands are addressed with 32-bit byte offsets from the start of a batch's matrix
    return p.K % SP_BK == 0 && p.K > 0 && p.a_sm >= 0 && p.b_sn >= 0 && p.b_sk >= 0 && (p.M - 1) * p.a_sm + p.K < ((int64_t)1 << 29) &&
           (p.N - 1) * p.b_sn + (p.K - 1) * p.b_sk + 1 < ((int64_t)1 << 29);
}

double gemm_f32_split_cost(const GemmArgs& p, int cus) {
    double best = 1e300;
    if (tuning().gemm_split == 0 || !split_takes(p)) return best;
    for (int f = 0; f < 3; ++f)
        best = std::min(best, split_cost(f, p.batch * ceil_div(p.M, (int64_t)kSplitForms[f].bm) * ceil_div(p.N, (int64_t)kSplitForms[f].bn), cus));
    return best;
}

bool launch_gemm_f32_split(GemmArgs p, bool b_kc, double other_cost, int cus, hipStream_t stream) {
    const int force = tuning().gemm_split;
    if (force == 0 || !split_takes(p)) return false;
    int best = -1;
    double best_cost = other_cost;
    for (int f = 0; f < 3; ++f) {
        const SplitForm& form = kSplitForms[f];
        const double cost = split_cost(f, p.batch * ceil_div(p.M, (int64_t)form.bm) * ceil_div(p.N, (int64_t)form.bn), cus);
        if (force > 0 ? force == form.bm : cost < best_cost) { best = f; best_cost = cost; }
    }
    if (best < 0) return false;
    const SplitForm& form = kSplitForms[best];
    p.tiles_m = ceil_div(p.M, (int64_t)form.bm);
    p.tiles_n = ceil_div(p.N, (int64_t)form.bn);
    p.nwg = p.batch * p.tiles_m * p.tiles_n;
    if (!grid_fits(p.nwg, best == 2 ? 512 : 256)) return false;
    const int64_t per_xcd = ceil_div(p.nwg, (int64_t)NUM_XCD), per_batch = p.tiles_m * p.tiles_n;
    p.group_m = choose_group_m(p.tiles_m, per_xcd < per_batch ? per_xcd : per_batch, (int64_t)form.resident * (cus / NUM_XCD), form.bm, form.bn, p.K * 4);
    const dim3 grid((unsigned)p.nwg);
    if (best == 0 && b_kc) hipLaunchKernelGGL((gemm_f32_split_kernel<2, 2, 2, 2, 1, 4, true>), grid, dim3(256), 0, stream, p);
    else if (best == 0) hipLaunchKernelGGL((gemm_f32_split_kernel<2, 2, 2, 2, 1, 4, false>), grid, dim3(256), 0, stream, p);
    else if (best == 1 && b_kc) hipLaunchKernelGGL((gemm_f32_split_kernel<4, 2, 2, 2, 1, 3, true>), grid, dim3(256), 0, stream, p);
    else if (best == 1) hipLaunchKernelGGL((gemm_f32_split_kernel<4, 2, 2, 2, 1, 3, false>), grid, dim3(256), 0, stream, p);
    else if (b_kc) hipLaunchKernelGGL((gemm_f32_split_kernel<4, 4, 4, 2, 2, 2, true>), grid, dim3(512), 0, stream, p);
    else hipLaunchKernelGGL((gemm_f32_split_kernel<4, 4, 4, 2, 2, 2, false>), grid, dim3(512), 0, stream, p);
    return true;
}

}  // namespace mi355x
