// fp32 GEMM on the bf16 matrix unit with constant weights that were split beforehand.
//
// The arithmetic is that of gemm_f32_split.hip (three bf16 parts of every value, six products, two sets of accumulators). B, packed once
// in fragment order (split_bf16.h), goes from memory straight into the registers of the MFMA; only A is split here, on its way into LDS.
// That takes B's splitting, its LDS writes and its fragment reads out of the loop, and one MFMA of 32 x 32 x 16 does the work of
// two of 16 x 16 x 32 at 1640 instead of 1415 TFLOP/s, the rate at which each runs with nothing else on the chip (273 and 236 TFLOP/s of
// split products: the clock gives way before the issue slots do).
//
//   * WAVES_M x WAVES_N waves own (32 TM) x (32 TN) outputs each; WAVES_K such groups share K, step by step, and their sums meet in LDS
//     once. A step is 32 k for each group: the tile is split into the stage the next step reads while this one is multiplied, one
//     barrier a step, placed between the two halves so that the fragments of the half after it are read under MFMAs.
//   * B's registers of a half are loaded again right after their last MFMA, for the half after the next.
// What bounds it: the clock under MFMAs where tiles fill the chip several times over, a launch's first loads and last stores
// (4 to 8 us, `fixed` below) where each CU has one tile. Against the kernels before it (MI355X_GEMM_PACKED=0): 8192 x 2304 x 768
// 180 -> 144 us (201 TFLOP/s), 8192 x 768 x 768 65 -> 52, 8192 x 3072 x 768 222 -> 178, 8192 x 768 x 3072 228 -> 187,
// 1024 x 30522 x 768 297 -> 235, 1500 x 1024 x 4096 135 -> 74, 1024 x 2304 x 768 36.5 -> 28.8, 1024 x 3072 x 768 42.4 -> 31.4,
// 1024 x 768 x 3072 41.5 -> 37.5, 128 x 2304 x 768 12.3 -> 8.6, 373 x 1024 x 256 7.4 -> 6.1; 187 products of 8 to 16384 rows 0.84 of the time.
// Twelve waves over 128 x 192 fill the chip evenly where the wider tiles do not (192 columns divide 768, 2304 and 3072): 8192 x 768 x 768 51.5 -> 47.7 us,
// 8192 x 2304 x 768 144 -> 138, 2151 x 2304 x 768 46.1 -> 41.5, 1505 x 3072 x 768 45.3 -> 39.5.
// Its error against float64 is smaller than theirs: 0.8e-7 (2-norm) where the fp32 MFMA has 5.0e-7 and 16 x 16 x 32 1.6e-7 (K = 768).
// Tried: B two steps ahead instead of one and A two (even), B's fragments through LDS, A packed beforehand too (its loads are half as
// long again: even), loads and splits placed between the MFMAs by hand (even or behind).
//   * An output register is 32 neighbouring columns of a row over 32 lanes: stores are whole 128-byte lines whatever N and the row
//     stride are, and a lane has one bias value per 32 columns.
#include "common.h"
#include "gemm_tile.h"
#include "gemm_args.h"
#include "split_bf16.h"

#include <algorithm>

namespace mi355x {

struct PackedGemmArgs {
    GemmArgs g;
    const char* packed;
    int kt;          // steps of 32 k
    int kt_stream;   // of 32 columns of the packed copy: as many, or those of all parts where a batch entry multiplies a part of K
};

template <int TM, int TN, int WAVES_M, int WAVES_N, int WAVES_K, int PER_SIMD>
__global__ __launch_bounds__(WAVES_M * WAVES_N * WAVES_K * WAVE, PER_SIMD) void gemm_f32_packed_kernel(PackedGemmArgs pa) {
    const GemmArgs& p = pa.g;
    constexpr int WAVES = WAVES_M * WAVES_N * WAVES_K, THREADS = WAVES * WAVE, BM = 32 * TM * WAVES_M, BN = 32 * TN * WAVES_N;
    constexpr int GROUP = BM / 32 * 2 * PK_FRAGMENT, STAGE = WAVES_K * GROUP;      // bytes of a 32-k tile of A; of all groups' tiles
    constexpr int BLOCKS = BM * BN / 1024;                                        // 32 x 32 blocks of the workgroup's tile
    constexpr int SUMS = WAVES_K > 1 ? WAVES_K * BLOCKS * 4096 : 0;
    constexpr int UNITS = BM * 4 * WAVES_K, PER_T = (UNITS + THREADS - 1) / THREADS;
    static_assert((UNITS % THREADS == 0 || UNITS < THREADS) && UNITS % WAVE == 0 && THREADS % (4 * WAVE) == 0, "whole units per thread, or one for some waves");
    __shared__ __attribute__((aligned(16))) char lds[2 * STAGE > SUMS ? 2 * STAGE : SUMS];

    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int li = lane % 32, lh = lane / 32;
    const int wm = wave % WAVES_M, wn = wave / WAVES_M % WAVES_N, wk = wave / (WAVES_M * WAVES_N);

    const uint32_t logical = (uint32_t)xcd_remap(blockIdx.x, p.nwg), tiles_per_batch = (uint32_t)(p.tiles_m * p.tiles_n);
    const uint32_t b = logical / tiles_per_batch, t = logical % tiles_per_batch;
    const int64_t b0 = b / (uint32_t)p.batch1, b1 = b % (uint32_t)p.batch1;
    int64_t tm, tn;
    tile_coords(t, p.tiles_m, p.tiles_n, p.group_m, tm, tn);
    const int64_t m0 = tm * BM, n0 = tn * BN;

    // operands as raw buffers with 32-bit offsets (launch precondition); bit 31 makes a load return zero and drops a store
    constexpr uint32_t OUT = 0x80000000u;
    const float* A = p.A + b0 * p.a_sb0 + b1 * p.a_sb1;
    const __amdgpu_buffer_rsrc_t a_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, 0x7fffffff, 0x00020000);
    const char* packed = pa.packed;
    int columns_all = (int)p.N;
    asm volatile("" : "+s"(packed), "+s"(columns_all));   // (here with the arguments that A needs: fetched after its first loads they hold up B's, 0.2 us)
    const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(packed), 0, 0x7fffffff, 0x00020000);

    // A: (k group, row, unit) of this thread's units, four lanes to the 128 bytes of a row; rows beyond the matrix are its last one
    uint32_t a_off[PER_T];
    int a_at[PER_T];
#pragma unroll
    for (int it = 0; it < PER_T; ++it) {
        const int idx = tid + it * THREADS, g = idx % 4, row = idx / 4 % BM, kg = idx / 4 / BM;
        const int64_t r = m0 + row < p.M ? m0 + row : p.M - 1;
        a_off[it] = (uint32_t)(r * p.a_sm + 32 * kg + 4 * g) * 4u;
        // (rows xor-ed with 0, 4, 8, 12 for g = 0..3: neighbouring lanes write to different banks, and reads keep theirs)
        a_at[it] = kg * GROUP + (row / 32 * 2 + g / 2) * PK_FRAGMENT + ((g & 1) * 32 + ((row % 32) ^ (4 * g))) * 16;
    }
    const int steps = (pa.kt + WAVES_K - 1) / WAVES_K;
    f32x4 va[PER_T][2];
    const bool loads = UNITS >= THREADS || tid < UNITS;   // (uniform)
    auto load_a = [&](int it, int st) {
        if (!loads) return;
        uint32_t off = a_off[it];
        if constexpr (WAVES_K > 1) {   // a group that has no tile in the last step multiplies zeros
            const int kg = (tid + it * THREADS) / 4 / BM;
            off = st * WAVES_K + kg < pa.kt ? off : OUT;
        }
        const int base = st * (32 * WAVES_K * 4);
#pragma unroll
        for (int h = 0; h < 2; ++h) va[it][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(a_rsrc, (int)(off + 64u * h), base, 0));
    };
    auto store_a = [&](char* stage, int it) {
        if (!loads) return;
        u32x4 part[SP_PLANES];
        split_unit8(va[it][0], va[it][1], part);
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q) *reinterpret_cast<u32x4*>(stage + a_at[it] + q * PK_PLANE) = part[q];
    };
    // B: one stream of fragments per 32 columns; columns beyond the matrix are its last block's
    const int n_blocks = (columns_all + 31) / 32;
    const uint32_t first_step = pa.kt_stream != pa.kt ? b * (uint32_t)pa.kt : 0u;
    uint32_t b_off[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) {
        const int block = min((int)(n0 / 32) + wn * TN + j, n_blocks - 1);
        b_off[j] = ((uint32_t)block * (uint32_t)pa.kt_stream + first_step) * (uint32_t)(2 * PK_FRAGMENT);
    }
    bf16x8 fa[2][TM][SP_PLANES], fb[2][TN][SP_PLANES];
    auto load_b = [&](auto s_tag, int j, int st) {
        constexpr int s = decltype(s_tag)::value;
        const uint32_t at = b_off[j] + (uint32_t)(min(st * WAVES_K + wk, pa.kt - 1) * 2 + s) * (uint32_t)PK_FRAGMENT;
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q)
            fb[s][j][q] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, lane * 16 + q * PK_PLANE, (int)at, 0));
    };
    int a_rd[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) a_rd[s] = wk * GROUP + (wm * TM * 2 + s) * PK_FRAGMENT + (lh * 32 + (li ^ (4 * (2 * s + lh)))) * 16;
    auto read_a = [&](auto s_tag, const char* stage) {
        constexpr int s = decltype(s_tag)::value;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int q = 0; q < SP_PLANES; ++q) fa[s][i][q] = *reinterpret_cast<const bf16x8*>(stage + a_rd[s] + i * 2 * PK_FRAGMENT + q * PK_PLANE);
    };

    f32x16 acc[TM][TN], small[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = small[i][j][r] = 0.f;
    auto multiply = [&](auto s_tag, int next) {
        constexpr int s = decltype(s_tag)::value;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
#pragma unroll
            for (int u = 0; u < PK_PRODUCTS; ++u)
#pragma unroll
                for (int i = 0; i < TM; ++i) {
                    f32x16& sum = u == 0 ? acc[i][j] : small[i][j];
                    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[s][i][PK_QA[u]], fb[s][j][PK_QB[u]], sum, 0, 0, 0);
                }
            load_b(s_tag, j, next);
        }
    };
    auto sync = [&]() {   // LDS only: loads from memory stay in flight
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };

    constexpr std::integral_constant<int, 0> first{};
    constexpr std::integral_constant<int, 1> second{};
    const int last = steps - 1;   // look-aheads are clamped to the last step, not switched off
#pragma unroll
    for (int it = 0; it < PER_T; ++it) load_a(it, 0);
#pragma unroll
    for (int j = 0; j < TN; ++j) load_b(first, j, 0);
#pragma unroll
    for (int j = 0; j < TN; ++j) load_b(second, j, 0);
#pragma unroll
    for (int it = 0; it < PER_T; ++it) {
        store_a(lds, it);
        load_a(it, min(1, last));
    }
    sync();
    read_a(first, lds);
    for (int st = 0; st < steps; ++st) {
        const int next = min(st + 1, last), after = min(st + 2, last);
        const char* stage = lds + (st & 1) * STAGE;
        char* other = lds + ((st + 1) & 1) * STAGE;
        read_a(second, stage);
#pragma unroll
        for (int it = 0; it < PER_T; ++it) {
            store_a(other, it);
            load_a(it, after);
        }
        multiply(first, next);
        sync();   // `other` is written, and everyone has read `stage`
        read_a(first, other);
        multiply(second, next);
    }

    // The sums of a block over steps `from` to `to` computed again with the fp32 MFMA, straight from global memory: for inputs that the
    // split form cannot hold. Only blocks that are not finite, with 32 k of loads in flight: bound by the fp32 MFMA. One row of NaN:
    // 128 x 768 x 3072 235 -> 42 us (20 without, the kernel before 21), 1024 x 768 x 3072 379 -> 82 (38, 39), 8192 x 768 x 3072 1470 -> 321
    // (186, the split kernel before 650).
    auto again = [&](int64_t bm, int64_t bn, int from, int to) __attribute__((always_inline)) {
        f32x16 sum;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum[r] = 0.f;
        const int64_t m = bm + li, n = bn + li;
        const float* ap = A + (m < p.M ? m : p.M - 1) * p.a_sm + 16 * lh;
        const float* bp = p.B + b0 * p.b_sb0 + (n < p.N ? n : p.N - 1) * p.b_sn + 16 * lh * p.b_sk;
        for (int st = from; st < to; ++st) {
            typedef f32x4 unaligned __attribute__((aligned(4)));
            f32x4 va[4], vb[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) va[c] = *reinterpret_cast<const f32x4*>(ap + 32 * st + 4 * c);
            if (p.b_sk == 1) {
#pragma unroll
                for (int c = 0; c < 4; ++c) vb[c] = *reinterpret_cast<const unaligned*>(bp + 32 * st + 4 * c);
            } else {
#pragma unroll
                for (int e = 0; e < 16; ++e) vb[e / 4][e % 4] = bp[(32 * st + e) * p.b_sk];
            }
#pragma unroll
            for (int e = 0; e < 16; ++e) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(va[e / 4][e % 4], vb[e / 4][e % 4], sum, 0, 0, 0);
        }
        return sum;
    };

    float* C = p.C + b0 * p.c_sb0 + b1 * p.c_sb1 + m0 * p.c_sm + n0;
    const float* R = (p.epi & MI355X_EPI_RESIDUAL) ? p.residual + b0 * p.r_sb0 + b1 * p.r_sb1 + m0 * p.r_sm + n0 : p.C;
    const __amdgpu_buffer_rsrc_t c_rsrc = __builtin_amdgcn_make_buffer_rsrc(C, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t r_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(R), 0, 0x7fffffff, 0x00020000);
    const int rows = (int)min((int64_t)BM, p.M - m0), columns = (int)min((int64_t)BN, p.N - n0);
    // `count` outputs of a column: rows m, m + 1, m + 2, m + 3, then eight rows on. No branch inside: loads and stores go out together.
    auto finish = [&](auto count_tag, auto act_tag, auto res_tag, const float* v, int m, int n, float bias) __attribute__((always_inline)) {
        constexpr int COUNT = decltype(count_tag)::value, ACT = decltype(act_tag)::value;
        constexpr bool RES = decltype(res_tag)::value;
        float res[COUNT];
        uint32_t row[COUNT];
#pragma unroll
        for (int r = 0; r < COUNT; ++r) row[r] = (uint32_t)(m + 8 * (r / 4) + r % 4);
        if constexpr (RES)
#pragma unroll
            for (int r = 0; r < COUNT; ++r) {
                const uint32_t off = (row[r] * (uint32_t)p.r_sm + (uint32_t)n) * 4u;
                res[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r_rsrc, (int)((int)row[r] < rows && n < columns ? off : OUT), 0, 0));
            }
#pragma unroll
        for (int r = 0; r < COUNT; ++r) {
            float o = apply_epilogue(fmaf(v[r], p.alpha, bias), ACT, 0.f);
            if constexpr (RES) o += res[r];
            const uint32_t off = (row[r] * (uint32_t)p.c_sm + (uint32_t)n) * 4u;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, o), c_rsrc, (int)((int)row[r] < rows && n < columns ? off : OUT), 0, 0);
        }
    };
    // f(activation, residual) with both known at compile time
    auto with_epilogue = [&](auto&& f) __attribute__((always_inline)) {
        auto act = [&](auto res) __attribute__((always_inline)) {
            if (p.epi & MI355X_EPI_GELU) f(std::integral_constant<int, MI355X_EPI_GELU>{}, res);
            else if (p.epi & MI355X_EPI_RELU) f(std::integral_constant<int, MI355X_EPI_RELU>{}, res);
            else f(std::integral_constant<int, 0>{}, res);
        };
        if (p.epi & MI355X_EPI_RESIDUAL) act(std::true_type{});
        else act(std::false_type{});
    };
    auto bias_of = [&](int n) { return (p.epi & MI355X_EPI_BIAS) && n < columns ? p.bias[n0 + n] : 0.f; };

    if constexpr (WAVES_K == 1) {
        float bias[TN], probe = 0.f;   // probe stays 0 while every sum is finite
#pragma unroll
        for (int j = 0; j < TN; ++j) bias[j] = bias_of(32 * (wn * TN + j) + li);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                acc[i][j] = (acc[i][j] + small[i][j]) * SP_UNSCALE;
#pragma unroll
                for (int r = 0; r < 16; ++r) probe = fmaf(acc[i][j][r], 0.f, probe);
            }
        if (__builtin_expect(__any(probe != 0.f), 0)) {   // (NaN compares unequal)
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    float block = 0.f;
#pragma unroll
                    for (int r = 0; r < 16; ++r) block = fmaf(acc[i][j][r], 0.f, block);
                    if (__any(block != 0.f)) acc[i][j] = again(m0 + 32 * (wm * TM + i), n0 + 32 * (wn * TN + j), 0, pa.kt);
                }
        }
        with_epilogue([&](auto act, auto res) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) {
                    float v[16];
#pragma unroll
                    for (int r = 0; r < 16; ++r) v[r] = acc[i][j][r];
                    finish(std::integral_constant<int, 16>{}, act, res, v, 32 * (wm * TM + i) + 4 * lh, 32 * (wn * TN + j) + li, bias[j]);
                }
        });
    } else {
        // [group][block][register / 4][lane]: the quads of all groups are added up by the thread that stores them
        constexpr int QUADS = BLOCKS * 256, PER = (QUADS + THREADS - 1) / THREADS;
        f32x4* sums = reinterpret_cast<f32x4*>(lds);
        __syncthreads();   // everyone has read its fragments
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                acc[i][j] = (acc[i][j] + small[i][j]) * SP_UNSCALE;
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    sums[((wk * BLOCKS + (wm * TM + i) * (TN * WAVES_N) + wn * TN + j) * 4 + q) * WAVE + lane] =
                        f32x4{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
            }
        float bias[PER];
#pragma unroll
        for (int it = 0; it < PER; ++it) {
            const int v = it * THREADS + tid;
            bias[it] = bias_of(32 * (v / 256 % (TN * WAVES_N)) + li);
        }
        __syncthreads();
        f32x4 sum[PER];
        float probe = 0.f;
#pragma unroll
        for (int it = 0; it < PER; ++it) {
            const int v = min(it * THREADS + tid, QUADS - 1);
            sum[it] = sums[v];
#pragma unroll
            for (int w = 1; w < WAVES_K; ++w) sum[it] += sums[w * QUADS + v];
#pragma unroll
            for (int r = 0; r < 4; ++r) probe = fmaf(sum[it][r], 0.f, probe);
        }
        if (__builtin_expect(__syncthreads_or(probe != 0.f), 0))
            for (int block = 0; block < BLOCKS; ++block) {   // each by all waves, a share of K each
                float of_block = 0.f;
#pragma unroll
                for (int it = 0; it < PER; ++it)
                    if (min(it * THREADS + tid, QUADS - 1) / 256 == block)
#pragma unroll
                        for (int r = 0; r < 4; ++r) of_block = fmaf(sum[it][r], 0.f, of_block);
                if (!__syncthreads_or(of_block != 0.f)) continue;   // (everyone has read the sums before)
                const f32x16 v = again(m0 + 32 * (block / (TN * WAVES_N)), n0 + 32 * (block % (TN * WAVES_N)), pa.kt * wave / WAVES, pa.kt * (wave + 1) / WAVES);
#pragma unroll
                for (int q = 0; q < 4; ++q) sums[(wave * 4 + q) * WAVE + lane] = f32x4{v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]};
                __syncthreads();
#pragma unroll
                for (int it = 0; it < PER; ++it) {
                    const int u = min(it * THREADS + tid, QUADS - 1);
                    if (u / 256 != block) continue;
                    sum[it] = sums[u % 256];
                    for (int w = 1; w < WAVES; ++w) sum[it] += sums[w * 256 + u % 256];
                }
            }
        with_epilogue([&](auto act, auto res) __attribute__((always_inline)) {
#pragma unroll
            for (int it = 0; it < PER; ++it) {
                const int v = it * THREADS + tid, block = v / 256;
                if (QUADS % THREADS && v >= QUADS) break;
                const float s[4] = {sum[it][0], sum[it][1], sum[it][2], sum[it][3]};
                finish(std::integral_constant<int, 4>{}, act, res, s, 32 * (block / (TN * WAVES_N)) + 8 * (v / WAVE % 4) + 4 * lh,
                       32 * (block % (TN * WAVES_N)) + li, bias[it]);
            }
        });
    }
}

// One unit (eight k of a row, a lane's share of a fragment) per thread: bound by the reads of B, once when a graph is prepared.
__global__ void pack_f32_kernel(const float* w, u32x4* packed, int64_t rows, int64_t K, int64_t s_row, int64_t s_k, int64_t units) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= units) return;
    const int l = (int)(i % WAVE), s = (int)(i / WAVE % 2), g = 2 * s + l / 32;
    const int64_t steps = K / 32, step = i / (2 * WAVE) % steps, block = i / (2 * WAVE) / steps, row = block * 32 + l % 32;
    f32x4 v[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int e = 0; e < 4; ++e) v[h][e] = row < rows ? w[row * s_row + (step * 32 + 16 * h + 4 * g + e) * s_k] : 0.f;
    u32x4 part[SP_PLANES];
    split_unit8(v[0], v[1], part);
#pragma unroll
    for (int q = 0; q < SP_PLANES; ++q) packed[((i / WAVE) * SP_PLANES + q) * WAVE + l] = part[q];
}

// Nanoseconds: `fixed` and `per_k` while every workgroup has a CU to itself, `again` and `again_k` for each further one on the same CU
// (by halves from six on, where they no longer run in step). Fitted over 600 products of M = 8 to 16384, N = 64 to 32000 and
// K = 64 to 4096.
struct PackedForm { int bm, bn, threads, resident; double fixed, per_k, again, again_k; };
static const PackedForm kPackedForms[] = {
    {128, 256, 512, 1, 8440, 56.0, 7580, 64.7}, {64, 256, 256, 2, 5220, 35.8, 3290, 30.8}, {64, 192, 512, 1, 7490, 25.8, 5920, 29.7},
    {64, 128, 512, 1, 4900, 16.5, 2570, 17.5},  {64, 64, 512, 1, 5180, 8.85, 3530, 12.1},  {64, 64, 256, 3, 3870, 15.0, 860, 10.6},
    {32, 64, 512, 1, 4260, 5.5, 1290, 6.25},    {32, 32, 512, 1, 4730, 3.69, 2050, 5.7},   {128, 128, 256, 2, 6040, 35.6, 3120, 31.7},
    {64, 128, 256, 2, 3660, 21.0, 1900, 16.2},
    {128, 192, 768, 1, 7600, 52.0, 2800, 53.5}};
constexpr int TWELVE_WAVES = 10;
constexpr int kPackedGroups[] = {1, 1, 2, 2, 4, 1, 4, 8, 1, 1, 1};   // of waves that share K
constexpr int kNumPackedForms = sizeof(kPackedForms) / sizeof(kPackedForms[0]);

static void launch_packed(int form, const PackedGemmArgs& p, hipStream_t st) {
    const dim3 grid((unsigned)p.g.nwg), block(kPackedForms[form].threads);
    switch (form) {
        case 0: hipLaunchKernelGGL((gemm_f32_packed_kernel<2, 2, 2, 4, 1, 2>), grid, block, 0, st, p); break;
        case 1: hipLaunchKernelGGL((gemm_f32_packed_kernel<2, 2, 1, 4, 1, 2>), grid, block, 0, st, p); break;
        case 2: hipLaunchKernelGGL((gemm_f32_packed_kernel<1, 3, 2, 2, 2, 2>), grid, block, 0, st, p); break;
        case 3: hipLaunchKernelGGL((gemm_f32_packed_kernel<2, 1, 1, 4, 2, 2>), grid, block, 0, st, p); break;
        case 4: hipLaunchKernelGGL((gemm_f32_packed_kernel<2, 1, 1, 2, 4, 2>), grid, block, 0, st, p); break;
        case 5: hipLaunchKernelGGL((gemm_f32_packed_kernel<1, 1, 2, 2, 1, 3>), grid, block, 0, st, p); break;
        case 6: hipLaunchKernelGGL((gemm_f32_packed_kernel<1, 1, 1, 2, 4, 2>), grid, block, 0, st, p); break;
        case 8: hipLaunchKernelGGL((gemm_f32_packed_kernel<2, 2, 2, 2, 1, 2>), grid, block, 0, st, p); break;
        case 9: hipLaunchKernelGGL((gemm_f32_packed_kernel<2, 1, 1, 4, 1, 2>), grid, block, 0, st, p); break;
        case 10: hipLaunchKernelGGL((gemm_f32_packed_kernel<2, 1, 2, 6, 1, 3>), grid, block, 0, st, p); break;
        default: hipLaunchKernelGGL((gemm_f32_packed_kernel<1, 1, 1, 1, 8, 2>), grid, block, 0, st, p); break;
    }
}

static double packed_cost(const PackedForm& f, int64_t nwg, int64_t K, int cus) {
    const int64_t up = ceil_div(nwg, (int64_t)cus);
    const double more = up <= 6 ? (double)(up - 1) : (double)nwg / cus - 0.5;
    return f.fixed + f.per_k * (double)K + more * (f.again + f.again_k * (double)K);
}

// What mi355x_gemm_f32 takes, from the rules of its kernels (with what those leave out because it is the same on both of their sides:
// a launch, first loads, last stores). Over the same products a median 7 % below what was measured; the few-tile kernel's is at times too
// long, by up to a tenth where weights come from beyond the L2 (1245 x 96 x 1056 9.2 us, packed 10.1): its share below is what keeps
// those there.
static double unpacked_cost(const GemmArgs& p, bool b_kc, int cus) {
    double best = 0.91 * gemm_f32_direct_cost(p, b_kc, cus);
    const bool nt = b_kc && p.N % 4 == 0;
    if (nt) best = std::min(best, gemm_f32_nt_cost(p, cus));
    const double split = gemm_f32_split_cost(p, cus);
    if (split < 1e300 && p.K >= (nt ? 256 : 128)) best = std::min(best, (nt ? 6000 : 8000) + split * (double)p.K);
    return best;
}

// Preconditions of the kernel besides pointer alignment
static bool packed_takes(const GemmArgs& p) {
    return p.K > 0 && p.K % 32 == 0 && p.a_sk == 1 && p.a_sm >= 0 && p.a_sm % 4 == 0 && p.a_sb0 % 4 == 0 && p.a_sb1 % 4 == 0 &&
           p.b_sb1 == 0 && (p.M - 1) * p.a_sm + p.K < ((int64_t)1 << 29) &&
           ceil_div(p.N, (int64_t)32) * (p.K / 32) * (2 * PK_FRAGMENT) < ((int64_t)1 << 31) &&
           p.c_sm >= 0 && p.c_sm < ((int64_t)1 << 22) && p.r_sm >= 0 && p.r_sm < ((int64_t)1 << 22);   // (rows of a tile of C, 32-bit byte offsets)
}

// The fastest form, -1 where mi355x_gemm_f32 is faster; or the one that is forced (MI355X_GEMM_PACKED). Few rows are bound by the weights'
// way into the CUs, of which the packed copy has half as many bytes again, and the estimates do not know it: with weights from beyond the
// L2 1 x 20149 x 832 took 14.5 us and packed 19.0, 5 x 20736 x 2432 38.5 and 53.4, 8 x 4576 x 2080 13.4 and 15.7, 20 x 7232 x 2368 17.2 and
// 20.0. Up to 16 rows (31 products, of which the packed form was ahead in 14, by 3 % on average behind) none is packed, up to 32 those that are
// well ahead (28 x 13792 x 1280 23.6 -> 19.1). Over 413 products that nothing was fitted to the pick is at most 4 % behind the kernels before
// and takes 0.88 of their time; against the fastest form it is 2.4 % behind over 187, up to 1.7 times where K is short and tiles are many
// (5190 x 23059 x 192 282 us packed, 485 as picked: the estimate of the kernels before is low there).
// `best_cost`: of what is chosen, either way.
static int choose_packed(const GemmArgs& p, int cus, double& best_cost) {
    const int force = tuning().gemm_packed;
    best_cost = 0;
    if (force > 0 && force <= kNumPackedForms && packed_takes(p)) return force - 1;
    best_cost = unpacked_cost(p, p.b_sk == 1, cus);
    if (!packed_takes(p) || force >= 0 || p.M <= 16) return -1;
    if (p.M <= 32) best_cost *= 0.8;
    int best = -1;
    for (int f = 0; f < kNumPackedForms; ++f) {
        // Twelve waves sum K in one go. In place of groups that share it their error is up to 1.4 times as large (a layer of 8192 x 768 x 3072 that is
        // 7 % faster so stays with two groups for it).
        if (f == TWELVE_WAVES && (best < 0 || kPackedGroups[best] > 1 || p.K < 512)) continue;   // (2048 x 13720 x 256 91 us so, 80)
        const PackedForm& form = kPackedForms[f];
        const double cost = packed_cost(form, p.batch * ceil_div(p.M, (int64_t)form.bm) * ceil_div(p.N, (int64_t)form.bn), p.K, cus);
        if (cost < best_cost) { best = f; best_cost = cost; }
    }
    if (best < 0 && p.M <= 32) best_cost /= 0.8;
    return best;
}

static int choose_packed(const GemmArgs& p, int cus) {
    double cost;
    return choose_packed(p, cus, cost);
}

// The same for a product in parts (batch entries of p): the packed forms and the few-tile kernel, no other -- those before have up to twice their
// error. -1: the few-tile kernel.
static int choose_part(const GemmArgs& p, bool packed, int cus, double& best_cost) {
    const int force = tuning().gemm_packed;
    best_cost = 0;
    if (force > 0 && force <= kNumPackedForms && packed && packed_takes(p)) return force - 1;
    best_cost = 0.91 * gemm_f32_direct_cost(p, p.b_sk == 1, cus);
    if (!packed || !packed_takes(p) || force >= 0 || p.M <= 16) return -1;
    int best = -1;
    for (int f = 0; f < kNumPackedForms; ++f) {
        if (f == TWELVE_WAVES) continue;   // (parts are for few tiles)
        const PackedForm& form = kPackedForms[f];
        const double cost = packed_cost(form, p.batch * ceil_div(p.M, (int64_t)form.bm) * ceil_div(p.N, (int64_t)form.bn), p.K, cus) * (p.M <= 32 ? 1.25 : 1);
        if (cost < best_cost) { best = f; best_cost = cost; }
    }
    return best;
}

static int launch_chosen(PackedGemmArgs& pa, int form, int cus, hipStream_t stream) {
    GemmArgs& p = pa.g;
    const PackedForm& f = kPackedForms[form];
    p.tiles_m = ceil_div(p.M, (int64_t)f.bm);
    p.tiles_n = ceil_div(p.N, (int64_t)f.bn);
    p.nwg = p.batch * p.tiles_m * p.tiles_n;
    if (!grid_fits(p.nwg, f.threads)) return -1;
    const int64_t per_xcd = ceil_div(p.nwg, (int64_t)NUM_XCD), per_batch = p.tiles_m * p.tiles_n;
    p.group_m = choose_group_m(p.tiles_m, per_xcd < per_batch ? per_xcd : per_batch, (int64_t)f.resident * (cus / NUM_XCD), f.bm, f.bn, p.K * 5);
    launch_packed(form, pa, stream);
    return check_launch("gemm_f32_packed_kernel");
}

}  // namespace mi355x

extern "C" int mi355x_pack_f32(const float* w, void* packed, int64_t rows, int64_t K, int64_t row_stride, int64_t k_stride, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(rows >= 0 && K >= 0 && K % 32 == 0, "pack: %lld rows of %lld values, no multiple of 32", (long long)rows, (long long)K);
    if (rows == 0 || K == 0) return MI355X_OK;
    MI355X_REQUIRE(w && packed && (reinterpret_cast<uintptr_t>(packed) & 15) == 0, "pack: null or unaligned pointer");
    const int64_t units = ceil_div(rows, (int64_t)32) * (K / 32) * 2 * WAVE;
    MI355X_REQUIRE(grid_fits(ceil_div(units, (int64_t)256), 256), "pack: grid too large");
    hipLaunchKernelGGL(pack_f32_kernel, dim3((unsigned)ceil_div(units, (int64_t)256)), dim3(256), 0, static_cast<hipStream_t>(stream), w,
                       static_cast<u32x4*>(packed), rows, K, row_stride, k_stride, units);
    return check_launch("pack_f32_kernel");
}

extern "C" int mi355x_gemm_packed_pays(int64_t batch, int64_t M, int64_t N, int64_t K, int b_kc) {
    using namespace mi355x;
    if (batch <= 0 || M <= 0 || N <= 0 || K <= 0) return 0;
    GemmArgs p = {};
    p.batch = batch; p.batch1 = 1; p.M = M; p.N = N; p.K = K;
    p.a_sm = K; p.a_sk = 1; p.b_sk = b_kc ? 1 : N; p.b_sn = b_kc ? K : 1; p.c_sm = N;
    const int cus = device_cus();
    return choose_packed(p, cus > 0 ? cus : 256) >= 0;
}

extern "C" int mi355x_gemm_packed_f32(const float* A, const void* packed, const float* B, float* C, const float* bias,
                                      const float* residual, int64_t batch0, int64_t batch1, int64_t M, int64_t N, int64_t K,
                                      const int64_t* a_strides, const int64_t* b_strides, const int64_t* c_strides,
                                      const int64_t* r_strides, float alpha, int epilogue, void* stream) {
    using namespace mi355x;
    PackedGemmArgs pa;
    GemmArgs& p = pa.g;
    auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    if (A && B && C && packed && a_strides && b_strides && c_strides && batch0 > 0 && batch1 > 0 && M > 0 && N > 0 && K > 0 &&
        (epilogue & ~(MI355X_EPI_BIAS | MI355X_EPI_RELU | MI355X_EPI_GELU | MI355X_EPI_RESIDUAL)) == 0 && (!(epilogue & MI355X_EPI_BIAS) || bias) &&
        (!(epilogue & MI355X_EPI_RESIDUAL) || (residual && r_strides)) && (c_strides[2] >= N || M == 1) && al16(A) && al16(packed) && b_strides[0] == 0) {
        MI355X_TRACE_INIT(p);
        p.A = A; p.B = B; p.C = C; p.bias = bias; p.residual = residual;
        p.batch = batch0 * batch1; p.batch1 = batch1; p.M = M; p.N = N; p.K = K;
        p.a_sb0 = a_strides[0]; p.a_sb1 = a_strides[1]; p.a_sm = a_strides[2]; p.a_sk = a_strides[3];
        p.b_sb0 = b_strides[0]; p.b_sb1 = b_strides[1]; p.b_sk = b_strides[2]; p.b_sn = b_strides[3];
        p.c_sb0 = c_strides[0]; p.c_sb1 = c_strides[1]; p.c_sm = c_strides[2];
        const bool res = epilogue & MI355X_EPI_RESIDUAL;
        p.r_sb0 = res ? r_strides[0] : 0; p.r_sb1 = res ? r_strides[1] : 0; p.r_sm = res ? r_strides[2] : 0;
        p.alpha = alpha; p.epi = epilogue;
        pa.packed = static_cast<const char*>(packed);
        pa.kt = pa.kt_stream = (int)(K / 32);
        const int cus = device_cus();
        if (cus <= 0) return set_error(MI355X_ERR_NOT_INITIALIZED, "gemm: no usable HIP device");
        const int form = choose_packed(p, cus);
        if (form >= 0) {
            const int status = launch_chosen(pa, form, cus, static_cast<hipStream_t>(stream));
            if (status >= 0) return status;
        }
    }
    return mi355x_gemm_f32(A, B, C, bias, residual, batch0, batch1, M, N, K, a_strides, b_strides, c_strides, r_strides, alpha, epilogue, stream);
}

// Between one and eight parts, of at least 256 k each, by the estimates of the kernels and what the normalization takes longer to read them.
// What the sums' bytes cost is three times what a warm measurement says: a program whose weights do not fit the memory-side cache pays for every further
// byte there (an encoder layer over 1024 tokens with FFN2 in four parts 117 us over one set of weights, 122 in one part, but 131 against 128 over three).
// Both launches, weights from beyond the L2: 16 x 768 x 3072 16.0 us in one part, 8.9 in eight; 128 rows 21.7, 12.9 in four; 512 rows 28.9, 22.5 in
// four; 865 rows 39.7, 30.3 in three; 16 x 1024 x 4096 19.6, 9.9 in eight; 16 x 768 x 768 8.0, 7.1 in three. None of 49 products is behind one part.
extern "C" int64_t mi355x_gemm_parts(int64_t M, int64_t N, int64_t K, int b_kc, int packed) {
    using namespace mi355x;
    if (M <= 0 || N <= 0 || K <= 0 || N % 4 || N > 1024) return 1;
    int cus = device_cus();
    if (cus <= 0) cus = 256;
    GemmArgs p = {};
    p.batch = p.batch1 = 1; p.M = M; p.N = N; p.K = K;
    p.a_sm = K; p.a_sk = 1; p.b_sk = b_kc ? 1 : N; p.b_sn = b_kc ? K : 1; p.c_sm = N;
    double best_cost;
    if (packed) choose_packed(p, cus, best_cost);
    else best_cost = unpacked_cost(p, p.b_sk == 1, cus);
    best_cost *= 0.95;
    int64_t best = 1;
    for (const int64_t parts : {2, 3, 4, 6, 8}) {
        if (K % (parts * 32) || K / parts < 256) continue;
        p.batch = parts; p.K = K / parts;
        double cost;
        choose_part(p, packed, cus, cost);
        cost += 200.0 + 50.0 * (double)parts + 4.0 * (double)parts * (double)M * (double)N / 3000.0;
        if (cost < best_cost) { best = parts; best_cost = cost; }
    }
    return best;
}

extern "C" int mi355x_gemm_parts_packed_pays(int64_t parts, int64_t M, int64_t N, int64_t K, int b_kc) {
    using namespace mi355x;
    if (parts <= 0 || M <= 0 || N <= 0 || K <= 0 || K % (32 * parts)) return 0;
    GemmArgs p = {};
    p.batch = parts; p.batch1 = 1; p.M = M; p.N = N; p.K = K / parts;
    p.a_sm = K; p.a_sk = 1; p.b_sk = b_kc ? 1 : N; p.b_sn = b_kc ? K : 1; p.c_sm = N;
    const int cus = device_cus();
    double cost;
    return choose_part(p, ceil_div(N, (int64_t)32) * (K / 32) * (2 * PK_FRAGMENT) < ((int64_t)1 << 31), cus > 0 ? cus : 256, cost) >= 0;
}

extern "C" int mi355x_gemm_parts_f32(const float* A, const float* B, const void* packed, float* P, int64_t parts, int64_t M, int64_t N, int64_t K,
                                     int64_t a_row_stride, int64_t b_k_stride, int64_t b_column_stride, float alpha, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(parts > 0 && M >= 0 && N >= 0 && K >= 0 && K % parts == 0, "gemm_parts: K = %lld in %lld parts", (long long)K, (long long)parts);
    const int64_t share = K / parts;
    const int64_t a[4] = {share, 0, a_row_stride, 1}, b[4] = {share * b_k_stride, 0, b_k_stride, b_column_stride}, c[3] = {M * N, 0, N};
    if (A && B && P && M > 0 && N > 0 && share > 0) {
        PackedGemmArgs pa = {};
        GemmArgs& p = pa.g;
        MI355X_TRACE_INIT(p);
        p.A = A; p.B = B; p.C = P;
        p.batch = parts; p.batch1 = 1; p.M = M; p.N = N; p.K = share;
        p.a_sb0 = a[0]; p.a_sm = a[2]; p.a_sk = 1;
        p.b_sb0 = b[0]; p.b_sk = b[2]; p.b_sn = b[3];
        p.c_sb0 = c[0]; p.c_sm = N;
        p.alpha = alpha; p.epi = MI355X_EPI_NONE;
        pa.packed = static_cast<const char*>(packed);
        pa.kt = (int)(share / 32); pa.kt_stream = (int)(K / 32);
        const int cus = device_cus();
        if (cus <= 0) return set_error(MI355X_ERR_NOT_INITIALIZED, "gemm: no usable HIP device");
        const bool takes = packed && share % 32 == 0 && ceil_div(N, (int64_t)32) * (K / 32) * (2 * PK_FRAGMENT) < ((int64_t)1 << 31) &&
                           ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(packed)) & 15) == 0;
        double cost;
        const int form = choose_part(p, takes, cus, cost);
        if (form >= 0) {
            const int status = launch_chosen(pa, form, cus, static_cast<hipStream_t>(stream));
            if (status >= 0) return status;
        }
        // (a copy that is left out in a product of many rows: a kernel of large tiles)
        const bool b_kc = b_k_stride == 1;
        if (form < 0 && (b_kc || b_column_stride == 1) && cost < 1.4 * unpacked_cost(p, b_kc, cus) &&
            launch_gemm_f32_direct(p, b_kc, 1e300, cus, static_cast<hipStream_t>(stream)))
            return check_launch("gemm_f32_direct_kernel");
    }
    return mi355x_gemm_f32(A, B, P, nullptr, nullptr, parts, 1, M, N, share, a, b, c, nullptr, alpha, MI355X_EPI_NONE, stream);
}
