// ONNX Conv, fp32, on the bf16 matrix unit with constant filters that were split beforehand.
//
// The arithmetic is that of gemm_f32_packed.hip: three bf16 parts of every value, six products, two sets of accumulators. The input
// under a tile of positions (a patch: every row and column that a tap of theirs reads, zeros where it is padding) is split once on its
// way into LDS, and all taps of a filter read it there, each at a constant distance from the position: the nine taps of a 3 x 3 filter
// cost one pass of loads and splits instead of nine. Filters, packed in fragment order, go from memory straight into registers.
//
//   * WAVES_M x WAVES_P waves own 32 filters x (32 TP) consecutive positions each; WAVES_K such groups take turns of 16 CHUNK channels,
//     and their sums meet in LDS once.
//   * A unit of LDS is one pixel's eight channels, its three parts side by side (48 bytes: neighbouring pixels, also every second one,
//     start at different banks). Filters over at most four channels (PIXELS) have units of one pixel's four channels, a plane for each
//     part, and an MFMA step is four neighbouring taps of a filter row.
//   * One stage: where several workgroups share a CU the others multiply while one splits; loads of the next channels are in flight
//     under the products.
//   * An output register is one filter at 32 neighbouring positions: stores are whole lines whatever the extent.
// What bounds it: the clock under MFMAs, and how evenly the tiles fill the chip (32 images of a 28 x 28 layer of 128 are 196 tiles of
// 64 x 256 for 256 CUs); of the rest splitting is 5 to 10 us of 45, waiting for filters 2 to 4. Against the kernels before it
// (MI355X_CONV_PACKED=0), 32 images, 3 x 3: 64 x 56 x 56 -> 64 67 -> 45 us (164 TFLOP/s), 128 x 28 x 28 -> 128 69 -> 42,
// 256 x 14 x 14 -> 256 73 -> 44, 512 x 7 x 7 -> 512 78 -> 48, 64 x 56 x 56 -> 128 by two 46 -> 36; 1 x 1 128 x 28 x 28 -> 256 by two
// 14.7 -> 10.3; 7 x 7 by two over 3 x 224 x 224 -> 64 140 -> 65, one image 13.7 -> 5.9; 131 random layers take 0.63 of the time.
// Tiles of 128 filters split a patch half as often, which shows where it is large, by two (against tiles of 64): 32 images 64 x 56 x 56 -> 128
// 37.0 -> 28 us, 128 x 28 x 28 -> 256 32.9 -> 26, 16 images 64 x 49 x 49 -> 128 18.1 -> 15.7; by one at most 5 % ahead, where the rule seldom takes them.
// Tried: no strips (the first layer 104 us, patches of 99 KB where 34 do); all groups splitting at once (2 % behind over 8 x 256 x
// 28 x 28, 11 % over 1 x 512 x 7 x 7); loads placed by the compiler, which puts them before their uses (82 us where it is 45 now);
// 128 x 256 tiles (never ahead for 3 x 3); a second set of accumulators in turn for the five small products (even).
#include "common.h"
#include "gemm_tile.h"
#include "conv_args.h"
#include "split_bf16.h"

#include <algorithm>
#include <numeric>

namespace mi355x {

struct PackedConvArgs {
    ConvArgs c;
    const char* packed;
    // Images are cut into `strips` of strip_w columns of positions each (OW a multiple), and the strips of all images lie on top of each
    // other: positions are numbered in that order. The patch: virtual rows, patch_h of them for each strip, of patch_w pixels; a pixel
    // samples the input at `sample` times its place, positions are `step` pixels apart; `pixels` is the most that a tile's patch has.
    int strips, strip_w, patch_h, patch_w, taps_h, step_h, step_w, sample_h, sample_w, pixels;
    FastDiv div_strips, div_strip, div_strip_w, div_patch_h, div_patch_w;
    int groups, stages;   // of 16 channels; of 16 CHUNK WAVES_K (in a part of the channels, if they are summed in parts)
    int64_t part_size;    // outputs of a part, one after the other
    // SKIP: a 1 x 1 convolution of another input with the same result, summed into the same sums
    const float* X2; const float* W2; const float* bias2; const char* packed2;
    int C2, H2, Wd2, stride2_h, stride2_w, groups2, stages2;   // (of 16 SKIP_CHUNK WAVES_K)
};
constexpr int SKIP_CHUNK = 2;

// ROWS x COLUMNS: taps of the filter; PIXELS: C <= 4
template <int ROWS, int COLUMNS, bool PIXELS>
struct PackedFilter {
    static constexpr int PER_ROW = PIXELS ? (COLUMNS + 3) / 4 : COLUMNS;
    static constexpr int STEPS = ROWS * PER_ROW;   // MFMA steps of 16 k: of a group of channels, or of the whole filter
};

template <class FILTER, bool PIXELS, int TP, int WAVES_M, int WAVES_P, int WAVES_K, int CHUNK, int PER_T, bool SKIP>
__global__ __launch_bounds__(WAVES_M * WAVES_P * WAVES_K * WAVE, 2) void conv2d_f32_packed_kernel(PackedConvArgs pa) {
    const ConvArgs& p = pa.c;
    constexpr int THREADS = WAVES_M * WAVES_P * WAVES_K * WAVE, BP = 32 * TP * WAVES_P;
    constexpr int STEPS = FILTER::STEPS * CHUNK, RING = STEPS % 3 == 0 ? 3 : 2;
    static_assert(STEPS % RING == 0 && (!PIXELS || (WAVES_K == 1 && CHUNK == 1)), "the filter ring comes round with the stage");
    extern __shared__ __attribute__((aligned(16))) char lds[];

    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int li = lane % 32, lh = lane / 32;
    const int wm = wave % WAVES_M, wp = wave / WAVES_M % WAVES_P, wk = wave / (WAVES_M * WAVES_P);
    // consecutive tiles share their positions
    const uint32_t number = (uint32_t)xcd_remap(blockIdx.x, p.nwg), tiles = (uint32_t)(p.tiles_m * p.tiles_p), part = number / tiles, logical = number - part * tiles;
    const int stage0 = PIXELS ? 0 : (int)part * pa.stages, stage_end = stage0 + pa.stages;
    const int m0 = (int)(logical % (uint32_t)p.tiles_m) * 32 * WAVES_M;
    const int p0 = (int)(logical / (uint32_t)p.tiles_m) * BP;

    constexpr uint32_t OUT = 0x80000000u;   // an offset that makes a load return zero and drops a store
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.X), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(pa.packed), 0, 0x7fffffff, 0x00020000);

    // a position's strip and its place there
    auto place = [&](int pp, uint32_t& strip, uint32_t& oy, uint32_t& ox) {
        strip = fdiv((uint32_t)pp, pa.div_strip);
        const uint32_t q = (uint32_t)pp - strip * (uint32_t)(p.OH * pa.strip_w);
        oy = fdiv(q, pa.div_strip_w);
        ox = q - oy * (uint32_t)pa.strip_w;
    };
    // its virtual row and column
    auto pixel_of = [&](int pp, int& row, int& column) {
        uint32_t strip, oy, ox;
        place(pp, strip, oy, ox);
        row = (int)strip * pa.patch_h + (int)oy * pa.step_h;
        column = (int)ox * pa.step_w;
    };
    // its image and its place there
    auto output_of = [&](int pp, uint32_t& n, uint32_t& oy, uint32_t& ox) {
        uint32_t strip;
        place(pp, strip, oy, ox);
        n = fdiv(strip, pa.div_strips);
        ox += (strip - n * (uint32_t)pa.strips) * (uint32_t)pa.strip_w;
    };
    int row0, row1, column0;
    pixel_of(p0, row0, column0);
    pixel_of(min(p0 + BP, (int)p.P) - 1, row1, column0);
    const int pixels = (row1 - row0 + pa.taps_h) * pa.patch_w;   // of this patch
    int at[TP];   // byte address of a position's first unit
#pragma unroll
    for (int j = 0; j < TP; ++j) {
        int row, column;
        pixel_of(min(p0 + 32 * (wp * TP + j) + li, (int)p.P - 1), row, column);
        const int pixel = (row - row0) * pa.patch_w + column;
        at[j] = PIXELS ? pixel * 8 + lh * 16 : (wk * CHUNK * 2 + lh) * pa.pixels * 48 + pixel * 48;
    }
    // byte offset of a pixel in its image plane and first channel
    auto sample = [&](int pixel) -> uint32_t {
        const uint32_t r = fdiv((uint32_t)pixel, pa.div_patch_w);
        const uint32_t row = (uint32_t)row0 + r, strip = fdiv(row, pa.div_patch_h), n = fdiv(strip, pa.div_strips);
        const int y = (int)(row - strip * (uint32_t)pa.patch_h) * pa.sample_h - p.pad_t;
        const int x = (int)((uint32_t)pixel - r * (uint32_t)pa.patch_w) * pa.sample_w - p.pad_l +
                      (int)((strip - n * (uint32_t)pa.strips) * (uint32_t)pa.strip_w) * p.stride_w;
        const bool in = (int)n < p.N && (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.Wd;
        return in ? 4u * (uint32_t)(((int)n * p.C * p.H + y) * p.Wd + x) : OUT;
    };
    const int plane = p.H * p.Wd * 4;

    f32x16 acc[TP], small[TP];
#pragma unroll
    for (int j = 0; j < TP; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = small[j][r] = 0.f;
    bf16x8 fw[RING][SP_PLANES], fx[2][SP_PLANES];
    const int blocks = (p.M + 31) / 32;
    const uint32_t w_block = (uint32_t)min(m0 / 32 + wm, blocks - 1) * (uint32_t)(pa.groups * FILTER::STEPS) * (uint32_t)PK_FRAGMENT;
    auto load_w = [&](int slot, int stage, int step) {   // `step` beyond the stage: of the next one
        int group = (stage * WAVES_K + wk) * CHUNK + step / FILTER::STEPS;
        if (step >= STEPS) group = ((stage + 1) * WAVES_K + wk) * CHUNK + (step - STEPS) / FILTER::STEPS;
        const uint32_t off = w_block + ((uint32_t)min(group, pa.groups - 1) * FILTER::STEPS + step % FILTER::STEPS) * (uint32_t)PK_FRAGMENT;
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q)
            fw[slot][q] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, lane * 16 + q * PK_PLANE, (int)off, 0));
    };
    auto read_x = [&](int slot, int j, int step, int base) {
        if constexpr (PIXELS) {
            const char* from = lds + at[j] + base + 8 * ((step / FILTER::PER_ROW) * pa.patch_w + 4 * (step % FILTER::PER_ROW));
#pragma unroll
            for (int q = 0; q < SP_PLANES; ++q) {   // (an odd pixel is not 16-byte aligned)
                typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                const u32x2 a = *reinterpret_cast<const u32x2*>(from + q * pa.pixels * 8), b = *reinterpret_cast<const u32x2*>(from + q * pa.pixels * 8 + 8);
                fx[slot][q] = __builtin_bit_cast(bf16x8, u32x4{a.x, a.y, b.x, b.y});
            }
        } else {
            const int tap = step % FILTER::STEPS, chunk = step / FILTER::STEPS;
            const char* from = lds + at[j] + base + (chunk * 2 * pa.pixels + (tap / FILTER::PER_ROW) * p.dil_h * pa.patch_w + (tap % FILTER::PER_ROW) * p.dil_w) * 48;
#pragma unroll
            for (int q = 0; q < SP_PLANES; ++q) fx[slot][q] = *reinterpret_cast<const bf16x8*>(from + q * 16);
        }
    };
    auto sync = [&]() {   // LDS only: loads from memory stay in flight
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    auto multiply = [&](int stage) {   // a block of positions is read under the products of the one before it
        int zero = 0;
        asm volatile("" : "+s"(zero));   // (the distances of the taps are added here, not kept in registers from stage to stage)
        read_x(0, 0, 0, zero);
        static_for<STEPS * TP>([&](auto tag) {
            constexpr int at_once = decltype(tag)::value, step = at_once / TP, j = at_once % TP, slot = step % RING;
            if constexpr (at_once + 1 < STEPS * TP) read_x((at_once + 1) % 2, (at_once + 1) % TP, (at_once + 1) / TP, zero);
            __builtin_amdgcn_sched_barrier(0);   // (left alone, the compiler moves loads down to their uses)
#pragma unroll
            for (int u = 0; u < PK_PRODUCTS; ++u) {
                f32x16& sum = u == 0 ? acc[j] : small[j];
                sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[slot][PK_QA[u]], fx[at_once % 2][PK_QB[u]], sum, 0, 0, 0);
            }
            if constexpr (j + 1 == TP) load_w(slot, stage, step + RING);
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    // SKIP: the other input at the tile's positions, SKIP_CHUNK times 16 channels to a group of waves at a time: loaded under the products before,
    // split into LDS (position by position, halves of 16 channels apart) when everyone has read what was there. (With the first of them loaded
    // ahead of the taps, where there are registers for that, 8 images of 128 x 28 x 28 take 20.3 us instead of 19.0, one of 512 x 7 x 7 22.3
    // instead of 22.6.) Bound by the loads and their latency: 3 us for 32 channels of a tile of 64 x 256, a fifth of it products.
    constexpr int SKIP_THREADS = THREADS / WAVES_K, SKIP_UNITS = 2 * SKIP_CHUNK * BP, PER_2 = SKIP ? SKIP_UNITS / SKIP_THREADS : 1;
    static_assert(!SKIP || SKIP_UNITS % SKIP_THREADS == 0, "whole units per thread");
    const __amdgpu_buffer_rsrc_t x2_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(pa.X2), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t w2_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(pa.packed2), 0, 0x7fffffff, 0x00020000);
    const int id2 = tid % SKIP_THREADS, plane2 = pa.H2 * pa.Wd2 * 4;
    const uint32_t w2_block = (uint32_t)min(m0 / 32 + wm, blocks - 1) * (uint32_t)pa.groups2 * (uint32_t)PK_FRAGMENT;
    f32x4 v2[PER_2][2];
    bf16x8 fw2[SKIP_CHUNK][SP_PLANES];
    auto load_w2 = [&](int stage) {
        const int first = (stage * WAVES_K + wk) * SKIP_CHUNK;   // group of 16 channels
#pragma unroll
        for (int g = 0; g < SKIP_CHUNK; ++g)
#pragma unroll
            for (int q = 0; q < SP_PLANES; ++q)
                fw2[g][q] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(w2_rsrc, lane * 16 + q * PK_PLANE,
                                                                                           (int)(w2_block + (uint32_t)min(first + g, pa.groups2 - 1) * (uint32_t)PK_FRAGMENT), 0));
    };
    auto load_x2 = [&](int stage) {
        const int first = (stage * WAVES_K + wk) * SKIP_CHUNK;
#pragma unroll
        for (int it = 0; it < PER_2; ++it) {
            const int unit = id2 + it * SKIP_THREADS, c = 16 * first + 8 * (unit / BP);
            uint32_t n, oy, ox;
            output_of(min(p0 + unit % BP, (int)p.P - 1), n, oy, ox);
            const uint32_t at_0 = 4u * (uint32_t)((((int)n * pa.C2 + c) * pa.H2 + (int)oy * pa.stride2_h) * pa.Wd2 + (int)ox * pa.stride2_w);
            const uint32_t off = c < pa.C2 ? at_0 : OUT;   // C2 is a multiple of eight
#pragma unroll
            for (int e = 0; e < 8; ++e)
                v2[it][e / 4][e % 4] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(x2_rsrc, (int)off, e * plane2, 0));
        }
    };

#pragma unroll
    for (int s = 0; s < RING; ++s) load_w(s, stage0, s);
    if constexpr (PIXELS) {
        // the whole patch at once, in turns of PER_T units per thread
        for (int first = tid; first < pixels; first += PER_T * THREADS) {
            float v[PER_T][4];
#pragma unroll
            for (int it = 0; it < PER_T; ++it) {
                const uint32_t off = sample(first + it * THREADS);
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    v[it][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(x_rsrc, (int)(c < p.C ? off : OUT), min(c, p.C - 1) * plane, 0));
            }
#pragma unroll
            for (int it = 0; it < PER_T; ++it) {
                uint32_t part[SP_PLANES][2];
#pragma unroll
                for (int h = 0; h < 2; ++h) split_pair(v[it][2 * h], v[it][2 * h + 1], part[0][h], part[1][h], part[2][h]);
                const int pixel = first + it * THREADS;
                if (pixel < pixels)
#pragma unroll
                    for (int q = 0; q < SP_PLANES; ++q) {
                        typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
                        *reinterpret_cast<u32x2*>(lds + (q * pa.pixels + pixel) * 8) = u32x2{part[q][0], part[q][1]};
                    }
            }
        }
        __syncthreads();
        multiply(0);
    } else {
        // A group's units: the halves of its chunk, pixels of each. With several groups half of them split while the other half multiplies.
        constexpr int GROUP_THREADS = THREADS / WAVES_K;
        const int units = 2 * CHUNK * pixels, id = tid % GROUP_THREADS;   // (<= PER_T GROUP_THREADS: launch precondition)
        const bool late = WAVES_K > 1 && wk >= WAVES_K / 2;
        uint32_t x_off[PER_T];
        int x_to[PER_T], x_c[PER_T];
#pragma unroll
        for (int it = 0; it < PER_T; ++it) {
            const int unit = id + it * GROUP_THREADS, half = CHUNK == 1 ? unit >= pixels : unit / pixels, pixel = unit - half * pixels;
            x_c[it] = 8 * half;
            x_to[it] = ((wk * CHUNK * 2 + half) * pa.pixels + pixel) * 48;
            x_off[it] = unit < units ? sample(pixel) : OUT;
            if (x_off[it] != OUT) x_off[it] += (uint32_t)(8 * half * plane);
        }
        f32x4 v[PER_T][2];
        auto load_x = [&](int stage) {
            const int first = (stage * WAVES_K + wk) * CHUNK * 16;
#pragma unroll
            for (int it = 0; it < PER_T; ++it) {
                if (it * GROUP_THREADS >= units) break;   // (uniform)
                const uint32_t off = first + x_c[it] < p.C ? x_off[it] : OUT;   // C is a multiple of eight
#pragma unroll
                for (int e = 0; e < 8; ++e)
                    v[it][e / 4][e % 4] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(x_rsrc, (int)off, (first + e) * plane, 0));
            }
        };
        load_x(stage0);
        if (late) sync();
        for (int stage = stage0; stage < stage_end; ++stage) {
            if (stage != stage0) sync();   // the group has read its last channels
#pragma unroll
            for (int it = 0; it < PER_T; ++it) {
                if (it * GROUP_THREADS >= units) break;
                if (id + it * GROUP_THREADS < units) {
                    u32x4 part[SP_PLANES];
                    split_unit8(v[it][0], v[it][1], part);
#pragma unroll
                    for (int q = 0; q < SP_PLANES; ++q) *reinterpret_cast<u32x4*>(lds + x_to[it] + q * 16) = part[q];
                }
            }
            sync();
            if (stage + 1 < stage_end) load_x(stage + 1);
            multiply(stage);
        }
        if (WAVES_K > 1 && !late) sync();   // as many barriers for every wave
    }

    if constexpr (SKIP) {
        load_x2(0);
        load_w2(0);
        for (int stage = 0; stage < pa.stages2; ++stage) {
            __syncthreads();   // everyone has read its last units
#pragma unroll
            for (int it = 0; it < PER_2; ++it) {
                u32x4 part[SP_PLANES];
                split_unit8(v2[it][0], v2[it][1], part);
#pragma unroll
                for (int q = 0; q < SP_PLANES; ++q) *reinterpret_cast<u32x4*>(lds + (wk * SKIP_UNITS + id2 + it * SKIP_THREADS) * 48 + q * 16) = part[q];
            }
            __syncthreads();
            if (stage + 1 < pa.stages2) load_x2(stage + 1);
#pragma unroll
            for (int g = 0; g < SKIP_CHUNK; ++g)
#pragma unroll
                for (int j = 0; j < TP; ++j) {
                    const char* from = lds + (wk * SKIP_UNITS + (2 * g + lh) * BP + 32 * (wp * TP + j) + li) * 48;
                    bf16x8 x[SP_PLANES];
#pragma unroll
                    for (int q = 0; q < SP_PLANES; ++q) x[q] = *reinterpret_cast<const bf16x8*>(from + q * 16);
#pragma unroll
                    for (int u = 0; u < PK_PRODUCTS; ++u) {
                        f32x16& sum = u == 0 ? acc[j] : small[j];
                        sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw2[g][PK_QA[u]], x[PK_QB[u]], sum, 0, 0, 0);
                    }
                }
            if (stage + 1 < pa.stages2) load_w2(stage + 1);
        }
    }

    // the sums of the groups, in order, into those of the first
    auto add_groups = [&]() __attribute__((always_inline)) {
        if constexpr (WAVES_K > 1) {
            constexpr int WAVES_1 = WAVES_M * WAVES_P;
            f32x4* sums = reinterpret_cast<f32x4*>(lds);
            __syncthreads();
            if (wk > 0)
#pragma unroll
                for (int j = 0; j < TP; ++j)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        sums[(((wave - WAVES_1) * TP + j) * 4 + q) * WAVE + lane] =
                            f32x4{acc[j][4 * q], acc[j][4 * q + 1], acc[j][4 * q + 2], acc[j][4 * q + 3]};
            __syncthreads();
            if (wk == 0)
#pragma unroll
                for (int g = 0; g < WAVES_K - 1; ++g)
#pragma unroll
                    for (int j = 0; j < TP; ++j)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const f32x4 s = sums[(((g * WAVES_1 + wave) * TP + j) * 4 + q) * WAVE + lane];
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[j][4 * q + e] += s[e];
                        }
        }
    };
#pragma unroll
    for (int j = 0; j < TP; ++j) acc[j] = (acc[j] + small[j]) * SP_UNSCALE;
    add_groups();
    float probe = 0.f;   // stays 0 while every sum is finite
#pragma unroll
    for (int j = 0; j < TP; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = fmaf(acc[j][r], 0.f, probe);
    const int mb = m0 + 32 * wm;
    // (NaN compares unequal) Again with the fp32 MFMA, straight from memory: inputs that the split cannot hold. Of a wave's own blocks
    // only those that are not finite; with several groups the whole tile, each over its share of the channels. One pixel of NaN: 32 x 128 x 28 x 28 -> 128 606 -> 156 us (44
    // without, the kernel before 71), 32 x 512 x 7 x 7 -> 512 1319 -> 186 (48, 80), 1 x 512 x 7 x 7 601 -> 54 (17, 22).
    bool finite = !__any(probe != 0.f);
    if constexpr (WAVES_K > 1) {
        constexpr int PER_WAVE = TP * 4 * WAVE;   // a wave's sums of a group, which it has read: room for its word to all groups
        uint32_t* said = reinterpret_cast<uint32_t*>(lds);
        if (wk == 0) said[wave * PER_WAVE * 4] = finite;
        __syncthreads();
        uint32_t all = 1;
#pragma unroll
        for (int w = 0; w < WAVES_M * WAVES_P; ++w) all &= said[w * PER_WAVE * 4];
        finite = __builtin_amdgcn_readfirstlane(all);
    }
    if (__builtin_expect(!finite, 0)) {
#pragma unroll
        for (int j = 0; j < TP; ++j) {
            float block = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) block = fmaf(acc[j][r], 0.f, block);
            if (WAVES_K == 1 && !__any(block != 0.f)) continue;
            const int pp = min(p0 + 32 * (wp * TP + j) + li, (int)p.P - 1);
            uint32_t n, oy, ox;
            output_of(pp, n, oy, ox);
            const int y0 = (int)oy * p.stride_h - p.pad_t, x0 = (int)ox * p.stride_w - p.pad_l;
            const int m = min(mb + li, p.M - 1);
            f32x16 sum;
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = 0.f;
            if constexpr (PIXELS) {
                const float* w = p.W + (int64_t)m * p.K;
                for (int k = 0; k < p.K; k += 2) {
                    const int kk = min(k + lh, p.K - 1);
                    const uint32_t c = fdiv((uint32_t)kk, p.div_khw), t = (uint32_t)kk - c * (uint32_t)(p.KH * p.KW), ty = fdiv(t, p.div_kw);
                    const int y = y0 + (int)ty * p.dil_h, x = x0 + (int)(t - ty * (uint32_t)p.KW) * p.dil_w;
                    const bool in = (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.Wd;
                    const float xv = in ? p.X[(((int64_t)n * p.C + c) * p.H + y) * p.Wd + x] : 0.f;
                    const bool counted = k + lh < p.K;
                    sum = __builtin_amdgcn_mfma_f32_32x32x2f32(counted ? w[kk] : 0.f, counted ? xv : 0.f, sum, 0, 0, 0);
                }
            } else {
                // All taps of CHANNELS channels at once, the upper lanes' CHANNELS further on: they are contiguous in a filter, and C is a
                // multiple of eight. (Filters span less than 2^31 bytes: their packed copy does.)
                constexpr int TAPS = FILTER::STEPS, CHANNELS = TAPS == 1 ? 16 : 4;
                const __amdgpu_buffer_rsrc_t f_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.W), 0, 0x7fffffff, 0x00020000);
                const uint32_t w_first = 4u * (uint32_t)(m * p.K + lh * CHANNELS * TAPS);
                uint32_t x_first[TAPS];
#pragma unroll
                for (int t = 0; t < TAPS; ++t) {
                    const int y = y0 + t / FILTER::PER_ROW * p.dil_h, x = x0 + t % FILTER::PER_ROW * p.dil_w;
                    const bool in = (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.Wd;
                    x_first[t] = in ? 4u * (uint32_t)(((int)n * p.C * p.H + y) * p.Wd + x) + (uint32_t)(lh * CHANNELS) * (uint32_t)plane : OUT;
                }
                const int c_end = min(p.C, stage_end * 16 * CHUNK * WAVES_K);
                for (int c = stage0 * 16 * CHUNK * WAVES_K + 2 * CHANNELS * wk; c < c_end; c += 2 * CHANNELS * WAVES_K) {
                    f32x4 wv[CHANNELS * TAPS / 4];
                    float xv[CHANNELS * TAPS];
#pragma unroll
                    for (int g = 0; g < CHANNELS * TAPS / 4; ++g) {
                        const bool counted = c + lh * CHANNELS + 4 * g / TAPS / 4 * 4 < p.C;
                        wv[g] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(f_rsrc, (int)(counted ? w_first : OUT), (c * TAPS + 4 * g) * 4, 0));
                    }
#pragma unroll
                    for (int i = 0; i < CHANNELS * TAPS; ++i) {
                        const int e = i / TAPS;
                        const bool counted = c + lh * CHANNELS + e / 4 * 4 < p.C;
                        xv[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(x_rsrc, (int)(counted ? x_first[i % TAPS] : OUT), min(c + e, p.C - 1) * plane, 0));
                    }
#pragma unroll
                    for (int i = 0; i < CHANNELS * TAPS; ++i) sum = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[i / 4][i % 4], xv[i], sum, 0, 0, 0);
                }
                if constexpr (SKIP) {   // eight channels at a time, the upper lanes' four further on
                    const float* w2 = pa.W2 + (int64_t)m * pa.C2 + 4 * lh;
                    const float* x2 = pa.X2 + (((int64_t)n * pa.C2 + 4 * lh) * pa.H2 + (int)oy * pa.stride2_h) * pa.Wd2 + (int)ox * pa.stride2_w;
                    for (int c = 8 * wk; c < pa.C2; c += 8 * WAVES_K)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            sum = __builtin_amdgcn_mfma_f32_32x32x2f32(w2[c + e], x2[(int64_t)(c + e) * pa.H2 * pa.Wd2], sum, 0, 0, 0);
                }
            }
            acc[j] = sum;
        }
        add_groups();
    }
    if (wk > 0) return;

    // acc[j][r]: filter 8 (r / 4) + 4 lh + r % 4 of the block, position li
    const __amdgpu_buffer_rsrc_t y_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.Y + part * pa.part_size, 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t r_rsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.epi & MI355X_EPI_RESIDUAL ? p.residual : p.Y), 0, 0x7fffffff, 0x00020000);
    float bias[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = mb + 8 * (r / 4) + 4 * lh + r % 4;
        bias[r] = (p.epi & MI355X_EPI_BIAS) && m < p.M ? p.bias[m] : 0.f;
        if constexpr (SKIP) bias[r] += pa.bias2 && m < p.M ? pa.bias2[m] : 0.f;
    }
#pragma unroll
    for (int j = 0; j < TP; ++j) {
        const int pp = p0 + 32 * (wp * TP + j) + li;
        uint32_t n, oy, ox;
        output_of(pp, n, oy, ox);
        const uint32_t out = n * (uint32_t)(p.M * p.OHW) + oy * (uint32_t)p.OW + ox;
        uint32_t off[16];
        float res[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m = mb + 8 * (r / 4) + 4 * lh + r % 4;
            off[r] = pp < p.P && m < p.M ? 4u * (out + (uint32_t)m * (uint32_t)p.OHW) : OUT;
        }
        if (p.epi & MI355X_EPI_RESIDUAL)
#pragma unroll
            for (int r = 0; r < 16; ++r) res[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r_rsrc, (int)off[r], 0, 0));
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float o = acc[j][r] + bias[r];
            if (p.epi & MI355X_EPI_RELU) o = fmaxf(o, 0.f);
            if (p.epi & MI355X_EPI_RESIDUAL) o += res[r];
            if (p.epi & MI355X_EPI_RELU_AFTER) o = fmaxf(o, 0.f);
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, o), y_rsrc, (int)off[r], 0, 0);
        }
    }
}

// The sums of a convolution that was computed in parts of its channels, with its epilogue; MEAN: and the mean over the positions, all that a
// global pooling after it keeps. One wave to a row of positions; bound by the launch and one trip to memory (512 rows of 49 in four parts 2.9 us).
template <bool MEAN>
__global__ __launch_bounds__(256) void conv_parts_kernel(const float* __restrict__ P, int parts, const float* __restrict__ bias, const float* __restrict__ residual,
                                                         float* __restrict__ Y, int64_t rows, int M, int positions, int epi) {
    const int lane = threadIdx.x % WAVE;
    const int64_t row = (int64_t)blockIdx.x * (256 / WAVE) + threadIdx.x / WAVE, size = rows * positions;
    if (row >= rows) return;   // (a whole wave)
    const float b = epi & MI355X_EPI_BIAS ? bias[row % M] : 0.f;
    float total = 0.f;
    for (int at = lane; at < positions; at += WAVE) {
        const int64_t i = row * positions + at;
        float v[4], res = epi & MI355X_EPI_RESIDUAL ? residual[i] : 0.f;
#pragma unroll
        for (int s = 0; s < 4; ++s) v[s] = s < parts ? P[s * size + i] : 0.f;
        float o = (v[0] + v[1]) + (v[2] + v[3]) + b;
        if (epi & MI355X_EPI_RELU) o = fmaxf(o, 0.f);
        o += res;
        if (epi & MI355X_EPI_RELU_AFTER) o = fmaxf(o, 0.f);
        if constexpr (MEAN) total += o;
        else Y[i] = o;
    }
    if constexpr (MEAN) {
        total = wave_sum(total);
        if (lane == 0) Y[row] = total * (1.0f / (float)positions);
    }
}

// One unit (a lane's share of a fragment) per thread, once when a graph is prepared. Filter block, group of channels, tap, plane, lane.
__global__ void pack_conv_f32_kernel(const float* w, u32x4* packed, int M, int C, int KH, int KW, int groups, int steps, int64_t units) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= units) return;
    const int l = (int)(i % WAVE), step = (int)(i / WAVE % steps), group = (int)(i / WAVE / steps % groups);
    const int m = (int)(i / WAVE / steps / groups) * 32 + l % 32, h = l / 32;
    f32x4 v[2];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        int c = 16 * group + 8 * h + e, r = step / KW, s = step % KW;
        if (C <= 4) {
            const int per_row = (KW + 3) / 4;
            c = e % 4; r = step / per_row; s = 4 * (step % per_row) + 2 * h + e / 4;
        }
        v[e / 4][e % 4] = m < M && c < C && s < KW ? w[(((int64_t)m * C + c) * KH + r) * KW + s] : 0.f;
    }
    u32x4 part[SP_PLANES];
    split_unit8(v[0], v[1], part);
#pragma unroll
    for (int q = 0; q < SP_PLANES; ++q) packed[((i / WAVE) * SP_PLANES + q) * WAVE + l] = part[q];
}

// What a thread can hold of a stage (units; 0: no such kernel) and nanoseconds, of each kind of filter: 3 x 3, 1 x 1, 7 x 7 over few channels. `fixed`,
// `per_step` (stages of the loop over channels, MFMA steps where there are few) and `per_pixel` (hundreds of a patch, times the stages) hold
// while every workgroup has a CU to itself, the others for each further one on the same CU (by halves from six on, as in
// gemm_f32_packed.hip). Fitted over 370 layers of 1 to 32 images, 5 to 256 columns, 1 to 512 channels and 16 to 768 filters, 3 % off on
// average; the pick is 2.5 % behind the fastest form over 144 others, up to 1.6 times for 1 x 1 and for few 7 x 7 filters.
struct PackedConvCost { int per_t; double fixed, per_step, per_pixel, again, again_step, again_pixel; };
// `skip`: nanoseconds of a stage of a 1 x 1 convolution that is summed too, from 21 ends of residual blocks (0: no such kernel).
struct PackedConvForm { int bm, bp, waves, waves_k; double skip; PackedConvCost kinds[3]; };
constexpr int WIDE = 128;   // filters of a tile, for which a patch is split half as often
constexpr PackedConvForm kPackedConvForms[] = {
    {64, 256, 4, 1, 3000, {{4, 6690, 3100, 328, 4980, 3590, 0}, {}, {6, 5450, 475, 84.5, 3160, 339, 59.9}}},
    {64, 256, 8, 2, 3000, {{4, 7300, 6020, 355, 6280, 9650, 0}, {}, {}}},
    {64, 128, 8, 2, 3000, {{4, 5760, 3210, 360, 3730, 5250, 0}, {}, {}}},
    {64, 128, 4, 1, 1900, {{6, 4760, 1700, 312, 1870, 2250, 0}, {4, 4930, 499, 691, 3020, 263, 0}, {4, 4390, 241, 78, 1390, 212, 23.6}}},
    {64, 64, 8, 4, 3000, {{6, 6010, 3150, 704, 3980, 5100, 0}, {}, {}}},
    {32, 128, 8, 4, 4800, {{6, 5940, 3110, 706, 4130, 5550, 0}, {}, {}}},
    {32, 64, 8, 4, 2900, {{6, 4570, 1700, 730, 2770, 3050, 107}, {4, 4780, 268, 1540, 2400, 93.3, 1720}, {}}},
    {32, 32, 8, 8, 3500, {{8, 5450, 1250, 1730, 4090, 2660, 372}, {4, 4970, 0, 3640, 0, 0, 7770}, {}}},
    {64, 64, 4, 1, 1150, {{6, 3640, 1070, 281, 1380, 1220, 20.4}, {4, 3520, 477, 549, 1090, 357, 88.1}, {4, 4380, 111, 0, 777, 129, 26.9}}},
    {WIDE, 128, 8, 1, 0, {{4, 7200, 3200, 155, 6000, 4700, 200}, {}, {}}},
    {WIDE, 64, 8, 2, 0, {{6, 5900, 3850, 245, 6000, 4300, 100}, {}, {}}}};
constexpr int kNumPackedConvForms = sizeof(kPackedConvForms) / sizeof(kPackedConvForms[0]);

enum { PC_3X3, PC_1X1, PC_7X7, PC_NONE };
static int packed_conv_kind(int64_t C, int64_t KH, int64_t KW, const int64_t* dilations) {
    const bool square = KH == KW;
    if (square && C <= 4 && C > 0 && dilations[1] == 1 && dilations[0] == 1) return KH == 7 ? PC_7X7 : PC_NONE;
    if (C <= 0 || C % 8) return PC_NONE;
    return square && KH == 3 ? PC_3X3 : square && KH == 1 ? PC_1X1 : PC_NONE;
}
static int packed_conv_chunk(int kind) { return kind == PC_1X1 ? 2 : 1; }
static int packed_conv_steps(int kind) { return kind == PC_3X3 ? 9 : kind == PC_1X1 ? 1 : 14; }

template <class FILTER, bool PIXELS, int CHUNK, int KIND, bool SKIP = false>
static void launch_packed_conv(int form, const PackedConvArgs& pa, int lds, hipStream_t st) {
#define MI355X_FORM(index, tp, wm, wp, wk)                                                                                             \
    case index:                                                                                                                        \
        if constexpr (kPackedConvForms[index].kinds[KIND].per_t > 0 && !(SKIP && kPackedConvForms[index].skip == 0))                   \
            hipLaunchKernelGGL((conv2d_f32_packed_kernel<FILTER, PIXELS, tp, wm, wp, wk, CHUNK, kPackedConvForms[index].kinds[KIND].per_t, SKIP>), \
                               dim3((unsigned)pa.c.nwg), dim3(wm * wp * wk * WAVE), lds, st, pa);                                      \
        break;
    switch (form) {
        MI355X_FORM(0, 4, 2, 2, 1)
        MI355X_FORM(1, 4, 2, 2, 2)
        MI355X_FORM(2, 2, 2, 2, 2)
        MI355X_FORM(3, 2, 2, 2, 1)
        MI355X_FORM(4, 2, 2, 1, 4)
        MI355X_FORM(5, 2, 1, 2, 4)
        MI355X_FORM(6, 1, 1, 2, 4)
        MI355X_FORM(7, 1, 1, 1, 8)
        MI355X_FORM(8, 1, 2, 2, 1)
        MI355X_FORM(9, 2, 4, 2, 1)
        MI355X_FORM(10, 2, 4, 1, 2)
    }
#undef MI355X_FORM
}

static int patch_width(const PackedConvArgs& pa, int kind, int strip_w) {
    return (strip_w - 1) * pa.step_w + (kind == PC_3X3 ? 2 * pa.c.dil_w + 1 : kind == PC_1X1 ? 1 : (pa.c.KW + 3) / 4 * 4);
}

// The most pixels of a patch under `bp` consecutive positions of strips of `strip_w` columns, tiles starting at multiples of bp.
static int64_t patch_pixels(const PackedConvArgs& pa, int kind, int strip_w, int bp) {
    const ConvArgs& p = pa.c;
    const int64_t strip = (int64_t)p.OH * strip_w, all_rows = p.P / strip_w;
    const int positions = (int)std::min<int64_t>(bp, p.P), start = strip_w - std::gcd(bp, strip_w);   // the furthest column a tile starts at
    const int rows = (int)std::min<int64_t>((start + positions - 1) / strip_w + 1, all_rows);
    const int ends = strip % bp == 0 ? 0 : std::min((rows - 1 + p.OH - 1) / p.OH, (int)(all_rows / p.OH) - 1);   // of strips, within a tile
    return (int64_t)((rows - 1) * pa.step_h + ends * std::max(0, pa.taps_h - pa.step_h) + pa.taps_h) * patch_width(pa, kind, strip_w);
}

// Strips for tiles of `bp` positions, and the pixels of their patches. Narrow strips have small patches, wide ones whole lines of output:
// strips of 16 columns and more, the narrower ones where the patch shrinks by an eighth.
static int64_t choose_strips(const PackedConvArgs& pa, int kind, int bp, int& strip_w) {
    strip_w = pa.c.OW;
    int64_t pixels = patch_pixels(pa, kind, strip_w, bp);
    if (kind == PC_1X1) return pixels;
    for (int strips = 2; strips <= 16 && pa.c.OW >= 16 * strips; ++strips) {
        if (pa.c.OW % strips) continue;
        const int64_t n = patch_pixels(pa, kind, pa.c.OW / strips, bp);
        if (8 * n < 7 * pixels) { strip_w = pa.c.OW / strips; pixels = n; }
    }
    return pixels;
}

static void set_strips(PackedConvArgs& pa, int kind, int strip_w, int64_t pixels) {
    const ConvArgs& p = pa.c;
    pa.strip_w = strip_w;
    pa.strips = p.OW / strip_w;
    pa.patch_h = (p.OH - 1) * pa.step_h + pa.taps_h;
    pa.patch_w = patch_width(pa, kind, strip_w);
    pa.pixels = (int)pixels;
    pa.div_strips = make_fastdiv(pa.strips); pa.div_strip = make_fastdiv((int64_t)p.OH * strip_w); pa.div_strip_w = make_fastdiv(strip_w);
    pa.div_patch_h = make_fastdiv(pa.patch_h); pa.div_patch_w = make_fastdiv(pa.patch_w);
}

// Bytes of LDS that a form needs for patches of `pixels`, 0 where it does not fit.
static int packed_conv_lds(int kind, const PackedConvForm& f, int64_t pixels, bool skip = false) {
    constexpr int64_t LDS_BYTES = 160 * 1024;
    const int per_t = f.kinds[kind].per_t;
    if (per_t == 0 || (skip && f.skip == 0)) return 0;
    int64_t bytes = pixels * 8 * SP_PLANES + 16;
    if (kind == PC_3X3 || kind == PC_1X1) {
        const int64_t halves = 2 * packed_conv_chunk(kind);
        if (halves * pixels > (int64_t)per_t * (f.waves / f.waves_k) * WAVE) return 0;
        bytes = halves * f.waves_k * pixels * 48;
    }
    bytes = std::max(bytes, (int64_t)(f.waves_k - 1) * f.bm * f.bp * 4);
    if (skip) bytes = std::max(bytes, (int64_t)f.waves_k * 2 * SKIP_CHUNK * f.bp * 48);
    return bytes <= LDS_BYTES ? (int)bytes : 0;
}

// Geometry of a call; false where the kernel does not take it.
static bool packed_conv_args(PackedConvArgs& pa, int& kind, int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW,
                             const int64_t* pads, const int64_t* strides, const int64_t* dilations) {
    for (int64_t v : {N, C, H, Wd, M, KH, KW})
        if (v < 1 || v >= ((int64_t)1 << 24)) return false;
    for (int i = 0; i < 4; ++i)
        if (pads[i] < 0 || pads[i] >= (1 << 16)) return false;
    for (int i = 0; i < 2; ++i)
        if (strides[i] < 1 || strides[i] >= (1 << 10) || dilations[i] < 1 || dilations[i] >= (1 << 10)) return false;
    kind = packed_conv_kind(C, KH, KW, dilations);
    if (kind == PC_NONE) return false;
    const int64_t eff_kh = (KH - 1) * dilations[0] + 1, eff_kw = (KW - 1) * dilations[1] + 1;
    const int64_t hin = H + pads[0] + pads[2], win = Wd + pads[1] + pads[3];
    if (hin < eff_kh || win < eff_kw) return false;
    const int64_t OH = (hin - eff_kh) / strides[0] + 1, OW = (win - eff_kw) / strides[1] + 1;
    // 32-bit byte offsets into every operand
    const int64_t limit = (int64_t)1 << 29;
    if (N * C >= limit || N * C * H >= limit || N * C * H * Wd >= limit || N * M >= limit || OH * OW >= limit || N * OH * OW >= limit ||
        N * M * OH >= limit || N * M * OH * OW >= limit) return false;
    ConvArgs& p = pa.c;
    p.N = (int)N; p.C = (int)C; p.H = (int)H; p.Wd = (int)Wd; p.M = (int)M; p.KH = (int)KH; p.KW = (int)KW;
    p.OH = (int)OH; p.OW = (int)OW; p.OHW = (int)(OH * OW);
    p.pad_t = (int)pads[0]; p.pad_l = (int)pads[1];
    p.stride_h = (int)strides[0]; p.stride_w = (int)strides[1];
    p.dil_h = (int)dilations[0]; p.dil_w = (int)dilations[1];
    p.K = (int)(C * KH * KW); p.P = N * OH * OW;
    p.div_khw = make_fastdiv(KH * KW); p.div_kw = make_fastdiv(KW);
    p.div_ohw = make_fastdiv(OH * OW); p.div_ow = make_fastdiv(OW);
    const bool pointwise = kind == PC_1X1;
    pa.step_h = pointwise ? 1 : p.stride_h; pa.step_w = pointwise ? 1 : p.stride_w;
    pa.sample_h = pointwise ? p.stride_h : 1; pa.sample_w = pointwise ? p.stride_w : 1;
    pa.taps_h = (int)eff_kh;
    if (N * OW * ((OH - 1) * pa.step_h + eff_kh) >= ((int64_t)1 << 30) || (OW - 1) * pa.step_w + eff_kw + 4 >= (1 << 20)) return false;
    pa.groups = C <= 4 ? 1 : (int)ceil_div(C, (int64_t)16);
    return ceil_div(M, (int64_t)32) * pa.groups * packed_conv_steps(kind) * PK_FRAGMENT < ((int64_t)1 << 31);
}

static int64_t skip_stages(const PackedConvArgs& pa, const PackedConvForm& f) { return ceil_div((int64_t)pa.groups2, (int64_t)SKIP_CHUNK * f.waves_k); }

static int64_t packed_conv_stages(const PackedConvArgs& pa, int kind, const PackedConvForm& f) {
    return ceil_div((int64_t)pa.groups, (int64_t)packed_conv_chunk(kind) * f.waves_k);
}

// What mi355x_conv2d_res_f32 takes. `summed_apart`: by the kernel that sums each sixteenth of the channels on its own.
// Over the same layers a median 1 % off for the gather and the direct kernel; the general kernel's tiles fitted over 139 layers.
static double unpacked_conv_cost(const ConvArgs& p, int cus, bool& summed_apart) {
    summed_apart = false;
    if (p.K % 32 == 0) {
        const double gather = conv2d_f32_gather_cost(p, cus), direct = conv2d_f32_direct_cost(p, cus);
        summed_apart = direct < 0.95 * gather;
        return summed_apart ? direct : gather;
    }
    static const struct { int bm, bn; double fixed, per_k, again, again_k; } tiles[] = {
        {64, 128, 8290, 54.7, 3950, 42.9}, {64, 64, 11300, 18, 490, 26.9}, {32, 64, 3620, 24.6, 1600, 14.3}, {16, 64, 3510, 24.9, 480, 7.65}};
    double best = 1e300, cost = 0;   // (the tile that choose_conv_tile takes)
    for (const auto& t : tiles) {
        const int64_t nwg = ceil_div((int64_t)p.M, (int64_t)t.bm) * ceil_div(p.P, (int64_t)t.bn);
        const double work = (double)ceil_div(nwg, (int64_t)cus * 2) * t.bm * t.bn * (1.0 + 24.0 * (1.0 / t.bm + 1.0 / t.bn));
        if (work >= best) continue;
        best = work;
        cost = t.fixed + t.per_k * p.K + (double)(ceil_div(nwg, (int64_t)cus) - 1) * (t.again + t.again_k * p.K);
    }
    return cost;
}

// The fastest form, -1 where mi355x_conv2d_res_f32 is faster than that and `besides` nanoseconds (or so close that the estimates do not tell: at 0.94 for every kind
// 3 of 131 layers were 5 to 14 % slower, 32 x 256 x 56 x 56 -> 64, 1 x 1, 38.2 -> 43.5 us; as it is 1 of 438, 4 x 1 x 244 x 244 -> 100, 63.6 -> 66.7;
// the gather kernel's estimate is up to a third too long for 1 x 1 filters, most for few of them). A form whose waves all sum the
// same channels does not take over from the kernel that sums them apart: its error was up to 1.3 times as large there, everywhere else and
// of the other forms it is 0.2 to 0.9 of the kernels' before. Nor does a wide form from one whose channels more groups share (64 x 56 x 56 -> 128 by two
// 1.35e-7 of the outputs' norm by one group, 1.0e-7 by two; 128 x 25 x 25 -> 256 would go from 1.0e-7 to 1.4e-7 with 33.6 -> 23.7 us).
// `best_cost`: of what is chosen, either way. `skip`: the fastest form that sums a 1 x 1 convolution too, with that, whatever the kernels before take.
static int choose_packed_conv(PackedConvArgs& pa, int kind, int cus, double besides, double& best_cost, bool skip = false) {
    const ConvArgs& p = pa.c;
    bool summed_apart;
    best_cost = (kind != PC_1X1 ? 0.9 : p.M > 64 ? 0.85 : 0.7) * unpacked_conv_cost(p, cus, summed_apart) - besides;
    if (skip) best_cost = 1e300;
    int best = -1, last_bp = 0, strip_w = 0;
    int64_t pixels = 0;
    for (int turn = 0; turn < 6; ++turn)   // (the wide forms last: they are held against the pick of the others)
        for (int i = 0; i < kNumPackedConvForms; ++i) {
            const PackedConvForm& f = kPackedConvForms[i];
            const int bp = turn < 4 ? 256 >> turn : 128 >> (turn - 4);
            if (f.bp != bp || (f.bm == WIDE) != (turn >= 4) || (summed_apart && f.waves_k == 1)) continue;
            if (f.bm == WIDE && best >= 0 && kPackedConvForms[best].waves_k > f.waves_k) continue;
            if (bp != last_bp) pixels = choose_strips(pa, kind, bp, strip_w);
            last_bp = bp;
            if (!packed_conv_lds(kind, f, pixels, skip)) continue;
            const PackedConvCost& c = f.kinds[kind];
            const int64_t nwg = ceil_div((int64_t)p.M, (int64_t)f.bm) * ceil_div(p.P, (int64_t)f.bp), up = ceil_div(nwg, (int64_t)cus);
            const double more = up <= 6 ? (double)(up - 1) : (double)nwg / cus - 0.5;
            const bool few = kind == PC_7X7;
            const double stages = few ? 1 : (double)packed_conv_stages(pa, kind, f), steps = few ? packed_conv_steps(kind) : stages;
            const double patch = stages * (double)pixels / 100;
            double cost = c.fixed + c.per_step * steps + c.per_pixel * patch + more * (c.again + c.again_step * steps + c.again_pixel * patch);
            if (skip) cost += (double)skip_stages(pa, f) * f.skip * (1 + 0.65 * more);
            if (cost < best_cost) { best = i; best_cost = cost; }
        }
    return best;
}

// The form that takes a call, -1 where mi355x_conv2d_res_f32 does: the fastest, or the one that is forced (MI355X_CONV_PACKED) if its
// patch fits. With its strips, its patch's pixels and its LDS.
static int packed_conv_form(PackedConvArgs& pa, int kind, int cus, double besides, int& strip_w, int64_t& pixels, int& lds, bool skip = false) {
    double cost;
    const int force = tuning().conv_packed, form = force >= 0 ? force - 1 : choose_packed_conv(pa, kind, cus, besides, cost, skip);
    if (form < 0 || form >= kNumPackedConvForms) return -1;
    pixels = choose_strips(pa, kind, kPackedConvForms[form].bp, strip_w);
    lds = packed_conv_lds(kind, kPackedConvForms[form], pixels, skip);
    return lds > 0 ? form : -1;
}

// The other input of a call with a 1 x 1 convolution summed too; false where the kernel does not take it. (After packed_conv_args.)
static bool skip_args(PackedConvArgs& pa, int kind, int64_t C2, int64_t H2, int64_t Wd2, const int64_t* strides2) {
    const ConvArgs& p = pa.c;
    if (kind != PC_3X3 || C2 < 8 || C2 % 8 || C2 >= (1 << 24) || H2 < 1 || H2 >= (1 << 20) || Wd2 < 1 || Wd2 >= (1 << 20)) return false;
    for (int i = 0; i < 2; ++i)
        if (strides2[i] < 1 || strides2[i] >= (1 << 10)) return false;
    if ((H2 - 1) / strides2[0] + 1 != p.OH || (Wd2 - 1) / strides2[1] + 1 != p.OW) return false;
    const int64_t limit = (int64_t)1 << 29;
    if (p.N * C2 >= limit || p.N * C2 * H2 >= limit || p.N * C2 * H2 * Wd2 >= limit) return false;
    pa.C2 = (int)C2; pa.H2 = (int)H2; pa.Wd2 = (int)Wd2; pa.stride2_h = (int)strides2[0]; pa.stride2_w = (int)strides2[1];
    pa.groups2 = (int)ceil_div(C2, (int64_t)16);
    return ceil_div((int64_t)p.M, (int64_t)32) * pa.groups2 * PK_FRAGMENT < ((int64_t)1 << 31);
}

// The same in parts of the channels, whose sums a launch of its own adds up (`mean`: in place of one that takes their mean): the form, its parts and their time.
// For one or a few images, of which the last layers are a few tiles with long sums; up to 256 positions, which a wave of the launch that adds up goes
// through in turns. Weights from beyond the L2: 1 x 512 x 7 x 7 -> 512 18.5 us in one part, 12.5 in four (with the mean after it 20.7 and 12.7), 1 x 256 x
// 14 x 14 -> 512 by two 12.7 and 11.3, 2 x 256 x 14 x 14 -> 256 13.2 and 11.8, 4 x 512 x 7 x 7 22.8 and 14.4. Of 20 layers none is behind.
// `parts`: 0 for as many as pay, which it is set to, or how many are asked for.
static int choose_conv_parts(PackedConvArgs& pa, int kind, int cus, bool mean, int64_t& parts, double& best_cost) {
    const ConvArgs& p = pa.c;
    const int64_t asked = parts;
    int best = -1, strip_w = 0;
    best_cost = 1e300;
    if (kind != PC_3X3 || p.OHW > 256) return -1;
    for (int i = 0; i < kNumPackedConvForms; ++i) {
        const PackedConvForm& f = kPackedConvForms[i];
        const int64_t pixels = choose_strips(pa, kind, f.bp, strip_w), all = packed_conv_stages(pa, kind, f);
        if (f.bm == WIDE || f.waves_k == 1 || !packed_conv_lds(kind, f, pixels)) continue;   // (forms whose groups share the channels: no more error than the kernels before)
        for (const int n : {2, 4}) {
            if ((asked && n != asked) || all % n || pa.groups % (n * f.waves_k)) continue;
            const PackedConvCost& c = f.kinds[kind];
            const int64_t nwg = n * ceil_div((int64_t)p.M, (int64_t)f.bm) * ceil_div(p.P, (int64_t)f.bp), up = ceil_div(nwg, (int64_t)cus);
            const double more = up <= 6 ? (double)(up - 1) : (double)nwg / cus - 0.5, stages = (double)(all / n), patch = stages * (double)pixels / 100;
            const double sums = (mean ? 300 : 2300) + 4.0 * (n + 2) * (double)p.M * (double)p.P / 2000.0;
            const double cost = c.fixed + c.per_step * stages + c.per_pixel * patch + more * (c.again + c.again_step * stages + c.again_pixel * patch) + sums;
            if (cost < best_cost) { best = i; parts = n; best_cost = cost; }
        }
    }
    return best;
}

// Nanoseconds of mi355x_pack_conv_f32 before the convolution (512 x 256 filters of one tap 3.8 us, 768 x 512 of nine 16.5).
constexpr double PACKING = 3000, PACKING_PER_WEIGHT = 0.004;

}  // namespace mi355x

extern "C" int64_t mi355x_conv2d_packed_pays(int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW,
                                             const int64_t* pads, const int64_t* strides, const int64_t* dilations, int constant) {
    using namespace mi355x;
    PackedConvArgs pa = {};
    int kind;
    if (!pads || !strides || !dilations || !packed_conv_args(pa, kind, N, C, H, Wd, M, KH, KW, pads, strides, dilations)) return 0;
    const int cus = device_cus();
    const double packing = constant ? 0 : PACKING + PACKING_PER_WEIGHT * (double)M * pa.c.K;
    int strip_w, lds;
    int64_t pixels;
    if (packed_conv_form(pa, kind, cus > 0 ? cus : 256, packing, strip_w, pixels, lds) < 0) return 0;
    return ceil_div(M, (int64_t)32) * pa.groups * packed_conv_steps(kind) * PK_FRAGMENT;
}

extern "C" int mi355x_pack_conv_f32(const float* w, void* packed, int64_t M, int64_t C, int64_t KH, int64_t KW, void* stream) {
    using namespace mi355x;
    const int64_t ones[2] = {1, 1};
    MI355X_REQUIRE(M >= 1 && M < (1 << 24) && C >= 1 && C < (1 << 24) && packed_conv_kind(C, KH, KW, ones) != PC_NONE,
                   "pack: no packed form of %lld filters of %lld x %lld x %lld", (long long)M, (long long)C, (long long)KH, (long long)KW);
    MI355X_REQUIRE(w && packed && (reinterpret_cast<uintptr_t>(packed) & 15) == 0, "pack: null or unaligned pointer");
    const int steps = packed_conv_steps(packed_conv_kind(C, KH, KW, ones)), groups = C <= 4 ? 1 : (int)ceil_div(C, (int64_t)16);
    const int64_t units = ceil_div(M, (int64_t)32) * groups * steps * WAVE;
    MI355X_REQUIRE(grid_fits(ceil_div(units, (int64_t)256), 256), "pack: grid too large");
    hipLaunchKernelGGL(pack_conv_f32_kernel, dim3((unsigned)ceil_div(units, (int64_t)256)), dim3(256), 0, static_cast<hipStream_t>(stream), w,
                       static_cast<u32x4*>(packed), (int)M, (int)C, (int)KH, (int)KW, groups, steps, units);
    return check_launch("pack_conv_f32_kernel");
}

extern "C" int mi355x_conv2d_packed_f32(const float* X, const void* packed, const float* W, const float* bias, const float* residual,
                                        float* Y, int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW,
                                        const int64_t* pads, const int64_t* strides, const int64_t* dilations, int epilogue, void* stream) {
    using namespace mi355x;
    if (X && W && Y && packed && pads && strides && dilations && (reinterpret_cast<uintptr_t>(packed) & 15) == 0 &&
        (epilogue & ~(MI355X_EPI_BIAS | MI355X_EPI_RELU | MI355X_EPI_RESIDUAL | MI355X_EPI_RELU_AFTER)) == 0 &&
        (!(epilogue & MI355X_EPI_BIAS) || bias) && (!(epilogue & MI355X_EPI_RESIDUAL) || residual)) {
        PackedConvArgs pa = {};
        ConvArgs& p = pa.c;
        int kind;
        if (packed_conv_args(pa, kind, N, C, H, Wd, M, KH, KW, pads, strides, dilations)) {
            const int cus = device_cus();
            if (cus <= 0) return set_error(MI355X_ERR_NOT_INITIALIZED, "conv2d: no usable HIP device");
            int strip_w, lds;
            int64_t pixels;
            const int form = packed_conv_form(pa, kind, cus, 0, strip_w, pixels, lds);
            if (form >= 0) {
                const PackedConvForm& f = kPackedConvForms[form];
                p.X = X; p.W = W; p.bias = bias; p.residual = residual; p.Y = Y; p.epi = epilogue;
                p.tiles_m = ceil_div(M, (int64_t)f.bm);
                p.tiles_p = ceil_div(p.P, (int64_t)f.bp);
                p.nwg = p.tiles_m * p.tiles_p;
                pa.packed = static_cast<const char*>(packed);
                pa.stages = (int)packed_conv_stages(pa, kind, f);
                hipStream_t st = static_cast<hipStream_t>(stream);
                if (grid_fits(p.nwg, f.waves * WAVE)) {
                    set_strips(pa, kind, strip_w, pixels);
                    switch (kind) {
                        case PC_3X3: launch_packed_conv<PackedFilter<3, 3, false>, false, 1, 0>(form, pa, lds, st); break;
                        case PC_1X1: launch_packed_conv<PackedFilter<1, 1, false>, false, 2, 1>(form, pa, lds, st); break;
                        default: launch_packed_conv<PackedFilter<7, 7, true>, true, 1, 2>(form, pa, lds, st); break;
                    }
                    return check_launch("conv2d_f32_packed_kernel");
                }
            }
        }
    }
    return mi355x_conv2d_res_f32(X, W, bias, residual, Y, N, C, H, Wd, M, KH, KW, pads, strides, dilations, epilogue, stream);
}

extern "C" int mi355x_conv2d_skip_pays(int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW, const int64_t* pads,
                                       const int64_t* strides, const int64_t* dilations, int64_t C2, int64_t H2, int64_t Wd2, const int64_t* strides2) {
    using namespace mi355x;
    PackedConvArgs pa = {}, pointwise = {};
    int kind, kind2;
    const int64_t none[4] = {0, 0, 0, 0}, ones[2] = {1, 1};
    if (!pads || !strides || !dilations || !strides2 || !packed_conv_args(pa, kind, N, C, H, Wd, M, KH, KW, pads, strides, dilations) ||
        !skip_args(pa, kind, C2, H2, Wd2, strides2) || !packed_conv_args(pointwise, kind2, N, C2, H2, Wd2, M, 1, 1, none, strides2, ones)) return 0;
    int cus = device_cus();
    if (cus <= 0) cus = 256;
    if (tuning().conv_packed >= 0) {
        int strip_w, lds;
        int64_t pixels;
        return packed_conv_form(pa, kind, cus, 0, strip_w, pixels, lds, true) >= 0;
    }
    double both, conv, alone;
    if (choose_packed_conv(pa, kind, cus, 0, both, true) < 0) return 0;
    choose_packed_conv(pa, kind, cus, 0, conv);
    choose_packed_conv(pointwise, kind2, cus, 0, alone);
    return both < conv + alone - 500;   // (one image: 128 x 28 x 28 13.5 us as two launches, 12.7 as one, 256 x 14 x 14 14.8 and 16.6; 32 images 57 and 49, 54 and 48)
}

extern "C" int mi355x_conv2d_skip_f32(const float* X, const float* W, const void* packed, const float* bias, const float* X2, const float* W2, const void* packed2,
                                      const float* bias2, float* scratch, float* Y, int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW,
                                      const int64_t* pads, const int64_t* strides, const int64_t* dilations, int64_t C2, int64_t H2, int64_t Wd2,
                                      const int64_t* strides2, int epilogue, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE((epilogue & ~(MI355X_EPI_BIAS | MI355X_EPI_RELU_AFTER)) == 0, "conv2d_skip: unknown epilogue bits 0x%x", epilogue);
    auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    PackedConvArgs pa = {};
    ConvArgs& p = pa.c;
    int kind;
    if (X && W && Y && packed && X2 && W2 && packed2 && al16(packed) && al16(packed2) && pads && strides && dilations && strides2 &&
        (!(epilogue & MI355X_EPI_BIAS) || bias) && packed_conv_args(pa, kind, N, C, H, Wd, M, KH, KW, pads, strides, dilations) &&
        skip_args(pa, kind, C2, H2, Wd2, strides2)) {
        const int cus = device_cus();
        if (cus <= 0) return set_error(MI355X_ERR_NOT_INITIALIZED, "conv2d: no usable HIP device");
        int strip_w, lds;
        int64_t pixels;
        const int form = packed_conv_form(pa, kind, cus, 0, strip_w, pixels, lds, true);
        if (form >= 0) {
            const PackedConvForm& f = kPackedConvForms[form];
            p.X = X; p.W = W; p.bias = bias; p.Y = Y; p.epi = epilogue;
            pa.X2 = X2; pa.W2 = W2; pa.packed2 = static_cast<const char*>(packed2); pa.bias2 = bias2;
            p.tiles_m = ceil_div(M, (int64_t)f.bm);
            p.tiles_p = ceil_div(p.P, (int64_t)f.bp);
            p.nwg = p.tiles_m * p.tiles_p;
            pa.packed = static_cast<const char*>(packed);
            pa.stages = (int)packed_conv_stages(pa, kind, f);
            pa.stages2 = (int)skip_stages(pa, f);
            if (grid_fits(p.nwg, f.waves * WAVE)) {
                set_strips(pa, kind, strip_w, pixels);
                launch_packed_conv<PackedFilter<3, 3, false>, false, 1, 0, true>(form, pa, lds, static_cast<hipStream_t>(stream));
                return check_launch("conv2d_f32_packed_kernel");
            }
        }
    }
    MI355X_REQUIRE(strides2 && scratch, "conv2d_skip: null pointer");
    const int64_t none[4] = {0, 0, 0, 0}, ones[2] = {1, 1};
    const int status = mi355x_conv2d_packed_f32(X2, packed2, W2, bias2, nullptr, scratch, N, C2, H2, Wd2, M, 1, 1, none, strides2, ones, bias2 ? MI355X_EPI_BIAS : 0, stream);
    if (status != MI355X_OK) return status;
    return mi355x_conv2d_packed_f32(X, packed, W, bias, scratch, Y, N, C, H, Wd, M, KH, KW, pads, strides, dilations, epilogue | MI355X_EPI_RESIDUAL, stream);
}

extern "C" int64_t mi355x_conv2d_parts(int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW, const int64_t* pads,
                                       const int64_t* strides, const int64_t* dilations, int mean) {
    using namespace mi355x;
    PackedConvArgs pa = {};
    int kind;
    int64_t parts = 0;
    if (!pads || !strides || !dilations || !packed_conv_args(pa, kind, N, C, H, Wd, M, KH, KW, pads, strides, dilations) || tuning().conv_packed >= 0) return 1;
    int cus = device_cus();
    if (cus <= 0) cus = 256;
    double apart, whole;
    if (choose_conv_parts(pa, kind, cus, mean, parts, apart) < 0) return 1;
    choose_packed_conv(pa, kind, cus, 0, whole);
    return apart < whole ? parts : 1;
}

extern "C" int mi355x_conv2d_parts_f32(const float* X, const float* W, const void* packed, const float* bias, const float* residual, float* P, int64_t parts, float* Y,
                                       int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW, const int64_t* pads, const int64_t* strides,
                                       const int64_t* dilations, int epilogue, int mean, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE((epilogue & ~(MI355X_EPI_BIAS | MI355X_EPI_RELU | MI355X_EPI_RESIDUAL | MI355X_EPI_RELU_AFTER)) == 0, "conv2d_parts: unknown epilogue bits 0x%x", epilogue);
    MI355X_REQUIRE((!(epilogue & MI355X_EPI_BIAS) || bias) && (!(epilogue & MI355X_EPI_RESIDUAL) || residual), "conv2d_parts: null bias or residual");
    MI355X_REQUIRE(parts >= 1, "conv2d_parts: %lld parts", (long long)parts);
    PackedConvArgs pa = {};
    ConvArgs& p = pa.c;
    int kind;
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (X && W && P && Y && packed && pads && strides && dilations && (reinterpret_cast<uintptr_t>(packed) & 15) == 0 &&
        packed_conv_args(pa, kind, N, C, H, Wd, M, KH, KW, pads, strides, dilations)) {
        const int cus = device_cus();
        if (cus <= 0) return set_error(MI355X_ERR_NOT_INITIALIZED, "conv2d: no usable HIP device");
        int strip_w;
        double cost;
        const int form = choose_conv_parts(pa, kind, cus, mean, parts, cost);   // (P has room for that many)
        const int64_t rows = N * M, positions = p.OHW;
        if (form >= 0 && grid_fits(ceil_div(rows, (int64_t)4), 256)) {
            const PackedConvForm& f = kPackedConvForms[form];
            const int64_t pixels = choose_strips(pa, kind, f.bp, strip_w);
            p.X = X; p.W = W; p.Y = P; p.epi = 0;
            p.tiles_m = ceil_div(M, (int64_t)f.bm);
            p.tiles_p = ceil_div(p.P, (int64_t)f.bp);
            p.nwg = parts * p.tiles_m * p.tiles_p;
            pa.packed = static_cast<const char*>(packed);
            pa.stages = (int)(packed_conv_stages(pa, kind, f) / parts);
            pa.part_size = rows * positions;
            if (grid_fits(p.nwg, f.waves * WAVE)) {
                set_strips(pa, kind, strip_w, pixels);
                launch_packed_conv<PackedFilter<3, 3, false>, false, 1, 0>(form, pa, packed_conv_lds(kind, f, pixels), st);
                const int status = check_launch("conv2d_f32_packed_kernel");
                if (status != MI355X_OK) return status;
                const dim3 grid((unsigned)ceil_div(rows, (int64_t)4));
                if (mean) hipLaunchKernelGGL(conv_parts_kernel<true>, grid, dim3(256), 0, st, P, (int)parts, bias, residual, Y, rows, (int)M, (int)positions, epilogue);
                else hipLaunchKernelGGL(conv_parts_kernel<false>, grid, dim3(256), 0, st, P, (int)parts, bias, residual, Y, rows, (int)M, (int)positions, epilogue);
                return check_launch("conv_parts_kernel");
            }
        }
    }
    MI355X_REQUIRE(!mean || P, "conv2d_parts: null pointer");
    const int status = mi355x_conv2d_packed_f32(X, packed, W, bias, residual, mean ? P : Y, N, C, H, Wd, M, KH, KW, pads, strides, dilations, epilogue, stream);
    if (status != MI355X_OK || !mean) return status;
    const int64_t OH = (H + pads[0] + pads[2] - (KH - 1) * dilations[0] - 1) / strides[0] + 1, OW = (Wd + pads[1] + pads[3] - (KW - 1) * dilations[1] - 1) / strides[1] + 1;
    return mi355x_reduce_mean_f32(P, Y, N * M, OH * OW, 1, stream);
}
