// ONNX Conv of 7 x 7 filters by two over three channels, Relu and MaxPool of 3 x 3 by two as one launch: the stem of an image classifier.
//
// Apart, the convolution writes four times what the pooling keeps (103 MB of 26 for 32 images of 224 x 224 and 64 filters) and the pooling reads
// it again. Here a workgroup computes the convolution under a tile of PT_H x PT_W pooled outputs, (2 PT_H + 1) x (2 PT_W + 1) positions of which
// the border is computed by its neighbours too, keeps it in LDS and stores the maxima.
//
// The arithmetic is that of conv2d_f32_packed.hip (three bf16 parts of every value, six products, two sets of accumulators; sums that are not
// finite again with the fp32 MFMA), with another order of k: a pixel's three channels side by side, so that the seven taps of a filter row are
// 21 values in a row, three units of eight, and the filter 11 MFMA steps of 16 where four channels and eight taps take 14.
//   * The input under the tile is split once on its way into LDS, a plane for each part; a position's unit is 16 bytes from any multiple of
//     four on (positions are 12 bytes apart: neighbouring lanes start three banks apart).
//   * Small tiles (64 positions) for one or two images, whose larger tiles would leave most CUs idle.
//   * Filters, packed in fragment order, go from memory straight into registers, three steps ahead.
// What bounds it: the matrix products at the clock they leave (38 of 61 us for 32 images, the tiles' shared borders among them), of the rest splitting the input
// and the maxima, which overlap with another workgroup's products only in part. Against the two launches before it, 224 x 224 by 64 filters: one image
// 13.0 -> 6.9 us, 4 images 23.7 -> 11.4, 8 images 36.1 -> 18.9, 32 images 89.6 -> 61.2; 96 x 96 8.8 -> 5.1; 20 images of 256 x 256 77 -> 56.
// (With nine reads for each maximum 65 us where walking down columns takes 61.)
// Padded positions, those outside the convolution's result, are -inf in LDS and take no part; NaN wins a maximum, as in pool_norm.hip.
#include "common.h"
#include "gemm_tile.h"
#include "conv_args.h"
#include "split_bf16.h"

namespace mi355x {

constexpr int CP_TAPS = 7, CP_CHANNELS = 3, CP_ROW = CP_TAPS * CP_CHANNELS, CP_UNITS = 3 * CP_TAPS, CP_STEPS = (CP_UNITS + 1) / 2;

struct ConvPoolArgs {
    const float* X; const char* packed; const float* W; const float* bias; float* Y;
    int N, H, Wd, M, OH, OW, PH, PW;                // input, convolution, pooled
    int pad_t, pad_l, pool_t, pool_l;
    int tiles_m, tiles_x, tiles_y, epi;
    int64_t nwg;
};

template <int PT_H, int PT_W, int WAVES_M, int WAVES_P, int TP>
__global__ __launch_bounds__(WAVES_M * WAVES_P * WAVE, 2) void conv2d_f32_pool_kernel(ConvPoolArgs p) {
    constexpr int THREADS = WAVES_M * WAVES_P * WAVE, CH = 2 * PT_H + 1, CW = 2 * PT_W + 1, POSITIONS = CH * CW, BP = 32 * TP * WAVES_P;
    static_assert(POSITIONS <= BP, "a place for every position");
    constexpr int PATCH_H = 2 * (CH - 1) + CP_TAPS, PATCH_W = 2 * (CW - 1) + CP_TAPS + 1;   // (one column more: units end in the eighth tap)
    constexpr int ROW = PATCH_W * CP_CHANNELS * 2, PLANE = PATCH_H * ROW;                   // bytes
    constexpr int PITCH = BP + 16, BM = 32 * WAVES_M, RING = 3;
    static_assert(PATCH_W % 2 == 0, "pairs of pixels");
    extern __shared__ __attribute__((aligned(16))) char lds[];

    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int li = lane % 32, lh = lane / 32;
    const int wm = wave % WAVES_M, wp = wave / WAVES_M;
    // consecutive tiles share their input, then are neighbours
    uint32_t t = (uint32_t)xcd_remap(blockIdx.x, p.nwg);
    const int m0 = (int)(t % (uint32_t)p.tiles_m) * BM;
    t /= (uint32_t)p.tiles_m;
    const int px0 = (int)(t % (uint32_t)p.tiles_x) * PT_W;
    t /= (uint32_t)p.tiles_x;
    const int py0 = (int)(t % (uint32_t)p.tiles_y) * PT_H, n = (int)(t / (uint32_t)p.tiles_y);
    const int cy0 = 2 * py0 - p.pool_t, cx0 = 2 * px0 - p.pool_l;   // the tile's first position, maybe a padded one
    const int y0 = 2 * cy0 - p.pad_t, x0 = 2 * cx0 - p.pad_l;       // its first tap

    constexpr uint32_t OUT = 0x80000000u;   // an offset that makes a load return zero
    const float* X = p.X + (int64_t)n * CP_CHANNELS * p.H * p.Wd;
    const int plane = p.H * p.Wd * 4;
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(X), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(p.packed), 0, 0x7fffffff, 0x00020000);

    bf16x8 fw[RING][SP_PLANES], fx[2][SP_PLANES];
    const uint32_t w_block = (uint32_t)min(m0 / 32 + wm, (p.M + 31) / 32 - 1) * (uint32_t)(CP_STEPS * PK_FRAGMENT);
    auto load_w = [&](int slot, int step) {
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q)
            fw[slot][q] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, lane * 16 + q * PK_PLANE, (int)(w_block + (uint32_t)(step * PK_FRAGMENT)), 0));
    };
#pragma unroll
    for (int s = 0; s < RING; ++s) load_w(s, s);

    // the patch, two pixels of a row at a time: six values, three words of each plane
    constexpr int PAIRS = PATCH_H * PATCH_W / 2, PER_T = (PAIRS + THREADS - 1) / THREADS;
    {
        float v[PER_T][6];
#pragma unroll
        for (int it = 0; it < PER_T; ++it) {
            const int pair = tid + it * THREADS, row = pair / (PATCH_W / 2), column = 2 * (pair % (PATCH_W / 2));
            const int y = y0 + row;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int x = x0 + column + h;
                const uint32_t off = pair < PAIRS && (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.Wd ? 4u * (uint32_t)(y * p.Wd + x) : OUT;
#pragma unroll
                for (int c = 0; c < CP_CHANNELS; ++c)
                    v[it][3 * h + c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(x_rsrc, (int)off, c * plane, 0));
            }
        }
#pragma unroll
        for (int it = 0; it < PER_T; ++it) {
            const int pair = tid + it * THREADS;
            uint32_t part[SP_PLANES][3];
#pragma unroll
            for (int h = 0; h < 3; ++h) split_pair(v[it][2 * h], v[it][2 * h + 1], part[0][h], part[1][h], part[2][h]);
            if (pair < PAIRS)
#pragma unroll
                for (int q = 0; q < SP_PLANES; ++q)
#pragma unroll
                    for (int h = 0; h < 3; ++h) *reinterpret_cast<uint32_t*>(lds + q * PLANE + pair * 12 + 4 * h) = part[q][h];
        }
    }

    // A lane's two halves multiply units 2 s and 2 s + 1 of the 21: the second follows the first in its row, or begins the next one. The last step has
    // one unit, which the upper half reads too (against zeros of the filter).
    int at[TP], at_next[TP], at_last[TP];
#pragma unroll
    for (int j = 0; j < TP; ++j) {
        const int pos = min(32 * (wp * TP + j) + li, POSITIONS - 1);
        at_last[j] = 2 * (pos / CW) * ROW + 2 * (pos % CW) * CP_CHANNELS * 2;
        at[j] = at_last[j] + lh * 16;
        at_next[j] = at_last[j] + lh * (ROW - 32);
    }
    auto read_x = [&](int slot, int j, int step) {
        const int unit = 2 * step, from = (step + 1 == CP_STEPS ? at_last[j] : unit % 3 == 2 ? at_next[j] : at[j]) + unit / 3 * ROW + unit % 3 * 16;
        typedef u32x2 words __attribute__((aligned(4)));
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q) {
            const u32x2 a = *reinterpret_cast<const words*>(lds + from + q * PLANE), b = *reinterpret_cast<const words*>(lds + from + q * PLANE + 8);
            fx[slot][q] = __builtin_bit_cast(bf16x8, u32x4{a.x, a.y, b.x, b.y});
        }
    };
    f32x16 acc[TP], small[TP];
#pragma unroll
    for (int j = 0; j < TP; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[j][r] = small[j][r] = 0.f;
    __syncthreads();
    read_x(0, 0, 0);
    static_for<CP_STEPS * TP>([&](auto tag) {
        constexpr int now = decltype(tag)::value, step = now / TP, j = now % TP, slot = step % RING;
        if constexpr (now + 1 < CP_STEPS * TP) read_x((now + 1) % 2, (now + 1) % TP, (now + 1) / TP);
        __builtin_amdgcn_sched_barrier(0);   // (left alone, the compiler moves loads down to their uses)
#pragma unroll
        for (int u = 0; u < PK_PRODUCTS; ++u) {
            f32x16& sum = u == 0 ? acc[j] : small[j];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fw[slot][PK_QA[u]], fx[now % 2][PK_QB[u]], sum, 0, 0, 0);
        }
        if constexpr (j + 1 == TP && step + RING < CP_STEPS) load_w(slot, step + RING);
        __builtin_amdgcn_sched_barrier(0);
    });

    const int mb = m0 + 32 * wm;
#pragma unroll
    for (int j = 0; j < TP; ++j) {
        acc[j] = (acc[j] + small[j]) * SP_UNSCALE;
        float probe = 0.f;   // stays 0 while every sum is finite
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = fmaf(acc[j][r], 0.f, probe);
        if (__builtin_expect(__any(probe != 0.f), 0)) {   // (NaN compares unequal) this block again with the fp32 MFMA, straight from memory
            const int pos = min(32 * (wp * TP + j) + li, POSITIONS - 1);
            const int iy = y0 + 2 * (pos / CW), ix = x0 + 2 * (pos % CW);
            const float* w = p.W + (int64_t)min(mb + li, p.M - 1) * (CP_ROW * CP_TAPS);
            f32x16 sum;
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = 0.f;
            for (int k = 0; k < CP_ROW * CP_TAPS; k += 2) {
                const int kk = min(k + lh, CP_ROW * CP_TAPS - 1), c = kk / (CP_TAPS * CP_TAPS), tap = kk % (CP_TAPS * CP_TAPS);
                const int y = iy + tap / CP_TAPS, x = ix + tap % CP_TAPS;
                const bool counted = k + lh < CP_ROW * CP_TAPS, in = counted && (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.Wd;
                const float xv = in ? X[((int64_t)c * p.H + y) * p.Wd + x] : 0.f;
                sum = __builtin_amdgcn_mfma_f32_32x32x2f32(counted ? w[kk] : 0.f, xv, sum, 0, 0, 0);
            }
            acc[j] = sum;
        }
    }

    // acc[j][r]: filter 8 (r / 4) + 4 lh + r % 4 of the block, position li
    float bias[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int m = mb + 8 * (r / 4) + 4 * lh + r % 4;
        bias[r] = (p.epi & MI355X_EPI_BIAS) && m < p.M ? p.bias[m] : 0.f;
    }
    float* result = reinterpret_cast<float*>(lds);   // [filter][position], in the place of the patch
    const bool inside = cy0 >= 0 && cx0 >= 0 && cy0 + CH <= p.OH && cx0 + CW <= p.OW;   // (uniform: most tiles)
    __syncthreads();
#pragma unroll
    for (int j = 0; j < TP; ++j) {
        const int pos = 32 * (wp * TP + j) + li;
        const bool in = inside || ((unsigned)(cy0 + pos / CW) < (unsigned)p.OH && (unsigned)(cx0 + pos % CW) < (unsigned)p.OW);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            float o = acc[j][r] + bias[r];
            if (p.epi & MI355X_EPI_RELU) o = fmaxf(o, 0.f);
            result[(32 * wm + 8 * (r / 4) + 4 * lh + r % 4) * PITCH + pos] = in ? o : -INFINITY;
        }
    }
    __syncthreads();
    // a thread walks down a column of pooled outputs of one filter: the largest of three neighbours in each row, then of three rows
    for (int i = tid; i < BM * PT_W; i += THREADS) {
        const int m = i / PT_W, px = i % PT_W;
        if (m0 + m >= p.M || px0 + px >= p.PW) continue;
        const float* from = result + m * PITCH + 2 * px;
        auto row = [&](int y) { return __builtin_elementwise_maximum(__builtin_elementwise_maximum(from[y * CW], from[y * CW + 1]), from[y * CW + 2]); };
        float* to = p.Y + (((int64_t)n * p.M + m0 + m) * p.PH + py0) * p.PW + px0 + px;
        float above = row(0);
#pragma unroll
        for (int py = 0; py < PT_H; ++py) {
            const float middle = row(2 * py + 1), below = row(2 * py + 2);
            if (py0 + py < p.PH) to[py * p.PW] = __builtin_elementwise_maximum(__builtin_elementwise_maximum(above, middle), below);
            above = below;
        }
    }
}

// One unit (a lane's share of a fragment) per thread, once when a graph is prepared. Filter block, step, lane.
__global__ void pack_conv_pool_f32_kernel(const float* w, u32x4* packed, int M, int units) {
    const int i = (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i >= units) return;
    const int l = i % WAVE, step = i / WAVE % CP_STEPS, m = i / WAVE / CP_STEPS * 32 + l % 32, unit = 2 * step + l / 32;
    f32x4 v[2];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int at = unit % 3 * 8 + e, r = unit / 3;
        v[e / 4][e % 4] = m < M && unit < CP_UNITS && at < CP_ROW ? w[((m * CP_CHANNELS + at % 3) * CP_TAPS + r) * CP_TAPS + at / 3] : 0.f;
    }
    u32x4 part[SP_PLANES];
    split_unit8(v[0], v[1], part);
#pragma unroll
    for (int q = 0; q < SP_PLANES; ++q) packed[((i / WAVE) * SP_PLANES + q) * WAVE + l] = part[q];
}

// Tiles, filters and positions of a workgroup, and nanoseconds: `fixed` while every workgroup has a CU to itself, `again` for each further one
// on the same CU (by halves from seven on), from 17 stems of 1 to 32 images of 96 to 256 columns; the pick is at most 6 % behind the fastest form there.
struct ConvPoolForm { int pt_h, pt_w, bm, bp; double fixed, again; };
constexpr ConvPoolForm kConvPoolForms[] = {{8, 7, 64, 256, 12150, 7700}, {7, 8, 64, 256, 11650, 7500}, {8, 7, 32, 256, 8000, 4050}, {7, 8, 32, 256, 7700, 3950},
                                           {5, 5, 64, 128, 7450, 3850}, {4, 3, 64, 64, 5200, 2300}, {3, 4, 64, 64, 5100, 2250}};
constexpr int kNumConvPoolForms = sizeof(kConvPoolForms) / sizeof(kConvPoolForms[0]);

template <int PT_H, int PT_W, int WAVES_M, int WAVES_P, int TP>
static void launch_conv_pool_form(const ConvPoolArgs& p, hipStream_t st) {
    constexpr int CH = 2 * PT_H + 1, CW = 2 * PT_W + 1, PATCH = SP_PLANES * (2 * (CH - 1) + CP_TAPS) * (2 * (CW - 1) + CP_TAPS + 1) * CP_CHANNELS * 2;
    constexpr int RESULT = 32 * WAVES_M * (32 * TP * WAVES_P + 16) * 4, LDS = PATCH > RESULT ? PATCH : RESULT;
    hipLaunchKernelGGL((conv2d_f32_pool_kernel<PT_H, PT_W, WAVES_M, WAVES_P, TP>), dim3((unsigned)p.nwg), dim3(WAVES_M * WAVES_P * WAVE), LDS, st, p);
}

static int64_t set_form(ConvPoolArgs& p, const ConvPoolForm& f) {
    p.tiles_m = (int)ceil_div(p.M, f.bm);
    p.tiles_x = (int)ceil_div(p.PW, f.pt_w);
    p.tiles_y = (int)ceil_div(p.PH, f.pt_h);
    p.nwg = (int64_t)p.N * p.tiles_m * p.tiles_x * p.tiles_y;
    return p.nwg;
}

// Geometry of a call; false where the kernel does not take it.
static bool conv_pool_args(ConvPoolArgs& p, int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW, const int64_t* pads,
                           const int64_t* strides, const int64_t* dilations, int64_t PKH, int64_t PKW, const int64_t* pool_pads,
                           const int64_t* pool_strides, const int64_t* pool_dilations) {
    for (int64_t v : {N, H, Wd, M})
        if (v < 1 || v >= (1 << 20)) return false;
    if (C != CP_CHANNELS || KH != CP_TAPS || KW != CP_TAPS || PKH != 3 || PKW != 3) return false;
    for (int i = 0; i < 2; ++i)
        if (strides[i] != 2 || dilations[i] != 1 || pool_strides[i] != 2 || pool_dilations[i] != 1) return false;
    for (int i = 0; i < 4; ++i)
        if (pads[i] < 0 || pads[i] >= CP_TAPS || pool_pads[i] < 0 || pool_pads[i] >= 3) return false;
    const int64_t hin = H + pads[0] + pads[2], win = Wd + pads[1] + pads[3];
    if (hin < KH || win < KW) return false;
    const int64_t OH = (hin - KH) / 2 + 1, OW = (win - KW) / 2 + 1;
    if (OH + pool_pads[0] + pool_pads[2] < 3 || OW + pool_pads[1] + pool_pads[3] < 3) return false;
    const int64_t PH = (OH + pool_pads[0] + pool_pads[2] - 3) / 2 + 1, PW = (OW + pool_pads[1] + pool_pads[3] - 3) / 2 + 1;
    if (C * H * Wd >= ((int64_t)1 << 29) || ceil_div(M, (int64_t)32) * CP_STEPS * PK_FRAGMENT >= ((int64_t)1 << 31)) return false;   // 32-bit byte offsets
    p.N = (int)N; p.H = (int)H; p.Wd = (int)Wd; p.M = (int)M; p.OH = (int)OH; p.OW = (int)OW; p.PH = (int)PH; p.PW = (int)PW;
    p.pad_t = (int)pads[0]; p.pad_l = (int)pads[1]; p.pool_t = (int)pool_pads[0]; p.pool_l = (int)pool_pads[1];
    return true;
}

// The fastest form, or the one that is forced (MI355X_CONV_POOL=n; 0: none, -1 is returned). Some form always: over 102 stems of 1 to 32 images of 96 to 224
// columns and 1 to 512 filters the launch takes 0.21 to 0.75 of the time of the two before it, also where most of a block of 32 filters is padding (one
// filter: one image of 224 x 224 9.0 -> 6.3 us, 32 images 125 -> 26; 512 filters, 32 of 96 x 96: 131 -> 98).
static int choose_conv_pool(ConvPoolArgs& p, int cus) {
    const int force = tuning().conv_pool;
    if (force >= 0) return force <= kNumConvPoolForms ? force - 1 : -1;
    int best = -1;
    double best_cost = 1e300;
    for (int i = 0; i < kNumConvPoolForms; ++i) {
        const ConvPoolForm& f = kConvPoolForms[i];
        const int64_t nwg = set_form(p, f), up = ceil_div(nwg, (int64_t)cus);
        const double more = up <= 6 ? (double)(up - 1) : (double)nwg / cus - 0.5;
        const double cost = f.fixed + more * f.again;
        if (cost < best_cost) { best = i; best_cost = cost; }
    }
    return best;
}

}  // namespace mi355x

extern "C" int64_t mi355x_conv2d_pool_packed_pays(int64_t N, int64_t C, int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW, const int64_t* pads,
                                                  const int64_t* strides, const int64_t* dilations, int64_t PKH, int64_t PKW, const int64_t* pool_pads,
                                                  const int64_t* pool_strides, const int64_t* pool_dilations) {
    using namespace mi355x;
    ConvPoolArgs p = {};
    if (!pads || !strides || !dilations || !pool_pads || !pool_strides || !pool_dilations ||
        !conv_pool_args(p, N, C, H, Wd, M, KH, KW, pads, strides, dilations, PKH, PKW, pool_pads, pool_strides, pool_dilations)) return 0;
    const int cus = device_cus();
    if (choose_conv_pool(p, cus > 0 ? cus : 256) < 0) return 0;
    return ceil_div(M, (int64_t)32) * CP_STEPS * PK_FRAGMENT;
}

extern "C" int mi355x_pack_conv_pool_f32(const float* w, void* packed, int64_t M, int64_t C, int64_t KH, int64_t KW, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(M >= 1 && M < (1 << 20) && C == CP_CHANNELS && KH == CP_TAPS && KW == CP_TAPS, "pack: %lld filters of %lld x %lld x %lld", (long long)M,
                   (long long)C, (long long)KH, (long long)KW);
    MI355X_REQUIRE(w && packed && (reinterpret_cast<uintptr_t>(packed) & 15) == 0, "pack: null or unaligned pointer");
    const int units = (int)ceil_div(M, (int64_t)32) * CP_STEPS * WAVE;
    hipLaunchKernelGGL(pack_conv_pool_f32_kernel, dim3((unsigned)ceil_div(units, 256)), dim3(256), 0, static_cast<hipStream_t>(stream), w, static_cast<u32x4*>(packed),
                       (int)M, units);
    return check_launch("pack_conv_pool_f32_kernel");
}

extern "C" int mi355x_conv2d_pool_packed_f32(const float* X, const float* W, const void* packed, const float* bias, float* scratch, float* Y, int64_t N, int64_t C,
                                             int64_t H, int64_t Wd, int64_t M, int64_t KH, int64_t KW, const int64_t* pads, const int64_t* strides,
                                             const int64_t* dilations, int epilogue, int64_t PKH, int64_t PKW, const int64_t* pool_pads,
                                             const int64_t* pool_strides, const int64_t* pool_dilations, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(pads && strides && dilations && pool_pads && pool_strides && pool_dilations, "conv2d_pool: null array");
    ConvPoolArgs p = {};
    if (X && W && Y && packed && (reinterpret_cast<uintptr_t>(packed) & 15) == 0 && (epilogue & ~(MI355X_EPI_BIAS | MI355X_EPI_RELU)) == 0 &&
        (!(epilogue & MI355X_EPI_BIAS) || bias) &&
        conv_pool_args(p, N, C, H, Wd, M, KH, KW, pads, strides, dilations, PKH, PKW, pool_pads, pool_strides, pool_dilations)) {
        const int cus = device_cus();
        if (cus <= 0) return set_error(MI355X_ERR_NOT_INITIALIZED, "conv2d: no usable HIP device");
        const int form = choose_conv_pool(p, cus);
        if (form >= 0 && grid_fits(set_form(p, kConvPoolForms[form]), 256)) {
            p.X = X; p.W = W; p.packed = static_cast<const char*>(packed); p.bias = bias; p.Y = Y; p.epi = epilogue;
            hipStream_t st = static_cast<hipStream_t>(stream);
            switch (form) {
                case 0: launch_conv_pool_form<8, 7, 2, 2, 4>(p, st); break;
                case 1: launch_conv_pool_form<7, 8, 2, 2, 4>(p, st); break;
                case 2: launch_conv_pool_form<8, 7, 1, 4, 2>(p, st); break;
                case 3: launch_conv_pool_form<7, 8, 1, 4, 2>(p, st); break;
                case 4: launch_conv_pool_form<5, 5, 2, 2, 2>(p, st); break;
                case 5: launch_conv_pool_form<4, 3, 2, 2, 1>(p, st); break;
                default: launch_conv_pool_form<3, 4, 2, 2, 1>(p, st); break;
            }
            return check_launch("conv2d_f32_pool_kernel");
        }
    }
    const int status = mi355x_conv2d_f32(X, W, bias, scratch, N, C, H, Wd, M, KH, KW, pads, strides, dilations, epilogue, stream);
    if (status != MI355X_OK) return status;
    const int64_t OH = (H + pads[0] + pads[2] - (KH - 1) * dilations[0] - 1) / strides[0] + 1, OW = (Wd + pads[1] + pads[3] - (KW - 1) * dilations[1] - 1) / strides[1] + 1;
    return mi355x_maxpool2d_f32(scratch, Y, N, M, OH, OW, PKH, PKW, pool_pads, pool_strides, pool_dilations, stream);
}
