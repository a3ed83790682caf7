// ONNX Conv, fp32, outputs of few tiles: operands straight from memory into registers, the channels split over sixteen waves.
//
// One image through the later layers of a classifier is 8 to 50 tiles of 64 x 64: on a chip of 256 CUs the gather kernel then takes
// the latency of its K steps, a barrier each, whatever the arithmetic. Here a workgroup owns 16 TM channels x 16 TP positions, each
// wave sums a sixteenth of the input channels with no barrier, and the partial sums meet in LDS once, in the order of the waves.
// A 3 x 3 filter takes four channels at a time: lane (li, lq) reads the nine weights of channel 4 g + lq, which are consecutive, and
// the nine input values under them, at offsets that hold for every g (out of the image: bit 31, which loads a zero); tap t is one
// MFMA. A 1 x 1 filter takes sixteen channels at a time, four consecutive ones per lane.
#include "common.h"
#include "gemm_tile.h"
#include "conv_args.h"

namespace mi355x {

constexpr int CD_WAVES = 16;

// (TAPS == 9: C a multiple of 4; TAPS == 1: of 16)
template <int TM, int TP, int TAPS>
__global__ __launch_bounds__(WAVE * CD_WAVES) void conv2d_f32_direct_kernel(ConvArgs p) {
    constexpr int TILES = TM * TP;
    constexpr int STEPS = TAPS == 9 ? 9 : 4;            // MFMA steps of a group of channels
    constexpr int GROUP = TAPS == 9 ? 4 : 16;           // its channels
    constexpr int RING = TAPS == 9 ? (TILES >= 4 ? 1 : 2) : 4;
    __shared__ __attribute__((aligned(16))) f32x4 red[CD_WAVES][TILES][WAVE];

    const int tid = threadIdx.x, lane = tid % WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int li = lane % 16, lq = lane / 16;
    // consecutive tiles walk along the positions: the XCD that reads a strip of weights uses it for all of them
    const uint32_t logical = (uint32_t)xcd_remap(blockIdx.x, p.nwg);
    const int m0 = (int)(logical / (uint32_t)p.tiles_p) * 16 * TM;
    const int64_t p0 = (int64_t)(logical % (uint32_t)p.tiles_p) * 16 * TP;
    const int hw = p.H * p.Wd;

    // raw buffers of 2^31 - 1 bytes (launch precondition: a tensor spans less)
    const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.W), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.X), 0, 0x7fffffff, 0x00020000);
    uint32_t w_off[TM], x_off[TP][TAPS];
#pragma unroll
    for (int i = 0; i < TM; ++i) w_off[i] = 4u * ((uint32_t)min(m0 + 16 * i + li, p.M - 1) * (uint32_t)p.K + (uint32_t)(TAPS == 9 ? 9 : 4) * lq);
#pragma unroll
    for (int j = 0; j < TP; ++j) {
        const int64_t pp = min(p0 + 16 * j + li, p.P - 1);
        const uint32_t n = fdiv((uint32_t)pp, p.div_ohw);
        const uint32_t q = (uint32_t)pp - n * (uint32_t)p.OHW;
        const uint32_t oy = fdiv(q, p.div_ow);
        const int iy = (int)oy * p.stride_h - p.pad_t, ix = (int)(q - oy * (uint32_t)p.OW) * p.stride_w - p.pad_l;
        const int base = ((int)n * p.C + (TAPS == 9 ? 1 : 4) * lq) * hw;
#pragma unroll
        for (int t = 0; t < TAPS; ++t) {
            const int y = iy + (TAPS == 9 ? t / 3 : 0) * p.dil_h, x = ix + (TAPS == 9 ? t % 3 : 0) * p.dil_w;
            const bool in = (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.Wd;
            x_off[j][t] = in ? 4u * (uint32_t)(base + y * p.Wd + x) : 0x80000000u;
        }
    }

    // the outputs this thread adds up at the end, four channels of one position; their bias and residual values set out now
    const int tile = tid / WAVE;
    const int oc = m0 + 16 * (tile / TP) + 4 * lq;
    const int64_t op = p0 + 16 * (tile % TP) + li;
    const bool stored = tile < TILES && op < p.P;
    int64_t off = 0;
    float bias[4] = {0.f, 0.f, 0.f, 0.f}, res[4] = {0.f, 0.f, 0.f, 0.f};
    if (stored) {
        const uint32_t n = fdiv((uint32_t)op, p.div_ohw);
        off = ((int64_t)n * p.M + oc) * p.OHW + ((uint32_t)op - n * (uint32_t)p.OHW);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (oc + r < p.M) {
                if (p.epi & MI355X_EPI_BIAS) bias[r] = p.bias[oc + r];
                if (p.epi & MI355X_EPI_RESIDUAL) res[r] = p.residual[off + (int64_t)r * p.OHW];
            }
    }

    const int groups = p.C / GROUP, per_wave = (groups + CD_WAVES - 1) / CD_WAVES;
    const int begin = wave * per_wave, end = min(begin + per_wave, groups);

    float vw[RING][TM][STEPS], vx[RING][TP][STEPS];
    auto load = [&](int slot, int g) {
        const int w_g = (TAPS == 9 ? 144 : 64) * g, x_g = 4 * GROUP * hw * g;
#pragma unroll
        for (int i = 0; i < TM; ++i) {
#pragma unroll
            for (int h = 0; h < STEPS / 4; ++h) {
                const f32x4 v = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(w_rsrc, (int)(w_off[i] + 16u * h), w_g, 0));
#pragma unroll
                for (int e = 0; e < 4; ++e) vw[slot][i][4 * h + e] = v[e];
            }
            if constexpr (STEPS == 9) vw[slot][i][8] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(w_rsrc, (int)(w_off[i] + 32u), w_g, 0));
        }
#pragma unroll
        for (int j = 0; j < TP; ++j)
#pragma unroll
            for (int s = 0; s < STEPS; ++s)
                vx[slot][j][s] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                    x_rsrc, (int)x_off[j][TAPS == 9 ? s : 0], x_g + (TAPS == 9 ? 0 : 4 * s * hw), 0));
    };
    f32x4 acc[TM][TP];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TP; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int u = 0; u < RING; ++u)
        if (begin + u < end) load(u, begin + u);
    for (int g = begin; g < end; g += RING) {
        static_for<RING>([&](auto u) {
            if (g + u < end) {
#pragma unroll
                for (int s = 0; s < STEPS; ++s)
#pragma unroll
                    for (int i = 0; i < TM; ++i)
#pragma unroll
                        for (int j = 0; j < TP; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vw[u][i][s], vx[u][j][s], acc[i][j], 0, 0, 0);
            }
            if (g + u + RING < end) load(u, g + u + RING);   // (uniform; a load that is all out of range costs the address unit as much as any)
        });
    }

#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TP; ++j) red[wave][i * TP + j][lane] = acc[i][j];
    __syncthreads();
    if (!stored) return;
    f32x4 v = red[0][tile][lane];
#pragma unroll
    for (int w = 1; w < CD_WAVES; ++w) v += red[w][tile][lane];
#pragma unroll
    for (int r = 0; r < 4; ++r)
        if (oc + r < p.M) {
            float o = apply_epilogue(v[r], p.epi, bias[r]);
            if (p.epi & MI355X_EPI_RESIDUAL) o += res[r];
            if (p.epi & MI355X_EPI_RELU_AFTER) o = fmaxf(o, 0.f);
            p.Y[off + (int64_t)r * p.OHW] = o;
        }
}

// Nanoseconds: `fixed` and `per_k` for the first round of workgroups, `again` and `again_k` for each further one (331 layers of 16 to
// 1024 channels, K = 16 to 9216, up to 40 rounds; weights not in the L2). A strided filter, which reads half of each line, takes up to
// 1.3 times as long over a long K. The rule picks no kernel that is more than 3 % behind in these, and is 0.1 % behind the best pick on
// average (over 500 others 5 % in one); with `again` left out it was 10 to 20 % behind in ten: 3 x 32 x 20 x 20 -> 512 10.7 -> 12.9 us,
// 1 x 1 5 x 512 x 33 x 33 -> 100 14.9 -> 17.5, 3 x 1024 x 33 x 33 -> 200 23.6 -> 28.5. Bound by what a CU draws from its L2, the nine
// 4-byte loads per four channels included: one image 64 x 56 x 56 -> 64 14.8 -> 7.9 us, 128 x 28 x 28 -> 128 23.5 -> 10.7,
// 256 x 14 x 14 -> 256 41.3 -> 12.4, 512 x 7 x 7 -> 512 77.0 -> 20.6, 1 x 1 256 x 14 x 14 -> 512 10.0 -> 4.1; four images
// 512 x 7 x 7 -> 512 76.8 -> 32.5, 128 x 28 x 28 -> 128 23.8 -> 20.8, 64 x 56 x 56 -> 64 would be 22.5 against 15.4 and stay.
// (Loads past a wave's share, which a branch now skips: 64 x 56 x 56 -> 64 9.0 us with them, 1 x 1 7.6.)
struct ConvDirectForm { int taps, tm, tp; double fixed, again, per_k, again_k; };
static const ConvDirectForm kConvDirectForms[] = {{9, 1, 1, 2900, 670, 4.15, 3.1}, {9, 2, 1, 3000, 1070, 6.2, 5.75}, {9, 2, 2, 3650, 1740, 7.3, 6.45},
                                                  {1, 1, 1, 3100, 730, 2.5, 3.0}, {1, 2, 1, 3200, 840, 4.2, 5.2}, {1, 2, 2, 3500, 2000, 5.55, 7.35}};

template <int TAPS>
static void launch_direct(int form, const ConvArgs& p, hipStream_t st) {
    const dim3 grid((unsigned)p.nwg), block(WAVE * CD_WAVES);
    if (form == 0) hipLaunchKernelGGL((conv2d_f32_direct_kernel<1, 1, TAPS>), grid, block, 0, st, p);
    else if (form == 1) hipLaunchKernelGGL((conv2d_f32_direct_kernel<2, 1, TAPS>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((conv2d_f32_direct_kernel<2, 2, TAPS>), grid, block, 0, st, p);
}

// The fastest form of these and its time; -1 where there is none.
static int choose_direct(const ConvArgs& p, int cus, double& best_cost) {
    const int force = tuning().conv_direct;
    const bool taps9 = p.KH == 3 && p.KW == 3 && p.C % 4 == 0, taps1 = p.KH == 1 && p.KW == 1 && p.C % 16 == 0;
    best_cost = 1e300;
    if (force == 0 || !(taps9 || taps1)) return -1;
    // both operands are addressed with 32-bit byte offsets
    if ((int64_t)p.M * p.K >= ((int64_t)1 << 29) || (int64_t)p.N * p.C * p.H * p.Wd >= ((int64_t)1 << 29)) return -1;
    int best = -1;
    for (int f = 0; f < 6; ++f) {
        const ConvDirectForm& form = kConvDirectForms[f];
        if (form.taps != (taps9 ? 9 : 1)) continue;
        const int64_t rounds = ceil_div(ceil_div((int64_t)p.M, (int64_t)16 * form.tm) * ceil_div(p.P, (int64_t)16 * form.tp), (int64_t)cus);
        const double strided = (p.stride_h > 1 || p.stride_w > 1) && p.K >= 500 && rounds > 1 ? 1.3 : 1.0;
        const double cost = form.fixed + form.again * (double)(rounds - 1) + strided * (double)p.K * (form.per_k + form.again_k * (double)(rounds - 1));
        if (force > 0 ? force == 10 * form.tm + form.tp : cost < best_cost) { best = f; best_cost = cost; }
    }
    return best;
}

double conv2d_f32_direct_cost(const ConvArgs& p, int cus) {
    double cost;
    choose_direct(p, cus, cost);
    return cost;
}

bool launch_conv2d_f32_direct(const ConvArgs& args, double other_cost, int cus, hipStream_t stream) {
    ConvArgs p = args;
    double cost;
    const int best = choose_direct(p, cus, cost);
    if (best < 0 || (tuning().conv_direct <= 0 && cost >= 0.95 * other_cost)) return false;
    p.tiles_m = ceil_div((int64_t)p.M, (int64_t)16 * kConvDirectForms[best].tm);
    p.tiles_p = ceil_div(p.P, (int64_t)16 * kConvDirectForms[best].tp);
    p.nwg = p.tiles_m * p.tiles_p;
    if (!grid_fits(p.nwg, WAVE * CD_WAVES)) return false;
    if (kConvDirectForms[best].taps == 9) launch_direct<9>(best % 3, p, stream);
    else launch_direct<1>(best % 3, p, stream);
    return true;
}

}  // namespace mi355x
