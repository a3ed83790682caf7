// Argument block and helpers shared by the fp32 convolution kernels.
#pragma once

#include "common.h"

namespace mi355x {

// n / d for 0 <= n < 2^31 as umulhi(n, mul) >> shr (d == 1 special-cased).
struct FastDiv {
    uint32_t d, mul, shr;
};
static FastDiv make_fastdiv(int64_t d) {
    FastDiv f;
    f.d = (uint32_t)d;
    if (d == 1) { f.mul = 0; f.shr = 0; return f; }
    uint32_t l = 0;
    while ((1ull << l) < (uint64_t)d) ++l;  // ceil(log2 d)
    const uint32_t p = 31 + l;
    f.mul = (uint32_t)(((1ull << p) + (uint64_t)d - 1) / (uint64_t)d);
    f.shr = p - 32;
    return f;
}
__device__ __forceinline__ uint32_t fdiv(uint32_t n, const FastDiv& f) {
    return f.d == 1 ? n : (__umulhi(n, f.mul) >> f.shr);
}

// The part of the epilogue after bias and activation: the residual (same layout as Y, hence the same
// offset) and the activation that follows it (the last two steps of a ResNet block).
__device__ __forceinline__ f32x4 conv_epilogue_tail4(f32x4 v, int epi, const float* residual, int64_t off) {
    if (epi & MI355X_EPI_RESIDUAL) v += __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(residual + off));
    if (epi & MI355X_EPI_RELU_AFTER) v = f32x4{fmaxf(v.x, 0.f), fmaxf(v.y, 0.f), fmaxf(v.z, 0.f), fmaxf(v.w, 0.f)};
    return v;
}
__device__ __forceinline__ float conv_epilogue_tail1(float v, int epi, const float* residual, int64_t off) {
    if (epi & MI355X_EPI_RESIDUAL) v += residual[off];
    if (epi & MI355X_EPI_RELU_AFTER) v = fmaxf(v, 0.f);
    return v;
}

struct ConvArgs {
    const float* X; const float* W; const float* bias; float* Y;
    const float* residual;   // laid out like Y; read only with MI355X_EPI_RESIDUAL
    int N, C, H, Wd, M, KH, KW, OH, OW;
    int pad_t, pad_l, stride_h, stride_w, dil_h, dil_w;
    int K;          // C*KH*KW
    int64_t P;      // N*OH*OW
    int OHW;
    FastDiv div_khw, div_kw, div_ohw, div_ow;
    int64_t tiles_m, tiles_p, nwg;
    int group_m;    // tile walk order, see tile_coords
    int epi;
    int vec_w;      // W tile may use 16-byte loads
    int vec_y;      // Y may use 16-byte stores (OH*OW % 4 == 0, aligned)
    int x_bytes;    // size of X (gather kernel only; below 2^31)
    // gather kernel: the first full_tiles workgroups take whole tiles, the rest 16-position slices from p_full on
    int64_t full_tiles, p_full;
    MI355X_TRACE_MEMBER
};

// Nanoseconds of the gather kernel (conv2d_f32.hip).
double conv2d_f32_gather_cost(const ConvArgs& p, int cus);

// Convolution whose output is few tiles (conv2d_f32_direct.hip), 3 x 3 and 1 x 1 filters: no staging, the channels split over the
// waves of a workgroup. `other_cost`: nanoseconds the caller's own kernel takes; nothing is launched where it is not behind.
double conv2d_f32_direct_cost(const ConvArgs& p, int cus);   // nanoseconds of its fastest form, 1e300 where it has none
bool launch_conv2d_f32_direct(const ConvArgs& p, double other_cost, int cus, hipStream_t stream);

}  // namespace mi355x
