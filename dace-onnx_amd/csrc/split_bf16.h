// fp32 values as three bf16 numbers, for the kernels that multiply on the bf16 matrix unit.
//
// A float has 24 significant bits, a bf16 eight, so x = hi + mid + lo (round to nearest, subtract, round again), exactly: values are
// multiplied by 2^16 before they are split, so that the last bit of the smallest float, 2^-149, is the smallest bf16 subnormal,
// 2^-133 (the MFMA takes subnormals as they are), and sums by 2^-32 after. Infinities, NaN and values from 2^112 on split into parts
// that make every sum they enter NaN or infinite, which is how a kernel finds them.
#pragma once

#include "common.h"

namespace mi355x {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int SP_PLANES = 3;
constexpr float SP_SCALE = 65536.f, SP_UNSCALE = 1.f / (SP_SCALE * SP_SCALE);

// two floats -> the three bf16 parts of SP_SCALE times them, packed
__device__ __forceinline__ void split_pair(float x, float y, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
    auto pack = [](float a, float b) { return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2)); };
    auto low = [](uint32_t v) { return __builtin_bit_cast(float, v << 16); };
    auto high = [](uint32_t v) { return __builtin_bit_cast(float, v & 0xffff0000u); };
    x *= SP_SCALE; y *= SP_SCALE;
    hi = pack(x, y);
    x -= low(hi); y -= high(hi);
    mid = pack(x, y);
    x -= low(mid); y -= high(mid);
    lo = pack(x, y);
}

// eight floats -> a 16-byte unit of each plane
__device__ __forceinline__ void split_unit8(const f32x4& a, const f32x4& b, u32x4 (&part)[SP_PLANES]) {
    const f32x4 v[2] = {a, b};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            uint32_t hi, mid, lo;
            split_pair(v[h][2 * s], v[h][2 * s + 1], hi, mid, lo);
            part[0][2 * h + s] = hi; part[1][2 * h + s] = mid; part[2][2 * h + s] = lo;
        }
}

// Packed constants (written once, by mi355x_pack_f32): rows in blocks of 32, k in steps of 32, and of each block and step two
// fragments of `v_mfma_f32_32x32x16_bf16`, three planes each. Lane l of fragment s holds row l % 32 and unit g = 2 s + l / 32, whose
// eight k are {4 g .. 4 g + 3, 16 + 4 g .. 16 + 4 g + 3}: with that order four neighbouring lanes of a kernel that splits its other
// operand itself load 64 contiguous bytes of a row and a unit is one LDS write. A wave reads a fragment as one 1 KB load.
constexpr int PK_PLANE = 1024, PK_FRAGMENT = SP_PLANES * PK_PLANE;

// The products of two split values that reach 2^-24 of the result, the largest one (its own set of accumulators) first.
constexpr int PK_PRODUCTS = 6;
constexpr int PK_QA[PK_PRODUCTS] = {0, 0, 1, 1, 0, 2}, PK_QB[PK_PRODUCTS] = {0, 1, 0, 1, 2, 0};

}  // namespace mi355x
