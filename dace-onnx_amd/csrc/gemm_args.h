// Argument block shared by the fp32 GEMM kernels.
#pragma once

#include "common.h"

namespace mi355x {

struct GemmArgs {
    const float* A; const float* B; float* C; const float* bias; const float* residual;
    int64_t batch, batch1;  // total batch entries, and the extent of the inner batch level
    int64_t M, N, K;
    int64_t a_sb0, a_sb1, a_sm, a_sk;
    int64_t b_sb0, b_sb1, b_sk, b_sn;
    int64_t c_sb0, c_sb1, c_sm;
    int64_t r_sb0, r_sb1, r_sm;
    int64_t tiles_m, tiles_n, nwg;
    int group_m;  // tile walk order, see tile_coords
    float alpha;
    int epi;
    MI355X_TRACE_MEMBER
};

// GEMM with both operands contiguous along k (gemm_f32_nt.hip). Returns false when
// the problem is outside what that kernel handles (nothing launched).
bool launch_gemm_f32_nt(GemmArgs p, int cus, hipStream_t stream);

// Nanoseconds that kernel takes, 1e300 where it takes no such product.
double gemm_f32_nt_cost(const GemmArgs& p, int cus);

// GEMM with both operands contiguous along k whose eight waves split K (gemm_f32_ksplit.hip): 32 x 96 tiles.
bool launch_gemm_f32_ksplit(GemmArgs p, int cus, hipStream_t stream);

// GEMM with A contiguous along k and B along k (b_kc) or n, on the bf16 matrix unit with every value split in three
// (gemm_f32_split.hip). `other_cost`: nanoseconds per k the caller's own kernel takes; nothing is launched where no form of
// this one is below it.
bool launch_gemm_f32_split(GemmArgs p, bool b_kc, double other_cost, int cus, hipStream_t stream);

// Nanoseconds per k of its fastest form, 1e300 where it takes no such product.
double gemm_f32_split_cost(const GemmArgs& p, int cus);

// GEMM with A contiguous along k and B along k (b_kc) or n whose outputs are few tiles (gemm_f32_direct.hip): no staging, K split
// over the waves of a workgroup. `other_cost`: nanoseconds the caller's own kernel takes; nothing is launched where it is not behind.
bool launch_gemm_f32_direct(GemmArgs p, bool b_kc, double other_cost, int cus, hipStream_t stream);

// Nanoseconds of its fastest form, 1e300 where it takes no such product.
double gemm_f32_direct_cost(const GemmArgs& p, bool b_kc, int cus);

}  // namespace mi355x
