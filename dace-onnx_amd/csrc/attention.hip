// Fused scaled-dot-product attention core, fp32:  O = softmax(scale * Q K^T [+ mask]) V
// for one (batch, head) per slice, head size = 64; 128 keys (BERT-base) in one pass, any other number of
// keys, and any number with a mask, in blocks of 128 with a running maximum and sum.
//
// The reference runs this as three library nodes -- MatMul, Softmax, MatMul
// (daceml/onnx/op_implementations/pure_implementations.py:130-235, 346-366) -- with
// the [B, H, S, S] score tensor written to and read from memory twice. Here a
// workgroup of 4 waves owns 64 query rows of one (batch, head): scores and
// probabilities never leave registers.
//
//   * K and V of the slice (128 x 64 each) are staged once in LDS, rows padded by 4
//     floats; Q operands come straight from global memory (16 query rows per wave,
//     nobody shares them).
//   * S = Q K^T uses the swapped-operand form of v_mfma_f32_16x16x4_f32: afterwards
//     lane (li, lq) holds S[q = li][key = 16 j + 4 lq + r] in acc[j][r] -- a query
//     row's 128 scores sit in 4 lanes x 32 registers. Row max and row sum are 31
//     register operations plus two cross-lane steps (lanes li, li+16, li+32, li+48).
//   * That register layout is exactly the A-operand layout of the second product
//     when the four keys of an MFMA step are taken as {16 j + r + 4 lq, lq = 0..3}:
//     acc[j][r] is used as the operand as it stands, no shuffle, no LDS round trip.
//     The matching V operand of lane (li, lq) is V[key = 16 j + 4 lq + r][4 li .. 4 li + 3]:
//     one 16-byte LDS read feeds four MFMAs (output tile t holds columns 4 li + t),
//     and a lane ends up with four consecutive output columns of a row: 16-byte stores.
#include "common.h"
#include "gemm_tile.h"
#include "split_bf16.h"

#include <algorithm>

namespace mi355x {

constexpr int AT_SK = 128, AT_D = 64, AT_BQ = 64, AT_PITCH = AT_D + LDS_PAD;
constexpr int AF_ROWS = 16, AF_KEYS = 16;

struct AttnArgs {
    const float* Q; const float* K; const float* V; float* O;
    int64_t batch1, Sq, Sk, q_blocks, nwg;
    int64_t q_sb0, q_sb1, q_sr, k_sb0, k_sb1, k_sr, v_sb0, v_sb1, v_sr, o_sb0, o_sb1, o_sr;
    const float* mask; int64_t m_sb0, m_sb1, m_sr;   // masked form: added to scale * Q K^T, keys contiguous, 0 strides broadcast
    float scale;   // (last: next to the mask's address the compiler keeps both in a local array and reads the mask through it)
};

__device__ __forceinline__ float quad_lanes_max(float v) {  // over lanes li, li+16, li+32, li+48
    v = fmaxf(v, __shfl_xor(v, 16, WAVE));
    return fmaxf(v, __shfl_xor(v, 32, WAVE));
}
__device__ __forceinline__ float quad_lanes_sum(float v) {
    v += __shfl_xor(v, 16, WAVE);
    return v + __shfl_xor(v, 32, WAVE);
}

// WAVES waves of 16 query rows each per workgroup: 4 (64 rows, two workgroups per 128-row slice) is what the library
// uses; 3 and 2 (48 and 32 rows: three and four workgroups per slice, the last one of three with two working waves)
// exist to measure whether more, smaller workgroups help, see MI355X_ATTN_WAVES in the launcher.
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void attention_f32_kernel(AttnArgs p) {
    constexpr int SK = AT_SK, D = AT_D, PITCH = AT_PITCH, NJ = SK / 16, NC = D / 16;
    constexpr int NT = 64 * WAVES, VECS = SK * D / 4, PER_T = (VECS + NT - 1) / NT;   // K / V tile: 16-byte vectors per thread
    __shared__ __attribute__((aligned(16))) float lds_k[SK * PITCH];
    __shared__ __attribute__((aligned(16))) float lds_v[SK * PITCH];

    const int tid = threadIdx.x;
    const int lane = tid % WAVE, wave = tid / WAVE;
    const int li = lane % 16, lq = lane / 16;

    // consecutive logical ids (the query blocks of one slice, neighbouring heads) share an XCD's L2
    const int64_t logical = xcd_remap(blockIdx.x, p.nwg);
    const int64_t slice = logical / p.q_blocks, qb = logical % p.q_blocks;
    const int64_t b0 = slice / p.batch1, b1 = slice % p.batch1;
    const float* __restrict__ Q = p.Q + b0 * p.q_sb0 + b1 * p.q_sb1;
    const float* __restrict__ K = p.K + b0 * p.k_sb0 + b1 * p.k_sb1;
    const float* __restrict__ V = p.V + b0 * p.v_sb0 + b1 * p.v_sb1;
    float* __restrict__ O = p.O + b0 * p.o_sb0 + b1 * p.o_sb1;
    const int64_t q0 = qb * (16 * WAVES) + 16 * wave;   // first query row of this wave

    // ---- loads: K and V tiles (PER_T + PER_T vectors per thread), Q operands (4 per lane) ----------------
    f32x4 rk[PER_T], rv[PER_T], rq[NC];
#pragma unroll
    for (int it = 0; it < PER_T; ++it) {
        const int idx = tid + it * NT, row = idx / (D / 4), c4 = idx % (D / 4);
        if (VECS % NT == 0 || idx < VECS) rk[it] = *reinterpret_cast<const f32x4*>(K + row * p.k_sr + 4 * c4);
    }
    {
        int64_t qrow = q0 + li;
        qrow = qrow < p.Sq ? qrow : p.Sq - 1;   // clamped; rows beyond Sq are computed and not stored
#pragma unroll
        for (int c = 0; c < NC; ++c) rq[c] = *reinterpret_cast<const f32x4*>(Q + qrow * p.q_sr + 16 * c + 4 * lq);
    }
#pragma unroll
    for (int it = 0; it < PER_T; ++it) {
        const int idx = tid + it * NT, row = idx / (D / 4), c4 = idx % (D / 4);
        if (VECS % NT == 0 || idx < VECS) rv[it] = *reinterpret_cast<const f32x4*>(V + row * p.v_sr + 4 * c4);
    }
#pragma unroll
    for (int it = 0; it < PER_T; ++it) {
        const int idx = tid + it * NT, row = idx / (D / 4), c4 = idx % (D / 4);
        if (VECS % NT == 0 || idx < VECS) *reinterpret_cast<f32x4*>(lds_k + row * PITCH + 4 * c4) = rk[it];
    }
#pragma unroll
    for (int it = 0; it < PER_T; ++it) {
        const int idx = tid + it * NT, row = idx / (D / 4), c4 = idx % (D / 4);
        if (VECS % NT == 0 || idx < VECS) *reinterpret_cast<f32x4*>(lds_v + row * PITCH + 4 * c4) = rv[it];
    }
    __syncthreads();
    if (q0 >= p.Sq) return;  // whole wave beyond the last query row (after the only barrier)

    // ---- S = Q K^T: acc[j][r] = S[q0 + li][16 j + 4 lq + r] -------------------------------------------
    f32x4 acc[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        f32x4 kf[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            kf[j] = *reinterpret_cast<const f32x4*>(lds_k + (16 * j + li) * PITCH + 16 * c + 4 * lq);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][s], rq[c][s], acc[j], 0, 0, 0);
    }

    // ---- softmax over the 128 keys of each query row ------------------------------------------------
    // exp(scale s - max) as 2^(c s - max'), c = scale log2(e): one multiply per score and the bare v_exp_f32
    // (the library expf costs half a dozen more instructions per value; 32 values per lane)
    const float c = p.scale * 1.44269504088896340736f;
    float m = -INFINITY;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        acc[j] *= c;
        m = fmaxf(m, fmaxf(fmaxf(acc[j].x, acc[j].y), fmaxf(acc[j].z, acc[j].w)));
    }
    m = quad_lanes_max(m);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        acc[j].x = __builtin_amdgcn_exp2f(acc[j].x - m);
        acc[j].y = __builtin_amdgcn_exp2f(acc[j].y - m);
        acc[j].z = __builtin_amdgcn_exp2f(acc[j].z - m);
        acc[j].w = __builtin_amdgcn_exp2f(acc[j].w - m);
        sum += (acc[j].x + acc[j].y) + (acc[j].z + acc[j].w);
    }
    const float inv = 1.0f / quad_lanes_sum(sum);
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[j] *= inv;

    // ---- O = P V: out[t][r] = O[q0 + 4 lq + r][4 li + t] -------------------------------------------------
    f32x4 out[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) out[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        f32x4 vf[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            vf[r] = *reinterpret_cast<const f32x4*>(lds_v + (16 * j + 4 * lq + r) * PITCH + 4 * li);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int t = 0; t < 4; ++t)
                out[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(acc[j][r], vf[r][t], out[t], 0, 0, 0);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int64_t qrow = q0 + 4 * lq + r;
        if (qrow < p.Sq)
            *reinterpret_cast<f32x4*>(O + qrow * p.o_sr + 4 * li) = f32x4{out[0][r], out[1][r], out[2][r], out[3][r]};
    }
}

// Any number of keys: the same workgroup walks the keys in blocks of 128 with a running row maximum and
// row sum (the probabilities of a block are exp(s - running max); when the maximum grows, the sums and the
// output accumulators are rescaled by exp(old max - new max); the division by the row sum happens once, at
// the end). Keys beyond Sk in the last block are loaded from the last valid row, their scores set to -inf
// and their values to zero. Every wave takes part in the barriers of every block, so there is no early exit
// for query rows beyond Sq: they are computed on the clamped last row and not stored.
//
// MASKED: scale * Q K^T + mask, the padding mask of a batch of unequal sentences (or any mask of the scores' shape up to
// broadcasting). The scores stay in natural units then and the difference to the maximum is scaled by log2(e): a mask of the
// type's lowest value times log2(e) would overflow, and a row of such keys only is a uniform softmax, as node by node. A block
// whose keys are all -inf leaves the running sums alone; a row of them only is NaN at the end (0 / 0), also as node by node.
// Both products are summed in two sets of accumulators and the second block by block, so that no sum is longer than in the two
// products it replaces: 2 x 12 heads, 69 queries, 300 keys, scores of standard deviation 8 9.2e-7 -> 5.3e-7 (2-norm against float64;
// 5.7e-7 as two products and a softmax), 16 x 12 of 512 4.6e-7 -> 2.3e-7 (4.6e-7). It costs 1 %.
// The bare exponential of a rounded argument is not seen in these (with the low part of the product 4.58e-7 for 4.59e-7, 5 % slower).
// The nodes one at a time (two products, the addition, the softmax) take 259 us on 16 x 12 slices of 512 x 512 scores, this 135.
// 128 keys go through here too: 8 x 12 slices 10.0 us, the one-pass kernel above without a mask 8.5, the nodes 22.5.
template <bool MASKED>
__device__ __forceinline__ void attention_blocks(const AttnArgs& p, int64_t slice, int64_t qb, float* lds_k, float* lds_v) {
    constexpr int SK = AT_SK, D = AT_D, PITCH = AT_PITCH, NJ = SK / 16, NC = D / 16, SETS = MASKED ? 2 : 1;
    const int tid = threadIdx.x;
    const int lane = tid % WAVE, wave = tid / WAVE;
    const int li = lane % 16, lq = lane / 16;
    const int64_t b0 = slice / p.batch1, b1 = slice % p.batch1;
    const float* __restrict__ Q = p.Q + b0 * p.q_sb0 + b1 * p.q_sb1;
    const float* __restrict__ K = p.K + b0 * p.k_sb0 + b1 * p.k_sb1;
    const float* __restrict__ V = p.V + b0 * p.v_sb0 + b1 * p.v_sb1;
    float* __restrict__ O = p.O + b0 * p.o_sb0 + b1 * p.o_sb1;
    const int64_t q0 = qb * AT_BQ + 16 * wave;   // first query row of this wave

    f32x4 rq[NC];
    {
        int64_t qrow = q0 + li;
        qrow = qrow < p.Sq ? qrow : p.Sq - 1;
#pragma unroll
        for (int c = 0; c < NC; ++c) rq[c] = *reinterpret_cast<const f32x4*>(Q + qrow * p.q_sr + 16 * c + 4 * lq);
    }
    f32x4 out[4];                       // out[t][r] = O[q0 + 4 lq + r][4 li + t], not yet divided by the row sum
#pragma unroll
    for (int t = 0; t < 4; ++t) out[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;   // of query row q0 + li (the same value in its four lanes)
    constexpr float LOG2E = 1.44269504088896340736f;
    const float c = MASKED ? p.scale : p.scale * LOG2E;   // unmasked: scores in units of log2, exp(scale s - m) = 2^(c s - m')
    const float* __restrict__ mask = nullptr;             // the mask's row of query q0 + li
    if constexpr (MASKED) {
        const int64_t qrow = q0 + li < p.Sq ? q0 + li : p.Sq - 1;
        mask = p.mask + b0 * p.m_sb0 + b1 * p.m_sb1 + qrow * p.m_sr;
    }

    for (int64_t key0 = 0; key0 < p.Sk; key0 += SK) {
        f32x4 rk[8], rv[8];
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int idx = tid + it * 256, c4 = idx % (D / 4);
            int64_t row = key0 + idx / (D / 4);
            row = row < p.Sk ? row : p.Sk - 1;
            rk[it] = *reinterpret_cast<const f32x4*>(K + row * p.k_sr + 4 * c4);
            rv[it] = *reinterpret_cast<const f32x4*>(V + row * p.v_sr + 4 * c4);
        }
        if (key0 + SK > p.Sk)   // (zero times an infinity of the last key's would be NaN)
#pragma unroll
            for (int it = 0; it < 8; ++it)
                if (key0 + (tid + it * 256) / (D / 4) >= p.Sk) rv[it] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (key0 > 0) __syncthreads();   // the previous block's operands have been read by everyone
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int idx = tid + it * 256, row = idx / (D / 4), c4 = idx % (D / 4);
            *reinterpret_cast<f32x4*>(lds_k + row * PITCH + 4 * c4) = rk[it];
            *reinterpret_cast<f32x4*>(lds_v + row * PITCH + 4 * c4) = rv[it];
        }
        __syncthreads();

        // ---- S = Q K^T of this block: acc[j][r] = S[q0 + li][key0 + 16 j + 4 lq + r]
        f32x4 scores[SETS][NJ];
#pragma unroll
        for (int h = 0; h < SETS; ++h)
#pragma unroll
            for (int j = 0; j < NJ; ++j) scores[h][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            f32x4 kf[NJ];
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                kf[j] = *reinterpret_cast<const f32x4*>(lds_k + (16 * j + li) * PITCH + 16 * c + 4 * lq);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    f32x4& sum = scores[c * SETS / NC][j];
                    sum = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[j][s], rq[c][s], sum, 0, 0, 0);
                }
        }
        f32x4 acc[NJ];
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[j] = MASKED ? scores[0][j] + scores[SETS - 1][j] : scores[0][j];
        const bool ragged = key0 + SK > p.Sk;   // uniform
        float m_blk = -INFINITY;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int64_t key = key0 + 16 * j + 4 * lq;
            acc[j] *= c;
            if constexpr (MASKED) {
                typedef f32x4 unaligned __attribute__((aligned(4)));
                auto at = [&](int64_t k) { return mask[k < p.Sk ? k : p.Sk - 1]; };
                if (!ragged) acc[j] += *reinterpret_cast<const unaligned*>(mask + key);
                else acc[j] += f32x4{at(key), at(key + 1), at(key + 2), at(key + 3)};
            }
            if (ragged) {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (key + r >= p.Sk) acc[j][r] = -INFINITY;
            }
            m_blk = fmaxf(m_blk, fmaxf(fmaxf(acc[j].x, acc[j].y), fmaxf(acc[j].z, acc[j].w)));
        }
        const float m_new = fmaxf(m_run, quad_lanes_max(m_blk));
        const float m_ref = MASKED && m_new == -INFINITY ? 0.f : m_new;   // nothing but -inf so far: 2^(-inf - 0) = 0
        auto power = [&](float v) { return __builtin_amdgcn_exp2f(MASKED ? (v - m_ref) * LOG2E : v - m_ref); };
        const float alpha = power(m_run);    // 0 for the first block
        float sum = 0.f;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            acc[j].x = power(acc[j].x);
            acc[j].y = power(acc[j].y);
            acc[j].z = power(acc[j].z);
            acc[j].w = power(acc[j].w);
            sum += (acc[j].x + acc[j].y) + (acc[j].z + acc[j].w);
        }
        l_run = l_run * alpha + quad_lanes_sum(sum);
        m_run = m_new;
        // ---- out = alpha out + P V of this block (masked: by way of accumulators of its own). The accumulators hold rows 4 lq + r:
        // that row's factor lives in lane 4 lq + r
        f32x4 sums[SETS][4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if constexpr (MASKED) sums[0][t] = sums[SETS - 1][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            else
#pragma unroll
                for (int r = 0; r < 4; ++r) out[t][r] *= __shfl(alpha, 4 * lq + r, WAVE);
        }
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            f32x4 vf[4];
#pragma unroll
            for (int r = 0; r < 4; ++r)
                vf[r] = *reinterpret_cast<const f32x4*>(lds_v + (16 * j + 4 * lq + r) * PITCH + 4 * li);
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    f32x4& sum = MASKED ? sums[j % SETS][t] : out[t];
                    sum = __builtin_amdgcn_mfma_f32_16x16x4f32(acc[j][r], vf[r][t], sum, 0, 0, 0);
                }
        }
        if constexpr (MASKED) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float a = __shfl(alpha, 4 * lq + r, WAVE);
#pragma unroll
                for (int t = 0; t < 4; ++t) out[t][r] = fmaf(out[t][r], a, sums[0][t][r] + sums[SETS - 1][t][r]);
            }
        }
    }
    const float inv = 1.0f / l_run;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const float a = __shfl(inv, 4 * lq + r, WAVE);
        const int64_t qrow = q0 + 4 * lq + r;
        if (qrow < p.Sq)
            *reinterpret_cast<f32x4*>(O + qrow * p.o_sr + 4 * li) = f32x4{out[0][r] * a, out[1][r] * a, out[2][r] * a, out[3][r] * a};
    }
}

template <bool MASKED>
__global__ __launch_bounds__(256) void attention_f32_blocks_kernel(AttnArgs p) {
    __shared__ __attribute__((aligned(16))) float lds_k[AT_SK * AT_PITCH];
    __shared__ __attribute__((aligned(16))) float lds_v[AT_SK * AT_PITCH];
    const int64_t logical = xcd_remap(blockIdx.x, p.nwg);
    attention_blocks<MASKED>(p, logical / p.q_blocks, logical % p.q_blocks, lds_k, lds_v);
}

// Few query blocks (a sentence, a small batch): 16 query rows to a workgroup, the keys in chunks of 16 shared by its waves, wave w taking
// chunks w, w + WAVES, ... with a running maximum and sum of its own. No wave waits for another before the end, where their sums meet
// in LDS; no operand passes through LDS: K and Q are read as the fragments of S = Q K^T lie (16 rows, 64 bytes of each), V as 16-byte vectors of
// four rows, whole lines both, and the probabilities are the next product's operand as they stand.
// Both products are those of the split form below, with MFMAs of 16 x 16 x 16, and so is the error (0.96 to 1.03 of it; 0.25 to 0.65 of the fp32
// kernels'). A chunk whose sums are not finite is multiplied again with the fp32 MFMA, by its wave, from the registers it is in.
// What bounds it: the chain of one wave (launch, first loads, splits, 48 MFMAs a chunk, two exchanges, the sum over the waves) while a CU has
// one workgroup, the splits beyond, which the kernels of 64 and 128 query rows make once for all of them. 1 x 12 slices of 16 x 16
// 7.1 -> 3.8 us, of 64 x 64 7.3 -> 4.5, of 128 x 128 7.8 -> 5.8, of 256 x 256 13.8 -> 7.9, 8 x 12 of 16 x 512 25 -> 11.5. (With fp32 MFMAs
// 3.3, 4.2, 5.5, 7.4, 10.3, but 1.2 to 1.6 times the error of the split form.)
template <bool MASKED, int WAVES>
__global__ __launch_bounds__(WAVE * WAVES) void attention_few_kernel(AttnArgs p) {
    constexpr int ROWS = AF_ROWS, KEYS = AF_KEYS, D = AT_D, NC = D / 16;
    constexpr float LOG2E = 1.44269504088896340736f;
    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int li = lane % 16, lq = lane / 16;

    const uint32_t logical = (uint32_t)xcd_remap(blockIdx.x, p.nwg);   // (grids are below 2^31)
    const uint32_t slice = logical / (uint32_t)p.q_blocks, qb = logical % (uint32_t)p.q_blocks;
    const int64_t b0 = slice / (uint32_t)p.batch1, b1 = slice % (uint32_t)p.batch1;
    const float* __restrict__ Q = p.Q + b0 * p.q_sb0 + b1 * p.q_sb1;
    const float* __restrict__ K = p.K + b0 * p.k_sb0 + b1 * p.k_sb1 + 4 * lq;
    const float* __restrict__ V = p.V + b0 * p.v_sb0 + b1 * p.v_sb1 + 4 * li;
    float* __restrict__ O = p.O + b0 * p.o_sb0 + b1 * p.o_sb1;
    const int64_t q0 = (int64_t)qb * ROWS, qrow = q0 + li < p.Sq ? q0 + li : p.Sq - 1;   // clamped: computed, not stored
    const float* __restrict__ mask = MASKED ? p.mask + b0 * p.m_sb0 + b1 * p.m_sb1 + qrow * p.m_sr : nullptr;

    typedef short bf16x4 __attribute__((ext_vector_type(4)));
    auto parts = [](float x, float y, float z, float w, bf16x4 (&f)[SP_PLANES]) __attribute__((always_inline)) {
        uint32_t part[SP_PLANES][2];
        split_pair(x, y, part[0][0], part[1][0], part[2][0]);
        split_pair(z, w, part[0][1], part[1][1], part[2][1]);
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q) f[q] = __builtin_bit_cast(bf16x4, (u32x2{part[q][0], part[q][1]}));
    };
    // of any lane (the sum of finite values may overflow: that is more work, not another result)
    auto not_finite = [](const f32x4& v) __attribute__((always_inline)) {
        return __any(fmaf(v[0], 0.f, fmaf(v[1], 0.f, fmaf(v[2], 0.f, v[3] * 0.f))) != 0.f) != 0;   // (NaN compares unequal)
    };
    f32x4 rk[NC], rv[4], rm, rq[NC];
    bf16x4 fq[NC][SP_PLANES];
    auto load_k = [&](int64_t key0) {   // keys beyond the last are the last one
        const float* row = K + (key0 + li < p.Sk ? key0 + li : p.Sk - 1) * p.k_sr;
#pragma unroll
        for (int c = 0; c < NC; ++c) rk[c] = *reinterpret_cast<const f32x4*>(row + 16 * c);
        if constexpr (MASKED) {
            typedef f32x4 unaligned __attribute__((aligned(4)));
            if (key0 + KEYS <= p.Sk) rm = *reinterpret_cast<const unaligned*>(mask + key0 + 4 * lq);
            else
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int64_t key = key0 + 4 * lq + r;
                    rm[r] = mask[key < p.Sk ? key : p.Sk - 1];
                }
        }
    };
    auto load_v = [&](int64_t key0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int64_t key = key0 + 4 * lq + r;
            rv[r] = *reinterpret_cast<const f32x4*>(V + (key < p.Sk ? key : p.Sk - 1) * p.v_sr);
        }
    };
    const int64_t first = (int64_t)wave * KEYS;
    if (first < p.Sk) {
        load_k(first);
#pragma unroll
        for (int c = 0; c < NC; ++c) rq[c] = *reinterpret_cast<const f32x4*>(Q + qrow * p.q_sr + 16 * c + 4 * lq);
        load_v(first);
#pragma unroll
        for (int c = 0; c < NC; ++c) parts(rq[c][0], rq[c][1], rq[c][2], rq[c][3], fq[c]);
    }
    f32x4 out[4];   // out[t][r] = O[q0 + 4 lq + r][4 li + t] of this wave's keys, not yet divided by the sum
#pragma unroll
    for (int t = 0; t < 4; ++t) out[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m_run = -INFINITY, l_run = 0.f;   // of query row q0 + li (the same value in its four lanes)
    for (int64_t key0 = first; key0 < p.Sk; key0 += WAVES * KEYS) {
        const int64_t next = key0 + WAVES * KEYS;   // uniform
        f32x4 s;   // S[q0 + li][key0 + 4 lq + r]
        {
            f32x4 sum[2], small[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) sum[h] = small[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                bf16x4 fk[SP_PLANES];
                parts(rk[c][0], rk[c][1], rk[c][2], rk[c][3], fk);
#pragma unroll
                for (int u = 0; u < PK_PRODUCTS; ++u) {
                    f32x4& to = u == 0 ? sum[c % 2] : small[c % 2];
                    to = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(fk[PK_QA[u]], fq[c][PK_QB[u]], to, 0, 0, 0);
                }
            }
            s = ((sum[0] + sum[1]) + (small[0] + small[1])) * SP_UNSCALE;
        }
        if (__builtin_expect(not_finite(s), 0)) {
            f32x4 set[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) set[c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < NC; ++c) set[c] = __builtin_amdgcn_mfma_f32_16x16x4f32(rk[c][e], rq[c][e], set[c], 0, 0, 0);
            s = (set[0] + set[1]) + (set[2] + set[3]);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if constexpr (MASKED) s[r] = fmaf(s[r], p.scale, rm[r]);
            else s[r] *= p.scale;
        }
        if (next < p.Sk) load_k(next);
        if (key0 + KEYS > p.Sk)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (key0 + 4 * lq + r >= p.Sk) s[r] = -INFINITY;
        const float m_new = fmaxf(m_run, quad_lanes_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;   // nothing but -inf so far: 2^(-inf - 0) = 0
        auto power = [&](float v) { return __builtin_amdgcn_exp2f((v - m_ref) * LOG2E); };
#pragma unroll
        for (int r = 0; r < 4; ++r) s[r] = power(s[r]);
        const float sum = quad_lanes_sum((s[0] + s[1]) + (s[2] + s[3]));
        if (key0 + KEYS > p.Sk)   // (zero times an infinity of the last key's would be NaN)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (key0 + 4 * lq + r >= p.Sk) rv[r] = f32x4{0.f, 0.f, 0.f, 0.f};
        f32x4 product[4];
        {
            bf16x4 fp[SP_PLANES];
            parts(s[0], s[1], s[2], s[3], fp);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                bf16x4 fv[SP_PLANES];
                parts(rv[0][t], rv[1][t], rv[2][t], rv[3][t], fv);
                f32x4 sum = f32x4{0.f, 0.f, 0.f, 0.f}, small = sum;
#pragma unroll
                for (int u = 0; u < PK_PRODUCTS; ++u) {
                    f32x4& to = u == 0 ? sum : small;
                    to = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(fp[PK_QA[u]], fv[PK_QB[u]], to, 0, 0, 0);
                }
                product[t] = (sum + small) * SP_UNSCALE;
            }
        }
        if (__builtin_expect(not_finite((product[0] + product[1]) + (product[2] + product[3])), 0)) {
#pragma unroll
            for (int t = 0; t < 4; ++t) product[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int t = 0; t < 4; ++t) product[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(s[r], rv[r][t], product[t], 0, 0, 0);
        }
        if (next < p.Sk) load_v(next);
        if (key0 == first) {
#pragma unroll
            for (int t = 0; t < 4; ++t) out[t] = product[t];
            l_run = sum;
        } else {
            const float alpha = power(m_run);
            l_run = fmaf(l_run, alpha, sum);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float a = __shfl(alpha, 4 * lq + r, WAVE);
#pragma unroll
                for (int t = 0; t < 4; ++t) out[t][r] = fmaf(out[t][r], a, product[t][r]);
            }
        }
        m_run = m_new;
    }
    if constexpr (WAVES == 1) {
        const float inv = 1.0f / l_run;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float a = __shfl(inv, 4 * lq + r, WAVE);
            if (q0 + 4 * lq + r < p.Sq)
                *reinterpret_cast<f32x4*>(O + (q0 + 4 * lq + r) * p.o_sr + 4 * li) = f32x4{out[0][r] * a, out[1][r] * a, out[2][r] * a, out[3][r] * a};
        }
    } else {
        // the sums of the waves, in their order: one with no key has a maximum of -inf and adds zeros
        constexpr int PER = ROWS * D / (WAVE * WAVES);   // outputs of a thread, of one row
        __shared__ __attribute__((aligned(16))) float part[WAVES][ROWS][D];
        __shared__ float part_m[WAVES][ROWS], part_l[WAVES][ROWS];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            *reinterpret_cast<f32x4*>(&part[wave][4 * lq + r][4 * li]) = f32x4{out[0][r], out[1][r], out[2][r], out[3][r]};
        if (lq == 0) {
            part_m[wave][li] = m_run;
            part_l[wave][li] = l_run;
        }
        __syncthreads();
        const int row = tid / (D / PER), col = tid % (D / PER) * PER;
        float m = part_m[0][row];
#pragma unroll
        for (int w = 1; w < WAVES; ++w) m = fmaxf(m, part_m[w][row]);
        const float m_ref = m == -INFINITY ? 0.f : m;
        float l = 0.f, sum[PER];
#pragma unroll
        for (int e = 0; e < PER; ++e) sum[e] = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; ++w) {
            const float a = __builtin_amdgcn_exp2f((part_m[w][row] - m_ref) * LOG2E);
            l = fmaf(part_l[w][row], a, l);
#pragma unroll
            for (int e = 0; e < PER; ++e) sum[e] = fmaf(part[w][row][col + e], a, sum[e]);
        }
        const float inv = 1.0f / l;
        if (q0 + row < p.Sq) {
            typedef float vec __attribute__((ext_vector_type(PER < 4 ? PER : 4)));
#pragma unroll
            for (int e = 0; e < PER; e += (PER < 4 ? PER : 4)) {
                vec v;
#pragma unroll
                for (int i = 0; i < (PER < 4 ? PER : 4); ++i) v[i] = sum[e + i] * inv;
                *reinterpret_cast<vec*>(O + (q0 + row) * p.o_sr + col + e) = v;
            }
        }
    }
}

// Many rows: both products on the bf16 matrix unit, every value split in three (split_bf16.h; the six products in two sets of accumulators,
// the second product block by block). A workgroup of four waves owns 128 query rows, 32 of them each, and walks the keys in blocks of 64:
//   * S^T = K Q^T, Q split once into registers, K on its way into LDS in fragment order. A lane then holds half of a query's scores of the
//     block, the lane 32 further on the other half: the maximum and the sum are register operations and one exchange.
//   * O^T = V^T P^T takes the probabilities from the registers that they are in, split there; V is read a column per lane, so that the
//     eight keys of a unit, in the order in which the scores lie, become one LDS write.
//   * Query rows are the columns of O^T: their factors exp(old maximum - new maximum) are the lane's own.
// Sums that are not finite (infinities, NaN, values past 2^112, scores past 2^96) send the workgroup through the fp32 kernel above.
// What bounds it: a wave's chain of 6 us a block, half of it MFMAs and half splits and exponentials on the vector unit, which the waves of two
// workgroups on a CU overlap to 3.4; 254 registers leave no room for a third. Against the kernels above, with a mask: 16 x 12 slices of
// 512 x 512 135 -> 87 us, 32 x 12 of 256 73 -> 48, 20 x 12 of 200 50 -> 31, 32 x 12 of 64 15.1 -> 10.4; without: 121 -> 87, 65 -> 48, 44 -> 30,
// 13.4 -> 10.0. 2-norm of the error against float64 5.9e-7 -> 4.0e-7 and 1.1e-6 -> 4.2e-7. Where a CU gets one workgroup or none its chain is the
// longer one: 1 x 12 of 512 28.7 with the kernel above, 33.8 here.
constexpr int AS_KEYS = 64, AS_ROWS = 128;

template <bool MASKED>
__global__ __launch_bounds__(256, 2) void attention_split_kernel(AttnArgs p) {
    constexpr int D = AT_D, K_BYTES = AS_KEYS / 32 * (D / 16) * PK_FRAGMENT, BLOCKS_LDS = 2 * AT_SK * AT_PITCH * 4;
    static_assert(2 * K_BYTES <= BLOCKS_LDS, "the fp32 form takes more");
    __shared__ __attribute__((aligned(16))) char lds[BLOCKS_LDS];
    char* const lds_k = lds;             // [32 keys][16 of D][part][lane]
    char* const lds_v = lds + K_BYTES;   // [32 of D][16 keys][part][lane]

    const int tid = threadIdx.x, lane = tid % WAVE, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const int li = lane % 32, lh = lane / 32;
    const int64_t logical = xcd_remap(blockIdx.x, p.nwg);
    const int64_t slice = logical / p.q_blocks, qb = logical % p.q_blocks;
    const int64_t b0 = slice / p.batch1, b1 = slice % p.batch1;
    // (a slice of K, of V and of the mask spans less than 2^31 bytes: launch precondition)
    const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.K + b0 * p.k_sb0 + b1 * p.k_sb1), 0, 0x7fffffff, 0x00020000);
    const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.V + b0 * p.v_sb0 + b1 * p.v_sb1), 0, 0x7fffffff, 0x00020000);
    const int keys = (int)p.Sk, k_row = (int)p.k_sr * 4, v_row = (int)p.v_sr * 4;
    const int64_t row = qb * AS_ROWS + 32 * wave + li, qrow = row < p.Sq ? row : p.Sq - 1;
    const __amdgpu_buffer_rsrc_t m_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(MASKED ? p.mask + b0 * p.m_sb0 + b1 * p.m_sb1 : p.K), 0, 0x7fffffff, 0x00020000);
    const int m_row = (int)(qrow * p.m_sr) * 4;

    auto fragments = [](f32x4 a, f32x4 b, bf16x8 (&f)[SP_PLANES]) __attribute__((always_inline)) {
        u32x4 part[SP_PLANES];
        split_unit8(a, b, part);
#pragma unroll
        for (int q = 0; q < SP_PLANES; ++q) f[q] = __builtin_bit_cast(bf16x8, part[q]);
    };
    bf16x8 fq[D / 16][SP_PLANES];
    {
        const float* Q = p.Q + b0 * p.q_sb0 + b1 * p.q_sb1 + qrow * p.q_sr + 8 * lh;
#pragma unroll
        for (int c = 0; c < D / 16; ++c) fragments(*reinterpret_cast<const f32x4*>(Q + 16 * c), *reinterpret_cast<const f32x4*>(Q + 16 * c + 4), fq[c]);
    }
    f32x16 out[2];   // O^T: columns 32 db + 8 (r / 4) + 4 lh + r % 4 of query row li, times 2^32, not yet divided by the sum
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) out[db][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;
    bool infinite = false;   // a product of Q and K, of any lane of the wave
    const float scale = p.scale * SP_UNSCALE;
    constexpr float LOG2E = 1.44269504088896340736f;

    f32x4 rk[2][2], rv[2][2];
    auto load = [&](int key0) {   // keys beyond the last are the last one
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int idx = tid + it * 256, key = min(key0 + idx / 8, keys - 1);
#pragma unroll
            for (int h = 0; h < 2; ++h)
                rk[it][h] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, key * k_row + 32 * (idx % 8) + 16 * h, 0, 0));
#pragma unroll
            for (int e = 0; e < 8; ++e) {   // a wave's rows: keys 4 lh .. 4 lh + 3 and 8 further on, of the 16 of a step
                const int at = min(key0 + 16 * (2 * it + wave / 2) + 8 * (e / 4) + 4 * (wave % 2) + e % 4, keys - 1);
                rv[it][e / 4][e % 4] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(v_rsrc, 4 * lane, at * v_row, 0));
            }
        }
    };
    load(0);
    for (int key0 = 0; key0 < keys; key0 += AS_KEYS) {
        const bool ragged = key0 + AS_KEYS > keys;   // uniform
        f32x4 add[2][4];   // the mask's values of the scores below
        if constexpr (MASKED) {
            if (!ragged) {
#pragma unroll
                for (int g = 0; g < 8; ++g)
                    add[g / 4][g % 4] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(m_rsrc, m_row + 4 * (key0 + 8 * g + 4 * lh), 0, 0));
            } else {
                auto at = [&](int key) {
                    return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(m_rsrc, m_row + 4 * min(key, keys - 1), 0, 0));
                };
#pragma unroll
                for (int g = 0; g < 8; ++g) {
                    const int key = key0 + 8 * g + 4 * lh;
                    add[g / 4][g % 4] = f32x4{at(key), at(key + 1), at(key + 2), at(key + 3)};
                }
            }
        }
        if (key0 > 0) __syncthreads();   // everyone has read the block before
#pragma unroll
        for (int it = 0; it < 2; ++it) {
            const int idx = tid + it * 256;
            u32x4 part[SP_PLANES];
            split_unit8(rk[it][0], rk[it][1], part);
            const int key = idx / 8, u = idx % 8;   // (rows xor-ed with 4 u: the eight units of a row go to different banks)
#pragma unroll
            for (int q = 0; q < SP_PLANES; ++q)
                *reinterpret_cast<u32x4*>(lds_k + ((key / 32 * (D / 16) + u / 2) * SP_PLANES + q) * PK_PLANE + (u % 2 * 32 + ((key % 32) ^ (4 * u))) * 16) = part[q];
            split_unit8(rv[it][0], rv[it][1], part);
            const int step = idx / 128, half = idx / 64 % 2, d = idx % 64;
#pragma unroll
            for (int q = 0; q < SP_PLANES; ++q)
                *reinterpret_cast<u32x4*>(lds_v + ((d / 32 * (AS_KEYS / 16) + step) * SP_PLANES + q) * PK_PLANE + (half * 32 + d % 32) * 16) = part[q];
        }
        __syncthreads();

        // ---- the scores of this block: s[kb][r] of key 32 kb + 8 (r / 4) + 4 lh + r % 4
        f32x16 s[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            f32x16 sum, small;
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = small[r] = 0.f;
#pragma unroll
            for (int c = 0; c < D / 16; ++c) {
                bf16x8 fk[SP_PLANES];
#pragma unroll
                for (int q = 0; q < SP_PLANES; ++q)
                    fk[q] = *reinterpret_cast<const bf16x8*>(lds_k + ((kb * (D / 16) + c) * SP_PLANES + q) * PK_PLANE + (lh * 32 + (li ^ (4 * (2 * c + lh)))) * 16);
#pragma unroll
                for (int u = 0; u < PK_PRODUCTS; ++u) {
                    f32x16& to = u == 0 ? sum : small;
                    to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fk[PK_QA[u]], fq[c][PK_QB[u]], to, 0, 0, 0);
                }
            }
            s[kb] = sum + small;
        }
        __builtin_amdgcn_sched_barrier(0);
        load(key0 + AS_KEYS);   // in flight under the rest of the block
        __builtin_amdgcn_sched_barrier(0);
        float m_blk = -INFINITY, largest = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) largest = fmaxf(largest, fabsf(s[kb][r]));
        infinite |= __any(largest == INFINITY) != 0;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if constexpr (MASKED) s[kb][r] = fmaf(s[kb][r], scale, add[kb][r / 4][r % 4]);
                else s[kb][r] *= scale;
            }
        if (ragged)
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (key0 + 32 * kb + 8 * (r / 4) + 4 * lh + r % 4 >= keys) s[kb][r] = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) m_blk = fmaxf(m_blk, s[kb][r]);
        const float m_new = fmaxf(m_run, fmaxf(m_blk, __shfl_xor(m_blk, 32, WAVE)));
        const float m_ref = m_new == -INFINITY ? 0.f : m_new;   // nothing but -inf so far: 2^(-inf - 0) = 0
        auto power = [&](float v) { return __builtin_amdgcn_exp2f((v - m_ref) * LOG2E); };
        const float alpha = power(m_run);   // 0 for the first block
        float part_sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[kb][r] = power(s[kb][r]);
                part_sum[r % 4] += s[kb][r];
            }
        const float half_sum = (part_sum[0] + part_sum[1]) + (part_sum[2] + part_sum[3]);
        l_run = l_run * alpha + (half_sum + __shfl_xor(half_sum, 32, WAVE));
        m_run = m_new;

        // ---- out = alpha out + V^T P^T
        bf16x8 fp[AS_KEYS / 16][SP_PLANES];
#pragma unroll
        for (int step = 0; step < AS_KEYS / 16; ++step) {
            f32x4 v[2];
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e / 4][e % 4] = s[step / 2][8 * (step % 2) + e];
            fragments(v[0], v[1], fp[step]);
        }
#pragma unroll
        for (int db = 0; db < 2; ++db) {
            f32x16 sum, small;
#pragma unroll
            for (int r = 0; r < 16; ++r) sum[r] = small[r] = 0.f;
#pragma unroll
            for (int step = 0; step < AS_KEYS / 16; ++step) {
                bf16x8 fv[SP_PLANES];
#pragma unroll
                for (int q = 0; q < SP_PLANES; ++q)
                    fv[q] = *reinterpret_cast<const bf16x8*>(lds_v + ((db * (AS_KEYS / 16) + step) * SP_PLANES + q) * PK_PLANE + lane * 16);
#pragma unroll
                for (int u = 0; u < PK_PRODUCTS; ++u) {
                    f32x16& to = u == 0 ? sum : small;
                    to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fv[PK_QA[u]], fp[step][PK_QB[u]], to, 0, 0, 0);
                }
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) out[db][r] = fmaf(out[db][r], alpha, sum[r] + small[r]);
        }
    }
    // A score that is NaN or positive infinity makes the probabilities NaN and the sums with them. One that the split form made negative
    // infinity would pass for a masked one. With all scores of a row masked that way 0 / 0 is the NaN that the fp32 kernel has there.
    float probe = 0.f;   // stays 0 while all sums are finite
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = fmaf(out[db][r], 0.f, probe);
    if (__syncthreads_or(probe != 0.f || infinite)) {   // (NaN compares unequal)
        for (int half = 0; half < AS_ROWS / AT_BQ; ++half) {
            __syncthreads();
            attention_blocks<MASKED>(p, slice, qb * (AS_ROWS / AT_BQ) + half, reinterpret_cast<float*>(lds), reinterpret_cast<float*>(lds) + AT_SK * AT_PITCH);
        }
        return;
    }
    if (row >= p.Sq) return;
    const float inv = SP_UNSCALE / l_run;
    float* O = p.O + b0 * p.o_sb0 + b1 * p.o_sb1 + row * p.o_sr + 4 * lh;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<f32x4*>(O + 32 * db + 8 * g) =
                f32x4{out[db][4 * g] * inv, out[db][4 * g + 1] * inv, out[db][4 * g + 2] * inv, out[db][4 * g + 3] * inv};
}

// Nanoseconds of a workgroup with a CU to itself and of each further one on it, by blocks of keys: fitted over 26 shapes of 12 to 512 slices, 33
// to 512 keys, both forms measured on each; of the two the form not taken is at most 4 % faster in these.
static double attention_cost(int64_t slices, int64_t Sq, int64_t Sk, int64_t rows, int64_t keys, double fixed, double block, double again, double again_block) {
    const double blocks = (double)ceil_div(Sk, keys), more = (double)(ceil_div(slices * ceil_div(Sq, rows), (int64_t)std::max(device_cus(), 1)) - 1);
    return fixed + blocks * block + more * (again + blocks * again_block);
}
static double split_cost(int64_t slices, int64_t Sq, int64_t Sk) { return attention_cost(slices, Sq, Sk, AS_ROWS, AS_KEYS, 3400, 3800, 1500, 3000); }
static double blocks_cost(int64_t slices, int64_t Sq, int64_t Sk, bool masked) {
    return (masked ? 1 : 0.88) * attention_cost(slices, Sq, Sk, AT_BQ, AT_SK, 2400, 6600, 2000, 4900);
}
static bool split_pays(int64_t slices, int64_t Sq, int64_t Sk, bool masked) { return split_cost(slices, Sq, Sk) < 0.95 * blocks_cost(slices, Sq, Sk, masked); }

// How many waves share the keys in the form for few query blocks, 0 where another form is ahead. A wave to a chunk up to four of them (a workgroup
// to a CU: up to eight); further workgroups on a CU cost what their chunks take. Over 100 shapes of 8 to 512 keys and 12 to 384 slices the pick is at
// most 5 % behind the fastest form but for one (4 x 12 slices of 100 x 100 with a mask: 15 %), and never behind the forms before this one.
static int few_waves(int64_t slices, int64_t Sq, int64_t Sk, bool masked) {
    const int64_t chunks = ceil_div(Sk, (int64_t)AF_KEYS), up = ceil_div(slices * ceil_div(Sq, (int64_t)AF_ROWS), (int64_t)std::max(device_cus(), 1));
    const int waves = chunks <= 1 ? 1 : chunks <= 2 ? 2 : chunks <= 4 || up > 1 ? 4 : 8;
    const double fixed[] = {2400, 2500, 3000, 3950}, chunk[] = {1400, 1500, 1470, 1850};
    const int form = waves == 1 ? 0 : waves == 2 ? 1 : waves == 4 ? 2 : 3;
    const double cost = fixed[form] + chunk[form] * (double)ceil_div(chunks, (int64_t)waves) + (masked ? 1.1 : 1) * (double)(up - 1) * (850 + 210 * (double)chunks);
    return cost < 0.95 * std::min(split_cost(slices, Sq, Sk), blocks_cost(slices, Sq, Sk, masked)) ? waves : 0;
}

// mask == nullptr: the unmasked product
static int launch_attention(const float* Q, const float* K, const float* V, float* O, const float* mask, int64_t batch0,
                            int64_t batch1, int64_t Sq, int64_t Sk, int64_t D, const int64_t* q_strides, const int64_t* k_strides,
                            const int64_t* v_strides, const int64_t* o_strides, const int64_t* mask_strides, float scale, void* stream) {
    MI355X_REQUIRE(batch0 >= 0 && batch1 >= 0 && Sq >= 0, "attention: negative extent");
    MI355X_REQUIRE(Sk >= 1 && D == AT_D, "attention: head size 64 and at least one key are required (got %lld keys x %lld)",
                   (long long)Sk, (long long)D);
    if (batch0 * batch1 == 0 || Sq == 0) return MI355X_OK;
    MI355X_REQUIRE(Q && K && V && O && q_strides && k_strides && v_strides && o_strides, "attention: null pointer");
    auto al16 = [](const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
    bool ok = al16(Q) && al16(K) && al16(V) && al16(O);
    for (int i = 0; i < 3; ++i)
        ok = ok && q_strides[i] % 4 == 0 && k_strides[i] % 4 == 0 && v_strides[i] % 4 == 0 && o_strides[i] % 4 == 0 &&
             q_strides[i] >= 0 && k_strides[i] >= 0 && v_strides[i] >= 0 && o_strides[i] >= 0;
    MI355X_REQUIRE(ok, "attention: operands must be 16-byte aligned with strides that are multiples of 4 floats");
    AttnArgs p;
    p.Q = Q; p.K = K; p.V = V; p.O = O;
    p.batch1 = batch1; p.Sq = Sq; p.Sk = Sk;
    p.q_blocks = ceil_div(Sq, (int64_t)AT_BQ);
    p.nwg = batch0 * batch1 * p.q_blocks;
    MI355X_REQUIRE(grid_fits(p.nwg, 256), "attention: grid too large");
    p.q_sb0 = q_strides[0]; p.q_sb1 = q_strides[1]; p.q_sr = q_strides[2];
    p.k_sb0 = k_strides[0]; p.k_sb1 = k_strides[1]; p.k_sr = k_strides[2];
    p.v_sb0 = v_strides[0]; p.v_sb1 = v_strides[1]; p.v_sr = v_strides[2];
    p.o_sb0 = o_strides[0]; p.o_sb1 = o_strides[1]; p.o_sr = o_strides[2];
    p.scale = scale;
    p.mask = mask;
    p.m_sb0 = mask ? mask_strides[0] : 0; p.m_sb1 = mask ? mask_strides[1] : 0; p.m_sr = mask ? mask_strides[2] : 0;
    const Tuning forced = tuning();
    const int64_t few_nwg = batch0 * batch1 * ceil_div(Sq, (int64_t)AF_ROWS);
    const int waves = forced.attn_few > 0 ? forced.attn_few : forced.attn_few < 0 && forced.attn_split < 0 && forced.attn_waves == 0 ? few_waves(batch0 * batch1, Sq, Sk, mask != nullptr) : 0;
    if (waves > 0 && grid_fits(few_nwg, WAVE * 8)) {
        p.q_blocks = ceil_div(Sq, (int64_t)AF_ROWS);
        p.nwg = few_nwg;
        auto launch = [&](auto count) {
            constexpr int W = decltype(count)::value;
            const dim3 grid((unsigned)p.nwg), block(WAVE * W);
            if (mask) hipLaunchKernelGGL((attention_few_kernel<true, W>), grid, block, 0, static_cast<hipStream_t>(stream), p);
            else hipLaunchKernelGGL((attention_few_kernel<false, W>), grid, block, 0, static_cast<hipStream_t>(stream), p);
        };
        if (waves == 1) launch(std::integral_constant<int, 1>{});
        else if (waves == 2) launch(std::integral_constant<int, 2>{});
        else if (waves <= 4) launch(std::integral_constant<int, 4>{});
        else launch(std::integral_constant<int, 8>{});
        return check_launch("attention_few_kernel");
    }
    const int64_t split_blocks = ceil_div(Sq, (int64_t)AS_ROWS), split_nwg = batch0 * batch1 * split_blocks;
    const int split = forced.attn_split;
    if (split != 0 && grid_fits(split_nwg, 256) && Sk < (1 << 24) && Sk * k_strides[2] < (1 << 29) && Sk * v_strides[2] < (1 << 29) && (!mask || (mask_strides[2] >= 0 && Sq * mask_strides[2] + Sk < (1 << 29))) && (split > 0 || (forced.attn_waves == 0 && split_pays(batch0 * batch1, Sq, Sk, mask != nullptr)))) {
        p.q_blocks = split_blocks;
        p.nwg = split_nwg;
        if (mask) hipLaunchKernelGGL(attention_split_kernel<true>, dim3((unsigned)p.nwg), dim3(256), 0, static_cast<hipStream_t>(stream), p);
        else hipLaunchKernelGGL(attention_split_kernel<false>, dim3((unsigned)p.nwg), dim3(256), 0, static_cast<hipStream_t>(stream), p);
        return check_launch("attention_split_kernel");
    }
    if (mask) {
        hipLaunchKernelGGL(attention_f32_blocks_kernel<true>, dim3((unsigned)p.nwg), dim3(256), 0, static_cast<hipStream_t>(stream), p);
        return check_launch("attention_f32_blocks_kernel");
    }
    if (Sk == AT_SK) {
        // MI355X_ATTN_WAVES = 2 / 3: 32 / 48 query rows per workgroup instead of 64 (measured on 8 x 12 slices of 128 rows:
        // 384 / 288 workgroups instead of 192 -- no faster, the time is one wave's chain of loads, 256 MFMAs and stores)
        const int rows_waves = forced.attn_waves == 2 || forced.attn_waves == 3 ? forced.attn_waves : 4;
        p.q_blocks = ceil_div(Sq, (int64_t)16 * rows_waves);
        p.nwg = batch0 * batch1 * p.q_blocks;
        MI355X_REQUIRE(grid_fits(p.nwg, 64 * rows_waves), "attention: grid too large");
        const dim3 g((unsigned)p.nwg);
        hipStream_t st = static_cast<hipStream_t>(stream);
        if (rows_waves == 2) hipLaunchKernelGGL(attention_f32_kernel<2>, g, dim3(128), 0, st, p);
        else if (rows_waves == 3) hipLaunchKernelGGL(attention_f32_kernel<3>, g, dim3(192), 0, st, p);
        else hipLaunchKernelGGL(attention_f32_kernel<4>, g, dim3(256), 0, st, p);
        return check_launch("attention_f32_kernel");
    }
    hipLaunchKernelGGL(attention_f32_blocks_kernel<false>, dim3((unsigned)p.nwg), dim3(256), 0, static_cast<hipStream_t>(stream), p);
    return check_launch("attention_f32_blocks_kernel");
}

}  // namespace mi355x

extern "C" int mi355x_attention_f32(const float* Q, const float* K, const float* V, float* O,
                                    int64_t batch0, int64_t batch1, int64_t Sq, int64_t Sk, int64_t D,
                                    const int64_t* q_strides, const int64_t* k_strides,
                                    const int64_t* v_strides, const int64_t* o_strides,
                                    float scale, void* stream) {
    return mi355x::launch_attention(Q, K, V, O, nullptr, batch0, batch1, Sq, Sk, D, q_strides, k_strides, v_strides, o_strides, nullptr, scale, stream);
}

extern "C" int mi355x_attention_masked_f32(const float* Q, const float* K, const float* V, float* O, const float* mask,
                                           int64_t batch0, int64_t batch1, int64_t Sq, int64_t Sk, int64_t D,
                                           const int64_t* q_strides, const int64_t* k_strides,
                                           const int64_t* v_strides, const int64_t* o_strides, const int64_t* mask_strides,
                                           float scale, void* stream) {
    using namespace mi355x;
    MI355X_REQUIRE(batch0 * batch1 == 0 || Sq == 0 || (mask && mask_strides), "attention: null mask");
    return launch_attention(Q, K, V, O, mask, batch0, batch1, Sq, Sk, D, q_strides, k_strides, v_strides, o_strides, mask_strides, scale, stream);
}
