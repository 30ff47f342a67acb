// Device code of one (32 rows x 32 columns) tile, shared by the partial kernel (sk_lse_partial.hip) and the loop kernel of
// small problems (sk_loop.hip): the contractions, the column term's MFMA operand and the online log-sum-exp update. Both
// files are built with -fno-honor-nans -mno-amdgpu-ieee (row maxima straight over MFMA results).
#pragma once

#include <type_traits>
#include <utility>

#include "sk_common.h"

namespace sk {
namespace {

__device__ __forceinline__ float ex2(float x) { return __builtin_amdgcn_exp2f(x); }

// A workgroup barrier that orders LDS only: the release / acquire fences are restricted to the local address
// space, so that the wave waits for its LDS accesses (lgkmcnt) but not for its global loads in flight. (The
// fences of __syncthreads also cover global memory and made every wave wait for all its outstanding operand
// loads at the barrier.) For barriers that protect LDS buffers only.
__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// max(a, b, c) as one v_max3_f32 (the compiler would pair the operands into a tree of two-operand maxima).
// Its operands are always written by VALU instructions (the column-term adds), never directly by an MFMA.
__device__ __forceinline__ float max3(float a, float b, float c) {
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Compile-time loop: f(integral_constant<int, i>) for i in [B, E).
template <int B, int E, class F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// The online log-sum-exp update of one row block and one tile, as kOps elementary steps:
//   j == 0:        the tile's 16 column terms of this lane from LDS (four 16-byte reads, shared by the row
//                  blocks; costed high so that the adds land a few MFMA slots later, past the LDS latency)
//   j in [1, 17):  a_r = acc_r + col_r
//   j in [17, 25): running max over a pair of scores
//   j in [25, 41): acc_r = exp2(c (a_r - m)), in place
//   j in [41, 56): the sum of the 16 exponentials as a pairwise tree (8 + 4 + 2 + 1 adds), long after the
//                  exponentials were issued, so no add waits on the transcendental unit
//   j == 56:       S = S exp2(c (M - m)) + sum, M = m
// With FOLD the matrix pipe has already added the column terms (one more MFMA per row block and tile, see
// Streamed) and steps 1-16 are empty; step 0 only starts the running max, costed so that the first reads of
// the accumulators come a few MFMA slots after the last MFMA of the tile.
// The max is subtracted before the scaling: a - m is exact for the scores near the maximum, so the dominant
// term is exactly 1 and S is relative to 2^(c M) exactly, which is what the merge of the slots assumes.
// (Folding the offset into one fma, exp2(c a - fl(c m)), would leave S relative to the rounded fl(c M): an
// error of up to half an ulp of c M in the log-sum-exp, which moves with M from one iteration to the next
// and holds float32 Sinkhorn several ulps away from its fixed point. With L2, c is a power of two, c m is
// exact, and the fma is exactly c (a - m).)
// Steps are spread over the MFMA slots of the next tile in proportion to their cost.
constexpr int kOps = 57;
template <bool FOLD>
constexpr int op_cost(int j) {
    return FOLD && j > 0 && j < 17 ? 0 : j == 0 ? (FOLD ? 6 : 8) : (j >= 25 && j < 41) ? 4 : j == 56 ? 4 : 1;
}
template <bool FOLD>
constexpr int block_cost() {
    int s = 0;
    for (int j = 0; j < kOps; ++j) s += op_cost<FOLD>(j);
    return s;
}
// First step of slot i of NS (steps of the row blocks interleaved: step k is step k / RB of block k % RB).
template <int RB, bool FOLD>
constexpr int op_begin(int i, int NS) {
    const int target = (int)((long long)i * RB * block_cost<FOLD>() / NS);
    int cost = 0, k = 0;
    while (k < RB * kOps && cost < target) {
        cost += op_cost<FOLD>(k / RB);
        ++k;
    }
    return k;
}

// col4(q) returns the column terms of accumulators 4q .. 4q + 3 of the tile being updated (unused with FOLD).
// With L2 the scores are in log2 units times the copy's unit t (the first cloud's log2-unit copy) and c = 1 / t,
// a power of two: the max is subtracted and the rescaling applied by one fma, exp2(fma(a, c, -c m)), exact in
// c m and equal to exp2(c (a - m)) bit for bit (for t = 1, exp2(a - m)).
template <int RB, bool L2, bool FOLD = false>
struct Online {
    float m[RB];
    float mc[RB];      // L2: c m
    f32x4 cv[4];
    template <int k, class ColFn>
    __device__ __forceinline__ void step(f32x16 (&acc)[RB], ColFn&& col4, float (&M)[RB], float (&S)[RB], float c) {
        constexpr int j = k / RB, b = k % RB;
        if constexpr (j == 0) {
            if constexpr (b == 0 && !FOLD)
#pragma unroll
                for (int q = 0; q < 4; ++q) cv[q] = col4(q);
            m[b] = M[b];
        } else if constexpr (j < 17) {
            if constexpr (!FOLD) {
                constexpr int r = j - 1;
                acc[b][r] = acc[b][r] + cv[r / 4][r % 4];
            }
        } else if constexpr (j < 25) {
            constexpr int p = j - 17;
            // With FOLD the operands come straight from the MFMAs: a compiler-visible maximum, so that the
            // compiler keeps the wait states between the matrix results and their first VALU read.
            if constexpr (FOLD)
                m[b] = __builtin_fmaxf(__builtin_fmaxf(m[b], acc[b][2 * p]), acc[b][2 * p + 1]);
            else
                m[b] = max3(m[b], acc[b][2 * p], acc[b][2 * p + 1]);
        } else if constexpr (j < 41) {
            constexpr int r = j - 25;
            if constexpr (L2) {
                if constexpr (r == 0) mc[b] = m[b] * c;
                acc[b][r] = ex2(fmaf(acc[b][r], c, -mc[b]));
            } else {
                acc[b][r] = ex2(c * (acc[b][r] - m[b]));
            }
        } else if constexpr (j < 56) {
            // tree level l (stride 2^l) pairs acc[2^(l+1) q] += acc[2^(l+1) q + 2^l]
            constexpr int t = j - 41;
            constexpr int l = t < 8 ? 0 : t < 12 ? 1 : t < 14 ? 2 : 3;
            constexpr int q = t - (l == 0 ? 0 : l == 1 ? 8 : l == 2 ? 12 : 14);
            constexpr int lo = q << (l + 1), hi = lo + (1 << l);
            acc[b][lo] = acc[b][lo] + acc[b][hi];
        } else {
            S[b] = fmaf(S[b], ex2(L2 ? fmaf(M[b], c, -mc[b]) : c * (M[b] - m[b])), acc[b][0]);
            M[b] = m[b];
        }
    }
};

// The contractions: operand type, pieces per coordinate, the products as (first-cloud piece, second-cloud
// piece) in issue order, and the MFMA.
template <int CT>
struct Contract;

template <>
struct Contract<kF16x2> {
    using T = f16x8;
    static constexpr int pieces = 2, products = 3;
    static constexpr int first[3] = {0, 0, 1};               // x0 y0, x0 y1, x1 y0
    static constexpr int second[3] = {0, 1, 0};
    static __device__ __forceinline__ f32x16 mfma(const T& a, const T& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
    }
};

template <>
struct Contract<kBF16x3> {
    using T = bf16x8;
    static constexpr int pieces = 3, products = 6;
    static constexpr int first[6] = {0, 0, 1, 0, 1, 2};     // x0 y0, x0 y1, x1 y0, x0 y2, x1 y1, x2 y0
    static constexpr int second[6] = {0, 1, 0, 2, 1, 0};
    static __device__ __forceinline__ f32x16 mfma(const T& a, const T& b, const f32x16& c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
    }
};

// The A operand of the column MFMA (v_mfma_f32_32x32x16_bf16 against B = 1 in k < kColPieces of every row): the
// column term q as bf16 pieces that sum to it exactly, (q0 / 4, q0 / 4, q0 / 4, q0 / 4, q1, q2, 0, 0) with
// q0 = bf16(q), q1 = bf16(q - q0), q2 = q - q0 - q1 (each piece the nearest bf16 to what the earlier ones leave:
// 8 + 8 + 8 significand bits, all of fp32's; q0 / 4 is exact for |q| >= 2^-124, and bf16 has fp32's exponent
// range, so no term is out of range).
// Why q0 comes in quarters: this MFMA floors its accumulator input onto the grid of half an ulp of its largest
// product, 2^(e - 24) for a largest product in [2^e, 2^(e+1)), and then rounds the sum to nearest; products
// below that grid are dropped. (Measured on gfx950 over 4.2 million (accumulator, term) pairs of either sign and
// magnitude ratios 2^-14 to 2^3: that rule reproduces every result bit for bit.) With q0 whole, an accumulator
// (the dot product) much smaller than the column term therefore comes out a quarter ulp low on average, a bias
// toward -inf that does not average out over a row's scores and, at eps far above the scores' spread, moved
// balanced potentials along their neutral mode. With the largest product q0 / 4 the grid is four times finer and
// the bias a sixteenth of an ulp (measured: -0.060 against -0.249 ulp of the result); a compensating piece
// below the grid would be dropped, so none is added.
constexpr int kColPieces = 6;
__device__ __forceinline__ bf16x8 column_operand(float v) {
    const __bf16 q0 = (__bf16)v;
    const float r1 = v - (float)q0;                       // exact
    const __bf16 q1 = (__bf16)r1;
    const __bf16 q2 = (__bf16)(r1 - (float)q1);           // exact: at most 8 significant bits remain
    const __bf16 qq = (__bf16)((float)q0 * 0.25f);        // exact
    return bf16x8{qq, qq, qq, qq, q1, q2, 0, 0};
}
// The B operand of the column MFMA: 1 in k < kColPieces of every row (lanes 0-31), zeros elsewhere.
__device__ __forceinline__ bf16x8 column_ones(int h) {
    const __bf16 one = h == 0 ? (__bf16)1.0f : (__bf16)0.0f;
    return bf16x8{one, one, one, one, one, one, 0, 0};
}

}  // namespace
}  // namespace sk
