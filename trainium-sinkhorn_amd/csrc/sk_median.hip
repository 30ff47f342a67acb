// Exact median of the squared-Euclidean cost over all pairs, on the GPU: the normalisation
// "cost / median(cost)" of src/trnopt/sinkhorn.py:229-233 (wot's), which the reference computes on the host
// by materialising the n x m float64 cost matrix (527 MB at 7,355 x 8,962) and calling np.median.
//
//     C_ij = max((|x_i|^2 + |y_j|^2) - 2 x_i . y_j, 0)        in float64, x and y already centred
//     median = (C_(k0) + C_(k1)) / 2,   k0 = floor((N - 1) / 2), k1 = floor(N / 2),  N = n m
//
// (np.median's definition: the middle element for odd N, the mean of the two middle ones for even N.)
//
// The float64 costs are only needed near the answer. Two passes over approximate costs A_ij, |A_ij - C_ij| <= E,
// find out where that is: the dot products come from the fp16 matrix cores (two fp16 pieces per scaled
// coordinate, three products, as in sk_lse_partial.hip), the rest in float32. An order statistic moves by at most
// E when every element does, so C_(k) lies within E of A_(k), and every pair whose cost can be C_(k0) or C_(k1)
// has A within [A_(k0) - 2 E, A_(k1) + 2 E]:
//   1. histogram of all A (16,384 bins of relative width 2^-10) -> the bins of ranks k0 and k1, widened by 2 E;
//   2. the pairs below that bracket counted, the pairs inside collected (0.1-0.3 % of them);
//   3. the float64 costs of the collected pairs, and their order statistics k0 - below and k1 - below by a radix
//      select (non-negative doubles order like their bit patterns), 11 bits at a time.
// E follows the largest norms, so the few points far outside the others are set aside first (near_limit): they take no part
// in 1 and 2, their pairs' float64 costs are sorted into below, inside and above the bracket one by one (far_kernel), and the
// answer is checked to lie inside it. Without that, one point 40 times the others' norm widened the bracket past the
// workspace: 7,355 x 8,962 d 30 with one point at 20 / 30 / 40 / 1,000 times 290 / 437 / 918 / 1,000 us, and 204 at all of
// them with it.
// When the bracket holds more pairs than the workspace (massive ties), radix-select passes over every float64 cost take
// over (select_pass_kernel): three digits, the third also keeping the keys that still match, and the other three over
// those keys (or over every cost again, if those are too many as well). Every launch goes on the caller's stream with no
// host round trip.
//
// From the norms to the answer, all launches back to back: 7,355 x 8,962 d 30 188 us (the histogram pass 37 of them,
// the collecting pass 52); 10,000 x 10,000 d 64 455 us; 7,000 x 7,000 d 128 271 us; 300 x 257 d 30 94 us. With three
// radix passes over every float64 cost (254 to 187 us each at 7,355 x 8,962, where their fma floor is 54) it was 704,
// 1,633, 1,529 and 121 us.

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "sk_common.h"

namespace {

using sk::f16x8;
using sk::fail;
using sk::hip_fail;

constexpr int kBins = 2048;                 // 11-bit digits
constexpr int kRowsPerBlock = 256;          // one row per thread
constexpr int kColTile = 32;                // column points per LDS tile
constexpr int kTargetBlocks = 1024;         // blocks a full pass aims for: columns per block follow
constexpr int kChunk = 8;                   // coordinates per register chunk of the row
constexpr int kPasses = 6;
constexpr int kKeepPass = 2;                // the full pass that keeps the keys matching its prefix
constexpr unsigned long long kCandMax = 1ull << 22;   // collected pairs, at most
constexpr int kShift[kPasses] = {53, 42, 31, 20, 9, 0};
constexpr int kWidth[kPasses] = {11, 11, 11, 11, 11, 9};

struct SelectState {
    unsigned long long prefix[2];   // bits of the answer known so far (above the current digit)
    unsigned long long k[2];        // rank still to find among the keys that match the prefix
    int same;                       // 1 while both ranks have the same prefix (one histogram serves both)
    int arrived;                    // workgroups of the current launch that have added their counts
};

// What the launches of one call hand on (device memory, the start of the workspace).
struct MedianState {
    SelectState cand;               // the select over the collected pairs
    SelectState full;               // the select over every pair (only with `fallback`)
    unsigned long long below;       // pairs below the bracket
    unsigned long long count;       // pairs inside it
    unsigned long long base;        // key of the bracket's lower end less E: subtracted from the collected keys
    int bits;                       // bits of the largest difference to base
    int fallback;                   // 1: the bracket held more pairs than the workspace, or not the ranks
    unsigned long long kept;        // keys that the third full pass kept
    unsigned far[2];                // points of x and of y set aside
    double vlo, vhi;                // an answer in here is right with points set aside
    int arrived;
    float lo, hi;                   // the bracket, in scaled units
    double scale;                   // power of two: (max |x| + max |y|) scale in [8, 16)
    double err;                     // E in scaled units
};

// |p|^2 of every point of both clouds (fma in ascending coordinate order) and each workgroup's maximum of them. One
// point per thread of the workgroup's 32, its rows first copied to LDS with coalesced loads. The first workgroup also
// writes the initial state and clears the histograms.
constexpr int kNormRows = 32;
__global__ __launch_bounds__(256) void norms_kernel(const double* __restrict__ x, int n, const double* __restrict__ y, int m,
                                                    int d, double* __restrict__ xx, double* __restrict__ yy,
                                                    double* __restrict__ block_max, int xblocks, MedianState* st,
                                                    unsigned* __restrict__ hist) {
    extern __shared__ double rows[];           // kNormRows x (d | 1): an odd row length, so that rows spread over banks
    const bool is_x = (int)blockIdx.x < xblocks;
    const double* p = is_x ? x : y;
    const int np = is_x ? n : m, i0 = (is_x ? (int)blockIdx.x : (int)blockIdx.x - xblocks) * kNormRows;
    const int nr = np - i0 < kNormRows ? np - i0 : kNormRows, ld = d | 1;
    if (blockIdx.x == 0) {
        for (int b = threadIdx.x; b < 2 * kBins; b += blockDim.x) hist[b] = 0u;
        if (threadIdx.x == 0) {
            const unsigned long long N = (unsigned long long)n * (unsigned long long)m;
            SelectState s = {};
            s.k[0] = (N - 1ull) / 2ull;
            s.k[1] = N / 2ull;
            s.same = 1;
            *st = MedianState{};
            st->cand = s;
            st->full = s;
        }
    }
    for (int e = threadIdx.x; e < nr * d; e += blockDim.x) {
        const int r = e / d;
        rows[r * ld + (e - r * d)] = p[(size_t)i0 * d + e];
    }
    __syncthreads();
    if (threadIdx.x >= 64) return;             // the first wave
    double s = 0.0;
    if ((int)threadIdx.x < nr) {
        for (int k = 0; k < d; ++k) s = fma(rows[threadIdx.x * ld + k], rows[threadIdx.x * ld + k], s);
        (is_x ? xx : yy)[i0 + threadIdx.x] = s;
    }
    for (int o = 32; o > 0; o >>= 1) s = fmax(s, __shfl_xor(s, o));
    if (threadIdx.x == 0) block_max[blockIdx.x] = s;
}

__device__ __forceinline__ unsigned long long cost_key(double c) {
    // max(c, 0); -0.0 and +0.0 are the same cost and the same key
    const unsigned long long b = (unsigned long long)__double_as_longlong(c > 0.0 ? c : 0.0);
    return b & 0x7fffffffffffffffull;
}

// The pairs' approximate costs A = |x|^2 + |y|^2 - 2 x . y, in units scaled so that (max |x| + max |y|)^2 lies in
// [64, 256). Histogram bins are the float's top bits: 1,024 per octave over the 16 octaves below 256.
constexpr int kHistBits = 14, kHistBins = 1 << kHistBits, kHistShift = 13;
constexpr unsigned kHistBase = (0x43800000u >> kHistShift) - (unsigned)kHistBins;    // 256 = 2^8 is past the last bin
// E over (max |x| + max |y|)^2 =: R^2. Two fp16 pieces leave a coordinate v within max(2^-23 |v|, 2^-25) and the product
// x1 y1 out: 2^-22 |x||y| + sqrt(d) 2^-25 (|x| + |y|) in all, below 2^-23 R^2 (R >= 8, d <= 128, |x||y| <= R^2 / 4);
// 3 d products summed in float32 err by at most 3 d 2^-24 |x||y| <= 2^-17.4 R^2; the cost's own float32 steps by 2^-22 R^2.
// Twice the dot product's error is below 2^-16 R^2.
constexpr double kCostErr = 0x1p-16;

constexpr float kOutside = 1.0e38f;          // the scaled |p|^2 of a point that takes no part

// The squared norm above which a cloud's points are set aside, from the largest of every 32 points (v, n of them): none
// unless the largest norm is more than 8 times the typical one (the geometric mean of the n, to a power of two of the
// square); then from 4 times, if that concerns at most an eighth of the n. By one wave, alike in every wave.
__device__ inline double near_limit(const double* __restrict__ v, int n) {
    double mx = 0.0;
    int exps = 0, cnt = 0;
    const int lane = (int)(threadIdx.x & 63);
    for (int e = lane; e < n; e += 64) {
        const double t = v[e];
        mx = fmax(mx, t);
        if (t > 0.0 && t < 1.0e300) {
            int x;
            frexp(t, &x);
            exps += x;
            ++cnt;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        mx = fmax(mx, __shfl_xor(mx, o));
        exps += __shfl_xor(exps, o);
        cnt += __shfl_xor(cnt, o);
    }
    const double typical = cnt > 0 ? ldexp(1.0, exps / cnt) : mx;
    if (!(mx > 64.0 * typical)) return mx;
    int far = 0;
    for (int e = lane; e < n; e += 64) far += v[e] > 16.0 * typical ? 1 : 0;
    for (int o = 32; o > 0; o >>= 1) far += __shfl_xor(far, o);
    return 8 * far <= n ? 16.0 * typical : mx;
}

// Both clouds laid out for the passes: a float64 copy with rows of dp coordinates (zeros after d; the columns' also to
// whole tiles), the fp16 pieces of the scaled coordinates in the order of the matrix cores (as sk_pack_cloud_f32's
// tiles: one thread per tile, K chunk and lane), the scaled |p|^2 in float32 (padding points and those set aside, which
// are listed: 1e38, above every cost).
__global__ __launch_bounds__(256) void layout_kernel(const double* __restrict__ x, int n, const double* __restrict__ y, int m,
                                                     int d, int dp, int mp, int nc, const double* __restrict__ xx,
                                                     const double* __restrict__ yy, const double* __restrict__ block_max,
                                                     int xblocks, int yblocks, double* __restrict__ xp,
                                                     double* __restrict__ yp, f16x8* __restrict__ xt,
                                                     f16x8* __restrict__ yt, float* __restrict__ xf, float* __restrict__ yf,
                                                     int ntx, int nty, MedianState* st, unsigned* __restrict__ far_x,
                                                     unsigned* __restrict__ far_y) {
    const double lim_x = near_limit(block_max, xblocks), lim_y = near_limit(block_max + xblocks, yblocks);
    const double R = sqrt(lim_x) + sqrt(lim_y);
    int e = 0;
    if (R > 0.0 && R < 1.0e300) frexp(R, &e);            // R in [2^(e - 1), 2^e)
    const double s = R > 0.0 && R < 1.0e300 ? ldexp(1.0, 4 - e) : 1.0;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->scale = s;
        st->err = kCostErr * (R * s) * (R * s);
    }
    // one wave per row, and one per tile: no index divisions
    const int lane = (int)(threadIdx.x & 63), wave = (int)(blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6));
    const int waves = (int)(gridDim.x * (blockDim.x >> 6));
    for (int side = 0; side < 2; ++side) {
        const double* p = side == 0 ? x : y;
        const int np = side == 0 ? n : m, rows = side == 0 ? n : mp, nt = side == 0 ? ntx : nty;
        double* out = side == 0 ? xp : yp;
        f16x8* tiles = side == 0 ? xt : yt;
        float* f = side == 0 ? xf : yf;
        for (int i = wave; i < rows; i += waves)
            for (int k = lane; k < dp; k += 64) out[(size_t)i * dp + k] = i < np && k < d ? p[(size_t)i * d + k] : 0.0;
        for (int T = wave; T < nt; T += waves) {
            const int row = T * SK_TILE + (lane & 31);
            const double nn = row < np ? (side == 0 ? xx : yy)[row] : 0.0;
            const bool far = nn > (side == 0 ? lim_x : lim_y), near = row < np && !far;
            for (int cc = 0; cc < nc; ++cc) {
                f16x8 p0, p1;
#pragma unroll
                for (int c = 0; c < 8; ++c) {
                    const int k = 16 * cc + 8 * (lane >> 5) + c;
                    const float v = near && k < d ? (float)(p[(size_t)row * d + k] * s) : 0.0f;
                    const _Float16 a = (_Float16)v;
                    p0[c] = a;
                    p1[c] = (_Float16)(v - (float)a);
                }
                f16x8* o = tiles + ((size_t)T * nc + cc) * 128 + lane;
                o[0] = p0;
                o[64] = p1;
            }
            if (lane < 32) {
                f[row] = near ? (float)(nn * s * s) : kOutside;
                if (far) (side == 0 ? far_x : far_y)[atomicAdd(&st->far[side], 1u)] = (unsigned)row;
            }
        }
    }
}

// One pass over the approximate costs, one workgroup of 8 waves per CU. The (64 rows -- 32 above kp 64 --, column tile) units, row by row, are
// cut into equal contiguous ranges, one per wave: the rows' pieces stay in registers, the column tiles come straight
// from L2 one tile ahead. COLLECT false: every cost into the workgroup's histogram in LDS, stored whole to its slab (summed by
// bracket_kernel; no global atomics). COLLECT true: the pairs below the bracket counted, those inside staged in LDS and
// copied out with one reservation per workgroup. Bound by the LDS atomics of the histogram (one per cost).
constexpr int kApproxWaves = 8, kApproxThreads = 64 * kApproxWaves;
constexpr int row_blocks_of(int nc) { return nc <= 4 ? 2 : 1; }   // 32-row blocks per wave (256 registers a lane)
constexpr unsigned kStage = 8192;               // collected pairs a workgroup stages in LDS

template <int NC, bool COLLECT>
__global__ __launch_bounds__(kApproxThreads) void approx_pass_kernel(
    const f16x8* __restrict__ xt, const f16x8* __restrict__ yt, const float* __restrict__ xf, const float* __restrict__ yf,
    int n, int m, int ntx, int nty, MedianState* st, unsigned* __restrict__ slabs, unsigned* __restrict__ pairs,
    unsigned long long cap) {
    __shared__ unsigned bins[COLLECT ? kStage : kHistBins];
    __shared__ unsigned fill;
    __shared__ unsigned long long base;
    const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
    if (COLLECT && st->fallback != 0) return;        // more pairs than cap in the bracket (written by the launch before)
    if (tid == 0) fill = 0u;
    if constexpr (!COLLECT)
        for (int b = tid; b < kHistBins; b += kApproxThreads) bins[b] = 0u;
    __syncthreads();
    float lo = 0.0f;
    unsigned lo_bits = 0u, span = 0u;
    if constexpr (COLLECT) {
        lo = st->lo;
        lo_bits = __float_as_uint(lo);
        span = __float_as_uint(st->hi) - lo_bits;
    }
    constexpr int RB = row_blocks_of(NC);
    const int rbs = (ntx + RB - 1) / RB;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned long long below = 0;
    bool full = false;                               // COLLECT: more pairs than cap, no use collecting any more
    const unsigned long long units = (unsigned long long)rbs * (unsigned)nty, waves = (unsigned long long)gridDim.x * kApproxWaves;
    const unsigned long long w = (unsigned long long)blockIdx.x * kApproxWaves + wave;
    const unsigned u1 = (unsigned)(units * (w + 1) / waves);
    for (unsigned u = (unsigned)(units * w / waves); u < u1;) {
        const int rb = (int)(u / (unsigned)nty), t0 = (int)(u - (unsigned)rb * (unsigned)nty);
        const int t1 = u1 - u < (unsigned)(nty - t0) ? t0 + (int)(u1 - u) : nty;
        u += (unsigned)(t1 - t0);
        f16x8 xv[RB][NC][2];
        float xr[RB];
        int row[RB];
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const int blk = RB * rb + b < ntx ? RB * rb + b : ntx - 1;
            const bool twice = RB * rb + b >= ntx;           // a missing block repeats the last one: kept out by its |x|^2
            row[b] = blk * SK_TILE + (lane & 31);
            xr[b] = twice ? kOutside : xf[row[b]];
#pragma unroll
            for (int c = 0; c < 2 * NC; ++c) xv[b][c / 2][c % 2] = xt[(size_t)blk * (NC * 128) + c * 64 + lane];
        }
        f16x8 ya[NC][2], yb[NC][2];
        sk::f32x4 qa[4], qb[4];
        auto load = [&](int t, f16x8 (&yv)[NC][2], sk::f32x4 (&q)[4]) {
            const int tc = t < t1 ? t : t1 - 1;
#pragma unroll
            for (int c = 0; c < 2 * NC; ++c) yv[c / 2][c % 2] = yt[(size_t)tc * (NC * 128) + c * 64 + lane];
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = *reinterpret_cast<const sk::f32x4*>(yf + tc * SK_TILE + 8 * k + 4 * h);
        };
        unsigned cnt = 0;
        auto tile = [&](int t, const f16x8 (&yv)[NC][2], const sk::f32x4 (&q)[4]) {
#pragma unroll
            for (int b = 0; b < RB; ++b) {
                sk::f32x16 acc = {};
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(yv[c][0], xv[b][c][0], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(yv[c][1], xv[b][c][0], acc, 0, 0, 0);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(yv[c][0], xv[b][c][1], acc, 0, 0, 0);
                }
                unsigned in = 0;                     // COLLECT: the lane's costs inside the bracket
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float a = fmaxf(fmaf(acc[r], -2.0f, q[r / 4][r % 4]) + xr[b], 0.0f);
                    if constexpr (!COLLECT) {
                        const unsigned v = __float_as_uint(a) >> kHistShift;
                        const unsigned c = v < kHistBase ? kHistBase : v;
                        atomicAdd(&bins[(c < kHistBase + kHistBins ? c : kHistBase + kHistBins - 1) - kHistBase], 1u);
                    } else {
                        cnt += a < lo ? 1u : 0u;
                        // non-negative floats order like their bits: lo <= a <= hi in one comparison
                        in |= __float_as_uint(a) - lo_bits <= span ? 1u << r : 0u;
                    }
                }
                if constexpr (COLLECT) {
                    if (in != 0u && !full) {
                        // (padding points cost 1e38, above every bracket)
                        const unsigned k = (unsigned)__popc(in);
                        unsigned p = atomicAdd(&fill, k);
                        const unsigned staged = p >= kStage ? 0u : p + k <= kStage ? k : kStage - p;
                        unsigned long long g = staged < k ? atomicAdd(&st->count, (unsigned long long)(k - staged)) : 0ull;
                        full = g >= cap;
                        do {
                            const int r = __ffs((int)in) - 1;
                            in &= in - 1u;
                            const unsigned col = (unsigned)(t * SK_TILE + 8 * (r >> 2) + 4 * h + (r & 3));
                            const unsigned idx = (unsigned)row[b] * (unsigned)m + col;
                            if (p < kStage) {
                                bins[p] = idx;
                            } else {
                                if (g < cap) pairs[g] = idx;
                                ++g;
                            }
                            ++p;
                        } while (in != 0u);
                    }
                }
            }
        };
        load(t0, ya, qa);
        for (int t = t0; t < t1; t += 2) {
            load(t + 1, yb, qb);
            tile(t, ya, qa);
            if (t + 1 >= t1) break;
            load(t + 2, ya, qa);
            tile(t + 1, yb, qb);
        }
        below += cnt;
    }
    if constexpr (!COLLECT) {
        __syncthreads();
        for (int b = tid; b < kHistBins; b += kApproxThreads) slabs[(size_t)blockIdx.x * kHistBins + b] = bins[b];
    } else {
        for (int o = 32; o > 0; o >>= 1) below += __shfl_xor(below, o);
        if (lane == 0 && below != 0) atomicAdd(&st->below, below);
        __syncthreads();
        const unsigned nf = fill < kStage ? fill : kStage;
        if (tid == 0 && nf != 0u) base = atomicAdd(&st->count, (unsigned long long)nf);
        __syncthreads();
        for (unsigned e = tid; e < nf; e += kApproxThreads)
            if (base + e < cap) pairs[base + e] = bins[e];
    }
}

// Hand-over within a launch without fences (as the loop's merges, sk_lse_partial.hip): data goes through device-scope
// atomics only, every wave waits for its own to complete, and the workgroup's arrival is counted after a barrier. A
// device-scope fence instead writes back and invalidates the XCD's L2, 5 us a launch here. True in the last workgroup.
__device__ inline bool last_to_arrive(int* counter, int blocks) {
    __shared__ int last;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x == 0)
        last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == blocks - 1 ? 1 : 0;
    __syncthreads();
    return last != 0;
}

// The slabs summed (64 bins per workgroup, a quarter of the slabs per wave), and by the last workgroup to finish the bins
// of the two ranks: the bracket.
constexpr int kSumBlocks = kHistBins / 64;
static_assert(kSumBlocks == 256, "one workgroup sum per thread of the last workgroup");
__global__ __launch_bounds__(256) void bracket_kernel(const unsigned* __restrict__ slabs, int nslabs, MedianState* st,
                                                      unsigned long long* __restrict__ total, unsigned long long cap) {
    __shared__ unsigned long long part[256];
    __shared__ int pick[2];
    const int tid = threadIdx.x, bin = (int)blockIdx.x * 64 + (tid & 63);
    unsigned long long s = 0;
    for (int k = tid >> 6; k < nslabs; k += 4 * 16) {
        unsigned v[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) v[e] = k + 4 * e < nslabs ? slabs[(size_t)(k + 4 * e) * kHistBins + bin] : 0u;
#pragma unroll
        for (int e = 0; e < 16; ++e) s += v[e];
    }
    part[tid] = s;
    __syncthreads();
    if (tid < 64) {
        const unsigned long long t = part[tid] + part[tid + 64] + part[tid + 128] + part[tid + 192];
        __hip_atomic_store(total + bin, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned long long sum = t;
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
        if (tid == 0) __hip_atomic_store(total + kHistBins + blockIdx.x, sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (!last_to_arrive(&st->arrived, kSumBlocks)) return;
    // the workgroups' sums scanned, one per thread: the workgroup whose bins hold a rank; then that one's 64 bins by a wave
    __shared__ unsigned long long before[2];
    const unsigned long long mine = __hip_atomic_load(total + kHistBins + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    part[tid] = mine;
    if (tid < 2) {
        pick[tid] = 0;
        before[tid] = 0;
    }
    __syncthreads();
    for (int off = 1; off < 256; off <<= 1) {
        const unsigned long long v = tid >= off ? part[tid - off] : 0ull;
        __syncthreads();
        part[tid] += v;
        __syncthreads();
    }
    for (int r = 0; r < 2; ++r) {
        const unsigned long long rank = st->full.k[r], b = part[tid] - mine;
        if (rank >= b && rank < b + mine) {
            pick[r] = tid;
            before[r] = b;
        }
    }
    __syncthreads();
    if (tid < 128) {
        const int r = tid >> 6, lane = tid & 63, first = pick[r] * 64;
        unsigned long long c = __hip_atomic_load(total + first + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int o = 1; o < 64; o <<= 1) {
            const unsigned long long v = __shfl_up(c, o);
            if (lane >= o) c += v;
        }
        const unsigned long long hit = __ballot(st->full.k[r] < before[r] + c);
        if (lane == 0) pick[r] = first + (hit != 0ull ? __ffsll((long long)hit) - 1 : 63);
    }
    __syncthreads();
    if (tid == 0) {
        const double err = st->err, s2 = st->scale * st->scale;
        const double l = pick[0] == 0 ? 0.0 : (double)__uint_as_float((kHistBase + (unsigned)pick[0]) << kHistShift);
        const double u = pick[1] == kHistBins - 1 ? 1.0e30
                                                  : (double)__uint_as_float((kHistBase + (unsigned)pick[1] + 1u) << kHistShift);
        // one float step outwards on top of 2 E; then E more for the float64 costs of the pairs inside
        const double lb = l - 2.0 * err, ub = u + 2.0 * err;
        st->lo = lb > 0.0 ? (float)(lb * (1.0 - 0x1p-22)) : 0.0f;
        st->hi = (float)(ub * (1.0 + 0x1p-22));
        const double c0 = (lb - 2.0 * err) / s2, c1 = (ub + 2.0 * err) / s2;
        const unsigned long long k0 = c0 > 0.0 ? (unsigned long long)__double_as_longlong(c0) : 0ull;
        const unsigned long long k1 = (unsigned long long)__double_as_longlong(c1 < 1.7e308 ? c1 : 1.7e308);
        st->vlo = st->lo > 0.0f ? ((double)st->lo + err) / s2 : 0.0;      // what is below costs less than this
        st->vhi = ((double)st->hi - err) / s2;                            // and what is above more than this
        st->base = k0;
        st->bits = k1 > k0 ? 64 - __clzll((long long)(k1 - k0)) : 1;
        // More pairs than the workspace holds in whole groups of 64 bins inside the bracket: not even tried. (The last
        // group, with the padding points', is never inside.)
        const unsigned l0 = __float_as_uint(st->lo) >> kHistShift, h0 = __float_as_uint(st->hi) >> kHistShift;
        const int first = (int)(l0 < kHistBase ? 0u : l0 - kHistBase) / 64 + 1;
        const int last = (int)(h0 < kHistBase ? 0u : h0 - kHistBase < kHistBins ? h0 - kHistBase : kHistBins - 1u) / 64 - 1;
        if (last >= first && part[last] - part[first - 1] > cap) st->fallback = 1;
    }
}

__device__ __forceinline__ unsigned long long exact_key(const double* __restrict__ xp, const double* __restrict__ yp,
                                                        const double* __restrict__ xx, const double* __restrict__ yy, unsigned i,
                                                        unsigned j, int dp) {
    const double2* xr = reinterpret_cast<const double2*>(xp + (size_t)i * dp);
    const double2* yr = reinterpret_cast<const double2*>(yp + (size_t)j * dp);
    double acc = 0.0;
    for (int k = 0; k < dp / 2; k += 4) {
        double2 a[4], b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a[q] = xr[k + q];
            b[q] = yr[k + q];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = fma(a[q].y, b[q].y, fma(a[q].x, b[q].x, acc));
    }
    return cost_key((xx[i] + yy[j]) - 2.0 * acc);
}

// The pairs of the points set aside, by their float64 costs: below the bracket, inside it, or above. Every x with the far y,
// every near y with the far x. Bound by gathering the other cloud's rows: the whole call with 2.0 / 3.3 / 7.4 / 8.2 million
// such pairs at 7,355 x 8,962 d 30 494 / 557 / 709 / 739 us, d 128 883 / 1,077 / 1,646 / 1,761; the full passes, taken above
// kFarPairs, 970 and 2,180.
constexpr unsigned long long kFarPairs = 1ull << 23;
__global__ __launch_bounds__(256) void far_kernel(const unsigned* __restrict__ far_x, const unsigned* __restrict__ far_y,
                                                  const float* __restrict__ yf, const double* __restrict__ xp,
                                                  const double* __restrict__ yp, const double* __restrict__ xx,
                                                  const double* __restrict__ yy, int n, int m, int dp, MedianState* st,
                                                  unsigned* __restrict__ pairs, unsigned long long cap) {
    const unsigned long long px = (unsigned long long)st->far[0] * (unsigned)m, py = (unsigned long long)st->far[1] * (unsigned)n;
    if (px + py == 0 || px + py > kFarPairs) {
        if (px + py != 0 && blockIdx.x == 0 && threadIdx.x == 0) st->fallback = 1;
        return;
    }
    const unsigned long long base = st->base;
    const int bits = st->bits;
    unsigned long long below = 0;
    for (unsigned long long e = (unsigned long long)blockIdx.x * 256 + threadIdx.x; e < px + py; e += (unsigned long long)gridDim.x * 256) {
        const bool of_x = e < px;
        const unsigned q = (unsigned)(of_x ? e : e - px), len = (unsigned)(of_x ? m : n), p = q / len, o = q - p * len;
        const unsigned i = of_x ? far_x[p] : o, j = of_x ? o : far_y[p];
        if (of_x && yf[j] == kOutside) continue;
        const unsigned long long key = exact_key(xp, yp, xx, yy, i, j, dp), v = key - base;
        if (key < base) {
            ++below;
        } else if (bits >= 64 || (v >> bits) == 0ull) {
            const unsigned long long g = atomicAdd(&st->count, 1ull);
            if (g < cap) pairs[g] = i * (unsigned)m + j;
        }
    }
    for (int o = 32; o > 0; o >>= 1) below += __shfl_xor(below, o);
    if ((threadIdx.x & 63) == 0 && below != 0) atomicAdd(&st->below, below);
}

// The float64 keys of the collected pairs, less the bracket's base; a key outside the bracket's bits (a cost further
// from its approximation than E, which no finite input gives) sends the call to the full passes, as do too many pairs
// and ranks that are not inside.
__global__ __launch_bounds__(256) void exact_kernel(const unsigned* __restrict__ pairs, const double* __restrict__ xp,
                                                    const double* __restrict__ yp, const double* __restrict__ xx,
                                                    const double* __restrict__ yy, int m, int dp, MedianState* st,
                                                    unsigned long long* __restrict__ keys, unsigned long long cap) {
    const unsigned long long count = st->count, below = st->below, base = st->base;
    const unsigned long long k0 = st->full.k[0], k1 = st->full.k[1];
    const bool ok = count <= cap && k0 >= below && k1 - below < count;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        if (ok) {
            st->cand.k[0] = k0 - below;
            st->cand.k[1] = k1 - below;
        } else {
            st->fallback = 1;
        }
    }
    if (!ok) return;
    const int bits = st->bits;
    for (unsigned long long e = (unsigned long long)blockIdx.x * 256 + threadIdx.x; e < count; e += (unsigned long long)gridDim.x * 256) {
        const unsigned idx = pairs[e];
        const unsigned i = idx / (unsigned)m, j = idx - i * (unsigned)m;
        const unsigned long long key = exact_key(xp, yp, xx, yy, i, j, dp);
        const unsigned long long v = key - base;
        if (key < base || (bits < 64 && (v >> bits) != 0ull)) st->fallback = 1;
        keys[e] = v;
    }
}

// Pick, for each rank, the digit whose bin holds it; narrow the prefix and the rank; clear the histograms. By the last
// workgroup (256 threads, eight bins each) of the launch that filled them.
__device__ inline void select_digit(SelectState* st, unsigned* hist, int shift, int width) {
    __shared__ unsigned long long part[256];
    __shared__ int pick[2];
    __shared__ unsigned long long below[2];
    const int tid = threadIdx.x;
    const int bins = 1 << width, per = (bins + 255) / 256;
    const int same = st->same, hists = same ? 1 : 2;      // one histogram, scanned once, while the ranks share a prefix
    for (int s = 0; s < hists; ++s) {
        const unsigned* hs = hist + s * kBins;
        unsigned c[kBins / 256];                 // all requested at once: the loads come from beyond this XCD's L2
        unsigned long long mine = 0;
#pragma unroll
        for (int b = 0; b < kBins / 256; ++b) {
            const bool in = b < per && tid * per + b < bins;
            c[b] = in ? __hip_atomic_load(hs + tid * per + b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0u;
        }
#pragma unroll
        for (int b = 0; b < kBins / 256; ++b) mine += c[b];
        part[tid] = mine;
        if (tid < 2 && (same || tid == s)) {
            pick[tid] = 0;
            below[tid] = 0ull;
        }
        __syncthreads();
        for (int off = 1; off < 256; off <<= 1) {
            const unsigned long long v = tid >= off ? part[tid - off] : 0ull;
            __syncthreads();
            part[tid] += v;
            __syncthreads();
        }
        for (int r = s; r < (same ? 2 : s + 1); ++r) {
            const unsigned long long k = st->k[r];
            unsigned long long before = part[tid] - mine;
            if (k >= before && k < before + mine) {
                int at = -1;
#pragma unroll
                for (int b = 0; b < kBins / 256; ++b)
                    if (at < 0) {
                        if (k < before + c[b]) at = b;
                        else before += c[b];
                    }
                pick[r] = tid * per + at;
                below[r] = before;
            }
        }
        __syncthreads();
    }
    if (tid == 0) {
        for (int s = 0; s < 2; ++s) {
            st->prefix[s] |= (unsigned long long)pick[s] << shift;
            st->k[s] -= below[s];
        }
        st->same = (same && pick[0] == pick[1]) ? 1 : 0;
        st->arrived = 0;
    }
    for (int b = tid; b < hists * kBins; b += 256) hist[b] = 0u;
}

// A workgroup's digit counts into the launch's, and the digit picked by the last workgroup to add its own (true there).
// same: as select_digit reads it.
__device__ inline bool add_counts(SelectState* st, const unsigned (&h)[2][kBins], int same, unsigned* hist, int shift, int width,
                                  int blocks) {
    for (int b = threadIdx.x; b < (same ? 1 : 2) * kBins; b += 256) {
        const unsigned v = (&h[0][0])[b];
        if (v != 0u) atomicAdd(&hist[b], v);
    }
    if (!last_to_arrive(&st->arrived, blocks)) return false;
    select_digit(st, hist, shift, width);
    return true;
}

// One digit of the select over the collected keys; digit q holds bits [bits - 11 (q + 1), bits - 11 q).
__global__ __launch_bounds__(256) void select_cand_kernel(const unsigned long long* __restrict__ keys, MedianState* st,
                                                          unsigned* __restrict__ hist, int q) {
    __shared__ unsigned h[2][kBins];
    const int top = st->bits - 11 * q;
    if (st->fallback != 0 || top <= 0) return;
    const int shift = top > 11 ? top - 11 : 0, width = top > 11 ? 11 : top;
    const unsigned long long c = st->count;
    const int tid = threadIdx.x;
    const int same = st->cand.same;
    const unsigned long long high = top >= 64 ? 0ull : ~((1ull << top) - 1ull);
    const unsigned long long p0 = st->cand.prefix[0] & high, p1 = st->cand.prefix[1] & high;
    const unsigned dmask = (1u << width) - 1u;
    for (int b = tid; b < (same ? 1 : 2) * kBins; b += 256) (&h[0][0])[b] = 0u;
    __syncthreads();
    for (unsigned long long e = (unsigned long long)blockIdx.x * 256 + tid; e < c; e += (unsigned long long)gridDim.x * 256) {
        const unsigned long long key = keys[e];
        const unsigned digit = (unsigned)(key >> shift) & dmask;
        if ((key & high) == p0) atomicAdd(&h[0][digit], 1u);
        if (!same && (key & high) == p1) atomicAdd(&h[1][digit], 1u);
    }
    __syncthreads();
    if (add_counts(&st->cand, h, same, hist, shift, width, (int)gridDim.x) && shift == 0 && tid == 0 && (st->far[0] | st->far[1]) != 0u) {
        const double a = __longlong_as_double((long long)(st->cand.prefix[0] + st->base));
        const double b = __longlong_as_double((long long)(st->cand.prefix[1] + st->base));
        if (!(a >= st->vlo && b <= st->vhi)) st->fallback = 1;
    }
}

// One digit pass over the workgroup's block of 256 rows x `cols` columns, on the zero-padded copies (rows of
// dp coordinates, a multiple of 8; the column copy padded to whole tiles of 32 points). Each thread keeps its
// row's dot products with a tile of 32 column points in registers and takes the row's coordinates 8 at a
// time; the column coordinates are the same for every lane, so they come through the scalar cache as
// operands of the fma (no LDS traffic). The dot products sum over k in ascending order, one fma each; the
// padding adds 0 * 0.
// The column copy is read through the constant address space: its addresses are the same for every lane, and
// this keeps them on scalar loads whatever else the kernel stores.
typedef __attribute__((address_space(4))) const double ConstDouble;

// KEEP: the pass also keeps the matching keys, if no workgroup has more than kKeepStage of them and all together no more
// than cap; the later passes then read those (`kept_keys`) instead of recomputing every cost. A call at 7,355 x 8,962 d 30
// that ends here takes 703 us by this way, 1,145 with six full passes.
constexpr unsigned kKeepStage = 2048;
template <bool KEEP>
__global__ __launch_bounds__(kRowsPerBlock) void select_pass_kernel(
    const double* __restrict__ xp, const double* __restrict__ yp, const double* __restrict__ xx,
    const double* __restrict__ yy, int n, int m, int dp, int cols, MedianState* ms, unsigned* __restrict__ hist, int shift,
    int width, double* __restrict__ out, unsigned long long* __restrict__ keys, unsigned long long cap, int kept_keys) {
    __shared__ unsigned h[2][kBins];
    __shared__ unsigned long long stage[KEEP ? kKeepStage : 1];
    __shared__ unsigned fill;
    __shared__ unsigned long long base;
    const int tid = threadIdx.x;
    SelectState* st = &ms->full;
    if (ms->fallback == 0) {                              // the collected pairs hold the answer
        if (shift == 0 && blockIdx.x == 0 && tid == 0) {
            const double a = __longlong_as_double((long long)(ms->cand.prefix[0] + ms->base));
            const double b = __longlong_as_double((long long)(ms->cand.prefix[1] + ms->base));
            *out = (a + b) * 0.5;
        }
        return;
    }
    const int same = st->same;
    const unsigned long long high = shift + width >= 64 ? 0ull : ~((1ull << (shift + width)) - 1ull);
    const unsigned long long p0 = st->prefix[0] & high, p1 = st->prefix[1] & high;
    const unsigned dmask = (1u << width) - 1u;
    for (int b = tid; b < 2 * kBins; b += kRowsPerBlock) (&h[0][0])[b] = 0u;
    if (tid == 0) fill = 0u;
    bool full = false;
    __syncthreads();
    const bool on_keys = kept_keys != 0 && ms->kept <= cap;
    if (on_keys) {
        const unsigned long long c = ms->kept;
        for (unsigned long long e = (unsigned long long)blockIdx.x * kRowsPerBlock + tid; e < c;
             e += (unsigned long long)gridDim.x * kRowsPerBlock) {
            const unsigned long long key = keys[e];
            const unsigned digit = (unsigned)(key >> shift) & dmask;
            if ((key & high) == p0) atomicAdd(&h[0][digit], 1u);
            if (!same && (key & high) == p1) atomicAdd(&h[1][digit], 1u);
        }
    }

    const int rbs = (n + kRowsPerBlock - 1) / kRowsPerBlock, cbs = (m + cols - 1) / cols;
    for (int blk = on_keys ? rbs * cbs : (int)blockIdx.x; blk < rbs * cbs; blk += gridDim.x) {
        const int i = blk % rbs * kRowsPerBlock + tid;
        const bool row_ok = i < n;
        const double xi2 = row_ok ? xx[i] : 0.0;
        const double* xr = xp + (size_t)(row_ok ? i : 0) * dp;
        const int j_begin = blk / rbs * cols;
        const long long j_lim = (long long)j_begin + cols;
        const int j_end = j_lim < m ? (int)j_lim : m;

        for (int j0 = j_begin; j0 < j_end; j0 += kColTile) {
            const int nj = j_end - j0 < kColTile ? j_end - j0 : kColTile;
            const ConstDouble* yt = (const ConstDouble*)(yp + (size_t)j0 * dp);
            double acc[kColTile];
#pragma unroll
            for (int jj = 0; jj < kColTile; ++jj) acc[jj] = 0.0;
            for (int k0 = 0; k0 < dp; k0 += kChunk) {
                double xv[kChunk];
#pragma unroll
                for (int e = 0; e < kChunk; ++e) xv[e] = xr[k0 + e];
#pragma unroll
                for (int jj = 0; jj < kColTile; ++jj) {
                    const ConstDouble* yr = yt + (size_t)jj * dp + k0;
                    double a = acc[jj];
#pragma unroll
                    for (int e = 0; e < kChunk; ++e) a = fma(xv[e], yr[e], a);
                    acc[jj] = a;
                }
            }
#pragma unroll
            for (int jj = 0; jj < kColTile; ++jj) {
                const bool ok = row_ok && jj < nj;
                const double c = (xi2 + (jj < nj ? yy[j0 + jj] : 0.0)) - 2.0 * acc[jj];
                const unsigned long long key = cost_key(c);
                const unsigned digit = (unsigned)(key >> shift) & dmask;
                const bool m0 = ok && (key & high) == p0;
                const bool m1 = ok && !same && (key & high) == p1;
                if (m0) atomicAdd(&h[0][digit], 1u);
                if (m1) atomicAdd(&h[1][digit], 1u);
                if constexpr (KEEP) {
                    if ((m0 || m1) && !full) {
                        const unsigned p = atomicAdd(&fill, 1u);
                        if (p < kKeepStage) stage[p] = key;
                        full = p >= kKeepStage;
                    }
                }
            }
        }
    }
    __syncthreads();
    if constexpr (KEEP) {
        const unsigned nf = fill;                          // past the stage: too many, cap and more
        if (tid == 0 && nf != 0u) base = atomicAdd(&ms->kept, nf <= kKeepStage ? (unsigned long long)nf : cap + 1ull);
        __syncthreads();
        if (nf <= kKeepStage)
            for (unsigned e = tid; e < nf; e += kRowsPerBlock)
                if (base + e < cap) keys[base + e] = stage[e];
    }
    if (add_counts(st, h, same, hist, shift, width, (int)gridDim.x) && shift == 0 && tid == 0) {
        const double a = __longlong_as_double((long long)st->prefix[0]);
        const double b = __longlong_as_double((long long)st->prefix[1]);
        *out = (a + b) * 0.5;
    }
}

size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }
int padded_dim(int d) { return (d + kChunk - 1) / kChunk * kChunk; }
int padded_cols(int m) { return (m + kColTile - 1) / kColTile * kColTile; }
unsigned long long cand_cap(int n, int m) {
    const unsigned long long N = (unsigned long long)n * (unsigned long long)m;
    return N < kCandMax ? N : kCandMax;
}

// The workspace of one call.
struct MedianLayout {
    int dp, mp, nc, ntx, nty, xblocks, yblocks, blocks;
    unsigned long long cap;
    size_t state, hist, xx, yy, bmax, xp, yp, xt, yt, xf, yf, farx, fary, total, slabs, keys, bytes;
};

MedianLayout median_layout(int n, int m, int d) {
    MedianLayout o;
    o.dp = padded_dim(d);
    o.mp = padded_cols(m);
    o.nc = (d + 15) / 16;
    o.ntx = (n + SK_TILE - 1) / SK_TILE;
    o.nty = (m + SK_TILE - 1) / SK_TILE;
    o.xblocks = (n + kNormRows - 1) / kNormRows;
    o.yblocks = (m + kNormRows - 1) / kNormRows;
    o.cap = cand_cap(n, m);
    const int rbk = row_blocks_of(o.nc);
    const long long units = (long long)((o.ntx + rbk - 1) / rbk) * o.nty;
    o.blocks = (int)std::min<long long>(256, (units + kApproxWaves - 1) / kApproxWaves);
    size_t p = 0;
    auto take = [&](size_t bytes) {
        const size_t at = p;
        p += align256(bytes);
        return at;
    };
    o.state = take(sizeof(MedianState));
    o.hist = take(2 * kBins * sizeof(unsigned));
    o.xx = take((size_t)n * 8);
    o.yy = take((size_t)m * 8);
    o.bmax = take((size_t)(o.xblocks + o.yblocks) * 8);
    o.xp = take((size_t)n * o.dp * 8);
    o.yp = take((size_t)o.mp * o.dp * 8);
    o.xt = take((size_t)o.ntx * o.nc * 2048);
    o.yt = take((size_t)o.nty * o.nc * 2048);
    o.xf = take((size_t)o.ntx * SK_TILE * 4);
    o.yf = take((size_t)o.nty * SK_TILE * 4);
    o.farx = take((size_t)n * 4);
    o.fary = take((size_t)m * 4);
    o.total = take((size_t)(kHistBins + kSumBlocks) * 8);
    // the histogram slabs, then (they are done with by then) the collected pairs
    o.slabs = take(std::max((size_t)o.blocks * kHistBins * 4, (size_t)o.cap * 4));
    o.keys = take((size_t)o.cap * 8);
    o.bytes = p;
    return o;
}

template <int NC>
void launch_approx(const MedianLayout& o, char* w, int n, int m, hipStream_t s) {
    const f16x8 *xt = (const f16x8*)(w + o.xt), *yt = (const f16x8*)(w + o.yt);
    const float *xf = (const float*)(w + o.xf), *yf = (const float*)(w + o.yf);
    MedianState* st = (MedianState*)(w + o.state);
    unsigned* slabs = (unsigned*)(w + o.slabs);
    hipLaunchKernelGGL((approx_pass_kernel<NC, false>), dim3(o.blocks), dim3(kApproxThreads), 0, s, xt, yt, xf, yf, n, m, o.ntx,
                       o.nty, st, slabs, slabs, o.cap);
    hipLaunchKernelGGL(bracket_kernel, dim3(kSumBlocks), dim3(256), 0, s, slabs, o.blocks, st,
                       (unsigned long long*)(w + o.total), o.cap);
    hipLaunchKernelGGL((approx_pass_kernel<NC, true>), dim3(o.blocks), dim3(kApproxThreads), 0, s, xt, yt, xf, yf, n, m, o.ntx,
                       o.nty, st, slabs, slabs, o.cap);
}

}  // namespace

extern "C" {

size_t sk_cost_median_workspace_bytes(int n, int m, int d) {
    if (n < 1 || m < 1 || d < 1 || d > SK_MEDIAN_D_MAX) return 0;
    return median_layout(n, m, d).bytes;
}

int sk_cost_median_f64(const double* xc, const double* yc, int n, int m, int d, double* out, void* ws,
                       size_t ws_bytes, void* stream) {
    if (xc == nullptr || yc == nullptr || out == nullptr || ws == nullptr)
        return fail(SK_E_ARG, "sk_cost_median_f64: null pointer");
    if (n < 1 || m < 1 || d < 1 || d > SK_MEDIAN_D_MAX)
        return fail(SK_E_SHAPE, "sk_cost_median_f64: need n, m >= 1 and 1 <= d <= SK_MEDIAN_D_MAX");
    if ((unsigned long long)n * (unsigned long long)m > 0xffffffffull)
        return fail(SK_E_SHAPE, "sk_cost_median_f64: n * m must be below 2^32");
    if (ws_bytes < sk_cost_median_workspace_bytes(n, m, d))
        return fail(SK_E_WORKSPACE, "sk_cost_median_f64: workspace too small");
    if (((uintptr_t)ws & 255) != 0) return fail(SK_E_ARG, "sk_cost_median_f64: workspace must be 256-byte aligned");
    const MedianLayout o = median_layout(n, m, d);
    char* w = (char*)ws;
    MedianState* st = (MedianState*)(w + o.state);
    unsigned* hist = (unsigned*)(w + o.hist);
    double *xx = (double*)(w + o.xx), *yy = (double*)(w + o.yy), *bmax = (double*)(w + o.bmax);
    double *xp = (double*)(w + o.xp), *yp = (double*)(w + o.yp);
    unsigned long long* keys = (unsigned long long*)(w + o.keys);
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(norms_kernel, dim3(o.xblocks + o.yblocks), dim3(256), kNormRows * (d | 1) * sizeof(double), s, xc, n, yc,
                       m, d, xx, yy, bmax, o.xblocks, st, hist);
    hipLaunchKernelGGL(layout_kernel, dim3(1024), dim3(256), 0, s, xc, n, yc, m, d, o.dp, o.mp, o.nc, xx, yy, bmax, o.xblocks,
                       o.yblocks, xp, yp, (f16x8*)(w + o.xt), (f16x8*)(w + o.yt), (float*)(w + o.xf), (float*)(w + o.yf),
                       o.ntx, o.nty, st, (unsigned*)(w + o.farx), (unsigned*)(w + o.fary));
    switch (o.nc) {
        case 1: launch_approx<1>(o, w, n, m, s); break;
        case 2: launch_approx<2>(o, w, n, m, s); break;
        case 3: launch_approx<3>(o, w, n, m, s); break;
        case 4: launch_approx<4>(o, w, n, m, s); break;
        case 5: launch_approx<5>(o, w, n, m, s); break;
        case 6: launch_approx<6>(o, w, n, m, s); break;
        case 7: launch_approx<7>(o, w, n, m, s); break;
        default: launch_approx<8>(o, w, n, m, s); break;
    }
    if (std::max(o.xblocks, o.yblocks) >= 8)          // else near_limit sets none aside
        hipLaunchKernelGGL(far_kernel, dim3(256), dim3(256), 0, s, (const unsigned*)(w + o.farx), (const unsigned*)(w + o.fary),
                           (const float*)(w + o.yf), xp, yp, xx, yy, n, m, o.dp, st, (unsigned*)(w + o.slabs), o.cap);
    hipLaunchKernelGGL(exact_kernel, dim3(1024), dim3(256), 0, s, (const unsigned*)(w + o.slabs), xp, yp, xx, yy, m, o.dp, st,
                       keys, o.cap);
    // Six digits at most; a typical bracket's keys differ in their low 43 bits (four digits, the other launches return).
    const int cand_blocks = (int)std::min<unsigned long long>(128ull, (o.cap + 255) / 256);
    for (int q = 0; q < kPasses; ++q)
        hipLaunchKernelGGL(select_cand_kernel, dim3(cand_blocks), dim3(256), 0, s, keys, st, hist, q);
    // The passes over every cost, which return at once unless the collected pairs did not hold the answer: blocks of 256
    // rows by a multiple of a column tile, about kTargetBlocks of them, shared out over the workgroups.
    const int rb = (n + kRowsPerBlock - 1) / kRowsPerBlock;
    const int want = (kTargetBlocks + rb - 1) / rb;
    int cols = (m + want - 1) / want;
    cols = (cols + kColTile - 1) / kColTile * kColTile;
    const long long blocks = (long long)rb * ((m + cols - 1) / cols);
    const dim3 grid((unsigned)std::min<long long>(blocks, kTargetBlocks));
    for (int q = 0; q < kPasses; ++q)
        hipLaunchKernelGGL(q == kKeepPass ? select_pass_kernel<true> : select_pass_kernel<false>, grid, dim3(kRowsPerBlock), 0, s,
                           xp, yp, xx, yy, n, m, o.dp, cols, st, hist, kShift[q], kWidth[q], out, keys, o.cap, q > kKeepPass ? 1 : 0);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SK_OK : hip_fail(e, "sk_cost_median_f64");
}

}  // extern "C"
