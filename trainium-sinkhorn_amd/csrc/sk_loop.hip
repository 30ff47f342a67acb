// The on-device loop of small problems as one launch for many iterations (both clouds at most one 32-row block per CU
// and kLoopMaxTiles column tiles; taken by the rule of loop_persists, sk_kernels.hip).
//
// What bounds the launch-by-launch loop there: a half-step at 2,048 x 2,048 d 64 is about 1.5 us of tiles, but its two
// launches take 11 us: each starts up, fetches its arguments and then the scalars they point to, and the slots, the
// potentials and the arguments pass between them through memory. Here one workgroup per 32-row block of x and of y
// stays for all the iterations; all that passes between workgroups is the new potentials, each as one 8-byte word
// {value, iteration tag} that its readers poll: the data is its own flag, so an exchange costs one store and one load
// across the XCDs and no barrier, fence or counter. 700 x 500 d 5: 16.2 -> 9.7 us an iteration, 100 x 90 13.0 -> 8.0,
// 2,048 x 2,048 d 64 20.3 -> 17.4 (launches of 10 iterations; loop_persists has more sizes and both sides of its line).
//
// Bit for bit the launch-by-launch loop: a row block's columns are summed in the same segments as the split of the
// partial kernel gives its row group (Split), each segment by one wave with the same instructions (sk_tile.h), and a
// row's segments are merged in the same order (merge_group); the control takes the same decisions from the same measures
// (control_decide), each workgroup for itself.
//
// Every wait ends. The launch has at most one workgroup per CU, which all run at once where the GPU is free or as soon as
// other streams' workgroups leave their CUs; a poll that has not seen its word after `polls` rounds gives up: its workgroup
// ends without publishing, so that every other one's polls end the same way. The first workgroup, which waits for all the
// others' last words before it writes the state, then writes done = 2 instead and nothing else: the state and the copy's header
// are those the launch began with, y's potentials are saved (`rows`), and launches queued behind do nothing. From there the
// iterations are run again: by one workgroup in a launch queued behind (repair_kernel, 3 us where there is nothing to do), so
// that whoever reads the potentials next, the caller or a kernel, finds them done; or, for a host that looks at the state
// anyway, as ordinary launches (launch_recover), at their speed. When workgroups of several processes share the GPU's CUs,
// each waiting for the rest of its own, that is what ends it, so the first iteration, after which all are known to run, has
// fewer polls in that second form. Four processes side by side, each in 2,048 x 2,048 d 64 solves: 5.4-6.9 ms a solve (launches
// 12.5-12.8), one in 25 with a give-up and then 17-69 ms; with a second's polls and the repair on the device up to 1.1 s.
//
// An ordinary launch, not a cooperative one: the first cooperative launch of a process makes the runtime open one more
// hardware queue, and from then on everything that uses several streams runs slower (four single-cell pairs on streams of
// their own 17 -> 54 ms). What it would add is that two such launches never share the GPU; they must not (each would hold CUs
// that the other waits for, until both give up), so a caller keeps them on one stream.
//
// Where CUs would be idle, `ranks` workgroups share a row block: each takes every ranks-th segment, and rank 0 merges them all,
// one exchange more and a ranks-th of the tiles (2,048 x 2,048 d 64, us an iteration: one rank 25.6, two 20.6, four 16.9).
//
// A potential's word is overwritten only after every reader has it: the next iteration's value is published by a
// workgroup that has read all of the other cloud's values, each published by a workgroup that had read all of this one's.

#include <stddef.h>

#include <atomic>

#include "sk_common.h"
#include "sk_epilogue.h"
#include "sk_tile.h"

namespace sk {
namespace {

constexpr int kMaxPolls = 1 << 20;                  // of a word before a workgroup gives up: about a second
constexpr int kFirstPolls = 1 << 11;                // in the first iteration, where giving up is cheap: a few ms
constexpr int kRowsOfBlock = 32;

typedef unsigned long long u64;

__device__ __forceinline__ void publish(u64* p, unsigned bits, unsigned tag) {
    __hip_atomic_store(p, (u64)bits | ((u64)tag << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ u64 peek(const u64* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// What every workgroup knows of the loop, in LDS; changed by thread 0 between barriers.
struct Ctl {
    sk_state st;          // this workgroup's copy
    float c, t, s2;       // the log2-unit copy: its score scale (0: none), unit, and the second cloud's scale
    int pending;          // its tiles are to be made by this iteration's f update
    int unseen;           // this launch has remade them without this workgroup waiting for it: it makes its rows itself
    int polls;            // rounds before a poll gives up,
    int abort;            // and whether one has
};

// This workgroup's place among the `of` workgroups that share a row block: segment s of the block is rank s % of's. The
// others' (M, S) reach rank 0, which merges and publishes the block, as two tagged words per row and segment.
struct Rank {
    int rank, of;
    u64* slots;           // of this row block: (segment, row, {M, S})
    unsigned tag;
};

// The tile loop of one segment, the rows' operands in xv, the first tile's in yv (load_y(t) requests tile t's): (M, S) per
// lane. A tile's operands are requested as soon as the last MFMA of the one before has read the registers.
template <int NC, int ROLE, bool L2, class LoadY>
__device__ __forceinline__ void segment(const f16x8 (&xv)[NC][2], f16x8 (&yv)[NC][2], LoadY&& load_y, const bf16x8* cols,
                                        const bf16x8& ones, int lane, int tb, int te, float c, float& M, float& S) {
    using C = Contract<kF16x2>;
    float Ms[1] = {kEmpty}, Ss[1] = {0.0f};
    auto none = [](int) { return f32x4{}; };
    for (int t = tb; t < te; ++t) {
        const bf16x8 colA = cols[t * 32 + (lane & 31)];
        f32x16 acc[1] = {f32x16{}};
#pragma unroll
        for (int cc = 0; cc < NC; ++cc)
#pragma unroll
            for (int p = 0; p < C::products; ++p) {
                const int rp = ROLE == 0 ? C::first[p] : C::second[p], cp = ROLE == 0 ? C::second[p] : C::first[p];
                acc[0] = C::mfma(yv[cc][cp], xv[cc][rp], acc[0]);
            }
        if (t + 1 < te) load_y(t + 1);
        acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(colA, ones, acc[0], 0, 0, 0);
        Online<1, L2, true> on;
        static_for<0, kOps>([&](auto K) { on.template step<decltype(K)::value>(acc, none, Ms, Ss, c); });
    }
    M = Ms[0];
    S = Ss[0];
}

// One update: rows of block rb (ROLE 0: x, 1: y) against the other cloud. Fills the merged maximum and sum of row tid for
// tid < 32. expect: the tag of the column potentials (0: the launch's first f update, which takes them from memory).
template <int NC, int ROLE>
__device__ __forceinline__ void update(const PartialArgs& a, const u64* ex, unsigned expect, int rb, const Rank& rk, Ctl& ctl, bf16x8* cols,
                                       float2* slots, float& Mr, float& Sr) {
    constexpr int W = loop_waves(NC), NT = 64 * W, TILE16 = NC * 2 * 64;
    const int tid = tid_x(), lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const float* sc = ROLE == 0 ? ctl.st.sc_x : ctl.st.sc_y;
    const float chs = sc[0] * kLog2e;
    const bool l2 = ctl.c != 0.0f && ctl.c == chs && ctl.s2 == packed_scale(ROLE == 0 ? a.yc : a.xr);
    const float t = ctl.t;
    const f16x8* xt = l2 && ROLE == 0 ? packed_log2_tiles<f16x8>(a.xr, a.nrb * 32, NC) : packed_tiles<f16x8>(a.xr);
    const f16x8* yt = l2 && ROLE == 1 ? packed_log2_tiles<f16x8>(a.yc, a.s.nt * 32, NC) : packed_tiles<f16x8>(a.yc);
    f16x8 xv[NC][2];
#pragma unroll
    for (int k = 0; k < NC * 2; ++k) xv[k / 2][k % 2] = xt[(size_t)rb * TILE16 + k * 64 + lane];
    const bool remake = l2 && ctl.pending != 0;          // this iteration's f update makes x's log2-unit copy
    if (ROLE == 0 && (remake || (l2 && ctl.unseen != 0))) {
        const BakeParams bp = bake_params(a.xr, a.yc, sc);
        const f16x8* own = packed_tiles<f16x8>(a.xr);
#pragma unroll
        for (int cc = 0; cc < NC; ++cc) {
            const size_t u = (size_t)rb * TILE16 + cc * 128 + lane;
            bake_pieces(own[u], own[u + 64], bp, xv[cc][0], xv[cc][1]);
        }
    }
    // The wave's first segment, its first tile requested before the wait for the potentials (unless that is in the making)
    const int g = rb / (kRowsPerGroup / kRowsOfBlock), p0 = first_wg(g, a.s), ns = last_wg(g, a.s) - p0 + 1;
    const int lo = g * a.s.nt, hi = lo + a.s.nt;
    auto bounds = [&](int s, int& tb, int& te) {
        const int q0 = __builtin_amdgcn_readfirstlane(unit_at(cost_start(p0 + s, a.s), a.s));
        const int q1 = __builtin_amdgcn_readfirstlane(unit_at(cost_start(p0 + s + 1, a.s), a.s));
        tb = (q0 > lo ? q0 : lo) - lo;
        te = (q1 < hi ? q1 : hi) - lo;
    };
    int tb = 0, te = 0;
    const int s0 = wave * rk.of + rk.rank, step = W * rk.of;
    if (s0 < ns) bounds(s0, tb, te);
    f16x8 yv[NC][2];
    auto load_y = [&](int q) {
        const f16x8* b0 = yt + (size_t)q * TILE16;
#pragma unroll
        for (int k = 0; k < NC * 2; ++k) yv[k / 2][k % 2] = b0[k * 64 + lane];
    };
    if (!(ROLE == 1 && remake)) load_y(tb);
    // Column terms, as partial_pass takes them
    const float sigma = packed_scale(a.xr) * packed_scale(a.yc);
    const float inv_sigma = l2 ? 1.0f / t : (1.0f / packed_scale(a.xr)) * (1.0f / packed_scale(a.yc));
    const float alpha = l2 ? 1.0f : 0.5f, beta = l2 ? 1.0f : 0.5f * sc[2], cs = l2 ? t : sigma;
    const float c = l2 ? inv_sigma : chs * inv_sigma;
    const float* u0 = l2 ? a.u2 : a.u;
    const float* v0 = l2 ? a.v2 : a.v;
    const int n = a.s.nt * 32;
    for (int j0 = 0; j0 < n; j0 += 4 * NT) {
        float u[4], v[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = j0 + q * NT + tid < n ? j0 + q * NT + tid : n - 1;
            v[q] = v0[j];
            u[q] = expect == 0u ? u0[j] : 0.0f;
        }
        if (expect != 0u) {
            bool all = false;
            for (int r = 0; !all && r < ctl.polls; ++r) {
                u64 w[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) w[q] = peek(ex + (j0 + q * NT + tid < n ? j0 + q * NT + tid : n - 1));
                all = true;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    all = all && (unsigned)(w[q] >> 32) == expect;
                    u[q] = __uint_as_float((unsigned)w[q]);
                }
            }
            if (!all) ctl.abort = 1;
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = j0 + q * NT + tid;
            const float term = fmaxf(cs * fmaf(beta, v[q], fmaf(0.0f, v[q], alpha * u[q])), kPadScore);
            if (j < n) cols[j] = column_operand(term);
        }
    }
    __syncthreads();
    if (rk.rank != 0 && ctl.abort != 0) return;          // publish nothing (rank 0's caller looks)
    if (remake) {
        if (ROLE == 0) {
            // The copy's tiles of this row block, now that every y workgroup has published, i.e. is done with the old copy;
            // out of this XCD's L2 before the rows' potentials are published (by the same wave).
            if (wave == 0 && rk.rank == 0) {
                f16x8* copy = const_cast<f16x8*>(xt) + (size_t)rb * TILE16;
#pragma unroll
                for (int k = 0; k < NC * 2; ++k) copy[k * 64 + lane] = xv[k / 2][k % 2];
                __threadfence();
            }
        } else {
            __threadfence();      // the copy that the other workgroups have made, not this L2's old lines
            load_y(tb);
        }
    }
    const bf16x8 ones = column_ones(lane >> 5);
    for (int s = s0; s < ns; s += step) {
        float M, S;
        if (l2)
            segment<NC, ROLE, true>(xv, yv, load_y, cols, ones, lane, tb, te, c, M, S);
        else
            segment<NC, ROLE, false>(xv, yv, load_y, cols, ones, lane, tb, te, c, M, S);
        if (s + step < ns) {
            bounds(s + step, tb, te);
            load_y(tb);
        }
        // as store_rows
        const float Mo = __shfl_xor(M, 32), So = __shfl_xor(S, 32);
        const float Mn = fmaxf(M, Mo);
        const float Sn = S * ex2(c * (M - Mn)) + So * ex2(c * (Mo - Mn));
        const float2 v = make_float2(fmaxf(Mn * inv_sigma, kEmpty), Sn);
        if (lane < 32) {
            if (rk.rank == 0) {
                slots[s * kRowsOfBlock + lane] = v;
            } else {
                u64* dst = rk.slots + 2 * (size_t)(s * kRowsOfBlock + lane);
                publish(dst, __float_as_uint(v.x), rk.tag);
                publish(dst + 1, __float_as_uint(v.y), rk.tag);
            }
        }
    }
    if (rk.rank == 0 && rk.of > 1)
        for (int k = tid; k < ns * kRowsOfBlock; k += NT) {
            if (k / kRowsOfBlock % rk.of == 0) continue;
            u64 m = 0, q = 0;
            bool all = false;
            for (int r = 0; !all && r < ctl.polls; ++r) {
                m = peek(rk.slots + 2 * (size_t)k);
                q = peek(rk.slots + 2 * (size_t)k + 1);
                all = (unsigned)(m >> 32) == rk.tag && (unsigned)(q >> 32) == rk.tag;
            }
            if (!all) ctl.abort = 1;
            slots[k] = make_float2(__uint_as_float((unsigned)m), __uint_as_float((unsigned)q));
        }
    __syncthreads();
    if (rk.rank == 0 && tid < kRowsOfBlock) {
        // as merge_group
        const float cm = l2 ? 1.0f : chs;
        float M = kEmpty, S = 0.0f;
        for (int q = 0; q < ns; q += kMergeBatch) {
            float2 v[kMergeBatch];
#pragma unroll
            for (int k = 0; k < kMergeBatch; ++k) v[k] = q + k < ns ? slots[(q + k) * kRowsOfBlock + tid] : make_float2(kEmpty, 0.0f);
            float Mn = M;
#pragma unroll
            for (int k = 0; k < kMergeBatch; ++k) Mn = fmaxf(Mn, v[k].x);
            float Sn = S * ep_ex2(cm * (M - Mn));
#pragma unroll
            for (int k = 0; k < kMergeBatch; ++k) Sn += v[k].y * ep_ex2(cm * (v[k].x - Mn));
            M = Mn;
            S = Sn;
        }
        Mr = M;
        Sr = S;
    }
}

// The control of one iteration (every workgroup for itself, from the same measures): advances ctl, true when the loop is
// done. ny: row blocks of y; msr their published measures {max change}, {low}, {high half of the error sum} (null: they are in
// lds_mx and lds_sm already).
template <int NT>
__device__ inline bool control(const PartialArgs& g, const u64* msr, unsigned tag, int ny, bool measured, Ctl& ctl, float* lds_mx,
                               double* lds_sm) {
    const int tid = tid_x();
    if (measured && msr != nullptr) {
        for (int b = tid; b < ny; b += NT) {
            u64 w[3];
            bool all = false;
            for (int r = 0; !all && r < ctl.polls; ++r) {
                all = true;
                for (int q = 0; q < 3; ++q) {
                    w[q] = peek(msr + 3 * b + q);
                    all = all && (unsigned)(w[q] >> 32) == tag;
                }
            }
            if (!all) ctl.abort = 1;
            lds_mx[b] = __uint_as_float((unsigned)w[0]);
            lds_sm[b] = __longlong_as_double((long long)((w[1] & 0xffffffffull) | (w[2] << 32)));
        }
        __syncthreads();
    }
    if (tid < 64) {
        float mx = 0.0f;
        double sm = 0.0;
        constexpr int kPer = kRowsPerGroup / kRowsOfBlock;
        if (measured && tid * kPer < ny) {        // one row group per lane, its sum as merge_group stores it
            double wsum[kPer / 2];
#pragma unroll
            for (int b = 0; b < kPer; ++b) {
                const int k = tid * kPer + b;
                const double v = k < ny ? lds_sm[k] : 0.0;
                wsum[b / 2] = b % 2 == 0 ? v : wsum[b / 2] + v;
                if (k < ny) mx = fmaxf(mx, lds_mx[k]);
            }
            double s = wsum[0];
#pragma unroll
            for (int b = 1; b < kPer / 2; ++b) s += wsum[b];
            sm = (double)(float)s;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            mx = fmaxf(mx, __shfl_xor(mx, o));
            sm += __shfl_xor(sm, o);
        }
        if (tid == 0) {
            sk_state& st = ctl.st;
            const LoopCfg& cfg = g.cfg;
            int stage = st.stage, stage_it = st.stage_it, conv = 0;
            double err;
            if (control_decide(cfg, st.it, st.sc_x[1], mx, sm, stage, stage_it, conv, err)) {
                st.err = err;
                st.checks += 1;
            }
            st.stage = stage;
            st.stage_it = stage_it;
            st.converged = conv;
            st.done = conv != 0 || st.it >= cfg.max_iters ? 1 : 0;
            if (st.done == 0) {
                const float ran = st.sc_x[0];
                set_scalars(&st, eps_for(cfg, st.it, stage), cfg.rho_x, cfg.rho_y);
                if (st.sc_x[0] != ran) {          // a new eps: the copy for it, made by the next f update
                    const BakeParams b = bake_params(g.yc, g.xr, st.sc_x);
                    ctl.c = b.valid ? b.c : 0.0f;
                    ctl.t = b.valid ? b.t : 1.0f;
                    ctl.s2 = packed_scale(g.xr);
                    ctl.pending = b.valid ? 1 : 0;
                }
            }
        }
    }
    __syncthreads();
    return ctl.st.done != 0;
}

// The head of the exchange (zero at loop init).
struct Notes {
    int gave_up;          // the launch (LoopArgs::id) of which a workgroup has given up last
    int repairs;          // launches run again since the loop's init
};
static_assert(sizeof(Notes) <= 8 * kLoopNoteWords, "the exchange begins with kLoopNoteWords words for it");

struct LoopArgs {
    PartialArgs f, g;
    u64 *ex, *ey, *msr;      // the potentials of x and y and (two turns of) the measures of y's row blocks, tagged words
    u64 *sx, *sy;            // the segments' (M, S) of the ranks above 0 (Rank)
    float2* rows;            // y's potentials where the launch began: gh and its log2-unit potential
    Notes* notes;
    int id;                  // of this launch, not 0: another one's for every launch of the process
    int iters, polls, first_polls, ranks;
    int slots_x, slots_y;    // segments of a row block, at most
};

// One row of an update from its merged maximum and sum: the new potential, and R in its log2-unit potential (R + Ll).
template <int ROLE>
__device__ __forceinline__ float row_of(const PartialArgs& a, const Ctl& ctl, float M, float S, float p2, float off, float l2lo,
                                        float& u2, bool& l2) {
    const float* sc = ROLE == 0 ? ctl.st.sc_x : ctl.st.sc_y;
    const float chs = sc[0] * kLog2e;
    l2 = ctl.c != 0.0f && ctl.c == chs && ctl.s2 == packed_scale(ROLE == 0 ? a.yc : a.xr);
    const Log2Split ls = lse_log2(S);
    double R = 0.0;
    const float h = row_value({sc[2], sc[3], chs, p2, off}, l2, true, (double)M + (l2 ? (double)loop_weight_offset(a.yc) : 0.0),
                              (double)ls.e + (double)ls.lm, R);
    u2 = (float)(R + (double)l2lo);
    return h;
}

// The measures of a block of y's rows, one row per lane of the first half wave: the largest change and the error sum.
__device__ __forceinline__ void row_measures(const Ctl& ctl, float old, float now, bool real, float w, float& dmax, double& derr) {
    dmax = real ? fabsf(now - old) : 0.0f;
    const float delta = fminf((old - now) * ctl.st.sc_y[1], kDeltaCap);
    derr = (double)fabsf(w * (expf(delta) - 1.0f));
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) {
        dmax = fmaxf(dmax, __shfl_xor(dmax, o));
        derr += __shfl_xor(derr, o);
    }
}

// Whether the control of the iteration that ends looks at its measures.
__device__ __forceinline__ bool takes_measures(const LoopCfg& cfg, int it) {
    return cfg.n_stages > 0 || (cfg.fixed_iters == 0 && it > cfg.n_sched);
}

// This iteration's f update has made a pending copy if it was for its eps. (Another eps: the copy of another loop on the same
// clouds, still pending.)
__device__ __forceinline__ bool made_copy(const PartialArgs& f, const Ctl& ctl) {
    return ctl.pending != 0 && ctl.c == ctl.st.sc_x[0] * kLog2e && ctl.s2 == packed_scale(f.yc);
}

// y's log2-unit potential at a new eps, from gh as the control derives it.
__device__ __forceinline__ float at_new_eps(const Ctl& ctl, float gh, float l2lo) {
    return (float)((double)gh * (0.5 * (double)(ctl.st.sc_x[0] * kLog2e)) + (double)l2lo);
}

// The state and the copy's header, by one thread.
__device__ __forceinline__ void write_back(const LoopArgs& a, const Ctl& ctl) {
    *a.g.state = ctl.st;
    float* h = reinterpret_cast<float*>(a.f.rebake);
    const bool p = ctl.pending != 0;
    h[2] = p ? 0.0f : ctl.c;
    h[3] = ctl.s2;
    if (!p) h[4] = ctl.t;
    h[7] = ctl.c;
    h[8] = ctl.t;
    reinterpret_cast<int*>(h)[6] = p ? 1 : 0;
}

template <int NC>
__global__ __launch_bounds__(64 * loop_waves(NC)) void loop_kernel(LoopArgs a) {
    constexpr int NT = 64 * loop_waves(NC);
    __shared__ __attribute__((aligned(16))) bf16x8 cols[kLoopMaxTiles * 32];
    __shared__ float2 slots[kLoopMaxTiles * kRowsOfBlock];      // a segment has a tile at least
    __shared__ float lds_mx[kLoopMaxBlocks];
    __shared__ double lds_sm[kLoopMaxBlocks];
    __shared__ Ctl ctl;
    const int tid = tid_x(), rank = wg_x() % a.ranks, w = wg_x() / a.ranks;
    // Row blocks this workgroup has segments of: without any in a pass it takes no part in it.
    auto segments = [&](const PartialArgs& p) {
        if (w >= p.nrb) return 0;
        const int g = w / (kRowsPerGroup / kRowsOfBlock);
        return last_wg(g, p.s) - first_wg(g, p.s) + 1;
    };
    const int nsx = segments(a.f), nsy = segments(a.g);
    const bool has_x = rank < nsx, has_y = rank < nsy;
    if (!has_x && !has_y) return;
    const int i = w * kRowsOfBlock + tid;
    const bool rx = has_x && rank == 0 && tid < kRowsOfBlock, ry = has_y && rank == 0 && tid < kRowsOfBlock;
    float fh = rx ? a.f.out[i] : 0.0f, fr = rx ? a.f.out2[i] : 0.0f, gh = ry ? a.g.out[i] : 0.0f, gr = ry ? a.g.out2[i] : 0.0f;
    sk_state* const gst = a.g.state;
    if (tid == 0) {
        // by one thread: workgroups that have given up already may be writing both
        const int was_done = coh_load(&gst->done);
        __threadfence();
        ctl.abort = coh_load(&a.notes->gave_up) == a.id ? 1 : 0;
        ctl.st = *gst;
        ctl.st.done = ctl.abort != 0 ? 0 : was_done;
        const CopyTag tag = copy_tag(reinterpret_cast<const float*>(a.f.xr), true);
        ctl.c = tag.c;
        ctl.t = tag.t;
        ctl.s2 = tag.s2;
        ctl.pending = tag.pending;
        ctl.unseen = 0;
        ctl.polls = a.first_polls;
    }
    u64* const sx = a.sx + (size_t)w * a.slots_x * kRowsOfBlock * 2;
    u64* const sy = a.sy + (size_t)w * a.slots_y * kRowsOfBlock * 2;
    const LoopCfg& cfg = a.g.cfg;
    const float x2 = rx ? a.f.xsq[i] : 0.0f, xo = rx && a.f.off != nullptr ? a.f.off[i] : 0.0f, xl = rx ? a.f.rows_l2lo[i] : 0.0f;
    const float y2 = ry ? a.g.xsq[i] : 0.0f, yo = ry && a.g.off != nullptr ? a.g.off[i] : 0.0f, yl = ry ? a.g.rows_l2lo[i] : 0.0f;
    const float yw = ry ? a.g.w[i] : 0.0f;
    __syncthreads();
    const bool done_before = ctl.st.done != 0, late = ctl.abort != 0;
    __syncthreads();                       // every wave has the same answer before one may set abort
    if (done_before) return;
    if (ry) a.rows[i] = make_float2(gh, gr);       // (a late workgroup's rows too: nothing has changed them)
    if (late) {
        if (w == 0 && rank == 0 && tid == 0) coh_store(&gst->done, 2);
        return;
    }
    unsigned ytag = 0u;                    // the tag of y's latest potentials (0: in memory)
    bool done = false;
    for (int k = 0; k < a.iters && !done; ++k) {
        const unsigned tag = 2u * (unsigned)ctl.st.it + 1u;
        float M = 0.0f, S = 1.0f;
        // the f update
        if (has_x) {
            update<NC, 0>(a.f, a.ey, ytag, w, {rank, a.ranks, sx, tag}, ctl, cols, slots, M, S);
            if (rx && ctl.abort == 0) {
                bool l2;
                fh = row_of<0>(a.f, ctl, M, S, x2, xo, xl, fr, l2);
                publish(a.ex + i, __float_as_uint(l2 ? fr : fh), tag);
            }
        }
        __syncthreads();
        if (ctl.abort != 0) break;
        if (tid == 0) {
            ctl.st.it += 1;
            ctl.st.stage_it += 1;
        }
        __syncthreads();
        // the g update
        const bool need = needs_control(ctl.st.it, ctl.st.stage, ctl.st.stage_it, cfg);
        u64* const msr = a.msr + 3 * (size_t)a.g.nrb * (ctl.st.it & 1);
        const bool measured = need && takes_measures(cfg, ctl.st.it);
        if (has_y) {
            update<NC, 1>(a.g, a.ex, tag, w, {rank, a.ranks, sy, tag}, ctl, cols, slots, M, S);
            if (ry && ctl.abort == 0) {
                bool l2;
                const float old = gh;
                gh = row_of<1>(a.g, ctl, M, S, y2, yo, yl, gr, l2);
                if (measured) {
                    float dmax;
                    double derr;
                    row_measures(ctl, old, gh, i < a.g.n_real, yw, dmax, derr);
                    if (tid == 0) {
                        const u64 e = (u64)__double_as_longlong(derr);
                        publish(msr + 3 * w, __float_as_uint(dmax), tag + 1u);
                        publish(msr + 3 * w + 1, (unsigned)e, tag + 1u);
                        publish(msr + 3 * w + 2, (unsigned)(e >> 32), tag + 1u);
                    }
                }
            }
        }
        __syncthreads();
        if (ctl.abort != 0) break;
        if (tid == 0) {
            if (made_copy(a.f, ctl)) {       // rank 0 its block's tiles itself, and a g update waits for all of them
                if (rank != 0 && !has_y) ctl.unseen = 1;
                ctl.pending = 0;
            }
        }
        const float ran = ctl.st.sc_x[0];
        if (need) {
            __syncthreads();
            done = control<NT>(a.g, msr, tag + 1u, a.g.nrb, measured, ctl, lds_mx, lds_sm);
            if (ctl.abort != 0) break;
        }
        if (ry) {
            // y's potentials in the units of the next f update
            if (!done && ctl.st.sc_x[0] != ran) gr = at_new_eps(ctl, gh, yl);
            const bool next_l2 = ctl.c != 0.0f && ctl.c == ctl.st.sc_x[0] * kLog2e && ctl.s2 == packed_scale(a.g.xr);
            publish(a.ey + i, __float_as_uint(next_l2 ? gr : gh), tag + 1u);
        }
        ytag = tag + 1u;
        if (k == 0 && tid == 0) ctl.polls = a.polls;
        __syncthreads();
    }
    if (rx) {
        a.f.out[i] = fh;
        a.f.out2[i] = fr;
    }
    if (ry) {
        a.g.out[i] = gh;
        a.g.out2[i] = gr;
    }
    // The state and the copy's header, once every workgroup has read them (they all have published y's last values, or
    // x's that those rest on). A workgroup that gives up after that, in its last control, has stored its rows above and owes
    // nobody anything.
    if (w == 0 && rank == 0 && ctl.abort == 0) {
        bool all = true;
        for (int j = tid; j < a.g.nrb; j += NT) {
            bool seen = false;
            for (int r = 0; !seen && r < ctl.polls; ++r) seen = (unsigned)(peek(a.ey + j * kRowsOfBlock) >> 32) == ytag;
            all = all && seen;
        }
        if (!all) ctl.abort = 1;
    }
    __syncthreads();
    if (ctl.abort != 0) {
        if (tid == 0) {
            coh_store(&a.notes->gave_up, a.id);
            __threadfence();
            if (w == 0 && rank == 0) coh_store(&gst->done, 2);
        }
        return;
    }
    if (w == 0 && rank == 0 && tid == 0) write_back(a, ctl);
}

// The iterations of a launch that gave up, by one workgroup: every row block in turn, with the same instructions in the same
// order, the potentials through memory (fences: the workgroup reads its own stores). 100 iterations at 2,048 x 2,048 d 64
// take 0.4 s, which nobody is meant to see.
template <int NC>
__global__ __launch_bounds__(64 * loop_waves(NC)) void repair_kernel(LoopArgs a) {
    constexpr int NT = 64 * loop_waves(NC);
    __shared__ __attribute__((aligned(16))) bf16x8 cols[kLoopMaxTiles * 32];
    __shared__ float2 slots[kLoopMaxTiles * kRowsOfBlock];
    __shared__ float lds_mx[kLoopMaxBlocks];
    __shared__ double lds_sm[kLoopMaxBlocks];
    __shared__ Ctl ctl;
    if (a.g.state->done != 2) return;
    const int tid = tid_x();
    const Rank alone = {0, 1, nullptr, 0u};
    const LoopCfg& cfg = a.g.cfg;
    if (tid == 0) {
        const CopyTag tag = copy_tag(reinterpret_cast<const float*>(a.f.xr), true);
        ctl.st = *a.g.state;
        ctl.st.done = 0;
        ctl.c = tag.c;
        ctl.t = tag.t;
        ctl.s2 = tag.s2;
        ctl.pending = tag.pending;
        ctl.unseen = 0;
        ctl.polls = 0;
        ctl.abort = 0;
        // (this loop's copy may be overwritten by a later eps's, whose f updates the launch has reached: made anew)
        if (ctl.c != 0.0f && ctl.c == ctl.st.sc_x[0] * kLog2e && ctl.s2 == packed_scale(a.f.yc)) ctl.pending = 1;
    }
    for (int i = tid; i < a.g.nrb * kRowsOfBlock; i += NT) {
        const float2 v = a.rows[i];
        a.g.out[i] = v.x;
        a.g.out2[i] = v.y;
    }
    __threadfence();
    __syncthreads();
    bool done = false;
    for (int k = 0; k < a.iters && !done; ++k) {
        for (int b = 0; b < a.f.nrb; ++b) {
            float M = 0.0f, S = 1.0f;
            update<NC, 0>(a.f, nullptr, 0u, b, alone, ctl, cols, slots, M, S);
            if (tid < kRowsOfBlock) {
                const int i = b * kRowsOfBlock + tid;
                float u2;
                bool l2;
                a.f.out[i] = row_of<0>(a.f, ctl, M, S, a.f.xsq[i], a.f.off != nullptr ? a.f.off[i] : 0.0f, a.f.rows_l2lo[i], u2, l2);
                a.f.out2[i] = u2;
            }
            __syncthreads();
        }
        __threadfence();
        if (tid == 0) {
            ctl.st.it += 1;
            ctl.st.stage_it += 1;
        }
        __syncthreads();
        const bool need = needs_control(ctl.st.it, ctl.st.stage, ctl.st.stage_it, cfg);
        const bool measured = need && takes_measures(cfg, ctl.st.it);
        for (int b = 0; b < a.g.nrb; ++b) {
            float M = 0.0f, S = 1.0f;
            update<NC, 1>(a.g, nullptr, 0u, b, alone, ctl, cols, slots, M, S);
            if (tid < kRowsOfBlock) {
                const int i = b * kRowsOfBlock + tid;
                float u2;
                bool l2;
                const float old = a.g.out[i];
                const float gh = row_of<1>(a.g, ctl, M, S, a.g.xsq[i], a.g.off != nullptr ? a.g.off[i] : 0.0f, a.g.rows_l2lo[i], u2, l2);
                a.g.out[i] = gh;
                a.g.out2[i] = u2;
                float dmax;
                double derr;
                row_measures(ctl, old, gh, i < a.g.n_real, a.g.w[i], dmax, derr);
                if (tid == 0) {
                    lds_mx[b] = dmax;
                    lds_sm[b] = derr;
                }
            }
            __syncthreads();
        }
        const float ran = ctl.st.sc_x[0];
        if (tid == 0 && made_copy(a.f, ctl)) ctl.pending = 0;
        __syncthreads();
        if (need) done = control<NT>(a.g, nullptr, 0u, a.g.nrb, measured, ctl, lds_mx, lds_sm);
        if (!done && ctl.st.sc_x[0] != ran)
            for (int i = tid; i < a.g.nrb * kRowsOfBlock; i += NT) a.g.out2[i] = at_new_eps(ctl, a.g.out[i], a.g.rows_l2lo[i]);
        __threadfence();
        __syncthreads();
    }
    if (tid == 0) {
        write_back(a, ctl);
        a.notes->repairs += 1;
    }
}

// Back to where a launch that gave up began, for launches to go on from. The copy's tiles may be those of an eps that the
// launch had reached: this loop's copy is made anew by the next f update, another's is dropped.
__global__ __launch_bounds__(256) void recover_kernel(LoopArgs a) {
    __shared__ int failed;
    const int tid = tid_x();
    if (tid == 0) failed = a.g.state->done == 2 ? 1 : 0;
    __syncthreads();
    if (failed == 0) return;
    for (int i = tid; i < a.g.nrb * kRowsOfBlock; i += 256) {
        const float2 v = a.rows[i];
        a.g.out[i] = v.x;
        a.g.out2[i] = v.y;
    }
    if (tid != 0) return;
    a.g.state->done = 0;
    a.notes->repairs += 1;
    float* h = reinterpret_cast<float*>(a.f.rebake);
    const CopyTag tag = copy_tag(h, true);
    h[2] = 0.0f;
    if (tag.c != 0.0f && tag.c == a.g.state->sc_x[0] * kLog2e && tag.s2 == packed_scale(a.f.yc)) {
        h[7] = tag.c;
        h[8] = tag.t;
        reinterpret_cast<int*>(h)[6] = 1;
    }
}

template <int NC>
hipError_t launch_nc(const LoopArgs& a, int workgroups, bool repair, hipStream_t st) {
    const dim3 threads(64 * loop_waves(NC));
    hipLaunchKernelGGL(loop_kernel<NC>, dim3(workgroups), threads, 0, st, a);
    if (repair) hipLaunchKernelGGL(repair_kernel<NC>, dim3(1), threads, 0, st, a);
    return hipGetLastError();
}

LoopArgs loop_args(const PartialArgs& f, const PartialArgs& g, void* exchange, int ranks, int slots_x, int slots_y) {
    LoopArgs a;
    a.f = f;
    a.g = g;
    a.notes = (Notes*)exchange;
    a.ex = (u64*)exchange + kLoopNoteWords;
    a.ey = a.ex + f.rows_pad;
    a.msr = a.ey + g.rows_pad;
    a.sx = a.msr + 6 * (size_t)g.nrb;
    a.sy = a.sx + (size_t)f.nrb * slots_x * kRowsOfBlock * 2;
    a.rows = (float2*)(a.sy + (size_t)g.nrb * slots_y * kRowsOfBlock * 2);
    a.slots_x = slots_x;
    a.slots_y = slots_y;
    a.ranks = ranks;
    a.id = a.iters = a.polls = a.first_polls = 0;
    return a;
}

}  // namespace

size_t loop_repairs_at() { return offsetof(Notes, repairs); }

hipError_t launch_recover(const PartialArgs& f, const PartialArgs& g, void* exchange, int ranks, int slots_x, int slots_y,
                          hipStream_t st) {
    hipLaunchKernelGGL(recover_kernel, dim3(1), dim3(256), 0, st, loop_args(f, g, exchange, ranks, slots_x, slots_y));
    return hipGetLastError();
}

hipError_t launch_loop(const PartialArgs& f, const PartialArgs& g, void* exchange, int iters, int nc, int ranks, int slots_x,
                       int slots_y, int polls, bool repair, hipStream_t st) {
    static std::atomic<unsigned> launches{0};
    LoopArgs a = loop_args(f, g, exchange, ranks, slots_x, slots_y);
    a.id = (int)(launches.fetch_add(1, std::memory_order_relaxed) << 1 | 1u);
    a.iters = iters;
    a.polls = polls > 0 ? polls : kMaxPolls;
    a.first_polls = repair || polls > 0 ? a.polls : kFirstPolls;
    const int wgs = (f.nrb > g.nrb ? f.nrb : g.nrb) * ranks;
    switch (nc) {
        case 1: return launch_nc<1>(a, wgs, repair, st);
        case 2: return launch_nc<2>(a, wgs, repair, st);
        case 3: return launch_nc<3>(a, wgs, repair, st);
        case 4: return launch_nc<4>(a, wgs, repair, st);
        case 5: return launch_nc<5>(a, wgs, repair, st);
        case 6: return launch_nc<6>(a, wgs, repair, st);
        case 7: return launch_nc<7>(a, wgs, repair, st);
        case 8: return launch_nc<8>(a, wgs, repair, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace sk
