// A solve's clouds from the caller's float64 points, on the GPU: the centre and the typical cost they are normalised by
// (src/trnopt/sinkhorn.py:220-238), then each cloud's normalised points packed for the half-steps with their squared norms
// (sinkhorn.py:131-165 does both on the host). Everything is float64 until the one rounding to float32 per value that
// the host made too.
//
// What bounds it: on the host the 10,000 x 64 clouds of a solve took 4.5 ms (the 20,000 sampled cost pairs 2.3 of them,
// the normalised copies, range checks, norms and casts the rest), as long as its 50 iterations. Here they cross the bus
// once, as they are, and are read three times from L2 or HBM (10 MB): that solve 9.6 -> 4.6 ms end to end, a 700 x 500
// d 16 one (20 iterations) 1.30 -> 0.71, a 7,355 x 8,962 d 30 one 8.4 -> 7.3.

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>

#include "sk_common.h"

namespace {

using sk::fail;
using sk::f16x8;
using sk::hip_fail;

constexpr int kThreads = 256;
// Workgroups of the statistics: bounded by what the last of them then has to add up.
constexpr int kSumBlocks = 128;         // workgroups of the coordinate sums, at most
constexpr int kSampleBlocks = 80;       // and of the sampled pairs

__device__ __forceinline__ void put(double* p, double v) {
    __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), (unsigned long long)__double_as_longlong(v), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ double get(const double* p) {
    return __longlong_as_double((long long)__hip_atomic_load(reinterpret_cast<const unsigned long long*>(p), __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT));
}

// Sums v over the workgroup in a fixed order; the result in thread 0.
__device__ inline double block_sum(double v, double* lds) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
    __syncthreads();
    double s = 0.0;
    if (threadIdx.x == 0)
        for (int w = 0; w < kThreads / 64; ++w) s += lds[w];
    return s;
}

__global__ void stats_init_kernel(int* counter) { *counter = 0; }

// stat[0 .. d): the mean of all points of both clouds; with `samples`, stat[d]: the mean squared distance of the pairs
// (x[pi], y[pj]), 1 if that is 0 (else stat[d] = 1). The first `sums` workgroups add up coordinates (each thread one
// coordinate of every few rows), the others sampled distances (one pair per thread at a time); the last workgroup to
// arrive adds the workgroups' sums in their order. Handed over as in sk_median.hip (device-scope atomics, no fences).
__global__ __launch_bounds__(kThreads) void stats_kernel(const double* __restrict__ x, int n, const double* __restrict__ y, int m,
                                                         int d, const int* __restrict__ pi, const int* __restrict__ pj,
                                                         int samples, int sums, double* __restrict__ part, int* counter,
                                                         double* __restrict__ stat) {
    __shared__ double lds[kThreads];
    __shared__ int last;
    const int tid = threadIdx.x, blocks = (int)gridDim.x;
    if ((int)blockIdx.x < sums) {
        const int rows_at_once = kThreads / d;             // d <= 128: two rows or more
        const int r = tid / d, k = tid - r * d;
        const long long total = (long long)n + m, per = (total + sums - 1) / sums;
        const long long r0 = blockIdx.x * per, r1 = r0 + per < total ? r0 + per : total;
        double s = 0.0;
        if (r < rows_at_once)
            for (long long i0 = r0 + r; i0 < r1; i0 += 8 * rows_at_once) {
                double v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const long long i = i0 + e * rows_at_once;
                    v[e] = i < r1 ? (i < n ? x[i * d + k] : y[(i - n) * d + k]) : 0.0;
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) s += v[e];
            }
        lds[tid] = s;
        __syncthreads();
        if (tid < d) {
            double t = 0.0;
            for (int q = 0; q < rows_at_once; ++q) t += lds[q * d + tid];
            put(part + (size_t)blockIdx.x * d + tid, t);
        }
    } else {
        double s = 0.0;
        for (int e = ((int)blockIdx.x - sums) * kThreads + tid; e < samples; e += (blocks - sums) * kThreads) {
            const double *a = x + (size_t)pi[e] * d, *b = y + (size_t)pj[e] * d;
            double t = 0.0;
#pragma unroll 8
            for (int k = 0; k < d; ++k) {
                const double q = a[k] - b[k];
                t = fma(q, q, t);
            }
            s += t;
        }
        s = block_sum(s, lds);
        if (tid == 0) put(part + (size_t)sums * d + (blockIdx.x - sums), s);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0)
        last = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == blocks - 1 ? 1 : 0;
    __syncthreads();
    if (last == 0) return;
    if (tid < d) {
        double t = 0.0;
        for (int b0 = 0; b0 < sums; b0 += 16) {
            double v[16];
#pragma unroll
            for (int b = 0; b < 16; ++b) v[b] = b0 + b < sums ? get(part + (size_t)(b0 + b) * d + tid) : 0.0;
#pragma unroll
            for (int b = 0; b < 16; ++b) t += v[b];
        }
        stat[tid] = t / (double)((long long)n + m);
    }
    const int sb = blocks - sums;
    double t = 0.0;
    for (int b = tid; b < sb; b += kThreads) t += get(part + (size_t)sums * d + b);
    __syncthreads();
    t = block_sum(t, lds);
    if (tid == 0) {
        const double mean = samples > 0 ? t / (double)samples : 1.0;
        stat[d] = mean > 0.0 ? mean : 1.0;
    }
}

__global__ __launch_bounds__(kThreads) void centre_kernel(const double* __restrict__ p, long long total, int d,
                                                          const double* __restrict__ centre, double* __restrict__ out) {
    for (long long e = (long long)blockIdx.x * kThreads + threadIdx.x; e < total; e += (long long)gridDim.x * kThreads)
        out[e] = p[e] - centre[total < (1LL << 31) ? (int)e % d : (int)(e % d)];
}

// The initial header of a packed cloud (sk_common.h) and its range slot.
__global__ void header_kernel(unsigned* __restrict__ header, unsigned long long* __restrict__ range) {
    if (threadIdx.x < 16) header[threadIdx.x] = threadIdx.x == 1 || threadIdx.x == 4 ? __float_as_uint(1.0f) : 0u;
    if (threadIdx.x == 0) *range = 0ull;
}

// |p|^2 of the normalised points p = (x - centre) / root (float64, cast; 0 on padding points), the largest |coordinate| as
// the packing sees it (float bits, header word 0) and in float64 (range; infinity for a NaN). One wave per point at a
// time, one atomic per workgroup.
__global__ __launch_bounds__(kThreads) void norm_kernel(const double* __restrict__ x, int n, int npad, int d,
                                                        const double* __restrict__ stat, float* __restrict__ sq,
                                                        unsigned* __restrict__ header, unsigned long long* __restrict__ range) {
    __shared__ double lds[kThreads / 64];
    const int lane = threadIdx.x & 63, waves = (int)gridDim.x * (kThreads / 64);
    const double root = sqrt(stat[d]);
    double mx = 0.0;
    for (int i = (int)blockIdx.x * (kThreads / 64) + (threadIdx.x >> 6); i < npad; i += waves) {
        double s = 0.0;
        if (i < n) {
            for (int k = lane; k < d; k += 64) {
                const double p = (x[(size_t)i * d + k] - stat[k]) / root;
                s = fma(p, p, s);
                mx = fabs(p) <= 1.0e308 ? fmax(mx, fabs(p)) : __builtin_inf();
            }
        }
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
        if (lane == 0) sq[i] = (float)s;
    }
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
    if (lane == 0) lds[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int w = 1; w < kThreads / 64; ++w) mx = fmax(mx, lds[w]);
    atomicMax(range, (unsigned long long)__double_as_longlong(mx));
    atomicMax(&header[0], __float_as_uint((float)mx));
}

// The packing of sk_pack_cloud_f32 (sk_kernels.hip) from the same points: one thread per tile, K chunk and lane.
__global__ __launch_bounds__(kThreads) void pack_kernel(const double* __restrict__ x, int n, int d,
                                                        const double* __restrict__ stat, char* __restrict__ dst, int npad,
                                                        int nc) {
    const long long idx = (long long)blockIdx.x * kThreads + threadIdx.x;
    const float s = sk::pack_scale(__uint_as_float(reinterpret_cast<const unsigned*>(dst)[0]));
    if (idx == 0) reinterpret_cast<float*>(dst)[1] = s;
    if (idx >= (long long)(npad / SK_TILE) * nc * 64) return;
    const double root = sqrt(stat[d]);
    const int lane = (int)(idx % 64), cc = (int)((idx / 64) % nc);
    const long long T = idx / (64 * nc), row = T * SK_TILE + (lane & 31);
    f16x8 p0, p1;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int k = 16 * cc + 8 * (lane >> 5) + e;
        const float v = row < n && k < d ? (float)((x[row * d + k] - stat[k]) / root) * s : 0.0f;   // s: a power of two
        const _Float16 a = (_Float16)v;
        p0[e] = a;
        p1[e] = (_Float16)(v - (float)a);
    }
    f16x8* o = reinterpret_cast<f16x8*>(dst + sk::kHeaderBytes) + (T * nc + cc) * 128 + lane;
    o[0] = p0;
    o[64] = p1;
}

int sum_blocks(long long rows) { return (int)std::max<long long>(1, std::min<long long>(kSumBlocks, rows / 64)); }
int sample_blocks(int samples) { return std::min(kSampleBlocks, (samples + kThreads - 1) / kThreads); }

int check_d(int d) {
    if (d < 1 || d > SK_KP_MAX) return fail(SK_E_SHAPE, "dimension %d must be in [1, %d]", d, SK_KP_MAX);
    return SK_OK;
}

}  // namespace

extern "C" {

size_t sk_cloud_stats_workspace_bytes(int d) {
    return d < 1 || d > SK_KP_MAX ? 0 : 256 + ((size_t)kSumBlocks * d + kSampleBlocks) * sizeof(double);
}

int sk_cloud_stats_f64(const double* x, int n, const double* y, int m, int d, const int* pairs_x, const int* pairs_y,
                       int samples, double* stat, void* ws, size_t ws_bytes, void* stream) {
    if (x == nullptr || y == nullptr || stat == nullptr || ws == nullptr || (samples > 0 && (pairs_x == nullptr || pairs_y == nullptr)))
        return fail(SK_E_ARG, "sk_cloud_stats_f64: null pointer");
    if (n < 1 || m < 1 || samples < 0) return fail(SK_E_SHAPE, "sk_cloud_stats_f64: n %d, m %d, samples %d", n, m, samples);
    if (int r = check_d(d)) return r;
    if (ws_bytes < sk_cloud_stats_workspace_bytes(d)) return fail(SK_E_WORKSPACE, "sk_cloud_stats_f64: workspace too small");
    if (((uintptr_t)ws & 255) != 0) return fail(SK_E_ARG, "sk_cloud_stats_f64: workspace must be 256-byte aligned");
    hipStream_t s = (hipStream_t)stream;
    int* counter = (int*)ws;
    double* part = (double*)((char*)ws + 256);
    const int sums = sum_blocks((long long)n + m), sb = sample_blocks(samples);
    hipLaunchKernelGGL(stats_init_kernel, dim3(1), dim3(1), 0, s, counter);
    hipLaunchKernelGGL(stats_kernel, dim3(sums + sb), dim3(kThreads), 0, s, x, n, y, m, d, pairs_x, pairs_y, samples, sums, part,
                       counter, stat);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SK_OK : hip_fail(e, "sk_cloud_stats_f64");
}

int sk_centre_f64(const double* pts, int n, int d, const double* centre, double* out, void* stream) {
    if (pts == nullptr || centre == nullptr || out == nullptr) return fail(SK_E_ARG, "sk_centre_f64: null pointer");
    if (n < 1 || d < 1) return fail(SK_E_SHAPE, "sk_centre_f64: n %d, d %d", n, d);
    const long long total = (long long)n * d;
    hipLaunchKernelGGL(centre_kernel, dim3((unsigned)std::min<long long>((total + kThreads - 1) / kThreads, 1024)), dim3(kThreads),
                       0, (hipStream_t)stream, pts, total, d, centre, out);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SK_OK : hip_fail(e, "sk_centre_f64");
}

int sk_prepare_cloud_f64(const double* pts, int n, int d, const double* stat, float* sq, void* pk, double* range,
                         void* stream) {
    if (pts == nullptr || stat == nullptr || sq == nullptr || pk == nullptr || range == nullptr)
        return fail(SK_E_ARG, "sk_prepare_cloud_f64: null pointer");
    if (n < 1) return fail(SK_E_SHAPE, "sk_prepare_cloud_f64: n %d", n);
    if (int r = check_d(d)) return r;
    if (((uintptr_t)pk & 15) != 0) return fail(SK_E_ARG, "sk_prepare_cloud_f64: pk must be 16-byte aligned");
    const int npad = sk_pad_points(n), nc = sk_pad_dim(d) / 16;
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(header_kernel, dim3(1), dim3(64), 0, s, (unsigned*)pk, (unsigned long long*)range);
    hipLaunchKernelGGL(norm_kernel, dim3(std::min((npad + 3) / 4, 512)), dim3(kThreads), 0, s, pts, n, npad, d, stat, sq,
                       (unsigned*)pk, (unsigned long long*)range);
    const long long units = (long long)(npad / SK_TILE) * nc * 64;
    hipLaunchKernelGGL(pack_kernel, dim3((unsigned)((units + kThreads - 1) / kThreads)), dim3(kThreads), 0, s, pts, n, d, stat,
                       (char*)pk, npad, nc);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? SK_OK : hip_fail(e, "sk_prepare_cloud_f64");
}

}  // extern "C"
