// krylov.hip -- FP64 vector kernels of the device Newton-Krylov solve (ImplicitEuler).
//
// The GMRES driver keeps its basis as nv vectors of length n at a fixed leading dimension
// ld.  Classical Gram-Schmidt needs the nv dot products <V_i, w> in one sweep: k_multidot
// reads w once per group of kGroup basis vectors and each basis vector once, with the
// group's accumulators in registers (the group index is a compile-time constant in the
// unrolled loop), and writes one partial per block and vector, which the kernel that needs the
// sums folds (k_gs_sweep, k_gs_normalize, k_reduce_rows).  Every sum has a fixed order.
#include "krylov.h"

#include <algorithm>

namespace gpf {

namespace {

constexpr int kGroup = 8;
constexpr int kWaves = kKrylovThreads / 64;

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

// max that propagates NaN (fmax drops it), so a non-finite residual is never read as small
__device__ __forceinline__ double nanmax(double a, double b) {
    if (a != a) return a;
    if (b != b) return b;
    return a > b ? a : b;
}

__device__ __forceinline__ double wave_max(double v) {
    for (int o = 32; o > 0; o >>= 1) v = nanmax(v, __shfl_xor(v, o));
    return v;
}

__global__ void __launch_bounds__(kKrylovThreads) k_multidot(const double* __restrict__ V, long ld, int nv,
                                                              const double* __restrict__ w, long n,
                                                              double* __restrict__ partial) {
    const int i0 = blockIdx.y * kGroup;
    const int cnt = min(kGroup, nv - i0);
    double acc[kGroup];
#pragma unroll
    for (int q = 0; q < kGroup; ++q) acc[q] = 0.0;
    const long stride = (long)gridDim.x * blockDim.x;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += stride) {
        const double we = w[e];
#pragma unroll
        for (int q = 0; q < kGroup; ++q)
            if (q < cnt) acc[q] += V[(long)(i0 + q) * ld + e] * we;
    }
    __shared__ double red[kGroup][kWaves];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < kGroup; ++q) {
        const double v = wave_sum(acc[q]);
        if (lane == 0) red[q][wv] = v;
    }
    __syncthreads();
    if ((int)threadIdx.x < cnt) {
        double t = 0.0;
        for (int k = 0; k < kWaves; ++k) t += red[threadIdx.x][k];
        partial[(long)(i0 + threadIdx.x) * gridDim.x + blockIdx.x] = t;
    }
}

__global__ void __launch_bounds__(kKrylovThreads) k_reduce_rows(const double* __restrict__ partial, long nblocks,
                                                                 double* __restrict__ out) {
    const double* row = partial + (long)blockIdx.x * nblocks;
    double v = 0.0;
    for (long b = threadIdx.x; b < nblocks; b += blockDim.x) v += row[b];
    __shared__ double red[kWaves];
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < kWaves; ++k) t += red[k];
        out[blockIdx.x] = t;
    }
}

// out may alias x or y
__global__ void __launch_bounds__(kKrylovThreads) k_axpby(double a, const double* x, double b, const double* y,
                                                           double* out, long n) {
    const long stride = (long)gridDim.x * blockDim.x;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += stride)
        out[e] = (x ? a * x[e] : 0.0) + b * y[e];
}

__global__ void __launch_bounds__(kKrylovThreads) k_normalize(const double* __restrict__ x,
                                                               const double* __restrict__ nrm2,
                                                               double* __restrict__ out, long n) {
    const double s2 = nrm2[0];
    const double inv = (s2 > 0.0) ? 1.0 / sqrt(s2) : 0.0;
    const long stride = (long)gridDim.x * blockDim.x;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += stride) out[e] = x[e] * inv;
}

__global__ void __launch_bounds__(kKrylovThreads) k_absmax(const double* __restrict__ x, long n,
                                                            double* __restrict__ partial) {
    double v = 0.0;
    const long stride = (long)gridDim.x * blockDim.x;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += stride) v = nanmax(v, fabs(x[e]));
    __shared__ double red[kWaves];
    v = wave_max(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < kWaves; ++k) t = nanmax(t, red[k]);
        partial[blockIdx.x] = t;
    }
}

__global__ void __launch_bounds__(kKrylovThreads) k_max_rows(const double* __restrict__ partial, long nblocks,
                                                              double* __restrict__ out) {
    double v = 0.0;
    for (long b = threadIdx.x; b < nblocks; b += blockDim.x) v = nanmax(v, partial[b]);
    __shared__ double red[kWaves];
    v = wave_max(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0.0;
        for (int k = 0; k < kWaves; ++k) t = nanmax(t, red[k]);
        out[0] = t;
    }
}

// ---------------------------------------------------------------------------
// one Arnoldi step's Gram-Schmidt sweeps (classical, twice) and normalisation
// ---------------------------------------------------------------------------
// Each sweep ends in sums over the whole vector that the next one needs.  Separate kernels for
// the partial sums, their reduction and the combination made nine launches of 2-4 us a step at
// 128^2; here the reduction is the head of the kernel that uses it (every block folds the
// partials again: at most 256 per vector), and a sweep's combination and the next sums share one
// pass, so a step has four.

// h[i] = sum_b partial[i * nb + b] for i < nv, into LDS: one wavefront per vector at a time
__device__ __forceinline__ void fold_partials(const double* __restrict__ partial, int nv, int nb, double* h) {
    const int lane = threadIdx.x & 63;
    for (int i = threadIdx.x >> 6; i < nv; i += kWaves) {
        double v = 0.0;
        for (int b = lane; b < nb; b += 64) v += partial[(long)i * nb + b];
        v = wave_sum(v);
        if (lane == 0) h[i] = v;
    }
    __syncthreads();
}

// w -= sum_i h[i] V_i with h folded from `partial`; then the partial sums of <V_i, w> (DOTS) or of
// <w, w> into `next`; block 0 leaves h in out
template <bool DOTS>
__global__ void __launch_bounds__(kKrylovThreads) k_gs_sweep(const double* __restrict__ V, long ld, int nv,
                                                              const double* __restrict__ partial, double* w, long n,
                                                              double* __restrict__ next, double* __restrict__ out) {
    __shared__ double h[kMaxKrylov + 1];
    __shared__ double red[kGroup][kWaves];
    const int nb = gridDim.x;
    fold_partials(partial, nv, nb, h);
    if (blockIdx.x == 0 && (int)threadIdx.x < nv) out[threadIdx.x] = h[threadIdx.x];
    const long stride = (long)gridDim.x * blockDim.x;
    const long first = blockIdx.x * (long)blockDim.x + threadIdx.x;
    double nrm = 0.0;
    for (long e = first; e < n; e += stride) {
        double acc = 0.0;
        for (int i = 0; i < nv; ++i) acc += h[i] * V[(long)i * ld + e];
        const double x = w[e] - acc;
        w[e] = x;
        if (!DOTS) nrm += x * x;
    }
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if constexpr (DOTS) {
        for (int i0 = 0; i0 < nv; i0 += kGroup) {
            const int cnt = min(kGroup, nv - i0);
            double acc[kGroup];
#pragma unroll
            for (int q = 0; q < kGroup; ++q) acc[q] = 0.0;
            for (long e = first; e < n; e += stride) {
                const double x = w[e];  // written by this thread above
#pragma unroll
                for (int q = 0; q < kGroup; ++q)
                    if (q < cnt) acc[q] += V[(long)(i0 + q) * ld + e] * x;
            }
#pragma unroll
            for (int q = 0; q < kGroup; ++q) {
                const double v = wave_sum(acc[q]);
                if (lane == 0) red[q][wv] = v;
            }
            __syncthreads();
            if ((int)threadIdx.x < cnt) {
                double t = 0.0;
                for (int k = 0; k < kWaves; ++k) t += red[threadIdx.x][k];
                next[(long)(i0 + threadIdx.x) * nb + blockIdx.x] = t;
            }
            __syncthreads();
        }
    } else {
        const double v = wave_sum(nrm);
        if (lane == 0) red[0][wv] = v;
        __syncthreads();
        if (threadIdx.x == 0) {
            double t = 0.0;
            for (int k = 0; k < kWaves; ++k) t += red[0][k];
            next[blockIdx.x] = t;
        }
    }
}

// out = sign x / |x| (0 where the norm is 0) with |x|^2 folded from `partial` (nb sums); block 0
// leaves |x|^2 in nrm2
__global__ void __launch_bounds__(kKrylovThreads) k_gs_normalize(const double* __restrict__ partial, int nb,
                                                                  const double* __restrict__ x, double sign,
                                                                  double* __restrict__ out, long n,
                                                                  double* __restrict__ nrm2) {
    __shared__ double h[1];
    fold_partials(partial, 1, nb, h);
    const double s2 = h[0];
    if (blockIdx.x == 0 && threadIdx.x == 0) nrm2[0] = s2;
    const double inv = (s2 > 0.0) ? sign / sqrt(s2) : 0.0;
    const long stride = (long)gridDim.x * blockDim.x;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += stride) out[e] = x[e] * inv;
}

// out = base + sum_i c[i] V_i (a null base reads as 0); out may alias base
__global__ void __launch_bounds__(kKrylovThreads) k_expand(const double* __restrict__ V, long ld, int nv, KrylovCoefs c,
                                                            const double* base, double* out, long n) {
    __shared__ double h[kMaxKrylov + 1];
    if ((int)threadIdx.x < nv) h[threadIdx.x] = c.v[threadIdx.x];
    __syncthreads();
    const long stride = (long)gridDim.x * blockDim.x;
    for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += stride) {
        double acc = 0.0;
        for (int i = 0; i < nv; ++i) acc += h[i] * V[(long)i * ld + e];
        out[e] = (base ? base[e] : 0.0) + acc;
    }
}

inline unsigned grid_for(long n) {
    long g = (n + kKrylovThreads - 1) / kKrylovThreads;
    if (g > 4096) g = 4096;
    if (g < 1) g = 1;
    return (unsigned)g;
}

}  // namespace

long krylov_blocks(long n) {
    long g = (n + kKrylovThreads - 1) / kKrylovThreads;
    if (g > 1024) g = 1024;
    if (g < 1) g = 1;
    return g;
}

hipError_t launch_multidot(const double* V, long ld, int nv, const double* w, long n, double* partial,
                           hipStream_t s) {
    if (nv <= 0) return hipSuccess;
    const unsigned groups = (unsigned)((nv + kGroup - 1) / kGroup);
    hipLaunchKernelGGL(k_multidot, dim3((unsigned)krylov_blocks(n), groups), dim3(kKrylovThreads), 0, s, V, ld, nv,
                       w, n, partial);
    return hipGetLastError();
}

hipError_t launch_reduce_rows(const double* partial, int nv, long nblocks, double* out, hipStream_t s) {
    if (nv <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_reduce_rows, dim3((unsigned)nv), dim3(kKrylovThreads), 0, s, partial, nblocks, out);
    return hipGetLastError();
}

hipError_t launch_axpby(double a, const double* x, double b, const double* y, double* out, long n, hipStream_t s) {
    hipLaunchKernelGGL(k_axpby, dim3(grid_for(n)), dim3(kKrylovThreads), 0, s, a, x, b, y, out, n);
    return hipGetLastError();
}

hipError_t launch_normalize(const double* x, const double* nrm2, double* out, long n, hipStream_t s) {
    hipLaunchKernelGGL(k_normalize, dim3(grid_for(n)), dim3(kKrylovThreads), 0, s, x, nrm2, out, n);
    return hipGetLastError();
}

hipError_t launch_absmax(const double* x, long n, double* partial, double* out, hipStream_t s) {
    const long nb = krylov_blocks(n);
    hipLaunchKernelGGL(k_absmax, dim3((unsigned)nb), dim3(kKrylovThreads), 0, s, x, n, partial);
    hipLaunchKernelGGL(k_max_rows, dim3(1), dim3(kKrylovThreads), 0, s, partial, nb, out);
    return hipGetLastError();
}

// Every block of the next kernel folds one partial per block and vector: at most 256 blocks, but
// for long vectors, whose sweeps are bound by memory (one wavefront per SIMD does not load fast
// enough), more, with 8 elements per thread, up to 1024 (us a step with at most 256, 512, 1024 and
// 2048: 128^3 of three fields 9009, 8600, 8431 and 8511, 2048^2 5146, 4640, 4449 and 4602)
long gs_blocks(long n) {
    const long most = std::clamp(n / (8L * kKrylovThreads), 256L, 1024L);
    return std::clamp((n + kKrylovThreads - 1) / kKrylovThreads, 1L, most);
}

hipError_t launch_gs_dots(const double* V, long ld, int nv, const double* w, long n, double* partial, hipStream_t s) {
    if (nv < 1 || nv > kMaxKrylov + 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_multidot, dim3((unsigned)gs_blocks(n), (unsigned)((nv + kGroup - 1) / kGroup)),
                       dim3(kKrylovThreads), 0, s, V, ld, nv, w, n, partial);
    return hipGetLastError();
}

hipError_t launch_gs_sweep(const double* V, long ld, int nv, const double* partial, double* w, long n, bool dots,
                           double* next, double* out, hipStream_t s) {
    if (nv < 1 || nv > kMaxKrylov + 1 || next == partial) return hipErrorInvalidValue;
    const dim3 grid((unsigned)gs_blocks(n));
    if (dots) hipLaunchKernelGGL(k_gs_sweep<true>, grid, dim3(kKrylovThreads), 0, s, V, ld, nv, partial, w, n, next, out);
    else hipLaunchKernelGGL(k_gs_sweep<false>, grid, dim3(kKrylovThreads), 0, s, V, ld, nv, partial, w, n, next, out);
    return hipGetLastError();
}

hipError_t launch_gs_normalize(const double* partial, const double* x, double sign, double* out, long n, double* nrm2,
                               hipStream_t s) {
    hipLaunchKernelGGL(k_gs_normalize, dim3(grid_for(n)), dim3(kKrylovThreads), 0, s, partial, (int)gs_blocks(n), x,
                       sign, out, n, nrm2);
    return hipGetLastError();
}

hipError_t launch_expand(const double* V, long ld, int nv, const KrylovCoefs& c, const double* base, double* out,
                         long n, hipStream_t s) {
    if (nv < 1 || nv > kMaxKrylov + 1) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_expand, dim3(grid_for(n)), dim3(kKrylovThreads), 0, s, V, ld, nv, c, base, out, n);
    return hipGetLastError();
}

}  // namespace gpf
