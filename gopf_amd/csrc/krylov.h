// krylov.h -- FP64 vector kernels of the device Newton-Krylov solve behind the
// ImplicitEuler stepper: block dot products against a set of basis vectors, linear
// combinations, normalisation and max-norm reductions.  All sums
// are formed in a fixed order (per-thread, then per-block tree, then one block over the
// block partials), so repeated solves give identical results.
#pragma once

#include <hip/hip_runtime.h>

namespace gpf {

// longest Krylov basis of one GMRES cycle (restart length)
constexpr int kMaxKrylov = 64;
constexpr int kKrylovThreads = 256;

// number of blocks (and partial sums per vector) the reductions below use for length n
long krylov_blocks(long n);

// partial[i * nblocks + b] = sum over block b's elements e of V[i * ld + e] * w[e],
// for i < nv; nblocks = krylov_blocks(n)
hipError_t launch_multidot(const double* V, long ld, int nv, const double* w, long n, double* partial,
                           hipStream_t s);
// out[i] = sum_b partial[i * nblocks + b], i < nv
hipError_t launch_reduce_rows(const double* partial, int nv, long nblocks, double* out, hipStream_t s);
// out = a x + b y; a null x reads as 0
hipError_t launch_axpby(double a, const double* x, double b, const double* y, double* out, long n,
                        hipStream_t s);
// out = x / sqrt(*nrm2), and 0 where *nrm2 is not positive (nrm2 in device memory)
hipError_t launch_normalize(const double* x, const double* nrm2, double* out, long n, hipStream_t s);
// out[0] = max_e |x[e]| (partial: krylov_blocks(n) doubles of scratch)
hipError_t launch_absmax(const double* x, long n, double* partial, double* out, hipStream_t s);

// The Arnoldi step of GMRES: gs_blocks(n) partial sums per vector, folded by the next kernel.
// launch_gs_dots: partial sums of <V_i, w>.  launch_gs_sweep: w -= sum_i h_i V_i with h folded from
// `partial` (left in out), then the partial sums of <V_i, w> (dots) or of <w, w> in next.
// launch_gs_normalize: out = sign x / |x| with |x|^2 folded from `partial` (left in nrm2).  out and
// nrm2 may be mapped host memory.
long gs_blocks(long n);
hipError_t launch_gs_dots(const double* V, long ld, int nv, const double* w, long n, double* partial, hipStream_t s);
hipError_t launch_gs_sweep(const double* V, long ld, int nv, const double* partial, double* w, long n, bool dots,
                           double* next, double* out, hipStream_t s);
hipError_t launch_gs_normalize(const double* partial, const double* x, double sign, double* out, long n, double* nrm2,
                               hipStream_t s);
// out = base + sum_{i < nv} c_i V_i (a null base reads as 0)
struct KrylovCoefs {
    double v[kMaxKrylov + 1];
};
hipError_t launch_expand(const double* V, long ld, int nv, const KrylovCoefs& c, const double* base, double* out,
                         long n, hipStream_t s);

}  // namespace gpf
