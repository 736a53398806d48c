// spectral_rowpoly.hip -- the forward row pass of ImplicitEuler's residual and of its directional
// derivative (FP64, every compiled length and the direct DFT).
//
// k_rows_poly transforms the rows of the fields and of their dense polynomials (the derived
// fields), or of the finite-difference derivative of both along a direction v:
//   field i:    v_i
//   derived d:  sum_k w_k g_d(x + o_k v),  o_k the stencil's offsets, w_k its weights over the step
// The transforms are linear, so the stencil's sum over residuals needs the sum over the
// pointwise sources only: one transform of each instead of one per stencil point (six by
// default), which with their launches were 9/10 of an ImplicitEuler step at 128^2 (10 steps:
// 27.4 -> 6.4 ms, with the middle pass and the shorter Gram-Schmidt).
#include "spectral_kernels.h"
#include "spectral_rowpoly.h"

namespace gpf {

namespace {

// real row of output o (fields, then derived fields) at element off
__device__ __forceinline__ double row_value(const RowPolyArgs& a, int o, const double (&c)[4][4], double x0, double x1,
                                            double v0, double v1) {
    if (o < a.nf) return a.npt ? (o == 0 ? v0 : v1) : (o == 0 ? x0 : x1);
    auto poly = [&](double y0, double y1) {
        if (a.nf == 1) return ((c[3][0] * y0 + c[2][0]) * y0 + c[1][0]) * y0 + c[0][0];
        return dense_poly<double>(c, y0, y1);
    };
    if (a.npt == 0) return poly(x0, x1);
    double s = 0.0;
    for (int k = 0; k < a.npt; ++k) s += a.w[k] * poly(x0 + a.off[k] * v0, x1 + a.off[k] * v1);
    return s;
}

__device__ __forceinline__ void pick_coefs(const RowPolyArgs& a, int d, double (&c)[4][4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            c[i][j] = (d == 0) ? a.dc[0][i][j] : (d == 1) ? a.dc[1][i][j] : (d == 2) ? a.dc[2][i][j] : a.dc[3][i][j];
}

// two outputs (2 blockIdx.y and the next) as one complex line, one row per line of threads, in
// the low-register schedule: at 128^2 a row is latency, and half the elements per thread shorten it
template <int N>
__global__ void __launch_bounds__(kMaxBlock) k_rows_poly(RowPolyArgs a) {
    extern __shared__ __align__(16) unsigned char smem[];
    cpx<double>* lds = reinterpret_cast<cpx<double>*>(smem);
    constexpr int E = LineShape<N, 1>::E;
    const int n = (N > 0) ? N : a.nx;
    const int TT = (N > 0) ? LineShape<N, 1>::T : n;
    const LineMap lm = line_map(true, a.TW, TT, n);
    const long row = (long)blockIdx.x * a.TW + lm.l;
    const bool valid = row < a.rows;
    const long rv = valid ? row : 0;
    const int oa = 2 * blockIdx.y, ob = oa + 1, nout = a.nf + a.nd;
    const bool two = ob < nout;
    cpx<double> v[E];
    double x0[E], x1[E], v0[E], v1[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const long off = rv * n + lm.t + TT * e;
        x0[e] = a.x[off];
        x1[e] = (a.nf > 1) ? a.x[a.n + off] : 0.0;
        v0[e] = a.npt ? a.v[off] : 0.0;
        v1[e] = (a.npt && a.nf > 1) ? a.v[a.n + off] : 0.0;
    }
    double ca[4][4], cb[4][4];
    pick_coefs(a, oa - a.nf, ca);
    pick_coefs(a, ob - a.nf, cb);
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const double A = row_value(a, oa, ca, x0[e], x1[e], v0[e], v1[e]);
        const double B = two ? row_value(a, ob, cb, x0[e], x1[e], v0[e], v1[e]) : 0.0;
        v[e] = mk<double>(A, B);
    }
    line_fft<double, N, -1, 1>(v, lds + lm.off, 1, n, lm.t, a.tw);
    cpx<double>* ma = (oa == 0) ? a.out[0] : a.out[2];
    cpx<double>* mb = two ? ((oa == 0) ? a.out[1] : a.out[3]) : nullptr;
    split_store<double, E>(v, lds + lm.off, n, lm.t, TT, row, valid, ma, ma + a.nmain, mb, mb ? mb + a.nmain : nullptr);
}

}  // namespace

hipError_t launch_rows_poly(const RowPolyArgs& a, hipStream_t s) {
    if (a.nf < 1 || a.nf > 2 || a.nd < 0 || a.nf + a.nd > kMaxArr || a.npt < 0 || a.npt > 8 || !a.x ||
        (a.npt && !a.v))
        return hipErrorInvalidValue;
    const int thr = a.TW * threads_per_line(a.nx, 1);
    const size_t smem = lds_elems(a.nx, a.TW) * sizeof(cpx<double>);
    const dim3 grid((unsigned)rows_blocks(a.rows, a.TW), (unsigned)((a.nf + a.nd + 1) / 2));
    auto go = [&](auto NC) -> hipError_t {
        return launch_k(k_rows_poly<decltype(NC)::value>, grid, dim3(thr), smem, s, a);
    };
    return ext_length(a.nx) ? dispatch_size<1>(a.nx, go) : dispatch_size<0>(a.nx, go);
}

}  // namespace gpf
