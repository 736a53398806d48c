// spectral_adjoint_kernels.h -- k_adj_mid (spectral_adjoint.h) and its launch template, instantiated
// per precision in spectral_adjoint{,64}.hip.
#pragma once

#include "spectral_adjoint.h"
#include "blockred.h"
#include "spectral_kernels.h"

namespace gpf {

namespace {

// The forward pencils, the multipliers with the scalars' sums and the inverse pencils of P and Q
// were three launches at 512^2 FP64 (5.4, 7.3 and 8.8 us, all latency); this one takes 12.1.  Two
// lines (P and Q) stay in registers, so the low-register schedule; formed in the pass, the
// multipliers' polynomials and division spilled the lines of 12 and 20 elements per thread.
template <typename T, int N, bool GRAD>
__global__ void __launch_bounds__(kMaxBlock) k_adj_mid(AdjMidArgs<T> m) {
    extern __shared__ __align__(16) unsigned char smem[];
    cpx<T>* lds = reinterpret_cast<cpx<T>*>(smem);
    constexpr int V = 1;
    constexpr int E = LineShape<N, V>::E;
    const AdjArgs<T>& a = m.a;
    const int n = (N > 0) ? N : m.p.n;
    const int TT = (N > 0) ? LineShape<N, V>::T : n;
    const TileInfo ti = decode_tile(m.p, blockIdx.x, gridDim.x);
    const LineMap lm = line_map(ti.es == 1, m.p.TW, TT, n);
    const bool valid = lm.l < ti.nvalid;
    // a line past the end of the tile works on the tile's first line, adds and stores nothing
    const long gb = (ti.s ? a.nmain : 0) + ti.base + (long)(valid ? lm.l : 0) * ti.sb + (long)lm.t * ti.es;
    const long se = (long)TT * ti.es;
    cpx<T> pv[E], qv[E];
#pragma unroll
    for (int e = 0; e < E; ++e) pv[e] = a.lam[gb + e * se];
    line_fft<T, N, -1, V>(pv, lds + lm.off, lm.es, n, lm.t, m.p.tw);
    double acc[kMaxAdjScalars];
#pragma unroll
    for (int s = 0; s < kMaxAdjScalars; ++s) acc[s] = 0.0;
    constexpr int C = (E % 4 == 0) ? 4 : (E % 5 == 0) ? 5 : 1;  // elements whose operands are in flight together
#pragma unroll
    for (int e0 = 0; e0 < E; e0 += C) {
        double2 mt[C];
        cpx<T> c1[C], c0[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            if (e0 + c >= E) break;
            const long i = gb + (e0 + c) * se;
            mt[c] = m.t.m[i];
            if constexpr (GRAD) {
                c1[c] = a.C1 ? a.C1[i] : mk<T>(T(0), T(0));
                c0[c] = a.C0 ? a.C0[i] : mk<T>(T(0), T(0));
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int e = e0 + c;
            if (e >= E) break;
            const double lx = (double)pv[e].x, ly = (double)pv[e].y;
            pv[e] = mk<T>((T)(mt[c].x * lx), (T)(mt[c].x * ly));
            qv[e] = mk<T>((T)(mt[c].y * lx), (T)(mt[c].y * ly));
            if constexpr (GRAD) {
                const long i = gb + e * se;
                double c1x = a.cscale * (double)c1[c].x, c0x = a.cscale * (double)c0[c].x;
                if (i == 0) {
                    if (a.C1 && a.mean1) c1x += a.cscale * *a.mean1;
                    if (a.C0 && a.mean0) c0x += a.cscale * *a.mean0;
                }
                // Re(conj(l) z) = l.x z.x + l.y z.y
                const double lc1 = lx * c1x + ly * (a.cscale * (double)c1[c].y);
                const double lc0 = lx * c0x + ly * (a.cscale * (double)c0[c].y);
#pragma unroll
                for (int s = 0; s < kMaxAdjScalars; ++s) {
                    if (s >= a.nscal) break;
                    const double2 g = m.t.g[(long)s * a.nk + i];
                    if (valid) acc[s] += g.x * lc1 + g.y * lc0;
                }
            }
        }
        asm volatile("" ::: "memory");
    }
    if constexpr (GRAD) {
        double* red = reinterpret_cast<double*>(lds + lds_elems(n, m.p.TW));
#pragma unroll
        for (int s = 0; s < kMaxAdjScalars; ++s) {
            if (s >= a.nscal) break;  // uniform over the block
            const double tot = block_sum(acc[s], red);
            if (threadIdx.x == 0) a.partial[(long)s * gridDim.x + blockIdx.x] += tot;
        }
    }
    // lines of more than 8 elements per thread: twiddles and LDS addresses formed anew for each
    // transform rather than kept live
    const cpx<T>* tw2 = m.p.tw;
    int t2 = lm.t;
    if constexpr (E > 8) asm volatile("" : "+s"(tw2), "+v"(t2));
    line_fft<T, N, +1, V>(pv, lds + lm.off, lm.es, n, t2, tw2);
    if (valid) {
#pragma unroll
        for (int e = 0; e < E; ++e) a.P[gb + e * se] = pv[e];
    }
    if constexpr (E > 8) asm volatile("" : "+s"(tw2), "+v"(t2));
    line_fft<T, N, +1, V>(qv, lds + lm.off, lm.es, n, t2, tw2);
    if (valid) {
#pragma unroll
        for (int e = 0; e < E; ++e) a.Q[gb + e * se] = qv[e];
    }
}

}  // namespace

template <typename T>
long adj_mid_blocks(const AdjMidArgs<T>& a) {
    return pencil_blocks(a.p.seg, a.p.nseg, a.p.TW, nullptr);
}

template <typename T>
hipError_t launch_adj_mid(const AdjMidArgs<T>& a0, int n, hipStream_t s) {
    AdjMidArgs<T> a = a0;
    if (!a.a.lam || !a.a.P || !a.a.Q || a.a.P == a.a.lam || a.a.Q == a.a.lam || !a.t.m) return hipErrorInvalidValue;
    if (a.a.nscal < 0 || a.a.nscal > kMaxAdjScalars) return hipErrorInvalidValue;
    a.p.n = n;
    a.p.lpt = 1;
    const long blocks = pencil_blocks(a.p.seg, a.p.nseg, a.p.TW, &a.p.tiles0);
    const int thr = a.p.TW * threads_per_line(n, 1);
    const bool grad = a.a.nscal > 0 && (a.a.C1 || a.a.C0);
    if (grad && !a.t.g) return hipErrorInvalidValue;
    const size_t smem = lds_elems(n, a.p.TW) * sizeof(cpx<T>) + (grad ? (size_t)thr * sizeof(double) : 0);
    auto go = [&](auto NC) -> hipError_t {
        constexpr int NN = decltype(NC)::value;
        if (grad) return launch_k(k_adj_mid<T, NN, true>, dim3(blocks), dim3(thr), smem, s, a);
        return launch_k(k_adj_mid<T, NN, false>, dim3(blocks), dim3(thr), smem, s, a);
    };
    return ext_length(n) ? dispatch_size<1>(n, go) : dispatch_size<0>(n, go);
}

}  // namespace gpf
