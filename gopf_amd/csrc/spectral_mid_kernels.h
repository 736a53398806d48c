// spectral_mid_kernels.h -- k_mid, the middle pass of the general path (spectral_mid.h), and its
// launch template.  Included by the spectral_mid*.hip units, one per precision and length set.
#pragma once

#include "kspace.h"
#include "spectral_kernels.h"
#include "spectral_mid.h"

namespace gpf {

namespace {

// Element access by byte offset from a uniform base: one offset register per element serves all
// arrays, where 64-bit element indexes cost two registers per element and array.  An array
// whose lines are shorter than kMidLong is below 4 GiB, so its offsets have 32 bits: 3D domains are
// cubes (the largest length before it, 800^3 in FP64: 4.1e9 bytes), sides of 2D domains at most 2560.
constexpr int kMidLong = 896;
template <int N>
using MidOff = std::conditional_t<(N >= kMidLong), unsigned long, unsigned>;

template <typename V, typename O>
__device__ __forceinline__ V ld(const V* p, O byte) {
    return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(p) + byte);
}
template <typename V, typename O>
__device__ __forceinline__ void st(V* p, O byte, V v) {
    *reinterpret_cast<V*>(reinterpret_cast<char*>(p) + byte) = v;
}

// the factor at the element whose complex value has byte offset o
template <typename T, typename O>
__device__ __forceinline__ double mid_factor(const MidField<T>& f, O o) {
    return f.s64 ? ld(f.s64, sizeof(T) == 8 ? o / 2 : o) : (double)ld(f.s, o / 2);
}

// the operands of one element of a stage besides the line spectra
template <typename T>
struct MidOperands {
    cpx<T> o1, start;  // k or fin; the value the stage starts from (k or init)
    double s;
};

template <typename T>
__device__ __forceinline__ MidTerm<T> mid_term(const MidField<T>& f, int q) {
    return (q == 0) ? f.t[0] : (q == 1) ? f.t[1] : (q == 2) ? f.t[2] : (q == 3) ? f.t[3] : (q == 4) ? f.t[4] : f.t[5];
}

// L(k) = -(2 pi |f|)^2 of element p of a line, from the grid's frequency table (kspace.h)
struct MidL {
    const double* axis;  // the table's part of the line's axis
    int vary;            // that axis: 0 x, 1 y, 2 z
    double fy, fx, fz;   // the fixed components
    __device__ __forceinline__ double f2(int p) const {
        const double v = axis[p];
        const double y = (vary == 1) ? v : fy, x = (vary == 0) ? v : fx, z = (vary == 2) ? v : fz;
        return y * y + x * x + z * z;
    }
    __device__ __forceinline__ double at(int p) const {
        return -(4.0 * 3.14159265358979323846 * 3.14159265358979323846) * f2(p);
    }
};

// the line of tile line l
__device__ __forceinline__ MidL mid_line(const KGrid& g, const TileInfo& ti, int l, int& kx) {
    MidL m;
    const int bl = ti.b0 + l;
    const int k0 = ksel(ti.ksrc0, ti.kfix0, ti.ia, bl, 0);
    const int k1 = ksel(ti.ksrc1, ti.kfix1, ti.ia, bl, 0);
    const int k2 = ksel(ti.ksrc2, ti.kfix2, ti.ia, bl, 0);
    double fr[3];
    ref_freq(g, k0, k1, k2, fr);
    m.vary = (ti.ksrc0 == 2) ? 0 : (ti.ksrc1 == 2) ? 1 : 2;
    m.axis = g.ftab + (m.vary == 1 ? 0 : m.vary == 0 ? g.ny : g.ny + g.nx / 2 + 1);
    m.fy = fr[0];
    m.fx = fr[1];
    m.fz = fr[2];
    kx = k0;
    return m;
}

// elements whose operands are in flight together: a divisor of E, bounded so that FP32 keeps
// four and FP64 two to three waves per SIMD
constexpr int mid_chunk(int E, int most) {
    int c = 1;
    for (int d = 1; d <= most; ++d)
        if (E % d == 0) c = d;
    return c;
}

// Bound by the stage operands' traffic (three to four arrays besides the line's own two).  It takes
// the place of the forward pencils, the stage pass and the first inverse pencils, each of which
// read and wrote its array again: 192^3 FP32, two fields, 100 us (19.5 + 2 x 30.9 + 21) -> 91 us
// and two of four launches fewer; 96^3 FP64, 27 us (9.2 + 18.3) -> 18.1 us a stage.
// One line of one field (blockIdx.y) per thread group, held in registers from its first load to
// its last store.  SINGLE: every field has one line term and at most one spectral one, neither
// with a LAP power (the precipitate's fields); its operands are loaded in chunks, the first
// before the forward transform so that it is in flight meanwhile, each next one before the last
// is used.  Otherwise the lines are transformed one after another and summed in FP64.
// HEAD: kMidScale / kMidResidual.
template <typename T, int N, int V, bool SINGLE, bool HEAD>
__global__ void __launch_bounds__(kMaxBlock) k_mid(MidArgs<T> a) {
    extern __shared__ __align__(16) unsigned char smem[];
    cpx<T>* lds = reinterpret_cast<cpx<T>*>(smem);
    constexpr int E = LineShape<N, V>::E;
    const int n = (N > 0) ? N : a.p.n;
    const int TT = (N > 0) ? LineShape<N, V>::T : n;
    const TileInfo ti = decode_tile(a.p, blockIdx.x, gridDim.x);
    const LineMap lm = line_map(ti.es == 1, a.p.TW, TT, n);
    const bool valid = lm.l < ti.nvalid;
    // a line past the end of the tile works on the tile's first line and stores nothing
    const int l = valid ? lm.l : 0;
    using Off = MidOff<N>;
    const Off o0 = (Off)(((ti.s ? a.nmain : 0) + ti.base + (long)l * ti.sb + (long)lm.t * ti.es) *
                                   (long)sizeof(cpx<T>));
    const Off so = (Off)((long)TT * ti.es * (long)sizeof(cpx<T>));
    auto off = [&](int e) { return o0 + so * (Off)e; };
    const int qf = blockIdx.y;
    const MidField<T>& f = (qf == 0) ? a.f[0] : (qf == 1) ? a.f[1] : (qf == 2) ? a.f[2] : a.f[3];
    const int op = a.op;
    MidL lap{};
    if (a.need_l) {
        int kx;
        lap = mid_line(a.g, ti, l, kx);
    }
    auto weight = [&](const MidTerm<T>& t, int e) {
        double m = t.coef;
        if (t.pw) m *= ipow(lap.at(lm.t + TT * e), t.pw);
        if (t.dmul) m *= t.dmul[0];
        return m;
    };
    const int nterm = f.nterm;
    cpx<T> v[E];
    auto load = [&](const cpx<T>* b) {
#pragma unroll
        for (int e = 0; e < E; ++e) v[e] = ld(b, off(e));
    };
    auto forward = [&]() { line_fft<T, N, -1, V>(v, lds + lm.off, lm.es, n, lm.t, a.p.tw); };
    if constexpr (HEAD) {
        load(f.t[0].b);
        if constexpr (SINGLE) {
            double s[E];
#pragma unroll
            for (int e = 0; e < E; ++e) s[e] = mid_factor(f, off(e));
            forward();
#pragma unroll
            for (int e = 0; e < E; ++e) v[e] = mk<T>((T)(s[e] * (double)v[e].x), (T)(s[e] * (double)v[e].y));
        } else {
            forward();
            double rx[E], ry[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if (valid && f.kn) st(f.kn, off(e), v[e]);
                rx[e] = (double)v[e].x;
                ry[e] = (double)v[e].y;
            }
            for (int q = 1; q < nterm; ++q) {
                const MidTerm<T> t = mid_term(f, q);
                if (t.b) load(t.b);
                if (t.line) forward();
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const double m = mid_factor(f, off(e)) * weight(t, e);
                    rx[e] += t.b ? m * (double)v[e].x : m;
                    if (t.b) ry[e] += m * (double)v[e].y;
                }
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                cpx<T> c = mk<T>(T(0), T(0));
                if (f.cc) c = ld(f.cc, off(e));
                v[e] = mk<T>((T)(rx[e] + (double)c.x), (T)(ry[e] + (double)c.y));
            }
        }
    } else {
        // the stage from R of element e and its operands; returns y
        auto finish = [&](int e, double rx, double ry, const MidOperands<T>& o) {
            // the right-hand side rounded to T, as RK4.Step stores it between its passes
            const double qx = (double)(T)rx, qy = (double)(T)ry;
            const Off i = off(e);
            cpx<T> y;
            if (op == kMidEuler) {
                y = mk<T>((T)(o.s * ((double)o.o1.x + a.bc * rx)), (T)(o.s * ((double)o.o1.y + a.bc * ry)));
            } else if (op == kMidStage3) {
                // fin is rounded to T before the division (rk4.go:57-67)
                const T fx = (T)((double)o.o1.x + a.bp * qx), fy = (T)((double)o.o1.y + a.bp * qy);
                y = mk<T>((T)(o.s * (double)fx), (T)(o.s * (double)fy));
            } else {
                if (valid) {
                    if (op == kMidStage0 && f.init) st(f.init, i, o.o1);
                    st(f.fin, i, mk<T>((T)((double)o.o1.x + a.bp * qx), (T)((double)o.o1.y + a.bp * qy)));
                }
                y = mk<T>((T)(o.s * ((double)o.start.x + a.bc * qx)), (T)(o.s * ((double)o.start.y + a.bc * qy)));
            }
            if (valid && f.kn) st(f.kn, i, y);
            return y;
        };
        const cpx<T>* p1 = (op == kMidStage0 || op == kMidEuler) ? f.k : f.fin;
        if constexpr (SINGLE) {
            constexpr int C = mid_chunk(E, sizeof(T) == 4 ? 4 : 2);
            const bool first = f.t[0].line != 0;  // the line is term 0 or 1
            const MidTerm<T> tl = first ? f.t[0] : f.t[1], ts = first ? f.t[1] : f.t[0];
            const cpx<T>* bs = (nterm > 1) ? ts.b : nullptr;
            const double wl = tl.dmul ? tl.coef * tl.dmul[0] : tl.coef;
            const double ws = ts.dmul ? ts.coef * ts.dmul[0] : ts.coef;
            cpx<T> o1[2][C], o2[2][C], ob[2][C];
            double os[2][C];
            auto fetch = [&](int h, int e0) {
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const Off i = off(e0 + c);
                    o1[h][c] = ld(p1, i);
                    o2[h][c] = (op == kMidStage12) ? ld((const cpx<T>*)f.init, i) : o1[h][c];
                    ob[h][c] = bs ? ld(bs, i) : mk<T>(T(0), T(0));
                    os[h][c] = mid_factor(f, i);
                }
            };
            load(tl.b);
            fetch(0, 0);
            forward();
#pragma unroll
            for (int j = 0; j < E / C; ++j) {
                if (j + 1 < E / C) fetch((j + 1) & 1, (j + 1) * C);
                asm volatile("" ::: "memory");  // at most two chunks of operands are live
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    const int e = j * C + c, h = j & 1;
                    const double rx = wl * (double)v[e].x + ws * (double)ob[h][c].x;
                    const double ry = wl * (double)v[e].y + ws * (double)ob[h][c].y;
                    v[e] = finish(e, rx, ry, MidOperands<T>{o1[h][c], o2[h][c], os[h][c]});
                }
                asm volatile("" ::: "memory");
            }
        } else {
            double rx[E], ry[E];
#pragma unroll
            for (int e = 0; e < E; ++e) rx[e] = ry[e] = 0.0;
            for (int q = 0; q < nterm; ++q) {
                const MidTerm<T> t = mid_term(f, q);
                if (t.b) load(t.b);
                if (t.line) forward();
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const double m = weight(t, e);
                    rx[e] += t.b ? m * (double)v[e].x : m;
                    if (t.b) ry[e] += m * (double)v[e].y;
                }
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const Off i = off(e);
                const cpx<T> c1 = ld(p1, i);
                const cpx<T> c2 = (op == kMidStage12) ? ld((const cpx<T>*)f.init, i) : c1;
                v[e] = finish(e, rx[e], ry[e], MidOperands<T>{c1, c2, mid_factor(f, i)});
                if (e % 4 == 3) asm volatile("" ::: "memory");
            }
        }
    }
    // the inverse transform's twiddles and LDS addresses are formed anew: kept from the forward
    // one, they would stay live through the stage (FP32 192: 175 VGPRs
    // against 126, two waves per SIMD against four)
    const cpx<T>* tw2 = a.p.tw;
    int t2 = lm.t;
    asm volatile("" : "+s"(tw2), "+v"(t2));
    line_fft<T, N, +1, V>(v, lds + lm.off, lm.es, n, t2, tw2);
    if (valid) {
#pragma unroll
        for (int e = 0; e < E; ++e) st(f.out, off(e), v[e]);
    }
}

}  // namespace

template <typename T, int SET>
hipError_t launch_mid_set(const MidArgs<T>& a0, int n, hipStream_t s) {
    if (a0.nf < 1 || a0.nf > kMaxArr) return hipErrorInvalidValue;
    if (n < kMidLong && (unsigned long long)a0.nk * sizeof(cpx<T>) >= (1ull << 32)) return hipErrorInvalidValue;
    MidArgs<T> a = a0;
    a.p.n = n;
    a.p.lpt = 1;
    bool single = true;
    for (int i = 0; i < a.nf; ++i) {
        const MidField<T>& f = a.f[i];
        int lines = 0;
        if (f.nterm < 0 || f.nterm > kMidTerms || !f.out) return hipErrorInvalidValue;
        for (int q = 0; q < f.nterm; ++q) {
            lines += f.t[q].line ? 1 : 0;
            if (f.t[q].line && !f.t[q].b) return hipErrorInvalidValue;
        }
        single = single && lines == 1 && f.nterm <= 2;
        for (int q = 0; q < f.nterm; ++q) single = single && f.t[q].b && f.t[q].pw == 0;
        if (a.op >= kMidScale && (f.nterm < 1 || !f.t[0].line)) return hipErrorInvalidValue;
        if (a.op == kMidScale && f.nterm != 1) return hipErrorInvalidValue;
        if (!f.s && !f.s64) return hipErrorInvalidValue;
    }
    if (a.op == kMidResidual) single = false;
    const long blocks = pencil_blocks(a.p.seg, a.p.nseg, a.p.TW, &a.p.tiles0);
    const int thr = a.p.TW * threads_per_line(n, 1);
    const size_t smem = lds_elems(n, a.p.TW) * sizeof(cpx<T>);
    const dim3 grid((unsigned)blocks, (unsigned)a.nf);
    return dispatch_size<SET>(n, [&](auto NC) -> hipError_t {
        constexpr int NN = decltype(NC)::value;
        if (a.op >= kMidScale) {
            if (single) return launch_k(k_mid<T, NN, 1, true, true>, grid, dim3(thr), smem, s, a);
            // the residual is ImplicitEuler's, which runs in FP64
            if constexpr (sizeof(T) == 8) return launch_k(k_mid<T, NN, 1, false, true>, grid, dim3(thr), smem, s, a);
            else return hipErrorInvalidValue;
        }
        if (single) return launch_k(k_mid<T, NN, 1, true, false>, grid, dim3(thr), smem, s, a);
        return launch_k(k_mid<T, NN, 1, false, false>, grid, dim3(thr), smem, s, a);
    });
}

extern template hipError_t launch_mid_set<float, 1>(const MidArgs<float>&, int, hipStream_t);
extern template hipError_t launch_mid_set<double, 1>(const MidArgs<double>&, int, hipStream_t);

template <typename T>
hipError_t launch_mid(const MidArgs<T>& a, int n, hipStream_t s) {
    return ext_length(n) ? launch_mid_set<T, 1>(a, n, s) : launch_mid_set<T, 0>(a, n, s);
}

}  // namespace gpf
