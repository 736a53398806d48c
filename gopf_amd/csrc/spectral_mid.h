// spectral_mid.h -- the middle pass of the general path along its last forward axis (z in 3D,
// y in 2D): forward transform of the lines, the k-space update, inverse transform of the
// result, in one launch (spectral_mid_kernels.h).  Separate passes wrote and read every
// derived field's spectrum and every updated spectrum once more each.
#pragma once

#include "spectral.h"

namespace gpf {

constexpr int kMidTerms = 6;

// what the pass forms at each k-point from the line spectra and R = sum_t coef_t L^pw_t B_t
enum MidOp {
    kMidStage0 = 0,   // RK4 stage 0: init = k (optional); fin = k + bp R; y = s (k + bc R)
    kMidStage12 = 1,  // RK4 stages 1, 2: fin += bp R; y = s (init + bc R)
    kMidStage3 = 2,   // RK4 stage 3: y = s (fin + bp R), stored to kn
    kMidEuler = 3,    // y = s (k + bc R), stored to kn
    kMidScale = 4,    // y = s B_0 (one line)
    kMidResidual = 5  // y = B_0 + sum_{t > 0} s coef_t L^pw_t B_t + cc (cc optional); kn = B_0
};

// one explicit term: B is transformed along the pass's axis first (line) or is a spectrum
// already; a null B is the constant 1
template <typename T>
struct MidTerm {
    const cpx<T>* b = nullptr;
    double coef = 1.0;
    int pw = 0;
    int line = 0;
    const double* dmul = nullptr;  // optional device-resident factor
};

// one output field of the pass; arrays are whole half spectra (main, then x-Nyquist)
template <typename T>
struct MidField {
    MidTerm<T> t[kMidTerms];
    int nterm = 0;
    const cpx<T>* k = nullptr;
    cpx<T>* init = nullptr;
    cpx<T>* fin = nullptr;
    cpx<T>* kn = nullptr;         // the updated spectrum (kMidResidual: B_0), stored when not null
    const T* s = nullptr;         // the factor table in the field precision, or
    const double* s64 = nullptr;  // in FP64 at both precisions
    const cpx<T>* cc = nullptr;
    cpx<T>* out = nullptr;        // y transformed back along the axis; never one of the fields' inputs
                                  // unless the launch has one field
};

template <typename T>
struct MidArgs {
    PencilArgs<T> p;              // tw, segments, TW, n (its arrays are unused)
    MidField<T> f[kMaxArr];
    int nf = 0;
    int op = 0;
    double bp = 0.0, bc = 0.0;
    int need_l = 0;               // some term has a LAP power
    KGrid g;
    long nmain = 0, nk = 0;       // elements of the main part of every array, and of the whole
};

// the pass along lines of length n (compiled lengths and the direct DFT up to 64)
template <typename T> hipError_t launch_mid(const MidArgs<T>& a, int n, hipStream_t s);

}  // namespace gpf
