// spectral_rowpoly.h -- forward row pass of the fields and their dense polynomials, or of the
// finite-difference derivative of both along a direction (ImplicitEuler).
#pragma once

#include "spectral.h"

namespace gpf {

struct RowPolyArgs {
    const cpx<double>* tw = nullptr;
    int nf = 0, nd = 0;                // one or two fields, nf + nd <= kMaxArr outputs
    const double* x = nullptr;         // the fields, n values each, one after the other
    const double* v = nullptr;         // the direction, laid out the same (npt > 0)
    long n = 0;
    int npt = 0;                       // stencil points; 0: the values themselves
    double off[8] = {}, w[8] = {};
    double dc[kMaxArr][4][4] = {};     // derived field d = sum_ij dc[d][i][j] f0^i f1^j
    cpx<double>* out[kMaxArr] = {};    // half spectra along x: the fields, then the derived fields
    long nmain = 0;
    long rows = 0;
    int nx = 0;
    int TW = 1;
};

hipError_t launch_rows_poly(const RowPolyArgs& a, hipStream_t s);

}  // namespace gpf
