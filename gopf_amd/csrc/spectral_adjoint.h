// spectral_adjoint.h -- the adjoint's reverse step along the last forward axis in one launch.
#pragma once

#include "pointwise.h"
#include "spectral.h"

namespace gpf {

// Per line of lam (transformed along every other axis): forward transform, P = m1 lam and
// Q = m2 lam, per scalar s the block sums of Re(conj(lam) (g1_s C1 + g0_s C0)), and the inverse
// transforms of P and Q along the axis into a.P and a.Q.  m1, m2 and the scalars' weights g1, g0
// depend on k only and come from tables (launch_adj_tables, once per run).
struct AdjTables {
    const double2* m = nullptr;  // m1, m2 of every k-point
    const double2* g = nullptr;  // per scalar, every k-point: g1, g0 (with the weights 1 / N and those of the half spectrum)
};
template <typename T>
struct AdjMidArgs {
    PencilArgs<T> p;  // tw, segments, TW
    AdjArgs<T> a;     // lam, P, Q, C1, C0 and their means, partial (adj_mid_blocks slots per scalar)
    AdjTables t;
};
template <typename T> long adj_mid_blocks(const AdjMidArgs<T>& a);
template <typename T> hipError_t launch_adj_mid(const AdjMidArgs<T>& a, int n, hipStream_t s);

}  // namespace gpf
