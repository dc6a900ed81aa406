// refine_pair.hpp -- what one refinement step does with a pair (i, j) of
// columns of X (see refine.hpp), shared by the kernels of all block sizes.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

namespace v2h {

struct RefPair {
    double rr;    // r_ij of the normalised columns
    double sa;    // coupling that is left when the step has made them orthogonal
    double dl;    // l_j - l_i; of equal ones +0 where i < j, else -0
    bool close;   // too close to be separated: within om in gap and coupling
};

// l, n: eigenvalue estimates and g^-1/2 of the two columns; g: G_ij; s, st: S_ij
// and S_ji, which round differently.  r_ij alone leaves s_ij = -l r_ij in S of a
// degenerate pair, which the step takes out with r_ij: kept beside the
// eigenvalues, it put errors of up to 3e-9 into U+.  upper: i < j.
__device__ __forceinline__ RefPair ref_pair(double li, double lj, double ni, double nj, double g, double s, double st,
                                            double om, bool upper) {
    RefPair p;
    const double nn = ni * nj, sv = 0.5 * (s + st) * nn;
    p.rr = -g * nn;
    p.dl = upper ? lj - li : -(li - lj);
    p.sa = fma(0.5 * (lj + li), p.rr, sv);
    p.close = !(fabs(p.dl) > om || fabs(p.sa) > om);
    return p;
}

// Rotation part of the correction of a separated pair, opposite for (i, j) and
// (j, i): the sign of dl turns a pair of equal estimates by 45 degrees, and with
// one sign for both X (I + E) would be singular.
__device__ __forceinline__ double ref_rotation(const RefPair& p) {
    const double ta = p.sa + p.sa;
    return ta / (p.dl + copysign(sqrt(fma(p.dl, p.dl, ta * ta)), p.dl));
}

}  // namespace v2h
