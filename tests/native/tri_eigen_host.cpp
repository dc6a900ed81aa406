// The tridiagonal eigensolver of the projection kernels (tri_eigen.hpp),
// compiled for the host: the threads of a workgroup one after the other.
#include <algorithm>
#include <cmath>
#include <vector>

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>
#define __builtin_amdgcn_rcp(q) (1.0 / (q))
using std::isfinite;
using std::max;
using std::min;

#include "tri_eigen.hpp"

using namespace v2h;

// Eigenvalues of the tridiagonal matrix (dd, ee) as the kernels take them:
// ascending in lam.  prev: the previous eigenvalues and their expected change
// (d + 1 values), or null.  Returns 1 where an eigenvalue did not converge.
extern "C" int tri_values_host(int d, const double* dd, const double* ee, const double* prev, double* lam) {
    std::vector<double> e2(d, 0.0);
    double lo = INFINITY, hi = -INFINITY, em = 0.0;
    for (int i = 0; i < d; i++) {
        const double el = i > 0 ? std::fabs(ee[i - 1]) : 0.0, er = i + 1 < d ? std::fabs(ee[i]) : 0.0;
        lo = std::fmin(lo, dd[i] - el - er);
        hi = std::fmax(hi, dd[i] + el + er);
        e2[i] = er * er;
        em = std::fmax(em, e2[i]);
    }
    const double tnorm = std::fmax(std::fabs(lo), std::fabs(hi)), pivmin = DBL_MIN * std::fmax(1.0, em);
    const double slack = 2.0 * kEps * tnorm * d + 2.0 * pivmin;
    bool bad = false;
    for (int l = 0; l < d; l++)
        lam[l] = tnorm > 0.0 ? tri_eigenvalue(l, d, dd, e2.data(), lo - slack, hi + slack, 2.0 * kEps * tnorm, pivmin,
                                              prev ? prev[l] : NAN, prev ? prev[d] : NAN, bad)
                             : 0.0;
    return bad ? 1 : 0;
}

// Eigenvectors of every cluster (columns of S, d x d), xs their squared norms.
extern "C" int tri_vectors_host(int d, const double* dd, const double* ee, const double* lam, double* S, double* xs) {
    std::vector<double> fac(5 * (size_t)d * d), e(ee, ee + d);
    double tnorm = 0.0;
    for (int i = 0; i < d; i++)
        tnorm = std::fmax(tnorm, std::fabs(dd[i]) + (i > 0 ? std::fabs(ee[i - 1]) : 0.0) +
                                     (i + 1 < d ? std::fabs(ee[i]) : 0.0));
    bool bad = false;
    for (int l = 0; l < d;) {
        int l1 = l;
        while (l1 + 1 < d && tri_linked(lam, l1 + 1, tnorm)) l1++;
        tri_vectors(l, l1, d, dd, e.data(), lam, xs, tnorm, S, fac.data(), bad);
        l = l1 + 1;
    }
    return bad ? 1 : 0;
}
