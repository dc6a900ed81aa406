// The pair corrections of the refinement (refine_pair.hpp) compiled for the
// host: one whole step on a small matrix.
#include <cmath>
#include <vector>

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime.h>

#include "refine_pair.hpp"

using namespace v2h;

// X <- X (I + E) with the corrections E of U (both d x d, row-major), E as the
// kernels form it (columns normalised first).  Returns the largest correction.
extern "C" double refine_step_host(int d, const double* U, double* X, double* E, double cluster_rel) {
    auto at = [d](const double* a, int i, int j) { return a[(size_t)i * d + j]; };
    std::vector<double> K(d * d), G(d * d), S(d * d), l(d), n(d), Y(X, X + d * d);
    auto product = [&](const double* a, bool ta, const double* b, double* c) {
        for (int i = 0; i < d; i++)
            for (int j = 0; j < d; j++) {
                double s = 0.0;
                for (int k = 0; k < d; k++) s = std::fma(ta ? at(a, k, i) : at(a, i, k), at(b, k, j), s);
                c[(size_t)i * d + j] = s;
            }
    };
    product(U, false, X, K.data());
    product(X, true, X, G.data());
    product(X, true, K.data(), S.data());
    double scale = 0.0, me = 0.0;
    for (int i = 0; i < d; i++) {
        l[i] = at(S.data(), i, i) / at(G.data(), i, i);
        n[i] = 1.0 / std::sqrt(at(G.data(), i, i));
        scale = std::fmax(scale, std::fabs(l[i]));
    }
    for (int i = 0; i < d; i++)
        for (int j = 0; j < d; j++) {
            double ev = n[j] - 1.0;
            if (i != j) {
                const RefPair p = ref_pair(l[i], l[j], n[i], n[j], at(G.data(), i, j), at(S.data(), i, j),
                                           at(S.data(), j, i), cluster_rel * scale, i < j);
                ev = 0.5 * p.rr + (p.close ? 0.0 : ref_rotation(p));
            }
            me = std::fmax(me, std::fabs(ev));
            E[(size_t)i * d + j] = i == j ? ev : n[i] * ev;
        }
    product(Y.data(), false, E, K.data());
    for (int e = 0; e < d * d; e++) X[e] = Y[e] + K[e];
    return me;
}

// Coupling of one pair that stays when the step is done, with its orthogonality.
extern "C" int pair_host(double li, double lj, double g, double s, double om, double* left) {
    const RefPair p = ref_pair(li, lj, 1.0, 1.0, g, s, s, om, true);
    *left = p.sa;
    return p.close ? 1 : 0;
}
