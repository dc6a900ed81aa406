// tri_eigen.hpp -- eigenvalues and eigenvectors of a symmetric tridiagonal T,
// one thread per eigenvalue: Sturm counts with bracketed Newton steps, then two
// steps of inverse iteration, orthogonalised within clusters of close
// eigenvalues.  The diagonal dd and off-diagonal ee (e2: its squares) are in
// LDS; eigenvectors and LU factors in global memory, column l of thread l.
#pragma once

#include <hip/hip_runtime.h>

#include <cfloat>
#include <cmath>
#include <cstdint>

namespace v2h {

namespace {

constexpr double kEps = DBL_EPSILON;
// Consecutive eigenvalues closer than kClusterRel |lambda| + kClusterAbs ||T||
// share a cluster; its eigenvectors are orthogonalised against each other.
constexpr double kClusterRel = 1e-5;
constexpr double kClusterAbs = 1e-11;
constexpr int kMaxPasses = 160;  // Sturm passes per eigenvalue (bisection needs about 60)
constexpr int kChunk = 8;        // inverse-iteration loads issued ahead of their use

// 1/q to about 1 ulp: hardware reciprocal and one Newton step.
__device__ __forceinline__ double recip(double q) {
    const double r = __builtin_amdgcn_rcp(q);
    const double e = fma(-q, r, 1.0);
    return fma(r, e, r);
}

// Deterministic start vectors for inverse iteration, uniform in [-1, 1).
__device__ __forceinline__ double start_value(uint32_t l, uint32_t i) {
    uint32_t h = (l * 0x9E3779B1u) ^ ((i + 0x7F4A7C15u) * 0x85EBCA77u);
    h ^= h >> 15;
    h *= 0x2C1B3C6Du;
    h ^= h >> 12;
    h *= 0x297A2D39u;
    h ^= h >> 15;
    return (double)(h & 0xFFFFFFu) * (1.0 / 8388608.0) - 1.0;
}

// Sturm count of T - s I (eigenvalues below s) and S = d/ds log|det(T - s I)|
// = sum_j 1 / (s - lambda_j), from the pivots q_i of the LDL^T recurrence.
__device__ int sturm(double s, int d, const double* dd, const double* e2, double pivmin, double& S) {
    double q = dd[0] - s;
    if (fabs(q) < pivmin) q = -pivmin;
    double r = recip(q);
    int c = q < 0.0;
    double dq = -1.0;
    double acc = dq * r;
    auto step = [&](double di, double e) {
        double qn = fma(-e, r, di - s);
        const double dqn = fma(e * dq, r * r, -1.0);
        if (fabs(qn) < pivmin) qn = -pivmin;
        r = recip(qn);
        dq = dqn;
        c += qn < 0.0;
        acc = fma(dq, r, acc);
    };
    int i = 1;
    for (; i + 4 <= d; i += 4) {  // the loads of four steps ahead of the recurrence
        double dv[4], ev[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            dv[u] = dd[i + u];
            ev[u] = e2[i + u - 1];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) step(dv[u], ev[u]);
    }
    for (; i < d; i++) step(dd[i], e2[i - 1]);
    S = acc;
    return c;
}

// Inverse-iteration helpers on one column x (stride d) of the work area, with
// the LU factors of T - sg I in F (5 planes of stride d^2, same column).
struct Column {
    double* x;
    double* F;
    size_t ld, plane;  // d, d^2
    __device__ double& X(int i) const { return x[(size_t)i * ld]; }
    __device__ double& f(int q, int i) const { return F[q * plane + (size_t)i * ld]; }
};

// x <- L^{-1} P (scale x); loads run kChunk rows ahead of the recurrence.
__device__ void apply_pl(const Column& c, int d, double scale) {
    double bc = c.X(0) * scale;
    for (int i0 = 0; i0 + 1 < d; i0 += kChunk) {
        double xn[kChunk], f0[kChunk], sw[kChunk];
#pragma unroll
        for (int u = 0; u < kChunk; u++) {
            const int i = min(i0 + u, d - 2);
            xn[u] = c.X(i + 1);
            f0[u] = c.f(0, i);
            sw[u] = c.f(4, i);
        }
#pragma unroll
        for (int u = 0; u < kChunk; u++) {
            const int i = i0 + u;
            if (i + 1 < d) {
                const double bn = xn[u] * scale;
                const bool s = sw[u] != 0.0;
                c.X(i) = s ? bn : bc;
                bc = s ? fma(-f0[u], bn, bc) : fma(-f0[u], bc, bn);
            }
        }
    }
    c.X(d - 1) = bc;
}

// x <- U^{-1} x; returns ||x||^2.
__device__ double apply_u(const Column& c, int d) {
    double x1 = 0.0, x2 = 0.0, s2 = 0.0;
    for (int i0 = d - 1; i0 >= 0; i0 -= kChunk) {
        double xb[kChunk], f1[kChunk], f2[kChunk], f3[kChunk];
#pragma unroll
        for (int u = 0; u < kChunk; u++) {
            const int i = max(i0 - u, 0);
            xb[u] = c.X(i);
            f1[u] = c.f(1, i);
            f2[u] = c.f(2, i);
            f3[u] = c.f(3, i);
        }
#pragma unroll
        for (int u = 0; u < kChunk; u++) {
            const int i = i0 - u;
            if (i >= 0) {
                const double xi = fma(-f3[u], x2, fma(-f2[u], x1, xb[u])) * f1[u];
                c.X(i) = xi;
                s2 = fma(xi, xi, s2);
                x2 = x1;
                x1 = xi;
            }
        }
    }
    return s2;
}

// x <- x - sum_m (y_m . x / ||y_m||^2) y_m over the cluster's earlier columns
// (twice); returns the new ||x||^2.
__device__ double orthogonalise(const Column& c, int d, const double* Sv, int l0, int l, const double* xs) {
    for (int pass = 0; pass < 2; pass++)
        for (int m = l0; m < l; m++) {
            const double* y = Sv + m;
            double dot = 0.0;
            for (int i0 = 0; i0 < d; i0 += kChunk) {
                double yv[kChunk], xv[kChunk];
#pragma unroll
                for (int u = 0; u < kChunk; u++) {
                    const int i = min(i0 + u, d - 1);
                    yv[u] = y[(size_t)i * d];
                    xv[u] = c.X(i);
                }
#pragma unroll
                for (int u = 0; u < kChunk; u++)
                    if (i0 + u < d) dot = fma(yv[u], xv[u], dot);
            }
            const double f = dot / xs[m];
            for (int i0 = 0; i0 < d; i0 += kChunk) {
                double yv[kChunk], xv[kChunk];
#pragma unroll
                for (int u = 0; u < kChunk; u++) {
                    const int i = min(i0 + u, d - 1);
                    yv[u] = y[(size_t)i * d];
                    xv[u] = c.X(i);
                }
#pragma unroll
                for (int u = 0; u < kChunk; u++)
                    if (i0 + u < d) c.X(i0 + u) = fma(-f, yv[u], xv[u]);
            }
        }
    double s2 = 0.0;
    for (int i0 = 0; i0 < d; i0 += kChunk) {
        double xv[kChunk];
#pragma unroll
        for (int u = 0; u < kChunk; u++) xv[u] = c.X(min(i0 + u, d - 1));
#pragma unroll
        for (int u = 0; u < kChunk; u++)
            if (i0 + u < d) s2 = fma(xv[u], xv[u], s2);
    }
    return s2;
}

// Eigenvalue l (ascending) of T inside [gl, gu]; lp: a previous value of it,
// dprev its expected change (either not finite: none).  bad: not converged.
__device__ __forceinline__ double tri_eigenvalue(int l, int d, const double* dd, const double* e2, double gl, double gu,
                                                 double abstol, double pivmin, double lp, double dprev, bool& bad) {
    double lam = 0.0;
    double lo = gl, hi = gu;
    int clo = 0, chi = d;
    int passes = 0;
    double s = 0.5 * (lo + hi), S = 0.0;
    bool haveS = false;
    auto eval = [&](double x, double& Sx) {
        const int c = sturm(x, d, dd, e2, pivmin, Sx);
        passes++;
        if (c <= l) {
            lo = x;
            clo = c;
        } else {
            hi = x;
            chi = c;
        }
        return c;
    };
    if (dprev >= 0.0 && isfinite(lp) && isfinite(dprev)) {
        // expanding search around the previous eigenvalue of this block
        double del = fmax(2.0 * dprev, 8.0 * abstol);
        s = fmin(fmax(lp, lo), hi);
        const int c0 = eval(s, S);
        haveS = true;
        for (int e = 0; e < 8; e++) {
            const double x = (c0 <= l) ? s + del : s - del;
            if (!(x > lo && x < hi)) break;
            double Sx;
            const int cx = eval(x, Sx);
            if ((c0 <= l) != (cx <= l)) break;
            del *= 4.0;
        }
    }
    lam = 0.5 * (lo + hi);
    double last = INFINITY;
    bool probed = false;
    while (passes < kMaxPasses) {
        if (hi - lo <= abstol) {
            lam = 0.5 * (lo + hi);
            break;
        }
        double sn = 0.0;
        bool newton = false;
        if (clo == l && chi == l + 1 && haveS) {
            const double step = -1.0 / S;
            sn = s + step;
            const bool inside = sn > lo && sn < hi;
            if (fabs(step) <= 2.0 * abstol) {
                if (inside) {
                    lam = sn;
                    break;
                }
                // Out of the bracket, by rounding at eigenvalue l or at a
                // neighbour of it: next to one of high multiplicity S is large and
                // the step small, however far eigenvalue l is.  A count across
                // s tells (bisecting instead: 33 passes per eigenvalue of a random
                // 224-row T, against 15).
                if (!probed) {
                    probed = true;
                    const double x = s <= lo ? lo + 2.0 * abstol : hi - 2.0 * abstol;
                    double Sx;
                    if (x > lo && x < hi) eval(x, Sx);
                    if (hi - lo <= 2.5 * abstol) {
                        lam = 0.5 * (lo + hi);
                        break;
                    }
                    continue;
                }
            }
            newton = inside && fabs(step) <= 0.5 * last;
            if (newton) {
                last = fabs(step);
                // a little past the root, so that the step there points back into
                // the bracket whatever its rounding (with the count above alone,
                // which every eigenvalue would take then, 16 passes instead of 15):
                // by more than the counts round, by less than is accepted
                const double over = sn + copysign(1.5 * abstol, step);
                if (over > lo && over < hi) sn = over;
            }
        }
        if (!newton) {
            sn = 0.5 * (lo + hi);
            last = INFINITY;
            probed = false;
        }
        s = sn;
        eval(s, S);
        haveS = true;
        lam = s;
    }
    if (passes >= kMaxPasses) bad = true;
    return lam;
}

// Whether eigenvalues l - 1 and l belong to one cluster.
__device__ __forceinline__ bool tri_linked(const double* lamv, int l, double tnorm) {
    return l > 0 && (lamv[l] - lamv[l - 1]) <= kClusterRel * fmax(fabs(lamv[l]), fabs(lamv[l - 1])) + kClusterAbs * tnorm;
}

// Shift of the inverse iteration for eigenvector l: its eigenvalue, kept apart
// from the shift before it in the cluster (sprev; -INFINITY at its first).
__device__ __forceinline__ double tri_shift(double lam, double sprev, double tnorm) {
    const double pert = 10.0 * kEps * fmax(fabs(lam), 1e-3 * tnorm);
    return lam <= sprev + pert ? sprev + pert : lam;
}

// First solve for eigenvector l: T - sg I = P L U with partial pivoting
// ([q][i]: 0 multiplier, 1 reciprocal pivot, 2-3 superdiagonals of U, 4
// interchange), fused with L^{-1} P applied to the start vector; then U^{-1}.
// Returns ||x||^2.
__device__ __forceinline__ double tri_solve(const Column& col, int l, int d, const double* dd, const double* ee,
                                            double sg, double tnorm) {
    const double ptol = kEps * tnorm;
    double dcur = dd[0] - sg, ucur = d > 1 ? ee[0] : 0.0;
    double bc = start_value((uint32_t)l, 0u);
    for (int i = 0; i + 1 < d; i++) {
        const double sub = ee[i];
        double dnext = dd[i + 1] - sg;
        double unext = (i + 2 < d) ? ee[i + 1] : 0.0;
        const double bn = start_value((uint32_t)l, (uint32_t)(i + 1));
        double f, u0, u1, u2, sw, xi;
        if (fabs(dcur) >= fabs(sub)) {
            if (fabs(dcur) < ptol) dcur = (dcur < 0.0) ? -ptol : ptol;
            f = sub * recip(dcur);
            u0 = dcur;
            u1 = ucur;
            u2 = 0.0;
            sw = 0.0;
            dnext = fma(-f, ucur, dnext);
            xi = bc;
            bc = fma(-f, bc, bn);
        } else {
            f = dcur * recip(sub);
            u0 = sub;
            u1 = dnext;
            u2 = unext;
            sw = 1.0;
            dnext = fma(-f, dnext, ucur);
            unext = -f * unext;
            xi = bn;
            bc = fma(-f, bn, bc);
        }
        col.f(0, i) = f;
        col.f(1, i) = recip(u0);
        col.f(2, i) = u1;
        col.f(3, i) = u2;
        col.f(4, i) = sw;
        col.X(i) = xi;
        dcur = dnext;
        ucur = unext;
    }
    if (fabs(dcur) < ptol) dcur = (dcur < 0.0) ? -ptol : ptol;
    col.f(1, d - 1) = recip(dcur);
    col.f(2, d - 1) = 0.0;
    col.f(3, d - 1) = 0.0;
    col.X(d - 1) = bc;
    return apply_u(col, d);
}

// Second solve, with the first one's factors, from x of squared norm s2.
__device__ __forceinline__ double tri_resolve(const Column& col, int d, double s2) {
    apply_pl(col, d, 1.0 / sqrt(s2));
    return apply_u(col, d);
}

// Eigenvectors l0 .. l1 of one cluster, unnormalised, to the columns of Sv;
// xs[l] = ||S(:, l)||^2.  fac: 5 d^2 doubles for the LU factors.
__device__ __forceinline__ void tri_vectors(int l0, int l1, int d, const double* dd, const double* ee,
                                            const double* lamv, double* xs, double tnorm, double* Sv, double* fac,
                                            bool& bad) {
    double sprev = -INFINITY;
    for (int l = l0; l <= l1; l++) {
        const double sg = tri_shift(lamv[l], sprev, tnorm);
        sprev = sg;
        const Column col{Sv + l, fac + l, (size_t)d, (size_t)d * d};
        double s2 = tri_solve(col, l, d, dd, ee, sg, tnorm);
        if (l > l0) s2 = orthogonalise(col, d, Sv, l0, l, xs);
        s2 = tri_resolve(col, d, s2);
        if (l > l0) s2 = orthogonalise(col, d, Sv, l0, l, xs);
        if (!(s2 > 0.0) || !isfinite(s2)) {
            bad = true;
            s2 = INFINITY;  // drops the vector from T+
        }
        xs[l] = s2;
    }
}

}  // namespace

}  // namespace v2h
