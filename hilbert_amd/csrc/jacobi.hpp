// jacobi.hpp -- rounds of the parallel cyclic Jacobi eigensolver (round-robin
// ordering) on a packed symmetric matrix.
#pragma once

#include <hip/hip_runtime.h>

namespace v2h {

// Packed upper triangle: element (i, j), i <= j, at j (j + 1) / 2 + i.
__device__ __forceinline__ int pk(int i, int j) { return i <= j ? (j * (j + 1) >> 1) + i : (i * (i + 1) >> 1) + j; }

// Pair k of round t for dp (even) indices: the circle method with index
// dp - 1 fixed.  Returns p < q.
__device__ __forceinline__ void round_pair(int t, int k, int dp, int& p, int& q) {
    int M = dp - 1;
    int a, b;
    if (k == 0) {
        a = t;
        b = M;
    } else {
        a = t + k;
        if (a >= M) a -= M;
        b = t - k;
        if (b < 0) b += M;
    }
    p = a < b ? a : b;
    q = a < b ? b : a;
}

// Triangular tile index e -> (P, Q), P <= Q.
__device__ __forceinline__ void tri_pair(int e, int& P, int& Q) {
    int qq = (int)((sqrtf(8.0f * (float)e + 1.0f) - 1.0f) * 0.5f);
    while ((qq + 1) * (qq + 2) / 2 <= e) qq++;
    while (qq * (qq + 1) / 2 > e) qq--;
    Q = qq;
    P = e - qq * (qq + 1) / 2;
}

// One round of two-sided rotations G_P A G_Q^T on the packed matrix A; the 2x2
// diagonal tiles are set to their closed form.
template <int NT>
__device__ void apply_round(double* A, const int* pp, const int* qq, const double* rc, const double* rs, int m) {
    const int ntile = m * (m + 1) / 2;
    for (int e = threadIdx.x; e < ntile; e += NT) {
        int P, Q;
        tri_pair(e, P, Q);
        const double cP = rc[P], sP = rs[P];
        const int p = pp[P], q = qq[P];
        if (P == Q) {
            const int ipp = pk(p, p), ipq = pk(p, q), iqq = pk(q, q);
            const double app = A[ipp], apq = A[ipq], aqq = A[iqq];
            if (rs[P] != 0.0) {
                const double t = rs[P] / rc[P];
                A[ipp] = app - t * apq;
                A[iqq] = aqq + t * apq;
                A[ipq] = 0.0;
            }
            continue;
        }
        const double cQ = rc[Q], sQ = rs[Q];
        const int r = pp[Q], s = qq[Q];
        const int i0 = pk(p, r), i1 = pk(p, s), i2 = pk(q, r), i3 = pk(q, s);
        double a0 = A[i0], a1 = A[i1], a2 = A[i2], a3 = A[i3];
        // rows (p, q) by P
        double b0 = cP * a0 - sP * a2, b1 = cP * a1 - sP * a3;
        double b2 = sP * a0 + cP * a2, b3 = sP * a1 + cP * a3;
        // columns (r, s) by Q
        A[i0] = cQ * b0 - sQ * b1;
        A[i1] = sQ * b0 + cQ * b1;
        A[i2] = cQ * b2 - sQ * b3;
        A[i3] = sQ * b2 + cQ * b3;
    }
}

}  // namespace v2h
