// eig_big.hip -- eigendecomposition of the blocks above 224 rows that the
// refinement does not take (refine.hpp), spread over the whole GPU.
//
// Such a block neither fits one workgroup's registers nor gives one workgroup
// enough bandwidth: in one workgroup a 288-row block took 166 ms by Jacobi and
// a 228-row one 10 ms by reflections.  Here one launch reduces one column of
// every block, each workgroup holding a share of the rows:
//
//   U = Q T Q^T   step k: every workgroup finishes the rank-2 update of step
//                 k - 1 for column k from v, p and row k (the same few vector
//                 operations in each), forms the reflector, applies the update
//                 to its own rows and multiplies them by the new v.  Row k is
//                 read by all and rewritten by none, so a step needs no barrier
//                 but its launch.
//   T = S L S^T   one thread per eigenvalue, 64 per workgroup (tri_eigen.hpp);
//                 the vectors of a cluster of close eigenvalues are
//                 orthogonalised by a workgroup
//   V = Q S       compact-WY products of 16 reflectors, 64 columns per workgroup
//   U+            the final product of the refinement, V being the accepted X
//
// Bound by the latency of the d - 1 steps (vector reductions and one pass over
// the rows each).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "refine.hpp"
#include "tri_eigen.hpp"

namespace v2h {

namespace {

constexpr int kNT = 256;
constexpr int kNB = 16;                 // reflectors per compact-WY product
constexpr int kMaxD = kBigMaxRows;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
// Workgroup sum in a fixed order; red: 4 doubles.
__device__ __forceinline__ double wg_sum(double v, double* red) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    return (red[0] + red[1]) + (red[2] + red[3]);
}

// The work area of a block (tri_work): reflectors, eigenvectors of T, five
// planes that first hold the matrix and at the end the triangular factors of
// the compact-WY products, then the vectors.
struct Area {
    double *hv, *S, *fac, *dd, *ee, *lam, *xs, *v, *p;
    __device__ __forceinline__ Area(double* tri_work, const RefBlock& b) {
        const size_t d = b.d, n2 = d * d;
        hv = tri_work + b.tri;
        S = hv + n2;
        fac = S + n2;
        dd = hv + 7 * n2;
        ee = dd + d;
        lam = ee + d;
        xs = lam + d;
        v = xs + d;      // two vectors
        p = v + 2 * d;   // two vectors
    }
};

// need[i] = block i of the list is projected here: every active one without the
// refinement, else the active ones that it has not accepted.
__global__ void k_big_need(BatchDev B, RefDev R, const int* list, int n, int refined, int* need) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const RefBlock b = R.blk[list[i]];
    const int route = R.route[b.gblock];
    need[i] = B.st[b.inst].active && in_pgroup(B, b.inst) && (!refined || route != kRouteAccepted);
    RefState& rs = R.rs[list[i]];
    if (need[i] || rs.phase == kPhaseFresh) rs.phase = 0;
}

// A = sym(U), also to slot U of the refinement's work area (its final product
// reads it), one 32 x 32 tile per workgroup.
__global__ __launch_bounds__(kNT) void k_big_load(BatchDev B, RefDev R, const int* list, const int* need) {
    __shared__ double tt[32][33];
    if (!need[blockIdx.z]) return;
    const RefBlock b = R.blk[list[blockIdx.z]];
    const int d = b.d, c = threadIdx.x & 31, r0 = threadIdx.x >> 5;
    const int i0 = blockIdx.y * 32, j0 = blockIdx.x * 32;
    if (i0 >= d || j0 >= d) return;
    const double* U = B.u + B.inst[b.inst].poff + b.off;
    double* A = Area(R.tri_work, b).fac;
    double* Us = R.work + b.w + (size_t)kSlotU * d * d;
    for (int r = r0; r < 32; r += kNT / 32)
        tt[r][c] = (j0 + r < d && i0 + c < d) ? U[(size_t)(j0 + r) * d + i0 + c] : 0.0;
    __syncthreads();
    for (int r = r0; r < 32; r += kNT / 32)
        if (i0 + r < d && j0 + c < d) {
            const size_t e = (size_t)(i0 + r) * d + j0 + c;
            const double s = 0.5 * (U[e] + tt[c][r]);
            A[e] = s;
            Us[e] = s;
        }
}

// Step k of the reduction (k = 0 .. d - 2; the last has no reflector).
__global__ __launch_bounds__(kNT) void k_big_step(RefDev R, const int* list, const int* need, int k) {
    __shared__ double vs[kMaxD], ws[kMaxD], us[kMaxD];
    __shared__ double red[4];
    if (!need[blockIdx.y]) return;
    const RefBlock b = R.blk[list[blockIdx.y]];
    const int d = b.d, t = threadIdx.x;
    if (k > d - 2) return;
    const Area W(R.tri_work, b);
    double* A = W.fac;
    const double *vp = W.v + (size_t)(k & 1) * d, *pp = W.p + (size_t)(k & 1) * d;
    double *vn = W.v + (size_t)((k + 1) & 1) * d, *pn = W.p + (size_t)((k + 1) & 1) * d;
    // the pending update A -= v w^T + w v^T of step k - 1 (rows k .. d - 1)
    double kk = 0.0;
    if (k > 0) {
        for (int i = k + t; i < d; i += kNT) kk = fma(vp[i], pp[i], kk);
        kk = 0.5 * W.hv[(size_t)(k - 1) * d + k - 1] * wg_sum(kk, red);
    }
    for (int i = k + t; i < d; i += kNT) {
        const double v = k > 0 ? vp[i] : 0.0;
        vs[i] = v;
        ws[i] = k > 0 ? fma(-kk, v, pp[i]) : 0.0;
    }
    __syncthreads();
    // column k of the updated matrix
    const double vk = vs[k], wk = ws[k];
    double sg = 0.0;
    for (int i = k + t; i < d; i += kNT) {
        const double a = fma(-ws[i], vk, fma(-vs[i], wk, A[(size_t)k * d + i]));
        us[i] = a;
        if (i > k + 1) sg = fma(a, a, sg);
    }
    sg = wg_sum(sg, red);  // also completes us
    const double alpha = us[k + 1];
    if (k == d - 2) {
        if (blockIdx.x == 0 && t == 0) {
            W.dd[k] = us[k];
            W.ee[k] = alpha;
            W.dd[d - 1] = fma(-2.0 * ws[d - 1], vs[d - 1], A[(size_t)(d - 1) * d + d - 1]);
        }
        return;
    }
    double tk = 0.0, sc = 0.0, beta = alpha;
    if (sg != 0.0) {
        beta = -copysign(sqrt(fma(alpha, alpha, sg)), alpha);
        tk = (beta - alpha) / beta;
        sc = 1.0 / (alpha - beta);
    }
    if (blockIdx.x == 0 && t == 0) {
        W.dd[k] = us[k];
        W.ee[k] = beta;
        W.hv[(size_t)k * d + k] = tk;
    }
    __syncthreads();
    for (int i = k + 1 + t; i < d; i += kNT) {
        const double v = tk == 0.0 ? 0.0 : (i == k + 1 ? 1.0 : us[i] * sc);
        us[i] = v;
        if (blockIdx.x == 0) {
            W.hv[(size_t)k * d + i] = v;
            vn[i] = v;
        }
    }
    __syncthreads();
    // rows i > k, each always in the same wavefront of the grid
    const int nw = gridDim.x * (kNT / 64), w = blockIdx.x * (kNT / 64) + (t >> 6), lane = t & 63;
    for (int i = w + ((k + nw - w) / nw) * nw; i < d; i += nw) {
        const double vi = vs[i], wi = ws[i];
        double* Ai = A + (size_t)i * d;
        double s = 0.0;
        for (int j = k + 1 + lane; j < d; j += 64) {
            const double a = fma(-wi, vs[j], fma(-vi, ws[j], Ai[j]));
            Ai[j] = a;
            s = fma(a, us[j], s);
        }
        s = wave_sum(s);
        if (lane == 0) pn[i] = tk * s;
    }
}

// Eigenvalues, one thread each, 64 per workgroup.
__global__ __launch_bounds__(64) void k_big_values(BatchDev B, RefDev R, const int* list, const int* need) {
    __shared__ double dd[kMaxD], e2[kMaxD];
    if (!need[blockIdx.y]) return;
    const RefBlock b = R.blk[list[blockIdx.y]];
    const int d = b.d, t = threadIdx.x, l = blockIdx.x * 64 + t;
    if ((int)blockIdx.x * 64 >= d) return;
    const Area W(R.tri_work, b);
    double lo = INFINITY, hi = -INFINITY, em = 0.0;
    for (int i = t; i < d; i += 64) {
        const double x = W.dd[i], el = i > 0 ? fabs(W.ee[i - 1]) : 0.0, er = i + 1 < d ? fabs(W.ee[i]) : 0.0;
        dd[i] = x;
        e2[i] = er * er;
        lo = fmin(lo, x - el - er);
        hi = fmax(hi, x + el + er);
        em = fmax(em, er * er);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        lo = fmin(lo, __shfl_xor(lo, o, 64));
        hi = fmax(hi, __shfl_xor(hi, o, 64));
        em = fmax(em, __shfl_xor(em, o, 64));
    }
    __syncthreads();
    if (l >= d) return;
    const double tnorm = fmax(fabs(lo), fabs(hi)), pivmin = DBL_MIN * fmax(1.0, em);
    const double slack = 2.0 * kEps * tnorm * d + 2.0 * pivmin;
    bool bad = false;
    double lam = 0.0;
    if (tnorm > 0.0)
        lam = tri_eigenvalue(l, d, dd, e2, lo - slack, hi + slack, 2.0 * kEps * tnorm, pivmin, NAN, NAN, bad);
    W.lam[l] = lam;
    (R.work + b.w + (size_t)kRefSlots * d * d)[l] = lam;  // read by the final product
    if (bad) atomicOr(&B.st[b.inst].status, (int)kStatusJacobiNotConverged);
}

// ||T||, the same value in every lane (as k_big_values and the kernels below
// need it: Gershgorin's bound on the largest |eigenvalue|).
__device__ __forceinline__ double big_norm(const Area& W, int d) {
    double m = 0.0;
    for (int i = threadIdx.x & 63; i < d; i += 64)
        m = fmax(m, fabs(W.dd[i]) + (i > 0 ? fabs(W.ee[i - 1]) : 0.0) + (i + 1 < d ? fabs(W.ee[i]) : 0.0));
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    return m;
}

// Inverse iteration, one thread per eigenvector: the first solve or (second) the
// one after it.  Between and after them k_big_ortho orthogonalises each
// cluster: as in tri_vectors, except that a whole cluster takes each step
// together.
__global__ __launch_bounds__(64) void k_big_vectors(BatchDev B, RefDev R, const int* list, const int* need,
                                                    int second) {
    __shared__ double dd[kMaxD], ee[kMaxD], lam[kMaxD];
    if (!need[blockIdx.y]) return;
    const RefBlock b = R.blk[list[blockIdx.y]];
    const int d = b.d, t = threadIdx.x, l = blockIdx.x * 64 + t;
    if ((int)blockIdx.x * 64 >= d) return;
    const Area W(R.tri_work, b);
    const double tnorm = big_norm(W, d);
    for (int i = t; i < d; i += 64) {
        dd[i] = W.dd[i];
        ee[i] = i + 1 < d ? W.ee[i] : 0.0;
        lam[i] = W.lam[i];
    }
    __syncthreads();
    if (l >= d) return;
    if (!(tnorm > 0.0)) {  // T = 0: any orthonormal basis
        for (int i = 0; i < d; i++) W.S[(size_t)i * d + l] = i == l ? 1.0 : 0.0;
        W.xs[l] = 1.0;
        return;
    }
    const Column col{W.S + l, W.fac + l, (size_t)d, (size_t)d * d};
    if (second) {
        const double s2 = tri_resolve(col, d, W.xs[l]);
        const bool bad = !(s2 > 0.0) || !isfinite(s2);
        W.xs[l] = bad ? INFINITY : s2;
        if (bad) atomicOr(&B.st[b.inst].status, (int)kStatusJacobiNotConverged);
        return;
    }
    int l0 = l;
    while (tri_linked(lam, l0, tnorm)) l0--;
    double sg = -INFINITY;
    for (int i = l0; i <= l; i++) sg = tri_shift(lam[i], sg, tnorm);
    W.xs[l] = tri_solve(col, l, d, dd, ee, sg, tnorm);
}

// Gram-Schmidt, twice, of the vectors of every cluster of close eigenvalues;
// workgroup g takes the clusters that begin at an eigenvalue 16 g .. 16 g + 15.
// 16 columns at a time are orthogonalised against the earlier ones, 64 by 64
// (coefficients of a wavefront per quarter of the rows, summed in LDS), then
// among each other.  A cluster of m vectors takes about 8 m^2 d products and
// reads its columns m / 16 times.  A whole projection of 300 rows: 3.8 ms, with
// 200 equal eigenvalues 12.5 ms, with 285 of them 29 ms; of 417 rows with 397
// equal ones 82 ms.  One thread per cluster, with dependent loads of single
// values, takes 1.8 s for 213 equal ones of 224 rows.
__global__ __launch_bounds__(kNT) void k_big_ortho(BatchDev B, RefDev R, const int* list, const int* need) {
    constexpr int kP = 16, kE = 64;  // columns of a panel, earlier columns at a time
    __shared__ double lam[kMaxD];
    __shared__ double part[4][kP][kE], cf[kP][kE + 1], red[4];
    if (!need[blockIdx.y]) return;
    const RefBlock b = R.blk[list[blockIdx.y]];
    const int d = b.d, t = threadIdx.x, lane = t & 63, w = t >> 6, q = t & 15, r = t >> 4;
    if ((int)blockIdx.x * 16 >= d) return;
    const Area W(R.tri_work, b);
    double* S = W.S;
    const double tnorm = big_norm(W, d);
    if (!(tnorm > 0.0)) return;
    for (int i = t; i < d; i += kNT) lam[i] = W.lam[i];
    __syncthreads();
    // (every branch and loop bound below is the same for the whole workgroup,
    // but for the rows and columns of a thread)
    for (int l0 = blockIdx.x * 16; l0 < min((int)blockIdx.x * 16 + 16, d); l0++) {
        if (tri_linked(lam, l0, tnorm)) continue;
        int l1 = l0;
        while (l1 + 1 < d && tri_linked(lam, l1 + 1, tnorm)) l1++;
        if (l1 == l0) continue;
        for (int p0 = l0; p0 <= l1; p0 += kP) {
            const int pb = min(kP, l1 + 1 - p0);
            for (int pass = 0; pass < 2; pass++) {
                for (int c0 = l0; c0 < p0; c0 += kE) {
                    const int nc = min(kE, p0 - c0);
                    double acc[kP];
#pragma unroll
                    for (int k = 0; k < kP; k++) acc[k] = 0.0;
                    for (int i = w; i < d; i += 4) {
                        const double* row = S + (size_t)i * d;
                        const double y = lane < nc ? row[c0 + lane] : 0.0;
#pragma unroll
                        for (int k = 0; k < kP; k++) acc[k] = fma(y, row[min(p0 + k, d - 1)], acc[k]);
                    }
#pragma unroll
                    for (int k = 0; k < kP; k++) part[w][k][lane] = acc[k];
                    __syncthreads();
                    for (int e = t; e < kP * kE; e += kNT) {
                        const int k = e / kE, c = e % kE;
                        const double s = (part[0][k][c] + part[1][k][c]) + (part[2][k][c] + part[3][k][c]);
                        cf[k][c] = c < nc ? s / W.xs[c0 + c] : 0.0;
                    }
                    __syncthreads();
                    if (q < pb)
                        for (int i = r; i < d; i += kNT / 16) {
                            double* row = S + (size_t)i * d;
                            double v = row[p0 + q];
                            for (int c = 0; c < nc; c++) v = fma(-cf[q][c], row[c0 + c], v);
                            row[p0 + q] = v;
                        }
                    __syncthreads();
                }
                for (int k = 0; k < pb; k++) {  // column k of the panel against those before it
                    if (k > 0) {
                        double s = 0.0;
                        if (q < k)
                            for (int i = r; i < d; i += kNT / 16)
                                s = fma(S[(size_t)i * d + p0 + q], S[(size_t)i * d + p0 + k], s);
                        part[0][q][r] = s;
                        __syncthreads();
                        if (t < k) {
                            s = 0.0;
                            for (int e = 0; e < kNT / 16; e++) s += part[0][t][e];
                            cf[0][t] = s / W.xs[p0 + t];
                        }
                        __syncthreads();
                    }
                    double s2 = 0.0;
                    for (int i = t; i < d; i += kNT) {
                        double* row = S + (size_t)i * d + p0;
                        double v = row[k];
                        for (int c = 0; c < k; c++) v = fma(-cf[0][c], row[c], v);
                        row[k] = v;
                        s2 = fma(v, v, s2);
                    }
                    s2 = wg_sum(s2, red);
                    if (t == 0) {
                        const bool bad = !(s2 > 0.0) || !isfinite(s2);
                        W.xs[p0 + k] = bad ? INFINITY : s2;  // INFINITY drops the vector
                        if (bad) atomicOr(&B.st[b.inst].status, (int)kStatusJacobiNotConverged);
                    }
                    __syncthreads();
                }
            }
        }
    }
}

// Triangular factor of H_kc .. H_kc+15 = I - Y T Y^T (dlarft forward order), one
// workgroup per 16 reflectors; to plane 0 of the factors, 256 values each.
__global__ __launch_bounds__(kNT) void k_big_wy(RefDev R, const int* list, const int* need) {
    __shared__ double Y[kNB][kNT + 1], gram[kNB][kNB], Tm[kNB][kNB], tau[kNB];
    if (!need[blockIdx.y]) return;
    const RefBlock b = R.blk[list[blockIdx.y]];
    const int d = b.d, t = threadIdx.x, kc = blockIdx.x * kNB, nref = d - 2;
    if (kc >= nref) return;
    const Area W(R.tri_work, b);
    const int nb = min(kNB, nref - kc), a = t / kNB, c = t - a * kNB;
    if (t < kNB) tau[t] = t < nb ? W.hv[(size_t)(kc + t) * d + kc + t] : 0.0;
    double s = 0.0;
    for (int i0 = kc + 1; i0 < d; i0 += kNT) {
        __syncthreads();
        for (int j = 0; j < kNB; j++) {
            const int i = i0 + t;
            Y[j][t] = (j < nb && i < d && i > kc + j) ? W.hv[(size_t)(kc + j) * d + i] : 0.0;
        }
        __syncthreads();
        const int n = min(kNT, d - i0);
        if (a < c)
            for (int i = 0; i < n; i++) s = fma(Y[a][i], Y[c][i], s);
    }
    gram[a][c] = s;
    Tm[a][c] = 0.0;
    __syncthreads();
    for (int i = 0; i < kNB; i++) {
        if (t < i) {
            double q = 0.0;
            for (int e = t; e < i; e++) q = fma(Tm[t][e], gram[e][i], q);
            Tm[t][i] = -tau[i] * q;
        }
        if (t == i) Tm[i][i] = tau[i];
        __syncthreads();
    }
    W.fac[(size_t)blockIdx.x * kNB * kNB + t] = Tm[a][c];
}

// V = Q S with normalised columns, 64 columns per workgroup: the compact-WY
// products from the last reflectors to the first; the rows of a column are
// dealt to the four wavefronts.
__global__ __launch_bounds__(kNT) void k_big_form_v(RefDev R, const int* list, const int* need) {
    __shared__ double Y[kNB][64 + 1], Tm[kNB][kNB], part[4][kNB][64];
    if (!need[blockIdx.y]) return;
    const int bi = list[blockIdx.y];
    const RefBlock b = R.blk[bi];
    const int d = b.d, t = threadIdx.x, lane = t & 63, w = t >> 6, col = blockIdx.x * 64 + lane;
    if ((int)blockIdx.x * 64 >= d) return;
    const Area W(R.tri_work, b);
    double* V = R.work + b.w + (size_t)kSlotV * d * d;
    const bool in = col < d;
    const double x2 = in ? W.xs[col] : 1.0, inv = x2 > 0.0 ? 1.0 / sqrt(x2) : 0.0;
    if (in)
        for (int i = w; i < d; i += 4) V[(size_t)i * d + col] = W.S[(size_t)i * d + col] * inv;
    const int nref = d - 2;
    for (int kc = ((nref - 1) / kNB) * kNB; kc >= 0; kc -= kNB) {
        const int nb = min(kNB, nref - kc);
        double wv[kNB];
#pragma unroll
        for (int j = 0; j < kNB; j++) wv[j] = 0.0;
        // wavefront w takes the rows i0 + 16 w .. + 15 of each chunk of 64
        auto stage = [&](int i0) {
            __syncthreads();
            for (int e = t; e < kNB * 64; e += kNT) {
                const int j = e >> 6, i = i0 + (e & 63);
                Y[j][e & 63] = (j < nb && i < d && i > kc + j) ? W.hv[(size_t)(kc + j) * d + i] : 0.0;
            }
            __syncthreads();
        };
        if (t < kNB * kNB) Tm[t / kNB][t % kNB] = W.fac[(size_t)(kc / kNB) * kNB * kNB + t];
        for (int i0 = kc + 1; i0 < d; i0 += 64) {
            stage(i0);
            if (in)
                for (int u = 0; u < 16; u++) {
                    const int r = 16 * w + u, i = i0 + r;
                    if (i >= d) break;
                    const double m = V[(size_t)i * d + col];
#pragma unroll
                    for (int j = 0; j < kNB; j++) wv[j] = fma(Y[j][r], m, wv[j]);
                }
        }
#pragma unroll
        for (int j = 0; j < kNB; j++) part[w][j][lane] = wv[j];
        __syncthreads();
        double w2[kNB];
#pragma unroll
        for (int j = 0; j < kNB; j++)
            wv[j] = (part[0][j][lane] + part[1][j][lane]) + (part[2][j][lane] + part[3][j][lane]);
#pragma unroll
        for (int a = 0; a < kNB; a++) {
            double s = 0.0;
#pragma unroll
            for (int c = 0; c < kNB; c++) s = fma(Tm[a][c], wv[c], s);
            w2[a] = s;
        }
        for (int i0 = kc + 1; i0 < d; i0 += 64) {
            stage(i0);
            if (in)
                for (int u = 0; u < 16; u++) {
                    const int r = 16 * w + u, i = i0 + r;
                    if (i >= d) break;
                    double m = V[(size_t)i * d + col];
#pragma unroll
                    for (int j = 0; j < kNB; j++) m = fma(-Y[j][r], w2[j], m);
                    V[(size_t)i * d + col] = m;
                }
        }
        __syncthreads();  // the next product's rows may be another wavefront's
    }
    if (blockIdx.x == 0 && t == 0) {
        RefState& rs = R.rs[bi];
        rs.vvalid = 1;
        rs.phase = kPhaseFresh;
        rs.xfinal = kSlotV;
        rs.coupled = 0;
    }
}

}  // namespace

void launch_big_need(const BatchDev& B, const RefDev& R, const int* list, int n, bool refined, int* need,
                     hipStream_t s) {
    hipLaunchKernelGGL(k_big_need, dim3((n + 255) / 256), dim3(256), 0, s, B, R, list, n, refined ? 1 : 0, need);
}

int launch_big_eig(const BatchDev& B, const RefDev& R, const int* list, const int* need, int n, int max_d,
                   hipStream_t s) {
    const int tiles = (max_d + 31) / 32, cols = (max_d + 63) / 64, wy = (max_d - 2 + kNB - 1) / kNB;
    hipLaunchKernelGGL(k_big_load, dim3(tiles, tiles, n), dim3(kNT), 0, s, B, R, list, need);
    // two rows per wavefront; at most 64 workgroups, each of which repeats the vector work
    const int wgs = std::min(64, (max_d + 7) / 8);
    for (int k = 0; k <= max_d - 2; k++)
        hipLaunchKernelGGL(k_big_step, dim3(wgs, n), dim3(kNT), 0, s, R, list, need, k);
    hipLaunchKernelGGL(k_big_values, dim3(cols, n), dim3(64), 0, s, B, R, list, need);
    for (int second = 0; second < 2; second++) {
        hipLaunchKernelGGL(k_big_vectors, dim3(cols, n), dim3(64), 0, s, B, R, list, need, second);
        hipLaunchKernelGGL(k_big_ortho, dim3((max_d + 15) / 16, n), dim3(kNT), 0, s, B, R, list, need);
    }
    hipLaunchKernelGGL(k_big_wy, dim3(wy, n), dim3(kNT), 0, s, R, list, need);
    hipLaunchKernelGGL(k_big_form_v, dim3(cols, n), dim3(kNT), 0, s, R, list, need);
    return max_d + 7;
}

}  // namespace v2h
