// orbopt.hip -- device kernels of the v2RDM-CASSCF orbital step.
//
// The step (orbopt_driver.cpp) keeps the density-fitted integrals of the full
// orbital space resident as dense slices B^Q (nq x nfull x nfull).  Every
// contraction is a product of row-major matrices (k_dgemm):
//   gO   (rs|tu), r..u in O          = BO^T BO             (O: core + active)
//   Z    Z[x r][Q] = sum_st d[x r s t] BO[Q][s t]
//   F    F[x][y] = sum_(r,Q) Z[x r][Q] BFO[y][r][Q] + sum_r D[x][r] h[y][occ r]
//   Jd   (pp|tu)                     = Bdiag BO
//   Kd   (ps|pu)                     = BFO[p] BFO[p]^T, batched over p
//   U    exp(K): Taylor terms and squarings
//   B^Q  U^T B^Q U, batched over Q; h the same
// and the per-rotation gradient and exact diagonal Hessian read those
// intermediates (k_oo_grad_hess).  The formulas restate the focas optimiser
// (focas/orbopt_gradient.cc, orbopt_hessian.cc) for every rotation class at
// once through the generalized Fock matrix and the second derivative of the
// energy along one rotation.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <stdexcept>
#include <string>

#include "orbopt.hpp"
#include "wave_ops.hpp"

namespace v2h {

namespace {

constexpr int kT = 64;    // output tile
constexpr int kKc = 16;   // K chunk staged in LDS
#ifndef V2H_DGEMM_MFMA
#define V2H_DGEMM_MFMA 1
#endif
constexpr bool kUseMfma = V2H_DGEMM_MFMA != 0;  // tiled products on the matrix cores

// kc > 0: split K; batch entry bz covers k in [bz kc, min(K, (bz + 1) kc)) and
// writes its partial product to C + bz sC (summed by k_dgemm_slices).
// dg is added on the diagonal of the result (m == n).
template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_dgemm(int M, int N, int K, double alpha, const double* __restrict__ A,
                                               int64_t lda, int64_t sA, const double* __restrict__ B, int64_t ldb,
                                               int64_t sB, double beta, double* __restrict__ C, int64_t ldc,
                                               int64_t sC, int kc, double dg) {
    __shared__ double As[kKc][kT + 1];
    __shared__ double Bs[kKc][kT + 1];
    const int64_t bz = blockIdx.z;
    A += bz * sA;
    B += bz * sB;
    C += bz * sC;
    const int kbeg = kc > 0 ? (int)bz * kc : 0;
    const int kend = kc > 0 ? min(K, kbeg + kc) : K;
    const int m0 = blockIdx.y * kT, n0 = blockIdx.x * kT;
    const int t = threadIdx.x, tx = t & 15, ty = t >> 4;
    double acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[i][j] = 0.0;
    for (int k0 = kbeg; k0 < kend; k0 += kKc) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int idx = t + 256 * e;
            int m, k;
            if (!TA) { m = idx >> 4; k = idx & 15; } else { k = idx >> 6; m = idx & 63; }
            double v = 0.0;
            if (m0 + m < M && k0 + k < kend)
                v = TA ? A[(int64_t)(k0 + k) * lda + (m0 + m)] : A[(int64_t)(m0 + m) * lda + (k0 + k)];
            As[k][m] = v;
            int n, k2;
            if (!TB) { k2 = idx >> 6; n = idx & 63; } else { n = idx >> 4; k2 = idx & 15; }
            double w = 0.0;
            if (n0 + n < N && k0 + k2 < kend)
                w = TB ? B[(int64_t)(n0 + n) * ldb + (k0 + k2)] : B[(int64_t)(k0 + k2) * ldb + (n0 + n)];
            Bs[k2][n] = w;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < kKc; kk++) {
            double a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; i++) a[i] = As[kk][ty + 16 * i];
#pragma unroll
            for (int j = 0; j < 4; j++) b[j] = Bs[kk][tx + 16 * j];
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i][j] = __fma_rn(a[i], b[j], acc[i][j]);
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int m = m0 + ty + 16 * i;
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int n = n0 + tx + 16 * j;
            if (n >= N) continue;
            double* c = C + (int64_t)m * ldc + n;
            double v = beta != 0.0 ? __fma_rn(alpha, acc[i][j], beta * *c) : alpha * acc[i][j];
            if (m == n) v += dg;
            *c = v;
        }
    }
}

// The same product on the FP64 matrix cores: four wavefronts per 64 x 64
// tile, each a 32 x 32 quarter as 2 x 2 MFMA 16 x 16 x 4 tiles, operands read
// from the same LDS staging.  v_mfma_f64_16x16x4f64 lane layout (checked on
// gfx950): lane l supplies A[l % 16][l / 16] and B[l / 16][l % 16] and holds
// D[4 r + l / 16][l % 16] in its register r.
typedef double v4d __attribute__((ext_vector_type(4)));

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_dgemm_mfma(int M, int N, int K, double alpha, const double* __restrict__ A,
                                                    int64_t lda, int64_t sA, const double* __restrict__ B,
                                                    int64_t ldb, int64_t sB, double beta, double* __restrict__ C,
                                                    int64_t ldc, int64_t sC, int kc, double dg) {
    // row strides: 16 mod 32 doubles keep the four k of an operand read on
    // different banks; an operand that is turned on its way in needs an odd one
    __shared__ double As[kKc][TA ? kT + 16 : kT + 1];
    __shared__ double Bs[kKc][TB ? kT + 1 : kT + 16];
    const int64_t bz = blockIdx.z;
    A += bz * sA;
    B += bz * sB;
    C += bz * sC;
    const int kbeg = kc > 0 ? (int)bz * kc : 0;
    const int kend = kc > 0 ? min(K, kbeg + kc) : K;
    const int m0 = blockIdx.y * kT, n0 = blockIdx.x * kT;
    const int t = threadIdx.x, l = t & 63, w = t >> 6;
    const int wm = (w >> 1) * 32, wn = (w & 1) * 32;
    const int li = l & 15, lk = l >> 4;
    v4d acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++) acc[i][j] = v4d{0.0, 0.0, 0.0, 0.0};
    // a chunk's loads go to registers first, so that the next chunk's are in
    // flight during this chunk's products (400 products of 100^3: 58 -> 40 us,
    // the split ones 36 -> 17)
    double ra[4], rb[4];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int idx = t + 256 * e;
            int m, k;
            if (!TA) { m = idx >> 4; k = idx & 15; } else { k = idx >> 6; m = idx & 63; }
            ra[e] = 0.0;
            if (m0 + m < M && k0 + k < kend)
                ra[e] = TA ? A[(int64_t)(k0 + k) * lda + (m0 + m)] : A[(int64_t)(m0 + m) * lda + (k0 + k)];
            int n, k2;
            if (!TB) { k2 = idx >> 6; n = idx & 63; } else { n = idx >> 4; k2 = idx & 15; }
            rb[e] = 0.0;
            if (n0 + n < N && k0 + k2 < kend)
                rb[e] = TB ? B[(int64_t)(n0 + n) * ldb + (k0 + k2)] : B[(int64_t)(k0 + k2) * ldb + (n0 + n)];
        }
    };
    // 16 x 16 parts outside the matrix take no products (100 = 64 + 36: 7 of
    // 8 per side instead of all 8)
    const bool i0 = m0 + wm < M, i1 = m0 + wm + 16 < M, j0 = n0 + wn < N, j1 = n0 + wn + 16 < N;
    if (kbeg < kend) fetch(kbeg);
    for (int k0 = kbeg; k0 < kend; k0 += kKc) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int idx = t + 256 * e;
            if (!TA) As[idx & 15][idx >> 4] = ra[e];
            else As[idx >> 6][idx & 63] = ra[e];
            if (!TB) Bs[idx >> 6][idx & 63] = rb[e];
            else Bs[idx & 15][idx >> 4] = rb[e];
        }
        __syncthreads();
        if (k0 + kKc < kend) fetch(k0 + kKc);
        if (i0 && j0) {  // (uniform in the wavefront, like i1 and j1)
#pragma unroll
            for (int kk = 0; kk < kKc; kk += 4) {
                const double a0 = As[kk + lk][wm + li], a1 = As[kk + lk][wm + 16 + li];
                const double b0 = Bs[kk + lk][wn + li], b1 = Bs[kk + lk][wn + 16 + li];
                acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
                if (j1) acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
                if (i1) acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
                if (i1 && j1) acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int m = m0 + wm + 16 * i + 4 * r + lk, n = n0 + wn + 16 * j + li;
                if (m >= M || n >= N) continue;
                double* c = C + (int64_t)m * ldc + n;
                double v = beta != 0.0 ? __fma_rn(alpha, acc[i][j][r], beta * *c) : alpha * acc[i][j][r];
                if (m == n) v += dg;
                *c = v;
            }
}

// Products with a small result (the chains of 100 x 100 products of the
// exponential, the 10 x 10 results over 400 slices): latency bounds them, so a
// workgroup takes one 16 x 16 tile, its four wavefronts share K, and each lane
// loads its MFMA operands straight from memory, 16 loads in flight; the four
// partial tiles are added in LDS.  A 100 x 100 product: 3.8 us; with the
// whole rows and columns staged in LDS and no matrix instructions 7.3.
constexpr int kSmallMax = 128;

template <bool TA, bool TB>
__global__ __launch_bounds__(256) void k_dgemm_small(int M, int N, int K, double alpha, const double* __restrict__ A,
                                                     int64_t lda, int64_t sA, const double* __restrict__ B,
                                                     int64_t ldb, int64_t sB, double* __restrict__ C, int64_t ldc,
                                                     int64_t sC, SmallPoly poly) {
    constexpr int kU = 8;
    __shared__ double part[4][256];
    const int64_t bz = blockIdx.z;
    const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
    const int t = threadIdx.x, l = t & 63, w = t >> 6, li = l & 15, lk = l >> 4;
    // a row or column outside the matrix repeats the last one (its results are
    // not stored); k outside reads the last one and counts as zero
    const int am = min(m0 + li, M - 1), bn = min(n0 + li, N - 1);
    const double* Ap = A + bz * sA + (TA ? am : am * lda);
    const double* Bp = B + bz * sB + (TB ? bn * ldb : bn);
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 4 * kU * w; k0 < K; k0 += 16 * kU) {
        double a[kU], b[kU];
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const int64_t k = min(k0 + 4 * u + lk, K - 1);
            a[u] = Ap[TA ? k * lda : k];
            b[u] = Bp[TB ? k : k * ldb];
        }
#pragma unroll
        for (int u = 0; u < kU; u++) {
            const bool in = k0 + 4 * u + lk < K;
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(in ? a[u] : 0.0, in ? b[u] : 0.0, acc, 0, 0, 0);
        }
    }
#pragma unroll
    for (int r = 0; r < 4; r++) part[w][(4 * r + lk) * 16 + li] = acc[r];
    __syncthreads();
    const int m = m0 + (t >> 4), n = n0 + (t & 15);
    if (m >= M || n >= N) return;
    const double sum = (part[0][t] + part[1][t]) + (part[2][t] + part[3][t]);
    const int64_t e = (int64_t)m * ldc + n;
    const double diag = m == n ? 1.0 : 0.0;
    const double m1 = poly.M1 ? poly.M1[e] : 0.0, m2 = poly.M2 ? poly.M2[e] : 0.0, m3 = poly.M3 ? poly.M3[e] : 0.0;
    // the identity last: one rounding at its size
    const double v = poly.c[0] * diag + (alpha * sum + (poly.c[1] * m1 + (poly.c[2] * m2 + poly.c[3] * m3)));
    C[bz * sC + e] = v;
    if (poly.Q) poly.Q[e] = poly.q[0] * diag + (poly.q[1] * m1 + (poly.q[2] * m2 + poly.q[3] * v));
}

// C[m][n] = alpha sum_s W[s][m][n] + beta C[m][n], slices summed in order
__global__ __launch_bounds__(256) void k_dgemm_slices(const double* __restrict__ W, int slices, int M, int N,
                                                      double alpha, double beta, double* __restrict__ C, int64_t ldc) {
    const int64_t mn = (int64_t)M * N;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < mn; e += (int64_t)gridDim.x * blockDim.x) {
        double s = 0.0;
#pragma unroll 8
        for (int k = 0; k < slices; k++) s += W[k * mn + e];
        const int m = (int)(e / N), n = (int)(e - (int64_t)m * N);
        double* c = C + (int64_t)m * ldc + n;
        *c = beta != 0.0 ? __fma_rn(alpha, s, beta * *c) : alpha * s;
    }
}

// Packed triangle <-> square, a row of a slice per wavefront (no divisions by
// runtime sizes per element; at 100 orbitals and 400 slices, 48 MB: pack
// 11.7 -> 7.9 us, unpack 21 -> 17.5, the upper half's strided reads).
__global__ __launch_bounds__(256) void k_df_unpack(const double* __restrict__ qmo, int nq, int nfull,
                                                   double* __restrict__ bd) {
    const int64_t nn = (int64_t)nfull * nfull, ntri = (int64_t)nfull * (nfull + 1) / 2;
    for (int Q = blockIdx.y; Q < nq; Q += gridDim.y) {
        const double* in = qmo + Q * ntri;
        for (int p = blockIdx.x * 4 + threadIdx.y; p < nfull; p += gridDim.x * 4) {
            const int64_t row = (int64_t)p * (p + 1) / 2;
            double* out = bd + Q * nn + (int64_t)p * nfull;
            for (int q = threadIdx.x; q < nfull; q += 64)
                out[q] = in[p >= q ? row + q : (int64_t)q * (q + 1) / 2 + p];
        }
    }
}

__global__ __launch_bounds__(256) void k_df_pack(const double* __restrict__ bd, int nq, int nfull,
                                                 double* __restrict__ qmo) {
    const int64_t nn = (int64_t)nfull * nfull, ntri = (int64_t)nfull * (nfull + 1) / 2;
    for (int Q = blockIdx.y; Q < nq; Q += gridDim.y) {
        for (int p = blockIdx.x * 4 + threadIdx.y; p < nfull; p += gridDim.x * 4) {
            const double* in = bd + Q * nn + (int64_t)p * nfull;
            double* out = qmo + Q * ntri + (int64_t)p * (p + 1) / 2;
            for (int q = threadIdx.x; q <= p; q += 64) out[q] = in[q];
        }
    }
}

// spin-free D of two active (Pitzer) orbitals
__device__ double oo_d1(const OoTables& t, const double* x, int i, int j) {
    const int64_t o = t.d1[i * t.n + j];
    return o < 0 ? 0.0 : x[o] + x[t.d1[t.n * t.n + i * t.n + j]];
}

__device__ double oo_ab(const OoTables& t, const double* x, int i, int j, int k, int l) {
    const int4 a = t.pair[i * t.n + j], b = t.pair[k * t.n + l];
    if (a.x != b.x) return 0.0;
    return x[t.offab[a.x] + (int64_t)a.y * t.gab[a.x] + b.y];
}

__device__ double oo_aa(const OoTables& t, const double* x, int i, int j, int k, int l) {
    const int4 a = t.pair[i * t.n + j], b = t.pair[k * t.n + l];
    if (a.z < 0 || b.z < 0 || a.x != b.x) return 0.0;
    const int64_t e = (int64_t)a.z * t.gaa[a.x] + b.z;
    return (double)(a.w * b.w) * (x[t.offaa[a.x] + e] + x[t.offbb[a.x] + e]);
}

// d_pqrs = sum <a+_p a+_r a_s a_q> over O positions (core first, then active)
__device__ double oo_raw_d(const OoTables& t, const double* x, int p, int q, int r, int s) {
    const int nc = t.ncore;
    const bool cp = p < nc, cq = q < nc, cr = r < nc, cs = s < nc;
    const int ncnt = (int)cp + (int)cq + (int)cr + (int)cs;
    if (ncnt == 0) {
        p -= nc; q -= nc; r -= nc; s -= nc;
        return oo_ab(t, x, p, r, q, s) + oo_ab(t, x, r, p, s, q) + oo_aa(t, x, p, r, q, s);
    }
    if (ncnt == 4) return 4.0 * (p == q && r == s) - 2.0 * (p == s && q == r);
    if (ncnt != 2) return 0.0;
    if (cp && cq) return p == q ? 2.0 * oo_d1(t, x, r - nc, s - nc) : 0.0;
    if (cr && cs) return r == s ? 2.0 * oo_d1(t, x, p - nc, q - nc) : 0.0;
    if (cp && cs) return p == s ? -oo_d1(t, x, q - nc, r - nc) : 0.0;
    if (cq && cr) return q == r ? -oo_d1(t, x, p - nc, s - nc) : 0.0;
    return 0.0;
}

__global__ __launch_bounds__(256) void k_oo_density(OoTables t, const double* __restrict__ x, double* __restrict__ D,
                                                    double* __restrict__ d) {
    const int no = t.no;
    const int64_t n2 = (int64_t)no * no, n4 = n2 * n2;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n4 + n2; e += (int64_t)gridDim.x * blockDim.x) {
        if (e >= n4) {
            const int64_t f = e - n4;
            const int a = (int)(f / no), b = (int)(f - (int64_t)a * no);
            double v;
            if (a < t.ncore || b < t.ncore) v = (a == b) ? 2.0 : 0.0;
            else v = oo_d1(t, x, a - t.ncore, b - t.ncore);
            if ((a < t.ncore) != (b < t.ncore)) v = 0.0;
            D[f] = v;
            continue;
        }
        const int p = (int)(e / (n2 * no));
        const int q = (int)((e / n2) % no);
        const int r = (int)((e / no) % no);
        const int s = (int)(e % no);
        d[e] = 0.25 * (oo_raw_d(t, x, p, q, r, s) + oo_raw_d(t, x, q, p, r, s) + oo_raw_d(t, x, p, q, s, r) +
                       oo_raw_d(t, x, q, p, s, r));
    }
}

// One row p of 64 slices per workgroup: read with the lanes along the row (the
// occupied orbitals of an irrep are neighbours there), turned in LDS, written
// with the lanes along Q (lanes along Q on both sides took
// 20.8 us at 100 orbitals, 26 of them occupied, 400 slices; this 12).
__global__ __launch_bounds__(256) void k_oo_gather(const double* __restrict__ bd, int nq, int nfull,
                                                   const int* __restrict__ occ, int no, const int* __restrict__ pos,
                                                   double* __restrict__ BO, double* __restrict__ BFO,
                                                   double* __restrict__ Bdiag) {
    __shared__ double tile[16][65];
    const int64_t nn = (int64_t)nfull * nfull;
    const int t = threadIdx.x, p = blockIdx.x, po = pos[p];
    for (int q0 = blockIdx.y * 64; q0 < nq; q0 += gridDim.y * 64) {
        const int m = min(64, nq - q0);
        const double* row = bd + q0 * nn + (int64_t)p * nfull;
        if (t < m) Bdiag[(int64_t)p * nq + q0 + t] = row[t * nn + p];
        for (int r0 = 0; r0 < no; r0 += 16) {
            const int r = t & 15;
            if (r0 + r < no) {
                const int col = occ[r0 + r];
                for (int Q = t >> 4; Q < m; Q += 16) {
                    const double v = row[Q * nn + col];
                    tile[r][Q] = v;
                    if (po >= 0) BO[((int64_t)(q0 + Q) * no + po) * no + r0 + r] = v;
                }
            }
            __syncthreads();
            const int Q = t & 63;
            if (Q < m)
                for (int r2 = t >> 6; r2 < 16 && r0 + r2 < no; r2 += 4)
                    BFO[((int64_t)p * no + r0 + r2) * nq + q0 + Q] = tile[r2][Q];
            __syncthreads();
        }
    }
}

__global__ __launch_bounds__(256) void k_oo_fock1(const double* __restrict__ D, const double* __restrict__ h,
                                                  const int* __restrict__ occ, int no, int nfull, double* __restrict__ F) {
    const int64_t total = (int64_t)no * nfull;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < total; e += (int64_t)gridDim.x * blockDim.x) {
        const int xo = (int)(e / nfull), y = (int)(e - (int64_t)xo * nfull);
        double acc = 0.0;
        for (int r = 0; r < no; r++) acc = __fma_rn(D[xo * no + r], h[(int64_t)y * nfull + occ[r]], acc);
        F[e] += acc;
    }
}

// One workgroup per rotation pair: its threads split the O^2 sums, combined in
// a fixed order (573 pairs with 26^2 terms: 9.5 us; 24 with a
// wavefront per pair).
__global__ __launch_bounds__(256) void k_oo_grad_hess(OoGradArgs a) {
    __shared__ double part[4][4];
    const int k = blockIdx.x, t = threadIdx.x;
    const int p = a.pairs[k].x, q = a.pairs[k].y;
    const int no = a.no, nf = a.nfull;
    const int n2 = no * no;
    const int ip = a.pos[p], iq = a.pos[q];
    const double* Jp = a.Jd + (int64_t)p * n2;
    const double* Jq = a.Jd + (int64_t)q * n2;
    const double* Kp = a.Kd + (int64_t)p * n2;
    const double* Kq = a.Kd + (int64_t)q * n2;
    const int64_t no3 = (int64_t)n2 * no;
    // (asked for before the sums, so that they arrive under them)
    const double Fpq = ip >= 0 ? a.F[(int64_t)ip * nf + q] : 0.0;
    const double Fqp = iq >= 0 ? a.F[(int64_t)iq * nf + p] : 0.0;
    const double Fpp = ip >= 0 ? a.F[(int64_t)ip * nf + p] : 0.0;
    const double Fqq = iq >= 0 ? a.F[(int64_t)iq * nf + q] : 0.0;
    const double Dpp = ip >= 0 ? a.D[ip * no + ip] : 0.0;
    const double Dqq = iq >= 0 ? a.D[iq * no + iq] : 0.0;
    const double Dpq = (ip >= 0 && iq >= 0) ? a.D[ip * no + iq] : 0.0;
    const double hpp = a.h[(int64_t)p * nf + p], hqq = a.h[(int64_t)q * nf + q], hpq = a.h[(int64_t)p * nf + q];
    double g12 = 0.0, g13 = 0.0, c12 = 0.0, c13 = 0.0;
    for (int e = t; e < n2; e += 256) {
        const int s = e / no, u = e - s * no;
        if (ip >= 0) {
            g12 = __fma_rn(a.d[((int64_t)ip * no + ip) * n2 + e], Jq[e], g12);
            g13 = __fma_rn(a.d[ip * no3 + (int64_t)s * n2 + (int64_t)ip * no + u], Kq[e], g13);
        }
        if (iq >= 0) {
            g12 = __fma_rn(a.d[((int64_t)iq * no + iq) * n2 + e], Jp[e], g12);
            g13 = __fma_rn(a.d[iq * no3 + (int64_t)s * n2 + (int64_t)iq * no + u], Kp[e], g13);
        }
        if (ip >= 0 && iq >= 0) {
            const int64_t row = ((int64_t)ip * no + iq) * n2;
            c12 = __fma_rn(a.d[row + e], a.gO[row + e], c12);
            c13 = __fma_rn(a.d[ip * no3 + (int64_t)s * n2 + (int64_t)iq * no + u],
                           a.gO[iq * no3 + (int64_t)s * n2 + (int64_t)ip * no + u], c13);
        }
    }
    g12 = wsum(g12);
    g13 = wsum(g13);
    c12 = wsum(c12);
    c13 = wsum(c13);
    if ((t & 63) == 0) {
        part[t >> 6][0] = g12;
        part[t >> 6][1] = g13;
        part[t >> 6][2] = c12;
        part[t >> 6][3] = c13;
    }
    __syncthreads();
    if (t != 0) return;
    auto total = [&](int i) { return (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]); };
    a.g[k] = 2.0 * (Fqp - Fpq);
    const double val = -2.0 * (Fpp + Fqq) + 2.0 * (Dpp * hqq + Dqq * hpp - 2.0 * Dpq * hpq);
    a.H[k] = val + 2.0 * (total(0) - 2.0 * total(2)) + 4.0 * (total(1) - 2.0 * total(3));
}

constexpr int kRed = 1024;

__device__ void block_sum2(double& a, double& b, double* sa, double* sb) {
    const int t = threadIdx.x;
    sa[t] = a;
    sb[t] = b;
    __syncthreads();
    for (int w = kRed / 2; w > 0; w >>= 1) {
        if (t < w) {
            sa[t] += sa[t + w];
            sb[t] += sb[t + w];
        }
        __syncthreads();
    }
    a = sa[0];
    b = sb[0];
}

__global__ __launch_bounds__(kRed) void k_oo_precondition(const double* __restrict__ g, const double* __restrict__ H,
                                                          int nrot, double r, double* __restrict__ kref,
                                                          double* __restrict__ kcur, double* __restrict__ ksave,
                                                          double* __restrict__ out) {
    __shared__ double sa[kRed], sb[kRed];
    double gg = 0.0, quad = 0.0;
    for (int k = threadIdx.x; k < nrot; k += kRed) {
        const double gk = g[k], hk = H[k], ck = kcur[k];
        gg = __fma_rn(gk, gk, gg);
        quad += gk * ck + 0.5 * ck * hk * ck;
        double hv = hk < 0.0 ? -hk : hk;
        if (hv < 1.0e-2) hv = 1.0e-2;
        const double kr = -gk / hv;
        kref[k] = kr;
        kcur[k] = r * kr;
        ksave[k] = r * kr;
    }
    block_sum2(gg, quad, sa, sb);
    if (threadIdx.x == 0) {
        out[0] = gg;
        out[1] = quad;
    }
}

__global__ __launch_bounds__(256) void k_oo_update_kappa(const double* __restrict__ kref, int nrot, double r,
                                                         double* __restrict__ kcur, double* __restrict__ ksave) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nrot) return;
    const double kn = r * kref[k] - kcur[k];
    kcur[k] = kn;
    ksave[k] += kn;
}

__global__ __launch_bounds__(256) void k_oo_fill(double* __restrict__ p, int64_t n, double v) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) p[e] = v;
}

__global__ __launch_bounds__(256) void k_oo_scatter_kappa(const double* __restrict__ kappa, const int2* __restrict__ pairs,
                                                          int nrot, double scale, int nfull, double* __restrict__ K) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= nrot) return;
    const int p = pairs[k].x, q = pairs[k].y;
    const double v = scale * kappa[k];
    K[(int64_t)p * nfull + q] = v;
    K[(int64_t)q * nfull + p] = -v;
}

// out[0] = ||K||_1 in one workgroup: eight threads share a column, with four
// partial sums each (5.6 us at 100
// orbitals, 24.6 with one thread per column).
__global__ __launch_bounds__(1024) void k_oo_norm1(const double* __restrict__ K, int nfull, double* __restrict__ out) {
    __shared__ double part[8][128];
    const int c = threadIdx.x & 127, g = threadIdx.x >> 7;
    double mx = 0.0;
    for (int j0 = 0; j0 < nfull; j0 += 128) {
        const int j = j0 + c;
        double s[4] = {0.0, 0.0, 0.0, 0.0};
        if (j < nfull)
            for (int i = g; i < nfull; i += 32)
#pragma unroll
                for (int u = 0; u < 4; u++)
                    if (i + 8 * u < nfull) s[u] += fabs(K[(int64_t)(i + 8 * u) * nfull + j]);
        part[g][c] = (s[0] + s[1]) + (s[2] + s[3]);
        __syncthreads();
        if (g == 0) {
            double sum = 0.0;
#pragma unroll
            for (int q = 0; q < 8; q++) sum += part[q][c];
            mx = sum > mx ? sum : mx;
        }
        __syncthreads();
    }
    if (g == 0) part[0][c] = mx;
    __syncthreads();
    for (int w = 64; w > 0; w >>= 1) {
        if (threadIdx.x < w) part[0][c] = fmax(part[0][c], part[0][c + w]);
        __syncthreads();
    }
    if (threadIdx.x == 0) out[0] = part[0][0];
}

__global__ __launch_bounds__(256) void k_oo_identity(double* __restrict__ U, int nfull) {
    const int64_t n = (int64_t)nfull * nfull;
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
        U[e] = (e / nfull == e % nfull) ? 1.0 : 0.0;
}

__global__ __launch_bounds__(256) void k_oo_axpy(double a, const double* x, double* y, int64_t n) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
        y[e] = __fma_rn(a, x[e], y[e]);
}

__global__ __launch_bounds__(256) void k_oo_sub(const double* __restrict__ x, const double* __restrict__ z,
                                                double* __restrict__ y, int64_t n) {
    for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x)
        y[e] = x[e] - z[e];
}

unsigned grid_for(int64_t n) {
    const int64_t b = (n + 255) / 256;
    return (unsigned)(b < 1 ? 1 : (b > 65536 ? 65536 : b));
}

}  // namespace

namespace {

void dgemm_raw(bool ta, bool tb, int M, int N, int K, double alpha, const double* A, int64_t lda, int64_t sA,
               const double* B, int64_t ldb, int64_t sB, double beta, double* C, int64_t ldc, int64_t sC, int batch,
               int kc, double dg, hipStream_t s) {
    if (M <= 0 || N <= 0 || batch <= 0) return;
    const int64_t gy = (M + kT - 1) / kT, gx = (N + kT - 1) / kT;
    if (gy > 65535 || batch > 65535 || gx > (int64_t)1 << 30)
        throw std::invalid_argument("launch_dgemm: shape " + std::to_string(M) + " x " + std::to_string(N) +
                                    " x batch " + std::to_string(batch) + " exceeds the grid");
    const dim3 grid((unsigned)gx, (unsigned)gy, (unsigned)batch);
    if (kUseMfma) {
        if (!ta && !tb) hipLaunchKernelGGL((k_dgemm_mfma<false, false>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, kc, dg);
        else if (ta && !tb) hipLaunchKernelGGL((k_dgemm_mfma<true, false>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, kc, dg);
        else if (!ta && tb) hipLaunchKernelGGL((k_dgemm_mfma<false, true>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, kc, dg);
        else hipLaunchKernelGGL((k_dgemm_mfma<true, true>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, kc, dg);
        return;
    }
    if (!ta && !tb) hipLaunchKernelGGL((k_dgemm<false, false>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, kc, dg);
    else if (ta && !tb) hipLaunchKernelGGL((k_dgemm<true, false>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, kc, dg);
    else if (!ta && tb) hipLaunchKernelGGL((k_dgemm<false, true>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, kc, dg);
    else hipLaunchKernelGGL((k_dgemm<true, true>), grid, dim3(256), 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, kc, dg);
}

void small_raw(bool ta, bool tb, int M, int N, int K, double alpha, const double* A, int64_t lda, int64_t sA,
               const double* B, int64_t ldb, int64_t sB, double* C, int64_t ldc, int64_t sC, int batch,
               const SmallPoly& p, hipStream_t s) {
    if (batch <= 0) return;
    const dim3 grid((unsigned)((N + 15) / 16), (unsigned)((M + 15) / 16), (unsigned)batch), block(256);
#define V2H_SMALL(TA, TB) \
    hipLaunchKernelGGL((k_dgemm_small<TA, TB>), grid, block, 0, s, M, N, K, alpha, A, lda, sA, B, ldb, sB, C, ldc, sC, p)
    if (ta) {
        if (tb) V2H_SMALL(true, true);
        else V2H_SMALL(true, false);
    } else {
        if (tb) V2H_SMALL(false, true);
        else V2H_SMALL(false, false);
    }
#undef V2H_SMALL
}

}  // namespace

void launch_dgemm(bool ta, bool tb, int M, int N, int K, double alpha, const double* A, int64_t lda, int64_t sA,
                  const double* B, int64_t ldb, int64_t sB, double beta, double* C, int64_t ldc, int64_t sC,
                  int batch, hipStream_t s, double dg) {
    // up to four tiles of the small kernel in a 64 x 64 tile's place (100 results of 26 x 26 over
    // K = 400: 14.5 us, 28 in the 64 x 64 tile)
    if (M > 0 && N > 0 && M <= 32 && N <= 32 && K > 0 && beta == 0.0 && batch <= 65535) {
        SmallPoly poly{};
        poly.c[0] = dg;
        small_raw(ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, C, ldc, sC, batch, poly, s);
        return;
    }
    dgemm_raw(ta, tb, M, N, K, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc, sC, batch, 0, dg, s);
}

int dgemm_split_slices(int M, int N, int K) {
    const int64_t tiles = (int64_t)((M + kT - 1) / kT) * ((N + kT - 1) / kT);
    int sl = (int)std::min<int64_t>(kMaxSlices, std::max<int64_t>(1, 512 / std::max<int64_t>(1, tiles)));
    sl = std::min(sl, std::max(1, K / 64));
    return sl;
}

void launch_dgemm_small(bool ta, int M, int N, int K, double alpha, const double* A, int64_t lda, const double* B,
                        int64_t ldb, double* C, int64_t ldc, hipStream_t s, double dg) {
    if (M <= 0 || N <= 0) return;
    if (M > kSmallMax || N > kSmallMax || K > kSmallMax || K < 1) {
        launch_dgemm(ta, false, M, N, K, alpha, A, lda, 0, B, ldb, 0, 0.0, C, ldc, 0, 1, s, dg);
        return;
    }
    SmallPoly poly{};
    poly.c[0] = dg;
    small_raw(ta, false, M, N, K, alpha, A, lda, 0, B, ldb, 0, C, ldc, 0, 1, poly, s);
}

double* launch_oo_exp_taylor(int n, const double* K, double* W, double* U, double* T, hipStream_t s) {
    if (n > kSmallMax) {
        // degree 14 by Horner's rule, T <- I + K T / k for k = 14 .. 1
        launch_oo_identity(U, n, s);
        for (int k = 14; k >= 1; k--) {
            launch_dgemm_small(false, n, n, n, 1.0 / k, K, n, U, n, T, n, s, 1.0);
            std::swap(U, T);
        }
        return U;
    }
    // degree 15 as a cubic in K^4 whose coefficients are cubics in K (Paterson
    // and Stockmeyer): six products of about 4 us each, which latency bounds,
    // instead of fourteen; its error is no larger (the identity is added last)
    const int64_t nn = (int64_t)n * n;
    double *K2 = W, *K3 = W + nn, *K4 = W + 2 * nn;
    double c[16] = {1.0};
    for (int k = 1; k < 16; k++) c[k] = c[k - 1] / k;
    auto mul = [&](const double* A, const double* B, double* C, const SmallPoly& p) {
        small_raw(false, false, n, n, n, 1.0, A, n, 0, B, n, 0, C, n, 0, 1, p, s);
    };
    mul(K, K, K2, SmallPoly{});
    SmallPoly p{};
    p.M1 = K;
    p.M2 = K2;
    p.Q = U;
    for (int i = 0; i < 4; i++) p.q[i] = c[12 + i];
    mul(K2, K, K3, p);
    mul(K2, K2, K4, SmallPoly{});
    p.Q = nullptr;
    p.M3 = K3;
    for (int j = 2; j >= 0; j--) {
        for (int i = 0; i < 4; i++) p.c[i] = c[4 * j + i];
        mul(K4, U, T, p);
        std::swap(U, T);
    }
    return U;
}

void launch_dgemm_split(bool ta, bool tb, int M, int N, int K, double alpha, const double* A, int64_t lda,
                        const double* B, int64_t ldb, double beta, double* C, int64_t ldc, double* work,
                        hipStream_t s) {
    const int sl = dgemm_split_slices(M, N, K);
    if (sl <= 1) {
        dgemm_raw(ta, tb, M, N, K, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1, 0, 0.0, s);
        return;
    }
    const int kc = ((K + sl - 1) / sl + kKc - 1) / kKc * kKc;
    const int slices = (K + kc - 1) / kc;
    dgemm_raw(ta, tb, M, N, K, 1.0, A, lda, 0, B, ldb, 0, 0.0, work, N, (int64_t)M * N, slices, kc, 0.0, s);
    const int64_t mn = (int64_t)M * N;
    hipLaunchKernelGGL(k_dgemm_slices, dim3(grid_for(mn)), dim3(256), 0, s, work, slices, M, N, alpha, beta, C, ldc);
}

namespace {
dim3 slice_grid(int nq, int nfull) {
    return dim3((unsigned)std::min(1024, (nfull + 3) / 4), (unsigned)std::min(nq, 65535));
}
}  // namespace

void launch_df_unpack(const double* qmo, int nq, int nfull, double* bd, hipStream_t s) {
    hipLaunchKernelGGL(k_df_unpack, slice_grid(nq, nfull), dim3(64, 4), 0, s, qmo, nq, nfull, bd);
}

void launch_df_pack(const double* bd, int nq, int nfull, double* qmo, hipStream_t s) {
    hipLaunchKernelGGL(k_df_pack, slice_grid(nq, nfull), dim3(64, 4), 0, s, bd, nq, nfull, qmo);
}

void launch_oo_density(const OoTables& t, const double* x, double* D, double* d, hipStream_t s) {
    const int64_t n2 = (int64_t)t.no * t.no;
    hipLaunchKernelGGL(k_oo_density, dim3(grid_for(n2 * n2 + n2)), dim3(256), 0, s, t, x, D, d);
}

void launch_oo_gather(const double* bd, int nq, int nfull, const int* occ, int no, const int* pos, double* BO,
                      double* BFO, double* Bdiag, hipStream_t s) {
    const dim3 grid((unsigned)nfull, (unsigned)std::min((nq + 63) / 64, 65535));
    hipLaunchKernelGGL(k_oo_gather, grid, dim3(256), 0, s, bd, nq, nfull, occ, no, pos, BO, BFO, Bdiag);
}

void launch_oo_fock1(const double* D, const double* h, const int* occ, int no, int nfull, double* F, hipStream_t s) {
    hipLaunchKernelGGL(k_oo_fock1, dim3(grid_for((int64_t)no * nfull)), dim3(256), 0, s, D, h, occ, no, nfull, F);
}

void launch_oo_grad_hess(const OoGradArgs& a, hipStream_t s) {
    if (a.nrot <= 0) return;
    hipLaunchKernelGGL(k_oo_grad_hess, dim3(a.nrot), dim3(256), 0, s, a);
}

void launch_oo_precondition(const double* g, const double* H, int nrot, double r, double* kref, double* kcur,
                            double* ksave, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_oo_precondition, dim3(1), dim3(kRed), 0, s, g, H, nrot, r, kref, kcur, ksave, out);
}

void launch_oo_update_kappa(const double* kref, int nrot, double r, double* kcur, double* ksave, hipStream_t s) {
    if (nrot <= 0) return;
    hipLaunchKernelGGL(k_oo_update_kappa, dim3((nrot + 255) / 256), dim3(256), 0, s, kref, nrot, r, kcur, ksave);
}

void launch_oo_kappa_matrix(const double* kappa, const int2* pairs, int nrot, double scale, int nfull, double* K,
                            double* out, hipStream_t s) {
    const int64_t nn = (int64_t)nfull * nfull;
    hipLaunchKernelGGL(k_oo_fill, dim3(grid_for(nn)), dim3(256), 0, s, K, nn, 0.0);
    if (nrot > 0)
        hipLaunchKernelGGL(k_oo_scatter_kappa, dim3((nrot + 255) / 256), dim3(256), 0, s, kappa, pairs, nrot, scale,
                           nfull, K);
    hipLaunchKernelGGL(k_oo_norm1, dim3(1), dim3(1024), 0, s, K, nfull, out);
}

void launch_oo_identity(double* U, int nfull, hipStream_t s) {
    hipLaunchKernelGGL(k_oo_identity, dim3(grid_for((int64_t)nfull * nfull)), dim3(256), 0, s, U, nfull);
}

void launch_oo_axpy(double a, const double* x, double* y, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_oo_axpy, dim3(grid_for(n)), dim3(256), 0, s, a, x, y, n);
}

void launch_oo_sub(const double* x, const double* z, double* y, int64_t n, hipStream_t s) {
    hipLaunchKernelGGL(k_oo_sub, dim3(grid_for(n)), dim3(256), 0, s, x, z, y, n);
}

}  // namespace v2h
