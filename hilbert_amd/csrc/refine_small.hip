// refine_small.hip -- the warm-started PSD projection of the blocks of up to
// 64 rows: one launch does the whole refinement of a block (see refine.hpp)
// inside one workgroup (17..64 rows) or one wavefront (up to 16 rows).
//
// A block of this size has too little work for the tile launches of
// refine.hip: its five products are 10 d^3 flops, 2.6 MFLOP at d = 64, 8.5 us
// of one CU's FP64 matrix rate, while 29 launches take longer than that even
// when they find nothing to do.  Here X and U stay in LDS through every step,
// G = X^T X and S = X^T U X stay in the MFMA accumulators (wavefront w holds
// rows 16 w .. 16 w + 15 of every product), and K = U X and then E take U's
// place in LDS, so a block of 64 rows needs 70 KB and two share a CU.  The
// row stride 16 n + 4 spreads both access patterns of the MFMA operands (16
// rows by 4 columns and 4 rows by 16 columns) over the LDS banks.
#include <hip/hip_runtime.h>

#include <cmath>

#include "refine.hpp"
#include "refine_pair.hpp"

namespace v2h {

namespace {

typedef double v4d __attribute__((ext_vector_type(4)));

// A block is accepted when its largest correction, the norms and the pairs
// inside clusters included, is below kSmallAcceptE: what the step leaves is of
// the order of its square, 1e-15 (the 1e-16 / 1e-8 noise of a correction
// across the narrowest gap that counts as separated stays below it).  With the
// 2e-7 of the large blocks, and norms left out, blocks of a few rows were up to
// 3e-10 off: their norms are the whole error that the step before has left.
constexpr double kSmallAcceptE = 3e-8;
constexpr double kSmallAcceptCpl = 2e-14;
constexpr int kSmallMoreSteps = 3;  // a step costs less here than the eigensolver many times over

__device__ __forceinline__ double nmax(double a, double b) { return (a != a) ? a : ((b != b) ? b : fmax(a, b)); }
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}
__device__ __forceinline__ double wave_nmax(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = nmax(v, __shfl_xor(v, o, 64));
    return v;
}

// A team of NTHR threads works on one block: a workgroup, or one wavefront
// (whose LDS accesses execute in order: only the compiler must be held back).
template <int NTHR>
__device__ __forceinline__ void team_sync() {
    if constexpr (NTHR == 64) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    } else {
        __syncthreads();
    }
}

// One block of d <= 16 NTILE rows.  UK, X: 16 NTILE rows of stride 16 NTILE + 4;
// lam, nrm: 16 NTILE; red: 4 per wavefront.
template <int NTILE, int NTHR>
__device__ __forceinline__ void ref_small(const BatchDev& B, const SmallDev& R, const RefParams& P, const RefBlock& b,
                                          double* UK, double* X, double* lam, double* nrm, double* red,
                                          int t) {
    constexpr int DP = 16 * NTILE, LD = DP + 4, NW = NTHR / 64;
    static_assert(NTILE <= NW, "one wavefront per 16 rows");
    const int d = b.d, l = t & 63, w = t >> 6, li = l & 15, lk = l >> 4;
    const bool live = NTHR == 64 || w < NTILE;
    const int m0 = 16 * w, dk = (d + 3) & ~3;  // products run over k < dk; rows and columns from d on are zero
    const InstDev I = B.inst[b.inst];
    const double mu = B.st[b.inst].mu;
    const double* U = B.u + I.poff + b.off;
    double* V = R.work + b.w;

    auto load_u = [&]() {
        for (int e = t; e < DP * DP; e += NTHR) {
            const int i = e / DP, j = e - i * DP;
            UK[i * LD + j] = (i < d && j < d) ? U[i * d + j] : 0.0;
        }
        team_sync<NTHR>();
        for (int e = t; e < DP * DP; e += NTHR) {
            const int i = e / DP, j = e - i * DP;
            if (i < j) {
                const double s = 0.5 * (UK[i * LD + j] + UK[j * LD + i]);
                UK[i * LD + j] = s;
                UK[j * LD + i] = s;
            }
        }
    };
    for (int e = t; e < DP * DP; e += NTHR) {
        const int i = e / DP, j = e - i * DP;
        X[i * LD + j] = (i < d && j < d) ? V[i * d + j] : 0.0;
    }
    load_u();
    team_sync<NTHR>();

    bool coupled = false;
    for (int step = 1;; step++) {
        v4d g[NTILE], s[NTILE];
        {
            v4d kx[NTILE];
#pragma unroll
            for (int c = 0; c < NTILE; c++) kx[c] = g[c] = s[c] = v4d{0.0, 0.0, 0.0, 0.0};
            if (live)
                for (int k0 = 0; k0 < dk; k0 += 4) {  // K = U X, G = X^T X
                    const double au = UK[(m0 + li) * LD + k0 + lk], ax = X[(k0 + lk) * LD + m0 + li];
#pragma unroll
                    for (int c = 0; c < NTILE; c++) {
                        const double bx = X[(k0 + lk) * LD + 16 * c + li];
                        kx[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(au, bx, kx[c], 0, 0, 0);
                        g[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ax, bx, g[c], 0, 0, 0);
                    }
                }
            team_sync<NTHR>();
            if (live)
#pragma unroll
                for (int c = 0; c < NTILE; c++)
#pragma unroll
                    for (int r = 0; r < 4; r++) UK[(m0 + 4 * r + lk) * LD + 16 * c + li] = kx[c][r];
            team_sync<NTHR>();
        }
        if (live) {
            for (int k0 = 0; k0 < dk; k0 += 4) {  // S = X^T K
                const double ax = X[(k0 + lk) * LD + m0 + li];
#pragma unroll
                for (int c = 0; c < NTILE; c++)
                    s[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ax, UK[(k0 + lk) * LD + 16 * c + li], s[c], 0, 0, 0);
            }
#pragma unroll
            for (int c = 0; c < NTILE; c++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    if (c == w && 4 * r + lk == li) {
                        lam[m0 + li] = m0 + li < d ? s[c][r] / g[c][r] : 0.0;
                        nrm[m0 + li] = m0 + li < d ? 1.0 / sqrt(g[c][r]) : 1.0;
                    }
        }
        team_sync<NTHR>();  // lam; every wavefront is done with K
        if (live)
#pragma unroll
            for (int c = 0; c < NTILE; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) UK[(m0 + 4 * r + lk) * LD + 16 * c + li] = s[c][r];
        team_sync<NTHR>();

        // Corrections E, as in k_ref_etile, from (S + S^T) / 2: S_ij and S_ji
        // round differently, and that difference over a narrow gap would stay
        // in E + E^T = I - G, that is, in the orthogonality of X.  A pair too
        // close to be separated stays coupled; where its whole cluster is
        // positive, the coupling is kept beside the eigenvalues (s: the middle
        // factor of U+ = X (L+ + C) X^T), where it is negative, it has no part in
        // U+, and only a coupling across zero (mc) rejects the block.
        const double scale = wave_nmax(l < DP ? fabs(lam[l]) : 0.0);
        const double om = P.cluster_rel * scale;
        const double keep = fmin(P.accept_cpl, kSmallAcceptCpl) * scale;  // couplings below this are dropped
        double me = 0.0, mc = 0.0, mk = 0.0, fr = 0.0;
        if (live) {
#pragma unroll
            for (int c = 0; c < NTILE; c++) {
                const int j = 16 * c + li;
                const double lj = lam[j], nj = nrm[j];
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int i = m0 + 4 * r + lk;
                    double ev = 0.0, ei = 0.0, mid = 0.0;  // correction, E, middle factor
                    if (i < d && j < d) {
                        const double ni = nrm[i], li_ = lam[i];
                        if (i == j) {
                            ev = ei = nj - 1.0;
                            mid = fmax(lj, 0.0);
                        } else {
                            const RefPair p = ref_pair(li_, lj, ni, nj, g[c][r], s[c][r], UK[j * LD + i], om, i < j);
                            ev = 0.5 * p.rr;
                            if (!p.close) {
                                ev += ref_rotation(p);
                            } else if (!(fabs(p.sa) <= keep)) {
                                const double lo = fmin(lj, li_), hi = fmax(lj, li_);
                                if (lo > DP * fabs(p.sa)) {
                                    mid = p.sa;
                                    mk = fmax(mk, fabs(p.sa));
                                } else if (!(hi < -DP * fabs(p.sa))) {
                                    mc = nmax(mc, fabs(p.sa));
                                }
                            }
                            ei = ni * ev;
                        }
                        fr = fma(ev, ev, fr);
                        me = nmax(me, fabs(ev));
                    }
                    g[c][r] = ei;
                    s[c][r] = mid;
                }
            }
        }
        team_sync<NTHR>();  // S is read
        if (live)
#pragma unroll
            for (int c = 0; c < NTILE; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) UK[(m0 + 4 * r + lk) * LD + 16 * c + li] = g[c][r];
        me = wave_nmax(me);
        mc = wave_nmax(mc);
        mk = wave_nmax(mk);
        fr = wave_sum(fr);
        if constexpr (NW > 1) {
            if (l == 0) {
                red[4 * w] = me;
                red[4 * w + 1] = mc;
                red[4 * w + 2] = mk;
                red[4 * w + 3] = fr;
            }
        }
        team_sync<NTHR>();  // E, red
        if constexpr (NW > 1) {
            me = red[0];
            mc = red[1];
            mk = red[2];
            fr = red[3];
#pragma unroll
            for (int q = 1; q < NTILE; q++) {
                me = nmax(me, red[4 * q]);
                mc = nmax(mc, red[4 * q + 1]);
                mk = fmax(mk, red[4 * q + 2]);
                fr += red[4 * q + 3];
            }
        }
        // (a NaN coupling comes with a NaN correction)
        const bool accept = me <= fmin(P.accept_e, kSmallAcceptE) && mc == 0.0;
        if (!(fr <= 4.0 + 0.1 * d) || (!accept && step >= P.max_steps + kSmallMoreSteps)) {
            if (t == 0) R.route[b.gblock] = kRouteRejected;
            return;
        }
        // X + X E
        v4d xn[NTILE];
        if (live) {
#pragma unroll
            for (int c = 0; c < NTILE; c++) xn[c] = v4d{0.0, 0.0, 0.0, 0.0};
            for (int k0 = 0; k0 < dk; k0 += 4) {
                const double ax = X[(m0 + li) * LD + k0 + lk];
#pragma unroll
                for (int c = 0; c < NTILE; c++)
                    xn[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ax, UK[(k0 + lk) * LD + 16 * c + li], xn[c], 0, 0, 0);
            }
#pragma unroll
            for (int c = 0; c < NTILE; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) xn[c][r] += X[(m0 + 4 * r + lk) * LD + 16 * c + li];
        }
        team_sync<NTHR>();
        if (live)
#pragma unroll
            for (int c = 0; c < NTILE; c++)
#pragma unroll
                for (int r = 0; r < 4; r++) X[(m0 + 4 * r + lk) * LD + 16 * c + li] = xn[c][r];
        if (!accept) load_u();
        team_sync<NTHR>();
        if (accept && mk > 0.0) {  // U's place takes X (L+ + C)
            if (live)
#pragma unroll
                for (int c = 0; c < NTILE; c++)
#pragma unroll
                    for (int r = 0; r < 4; r++) UK[(m0 + 4 * r + lk) * LD + 16 * c + li] = s[c][r];
            team_sync<NTHR>();
            if (live) {
#pragma unroll
                for (int c = 0; c < NTILE; c++) xn[c] = v4d{0.0, 0.0, 0.0, 0.0};
                for (int k0 = 0; k0 < dk; k0 += 4) {
                    const double ax = X[(m0 + li) * LD + k0 + lk];
#pragma unroll
                    for (int c = 0; c < NTILE; c++)
                        xn[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ax, UK[(k0 + lk) * LD + 16 * c + li], xn[c], 0, 0, 0);
                }
            }
            team_sync<NTHR>();
            if (live)
#pragma unroll
                for (int c = 0; c < NTILE; c++)
#pragma unroll
                    for (int r = 0; r < 4; r++) UK[(m0 + 4 * r + lk) * LD + 16 * c + li] = xn[c][r];
            team_sync<NTHR>();
            coupled = true;
        }
        if (accept) break;
    }

    // x = X diag(l+) X^T / mu, z = U+ - sym(U), v1 = c - z; the accepted X is
    // the start of the next iteration
    double ex = 0.0, dr = 0.0;
    if (live) {
        const double inv_mu = 1.0 / mu;
        double* Xo = B.x + I.poff + b.off;
        double* Z = B.z + I.poff + b.off;
        double* V1 = B.v1 + I.poff + b.off;
        const double* Cc = B.c + I.poff + b.off;
        v4d a[NTILE];
#pragma unroll
        for (int c = 0; c < NTILE; c++) a[c] = v4d{0.0, 0.0, 0.0, 0.0};
        for (int k0 = 0; k0 < dk; k0 += 4) {
            const double ax = coupled ? UK[(m0 + li) * LD + k0 + lk] * inv_mu
                                      : X[(m0 + li) * LD + k0 + lk] * (fmax(lam[k0 + lk], 0.0) * inv_mu);
#pragma unroll
            for (int c = 0; c < NTILE; c++)
                a[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(ax, X[(16 * c + li) * LD + k0 + lk], a[c], 0, 0, 0);
        }
#pragma unroll
        for (int c = 0; c < NTILE; c++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int i = m0 + 4 * r + lk, j = 16 * c + li;
                if (i < d && j < d) {
                    const int e = i * d + j;
                    const double uij = U[e], xn = a[c][r];
                    const double zn = mu * xn - 0.5 * (uij + U[j * d + i]);
                    const double res = (uij - mu * Xo[e]) + zn;
                    Xo[e] = xn;
                    Z[e] = zn;
                    const double ce = Cc[e];
                    V1[e] = ce - zn;
                    ex += ce * xn;
                    dr += res * res;
                    V[e] = X[i * LD + j];
                }
            }
    }
    ex = wave_sum(ex);
    dr = wave_sum(dr);
    if constexpr (NW > 1) {
        __syncthreads();  // the readers of red in the last step are done
        if (l == 0) {
            red[2 * w] = ex;
            red[2 * w + 1] = dr;
        }
        __syncthreads();
        ex = red[0];
        dr = red[1];
#pragma unroll
        for (int q = 1; q < NTILE; q++) {
            ex += red[2 * q];
            dr += red[2 * q + 1];
        }
    }
    if (t == 0) {
        B.proj_part[2 * (size_t)b.gblock] = ex;
        B.proj_part[2 * (size_t)b.gblock + 1] = dr;
        B.st[b.inst].pending = 1;
        R.route[b.gblock] = kRouteAccepted;
    }
}

// A block without eigenvectors goes to the fallback; false: nothing to refine.
__device__ __forceinline__ bool ref_small_begin(const BatchDev& B, const SmallDev& R, const RefBlock& b,
                                                int vvalid, int t) {
    if (!B.st[b.inst].active || !in_pgroup(B, b.inst)) return false;
    if (vvalid) return true;
    if (t == 0) R.route[b.gblock] = kRouteFallback;
    return false;
}

// The first n1 workgroups take one block of 17..64 rows each (MT: 16-row tiles
// of the largest), the others four blocks of up to 16 rows, one per wavefront:
// one launch, so that neither class waits for the other.
template <int MT>
__global__ __launch_bounds__(256, 2) void k_ref_small(BatchDev B, SmallDev R, RefParams P, int n1, int n) {
    constexpr int DP = 16 * MT, kMat = DP * (DP + 4) > 4 * 320 ? DP * (DP + 4) : 4 * 320;
    __shared__ double UK[kMat], X[kMat], lam[64], nrm[64], red[16];
    if ((int)blockIdx.x >= n1) {
        const int w = threadIdx.x >> 6, t = threadIdx.x & 63;
        const int q = n1 + 4 * ((int)blockIdx.x - n1) + w;
        if (q >= n) return;
        const RefBlock b = R.blk[q];
        if (!ref_small_begin(B, R, b, R.vvalid[q], t)) return;
        return ref_small<1, 64>(B, R, P, b, UK + w * 320, X + w * 320, lam + w * 16, nrm + w * 16, nullptr, t);
    }
    if constexpr (MT > 1) {
        const int bi = blockIdx.x, t = threadIdx.x;
        const RefBlock b = R.blk[bi];
        if (!ref_small_begin(B, R, b, R.vvalid[bi], t)) return;
        if constexpr (MT >= 4)
            if (b.d > 48) return ref_small<4, 256>(B, R, P, b, UK, X, lam, nrm, red, t);
        if constexpr (MT >= 3)
            if (b.d > 32) return ref_small<3, 256>(B, R, P, b, UK, X, lam, nrm, red, t);
        ref_small<2, 256>(B, R, P, b, UK, X, lam, nrm, red, t);
    }
}

__global__ void k_ref_small_forget(SmallDev R, int n, int inst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && R.blk[i].inst == inst) R.vvalid[i] = 0;
}

}  // namespace

void launch_ref_small_forget(const SmallDev& R, int n, int inst, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_ref_small_forget, dim3((n + 255) / 256), dim3(256), 0, s, R, n, inst);
}

void launch_ref_small(const BatchDev& B, const SmallDev& R, const RefParams& P, int n1, int n, int max_d,
                      hipStream_t s) {
    if (n <= 0) return;
    const dim3 grid(n1 + (n - n1 + 3) / 4);
    if (max_d <= 16)
        hipLaunchKernelGGL(k_ref_small<1>, grid, dim3(256), 0, s, B, R, P, n1, n);
    else if (max_d <= 32)
        hipLaunchKernelGGL(k_ref_small<2>, grid, dim3(256), 0, s, B, R, P, n1, n);
    else if (max_d <= 48)
        hipLaunchKernelGGL(k_ref_small<3>, grid, dim3(256), 0, s, B, R, P, n1, n);
    else
        hipLaunchKernelGGL(k_ref_small<4>, grid, dim3(256), 0, s, B, R, P, n1, n);
}

}  // namespace v2h
