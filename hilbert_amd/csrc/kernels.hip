// kernels.hip -- CDNA4 (gfx950) kernels of the batched BPSDP solve.
//
// * Gather kernels over SELL-64 tables (one wavefront per 64 rows, or per
//   long row).  Every CG step is two launches, k_cg_at and k_cg_a, whose last
//   workgroup of an instance sums the partial dot products in a fixed order
//   (deterministic) and advances the CG state; k_cg_init forms the first
//   residual.
// * k_pre (+ k_pre_reduce): A [v1, x, A^T y] in one pass (rhs pieces, A x),
//   then the end-of-iteration bookkeeping (errors, energies, mu, convergence,
//   CG threshold).
// * k_post : A^T y and U = mu x + A^T y - c.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>

#include "common.hpp"
#include "kernels.hpp"
#include "sell.hpp"
#include "wave_ops.hpp"

namespace v2h {

namespace {

constexpr int kWG = 256;         // gather workgroup: 4 wavefronts
constexpr uint32_t kMarker = 255;

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// Workgroup id remapped so that each XCD (blocks are dealt round-robin over
// the 8 XCDs) runs a contiguous range of logical workgroups, keeping one
// instance's vectors in one XCD's L2.
__device__ __forceinline__ int xcd_remap(int bid, int n) {
    int per = n >> 3, rem = n & 7;
    int x = bid & 7, loc = bid >> 3;
    return x * per + (x < rem ? x : rem) + loc;
}

// Logical workgroup of this block under the launch plan (runs of the
// workgroups of selected instances; identity without a plan).
__device__ __forceinline__ int unit_wg(const UnitsDev& U) {
    const int c = U.remap ? xcd_remap(blockIdx.x, U.grid) : (int)blockIdx.x;
    if (U.plan == nullptr) return c;
    int lo = 0, hi = U.plan_m;  // plan[lo] <= c < plan[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (U.plan[mid] <= c)
            lo = mid;
        else
            hi = mid;
    }
    return U.plan[U.plan_m + 1 + lo] + (c - U.plan[lo]);
}

// Gather over one SELL slice (lane = row) or one long row (whole wave).
// Load(col, coef) accumulates into the caller's accumulators.
template <class Load>
__device__ __forceinline__ int64_t gather_unit(const SellDev& S, const double* coef, int unit, int lane,
                                               Load&& load, bool& is_long) {
    is_long = (unit & kLongFlag) != 0;
    if (!is_long) {
        uint32_t beg = S.slice_start[unit], end = S.slice_start[unit + 1];
        const uint32_t* e = S.ent + (size_t)beg * 64 + lane;
        int w = (int)(end - beg);
        bool skip = false;
        int k = 0;
        for (; k + 4 <= w; k += 4) {
            uint32_t v0 = e[(size_t)(k + 0) * 64], v1 = e[(size_t)(k + 1) * 64];
            uint32_t v2 = e[(size_t)(k + 2) * 64], v3 = e[(size_t)(k + 3) * 64];
            skip |= (v0 >> 24) == kMarker;
            load(v0 & 0xFFFFFFu, coef[v0 >> 24]);
            load(v1 & 0xFFFFFFu, coef[v1 >> 24]);
            load(v2 & 0xFFFFFFu, coef[v2 >> 24]);
            load(v3 & 0xFFFFFFu, coef[v3 >> 24]);
        }
        for (; k < w; k++) {
            uint32_t v = e[(size_t)k * 64];
            skip |= (v >> 24) == kMarker;
            load(v & 0xFFFFFFu, coef[v >> 24]);
        }
        int64_t row = (int64_t)unit * 64 + lane;
        return (skip || row >= S.nrows) ? -1 : row;
    }
    int li = unit & ~kLongFlag;
    uint32_t beg = S.long_start[li], end = S.long_start[li + 1];
    for (uint32_t e = beg + lane; e < end; e += 64) {
        uint32_t v = S.long_ent[e];
        load(v & 0xFFFFFFu, coef[v >> 24]);
    }
    return S.long_row[li];  // caller reduces the accumulators over the wave
}

template <int N>
__device__ __forceinline__ void block_partials(const double (&v)[N], double* red, double* out) {
    // red: [4][N] in LDS; out: N partials written by thread 0
    int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    double s[N];
#pragma unroll
    for (int i = 0; i < N; i++) s[i] = wave_sum(v[i]);
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < N; i++) red[wv * N + i] = s[i];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 0; i < N; i++) out[i] = ((red[i] + red[N + i]) + red[2 * N + i]) + red[3 * N + i];
    }
}

// Sum the nwg partial records (N doubles each) of one instance in a fixed
// order; every thread of the workgroup receives tot[N].  Runs in its own
// launch after the producing kernel: the kernel boundary makes every XCD's
// writes visible without device-scope fences inside the producer.
template <int N>
__device__ void reduce_partials(const double* parts, int nwg, double* red, double (&tot)[N]) {
    double s[N];
#pragma unroll
    for (int i = 0; i < N; i++) s[i] = 0.0;
    for (int k = threadIdx.x; k < nwg; k += blockDim.x) {
#pragma unroll
        for (int i = 0; i < N; i++) s[i] += parts[(size_t)k * N + i];
    }
    int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < N; i++) s[i] = wave_sum(s[i]);
    if (lane == 0) {
#pragma unroll
        for (int i = 0; i < N; i++) red[wv * N + i] = s[i];
    }
    __syncthreads();
    int nw = blockDim.x >> 6;
#pragma unroll
    for (int i = 0; i < N; i++) {
        double t = 0.0;
        for (int q = 0; q < nw; q++) t += red[q * N + i];
        tot[i] = t;
    }
}

__device__ __forceinline__ void load_coef(double* dst, const double* src) {
    for (int i = threadIdx.x; i < 256; i += blockDim.x) dst[i] = src[i];
    __syncthreads();
}

// ------------------------------------------------------------------------
// Gather launches.  Every wavefront starts from its UnitRec (one scalar load:
// table entries, coefficient table, first row), so its table loads, the
// workgroup's coefficient table and the instance state are in flight together;
// the first kPre entries of each lane are loaded before the set-up barrier.

constexpr int kPre = 4;

struct WaveGather {
    UnitRec R;
    int lane;
    bool is_long;
    uint32_t pre[kPre];
    __device__ __forceinline__ WaveGather(const UnitRec& r, int l) : R(r), lane(l) {
        is_long = (R.meta & kRecLong) != 0u;
        const int w = is_long ? 0 : (int)(R.meta & 0xFFFFu);
#pragma unroll
        for (int k = 0; k < kPre; k++) pre[k] = (k < w) ? R.ent[(size_t)k * 64 + lane] : 0u;
    }
    // first row of this lane (slices), before the entries are known
    __device__ __forceinline__ int64_t lane_row() const {
        const int nvalid = (int)((R.meta >> 16) & 0x7Fu);
        return (!is_long && lane < nvalid) ? (int64_t)R.row + lane : -1;
    }
    // Load(col, coef) over the lane's entries; returns the row the lane
    // writes (slices: -1 for padding lanes and long-row markers; long rows:
    // the row, after the caller's wave reduction, on lane 0).
    template <class Load>
    __device__ __forceinline__ int64_t run(const double* coef, Load&& load) {
        if (!is_long) {
            const int w = (int)(R.meta & 0xFFFFu);
            const bool skip = w > 0 && (pre[0] >> 24) == kMarker;
#pragma unroll
            for (int k = 0; k < kPre; k++)
                if (k < w) load(pre[k] & 0xFFFFFFu, coef[pre[k] >> 24]);
            const uint32_t* e = R.ent + lane;
            int k = kPre;
            for (; k + 4 <= w; k += 4) {
                const uint32_t v0 = e[(size_t)(k + 0) * 64], v1 = e[(size_t)(k + 1) * 64];
                const uint32_t v2 = e[(size_t)(k + 2) * 64], v3 = e[(size_t)(k + 3) * 64];
                load(v0 & 0xFFFFFFu, coef[v0 >> 24]);
                load(v1 & 0xFFFFFFu, coef[v1 >> 24]);
                load(v2 & 0xFFFFFFu, coef[v2 >> 24]);
                load(v3 & 0xFFFFFFu, coef[v3 >> 24]);
            }
            for (; k < w; k++) {
                const uint32_t v = e[(size_t)k * 64];
                load(v & 0xFFFFFFu, coef[v >> 24]);
            }
            return skip ? -1 : lane_row();
        }
        const int n = (int)(R.meta & ~kRecLong);
        for (int k = lane; k < n; k += 64) {
            const uint32_t v = R.ent[k];
            load(v & 0xFFFFFFu, coef[v >> 24]);
        }
        return R.row;
    }
};

// Coefficient table of the workgroup's structure into LDS (every wavefront of
// a workgroup belongs to one instance).
__device__ __forceinline__ void put_coef(double* coef, double v) {
    coef[threadIdx.x] = v;
    __syncthreads();
}

// Draws a ticket; true for the last of n, which takes the counter back to 0.
__device__ __forceinline__ bool draw_last(int* t, int n) {
    if (__hip_atomic_fetch_add(t, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != n - 1) return false;
    __hip_atomic_store(t, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return true;
}

// Sum over the workgroups of one instance of v (each workgroup's over its
// threads, in LDS red[4]) within the launch that produces it: the partial
// value goes past the XCDs' L2s to memory, then the workgroup draws a ticket of
// its group of 32, the last of a group one of the instance, and the very last
// sums the nwg partial values in a fixed order.  True in that workgroup, whose
// threads then all hold the total in v.  Every workgroup of the instance must
// call it.  One launch less per reduction than a reducing kernel (4 to 5 us each
// on an idle GPU, two per CG step).  Tickets of one counter are drawn one after
// the other (about 12 ns each): with one per instance, 1900 workgroups took 25 us
// longer, and 32 counters on one line 130 us for 24 000.
__device__ __forceinline__ bool last_sum(const BatchDev& B, const UnitsDev& U, int inst, int wg, double* red,
                                         double& v) {
    __shared__ int last;
    const int wg0 = U.wg_begin[inst], nwg = U.wg_begin[inst + 1] - wg0;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    v = wave_sum(v);
    if (lane == 0) red[wv] = v;
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_store(B.partials + wg, (red[0] + red[1]) + (red[2] + red[3]), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the value has reached memory
        const int grp = (wg - wg0) / kTicketGroup, ngrp = (nwg + kTicketGroup - 1) / kTicketGroup;
        const int size = min(kTicketGroup, nwg - grp * kTicketGroup);
        // groups of an instance from wg0 / kTicketGroup + inst on: no two share a counter
        int* t = B.ticket + (size_t)(U.ninst + wg0 / kTicketGroup + inst + grp) * kTicketStride;
        last = draw_last(t, size) && draw_last(B.ticket + (size_t)inst * kTicketStride, ngrp);
    }
    __syncthreads();
    if (!last) return false;
    double s = 0.0;
    for (int k = threadIdx.x; k < nwg; k += kWG)
        s += __hip_atomic_load(B.partials + wg0 + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s = wave_sum(s);
    if (lane == 0) red[wv] = s;
    __syncthreads();
    v = (red[0] + red[1]) + (red[2] + red[3]);
    return true;
}

// The CG on A A^T y = A (c - z) + mu (b - A x), warm-started, with two launches
// and two reductions per step:
//   k_cg_at   q <- A^T r + beta q (= A^T p); alpha = |r|^2 / |q|^2
//   k_cg_a    w = A q; p <- r + beta p, y <- y + alpha p, r <- r - alpha w;
//             beta = |r|^2 / |r_old|^2, stop test
// |q|^2 = p . A A^T p, so alpha is known before w: w is never stored, and the
// gather of A^T reads 8 contiguous bytes per row (r) instead of r, w and p (24 of
// a 32-byte row) to form p on the fly.  Per step and instance 8 (3 n_p + 7 n_d)
// bytes of vectors instead of 8 (2 n_p + 12 n_d).  Bound by HBM (and L2 for the
// gathers) in large batches, by launch latency for one small SDP.

// r = d0 + mu e, |r|^2
__global__ __launch_bounds__(kWG) void k_cg_init(BatchDev B, UnitsDev U) {
    const int wg = unit_wg(U);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int inst = U.wg_inst[wg];
    const UnitRec R = U.rec[(size_t)wg * 4 + wv];
    InstState& st = B.st[inst];
    if (!st.active || st.cg_done || B.inst[inst].small) return;
    __shared__ double red[4];
    // the slices cover every row (the long ones too, as lanes of theirs)
    const bool in = (R.meta & kRecLong) == 0u && lane < (int)((R.meta >> 16) & 0x7Fu);
    double rr = 0.0;
    if (in) {
        const int64_t g = B.inst[inst].doff + R.row + lane;
        const double r = __fma_rn(st.mu, B.e[g], B.d0[g]);
        B.r[g] = r;
        rr = r * r;
    }
    if (!last_sum(B, U, inst, wg, red, rr) || threadIdx.x != 0) return;
    st.rr = rr;
    if (!isfinite(rr)) st.status |= kStatusNonFinite;
    if (!(rr > st.cg_thr) || !isfinite(rr) || B.opt.cg_maxiter <= 0) {
        st.cg_done = 1;
        st.cg_last = 0;
    }
}

__global__ __launch_bounds__(kWG) void k_cg_at(BatchDev B, UnitsDev U) {
    static_assert(kWG == 256, "one coefficient per thread");
    const int wg = unit_wg(U);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int inst = U.wg_inst[wg];
    const UnitRec R = U.rec[(size_t)wg * 4 + wv];
    const double cv = R.coef[threadIdx.x];
    WaveGather G(R, lane);
    InstState& st = B.st[inst];
    const InstDev I = B.inst[inst];
    if (!st.active || I.small || st.cg_done) return;
    __shared__ double coef[256];
    __shared__ double red[4];
    put_coef(coef, cv);
    const double be = st.be;
    const bool first = st.cg_iter == 0;
    double* q = B.q + I.poff;
    const int64_t r0 = G.lane_row();
    double qo = (!first && r0 >= 0) ? q[r0] : 0.0;  // loaded with the gather
    const double* r = B.r + I.doff;
    double acc = 0.0;
    int64_t row = G.run(coef, [&](uint32_t col, double cf) { acc = __fma_rn(cf, r[col], acc); });
    if (G.is_long) {
        acc = wave_sum(acc);
        if (lane != 0) row = -1;
        if (!first && row >= 0) qo = q[row];
    }
    double qq = 0.0;
    if (row >= 0) {
        const double qn = first ? acc : __fma_rn(be, qo, acc);
        q[row] = qn;
        qq = qn * qn;
    }
    if (!last_sum(B, U, inst, wg, red, qq) || threadIdx.x != 0) return;
    if (!isfinite(qq)) st.status |= kStatusNonFinite;
    if (qq > 0.0 && isfinite(qq)) {
        st.al = st.rr / qq;
    } else {  // r is in the null space of A^T: nothing left to reduce
        st.cg_done = 1;
        st.cg_last = st.cg_iter;
        st.iiter += st.cg_iter;
    }
}

__global__ __launch_bounds__(kWG) void k_cg_a(BatchDev B, UnitsDev U) {
    const int wg = unit_wg(U);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int inst = U.wg_inst[wg];
    const UnitRec R = U.rec[(size_t)wg * 4 + wv];
    const double cv = R.coef[threadIdx.x];
    WaveGather G(R, lane);
    InstState& st = B.st[inst];
    const InstDev I = B.inst[inst];
    if (!st.active || I.small || st.cg_done) return;
    __shared__ double coef[256];
    __shared__ double red[4];
    put_coef(coef, cv);
    const double al = st.al, be = st.be;
    const bool first = st.cg_iter == 0;
    // the own row's state is loaded with the gather
    const int64_t r0 = G.lane_row();
    double r = 0.0, p = 0.0, y = 0.0;
    if (r0 >= 0) {
        const int64_t g = I.doff + r0;
        r = B.r[g];
        y = B.y[g];
        if (!first) p = B.p[g];
    }
    const double* q = B.q + I.poff;
    double acc = 0.0;
    int64_t row = G.run(coef, [&](uint32_t col, double cf) { acc = __fma_rn(cf, q[col], acc); });
    if (G.is_long) {
        acc = wave_sum(acc);
        if (lane != 0) row = -1;
        if (row >= 0) {
            const int64_t g = I.doff + row;
            r = B.r[g];
            y = B.y[g];
            if (!first) p = B.p[g];
        }
    }
    double rr = 0.0;
    if (row >= 0) {
        const int64_t g = I.doff + row;
        const double pn = first ? r : __fma_rn(be, p, r);
        const double rn = __fma_rn(-al, acc, r);
        B.p[g] = pn;
        B.y[g] = __fma_rn(al, pn, y);
        B.r[g] = rn;
        rr = rn * rn;
    }
    if (!last_sum(B, U, inst, wg, red, rr) || threadIdx.x != 0) return;
    const int s = st.cg_iter + 1;
    bool go_on = rr > st.cg_thr && s < B.opt.cg_maxiter;
    if (!isfinite(rr)) {
        st.status |= kStatusNonFinite;
        go_on = false;
    }
    st.be = rr / st.rr;
    st.rr = rr;
    st.cg_iter = s;
    if (!go_on) {
        st.cg_done = 1;
        st.cg_last = s;
        st.iiter += s;
    }
}

// A slice of pieces (sell.hpp) in the registers of a wavefront.
struct PieceSlice {
    uint32_t e[kPiece];
    int32_t dst;
    int w;
    __device__ __forceinline__ void load(const PieceDev& T, int u, int lane) {
        w = 0;
        dst = kNoPiece;
#pragma unroll
        for (int k = 0; k < kPiece; k++) e[k] = 0u;
        if (u >= T.nslices) return;
        const uint32_t s = T.slice[u];
        w = (int)(s >> 28);
        dst = T.dst[u * 64 + lane];
        const uint32_t* p = T.ent + (s & 0x0FFFFFFFu) + lane;
#pragma unroll
        for (int k = 0; k < kPiece; k++)
            if (k < w) e[k] = p[64 * k];
    }
    // (the empty asm keeps the addresses, which no step changes, from being held
    // in registers too)
    __device__ __forceinline__ double sum(const double* coef, const double* v) const {
        uint32_t x[kPiece];
#pragma unroll
        for (int k = 0; k < kPiece; k++) {
            x[k] = e[k];
            asm volatile("" : "+v"(x[k]));
        }
        double a = coef[x[0] >> 24] * v[x[0] & 0xFFFFFFu];
        if (w > 1) {  // (uniform)
            const double b = coef[x[1] >> 24] * v[x[1] & 0xFFFFFFu];
            if (w > 2) {
                a = __fma_rn(coef[x[2] >> 24], v[x[2] & 0xFFFFFFu], a);
                a = __fma_rn(coef[x[3] >> 24], v[x[3] & 0xFFFFFFu], a);
            }
            a += b;
        }
        return a;
    }
};

// The whole CG of a small instance (list[blockIdx.x]) in one workgroup, r, q and
// partial sums in LDS: a step is two passes over the pieces of the gather
// tables, each with a pass over the rows of several pieces and a workgroup sum;
// no step is launched that is not needed and the host looks at no CG.  A
// wavefront has at most kSmallHeld slices in each direction and keeps them and
// its rows' p and y in registers, so nothing but LDS is read in a step: beyond
// that (streaming the slices from L2) a step takes as long as its two launches
// would.  Bound by the latency of the LDS gathers, barriers and sums: (6e,6o) C2v,
// 22 steps, 118 us, against 310 us in two launches a step and 222 us streaming.
constexpr int kSmallNT = 1024, kSmallHeld = 6;
__global__ __launch_bounds__(kSmallNT) void k_cg_small(BatchDev B, const int* list) {
    extern __shared__ double sm[];
    constexpr int NW = kSmallNT / 64, KU = kSmallHeld;
    const int inst = list[blockIdx.x];
    InstState& st = B.st[inst];
    if (!st.active || !in_pgroup(B, inst)) return;
    const InstDev I = B.inst[inst];
    const StructDev& S = B.structs[I.sid];
    const PieceDev TA = S.pA, TT = S.pAT;
    const int nd = (int)S.n_dual;
    double *coefA = sm, *coefT = sm + 256, *red = sm + 512, *r = sm + 544, *q = r + nd, *part = q + S.n_primal;
    double* Y = B.y + I.doff;
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    int half = 0;  // alternating sum buffers: one barrier per sum
    auto wg_sum = [&](double v) {
        double* b = red + 16 * half;
        half ^= 1;
        v = wsum(v);
        if (lane == 0) b[wv] = v;
        __syncthreads();
        double s4[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < NW; k++) s4[k & 3] += b[k];
        return (s4[0] + s4[1]) + (s4[2] + s4[3]);
    };
    if (t < 256) {
        coefA[t] = S.A.coef[t];
        coefT[t] = S.AT.coef[t];
    }
    PieceSlice hA[KU], hT[KU];
    double yh[KU], ph[KU], ym = 0.0, pm = 0.0;  // of the held pieces' rows and of multi row t
#pragma unroll
    for (int m = 0; m < KU; m++) {
        hA[m].load(TA, wv + NW * m, lane);
        hT[m].load(TT, wv + NW * m, lane);
        yh[m] = hA[m].dst >= 0 ? Y[hA[m].dst] : 0.0;
        ph[m] = 0.0;
    }
    // the multi rows of the two operators that are this thread's
    int3 mA = make_int3(-1, 0, 0), mT = mA;
    if (t < TA.nmulti) mA = make_int3(TA.multi[3 * t], TA.multi[3 * t + 1], TA.multi[3 * t + 2]);
    if (t < TT.nmulti) mT = make_int3(TT.multi[3 * t], TT.multi[3 * t + 1], TT.multi[3 * t + 2]);
    if (mA.x >= 0) ym = Y[mA.x];
    const double mu = st.mu, thr = st.cg_thr;
    double rr = 0.0;
    for (int i = t; i < nd; i += kSmallNT) {
        const double v = __fma_rn(mu, B.e[I.doff + i], B.d0[I.doff + i]);
        r[i] = v;
        rr = __fma_rn(v, v, rr);
    }
    rr = wg_sum(rr);
    // one(row, sum, p, y) for every row of the operator applied to v
    auto apply = [&](const PieceSlice(&h)[KU], const int3& mr, bool multi, const double* coef, const double* v,
                     auto&& one) {
#pragma unroll
        for (int m = 0; m < KU; m++) {
            if (h[m].w == 0) continue;  // (uniform)
            const double a = h[m].sum(coef, v);
            int dst = h[m].dst;
            asm volatile("" : "+v"(dst));
            if (dst >= 0) one(dst, a, ph[m], yh[m]);
            else if (dst != kNoPiece) part[-1 - dst] = a;
        }
        if (!multi) return;
        __syncthreads();
        if (mr.x >= 0) {
            double a = part[mr.y];
            for (int k = 1; k < mr.z; k++) a += part[mr.y + k];
            one(mr.x, a, pm, ym);
        }
    };
    double be = 0.0;
    int s = 0, bad = !isfinite(rr);
    while (!bad && rr > thr && s < B.opt.cg_maxiter) {
        double qq = 0.0;
        apply(hT, mT, TT.nmulti > 0, coefT, r, [&](int row, double a, double&, double&) {
            const double qn = s > 0 ? __fma_rn(be, q[row], a) : a;
            q[row] = qn;
            qq = __fma_rn(qn, qn, qq);
        });
        qq = wg_sum(qq);
        bad = !isfinite(qq);
        if (bad || !(qq > 0.0)) break;  // 0: r is in the null space of A^T
        const double al = rr / qq;
        double rn2 = 0.0;
        apply(hA, mA, TA.nmulti > 0, coefA, q, [&](int row, double a, double& p, double& y) {
            const double ro = r[row], rn = __fma_rn(-al, a, ro);
            p = s > 0 ? __fma_rn(be, p, ro) : ro;
            y = __fma_rn(al, p, y);
            r[row] = rn;
            rn2 = __fma_rn(rn, rn, rn2);
        });
        rn2 = wg_sum(rn2);
        be = rn2 / rr;
        rr = rn2;
        s++;
        bad = !isfinite(rr);
    }
#pragma unroll
    for (int m = 0; m < KU; m++)
        if (hA[m].dst >= 0) Y[hA[m].dst] = yh[m];
    if (mA.x >= 0) Y[mA.x] = ym;
    if (t == 0) {
        if (bad) st.status |= kStatusNonFinite;
        st.rr = rr;
        st.cg_iter = st.cg_last = s;
        st.iiter += s;
        st.cg_done = 1;
    }
}

// Start of an outer iteration: A [v1, x, aty] -> d0, e; finishes the
// previous iteration (errors, energies, mu, convergence) and sets up the CG.
__global__ __launch_bounds__(kWG) void k_pre(BatchDev B, UnitsDev U) {
    const int wg = unit_wg(U);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int inst = U.wg_inst[wg];
    const UnitRec R = U.rec[(size_t)wg * 4 + wv];
    const double cv = R.coef[threadIdx.x];
    WaveGather G(R, lane);
    const InstState& st = B.st[inst];
    const InstDev I = B.inst[inst];
    if (!st.active) return;
    __shared__ double coef[256];
    __shared__ double red[4 * 4];
    put_coef(coef, cv);
    const double *v1 = B.v1 + I.poff, *x = B.x + I.poff, *aty = B.aty + I.poff;
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    int64_t row = G.run(coef, [&](uint32_t col, double cf) {
        a0 = __fma_rn(cf, v1[col], a0);
        a1 = __fma_rn(cf, x[col], a1);
        a2 = __fma_rn(cf, aty[col], a2);
    });
    if (G.is_long) {
        a0 = wave_sum(a0);
        a1 = wave_sum(a1);
        a2 = wave_sum(a2);
        if (lane != 0) row = -1;
    }
    double d4[4] = {0.0, 0.0, 0.0, 0.0};
    if (row >= 0) {
        const int64_t g = I.doff + row;
        const double bv = B.structs[I.sid].b[row];
        const double e = bv - a1;
        B.d0[g] = a0 - a2;
        B.e[g] = e;
        d4[0] = a0 * a0;
        d4[1] = a0 * e;
        d4[2] = e * e;
        d4[3] = bv * B.y[g];
    }
    block_partials<4>(d4, red, B.partials + (size_t)wg * 4);
}

// Iteration start, part 2 (one workgroup per instance): book-keeping of the
// finished iteration (errors, energies, mu, convergence) and CG set-up.
__global__ __launch_bounds__(kWG) void k_pre_reduce(BatchDev B, UnitsDev U) {
    const int inst = blockIdx.x;
    InstState& st = B.st[inst];
    if (!st.active || !in_pgroup(B, inst)) return;
    const InstDev I = B.inst[inst];
    __shared__ double red[4 * 4];
    double tot[4];
    reduce_partials<4>(B.partials + (size_t)U.wg_begin[inst] * 4, U.wg_begin[inst + 1] - U.wg_begin[inst], red, tot);
    if (threadIdx.x == 0) {
        const SolverOptions& o = B.opt;
        if (st.pending) {
            double ep = sqrt(tot[2]) / st.bnorm;
            double Ep = 0.0, dres = 0.0;
            for (int k = 0; k < I.nblocks; k++) {
                Ep += B.proj_part[2 * (size_t)(I.block_first + k)];
                dres += B.proj_part[2 * (size_t)(I.block_first + k) + 1];
            }
            double ed = sqrt(dres) / st.cnorm;
            st.eps_p = ep;
            st.eps_d = ed;
            st.e_primal = Ep;
            st.e_dual = tot[3];
            st.oiter += 1;
            st.maxiter_left -= 1;
            if (o.mu_update_frequency > 0 && st.oiter % o.mu_update_frequency == 0 && ed > 0.0 && ep > 0.0)
                st.mu *= ep / ed;
            if (fabs(Ep - tot[3]) < o.e_convergence && ep < o.r_convergence && ed < o.r_convergence) {
                st.converged = 1;
                st.active = 0;
            }
            if (!isfinite(Ep) || !isfinite(ep) || !isfinite(ed)) {
                st.status |= kStatusNonFinite;
                st.active = 0;
            }
            if (st.oiter >= o.maxiter || st.maxiter_left <= 0) st.active = 0;
        }
        st.pending = 0;
        double e = st.oiter == 0 ? 1.0 : fmax(st.eps_p, st.eps_d);
        double tol = o.cg_tol_factor * e;
        if (tol > kCgTolCap) tol = kCgTolCap;
        if (tol < o.cg_convergence) tol = o.cg_convergence;
        double mu = st.mu;
        double rhs2 = tot[0] + 2.0 * mu * tot[1] + mu * mu * tot[2];
        st.cg_thr = tol * tol * rhs2;
        st.be = 0.0;
        st.cg_iter = 0;
        st.cg_done = 0;
    }
}

// After the CG: aty = A^T y, u = mu x + aty - c.
__global__ __launch_bounds__(kWG) void k_post(BatchDev B, UnitsDev U) {
    const int wg = unit_wg(U);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int inst = U.wg_inst[wg];
    const UnitRec R = U.rec[(size_t)wg * 4 + wv];
    const double cv = R.coef[threadIdx.x];
    WaveGather G(R, lane);
    const InstState& st = B.st[inst];
    const InstDev I = B.inst[inst];
    if (!st.active) return;
    __shared__ double coef[256];
    put_coef(coef, cv);
    const double* y = B.y + I.doff;
    double acc = 0.0;
    int64_t row = G.run(coef, [&](uint32_t col, double cf) { acc = __fma_rn(cf, y[col], acc); });
    if (G.is_long) {
        acc = wave_sum(acc);
        if (lane != 0) row = -1;
    }
    if (row >= 0) {
        const int64_t g = I.poff + row;
        B.aty[g] = acc;
        B.u[g] = __fma_rn(st.mu, B.x[g], acc) - B.c[g];
    }
}

// Plain out = A in  or  out = A^T in, for one instance (API and tests).
__global__ __launch_bounds__(kWG) void k_spmv_plain(SellDev S, const int4* units, int wg0, const double* in,
                                                    double* out) {
    __shared__ double coef[256];
    load_coef(coef, S.coef);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int unit = ((const int*)&units[wg0 + blockIdx.x])[wv];
    if (unit < 0) return;
    double acc = 0.0;
    bool lng;
    int64_t row = gather_unit(S, coef, unit, lane, [&](uint32_t col, double cf) { acc = __fma_rn(cf, in[col], acc); }, lng);
    if (lng) {
        acc = wave_sum(acc);
        if (lane != 0) row = -1;
    }
    if (row >= 0) out[row] = acc;
}

template <int NT>
__device__ __forceinline__ double block_sum(double v, double* red) {
    v = wave_sum(v);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < NT / 64; q++) t += red[q];
    return t;
}

// ------------------------------------------------------------------------
// small kernels

__global__ void k_fill(double* p, int64_t n, double v) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t st = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += st) p[i] = v;
}

__global__ void k_copy(double* dst, const double* src, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t st = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += st) dst[i] = src[i];
}

// c[e] = src[i1[e]] - src[i2[e]] (index < 0 reads 0)
__global__ void k_pack_cost(const int32_t* i1, const int32_t* i2, const double* src, double* c, int64_t n) {
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t st = (int64_t)gridDim.x * blockDim.x;
    for (; e < n; e += st) {
        int32_t a = i1[e], b = i2[e];
        double v = a >= 0 ? src[a] : 0.0;
        if (b >= 0) v -= src[b];
        c[e] = v;
    }
}

// dsrc[t] = sum over the primal elements e that read src[t] of +-xbar[e]
__global__ void k_cost_adjoint(const int32_t* ptr, const int32_t* ent, const double* xbar, double* dsrc, int64_t nsrc) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t st = (int64_t)gridDim.x * blockDim.x;
    for (; t < nsrc; t += st) {
        double v = 0.0;
        for (int32_t k = ptr[t]; k < ptr[t + 1]; k++) {
            uint32_t e = (uint32_t)ent[k];
            double xv = xbar[e & 0x7FFFFFFFu];
            v += (e & 0x80000000u) ? -xv : xv;
        }
        dsrc[t] = v;
    }
}

// a . b in two launches with a fixed summation order: kDotParts workgroups
// each reduce one contiguous chunk into out[1 + part], then one workgroup
// sums the parts in order into out[0].
constexpr int kDotParts = 256;
__global__ __launch_bounds__(256) void k_dot_part(const double* a, const double* b, int64_t n, double* out) {
    __shared__ double red[4];
    const int64_t chunk = (n + kDotParts - 1) / kDotParts;
    const int64_t lo = (int64_t)blockIdx.x * chunk, hi = lo + chunk < n ? lo + chunk : n;
    double s = 0.0;
    for (int64_t i = lo + threadIdx.x; i < hi; i += 256) s = fma(a[i], b[i], s);
    s = block_sum<256>(s, red);
    if (threadIdx.x == 0) out[1 + blockIdx.x] = s;
}
__global__ __launch_bounds__(256) void k_dot_final(double* out) {
    __shared__ double red[4];
    const double s = block_sum<256>(out[1 + threadIdx.x], red);
    if (threadIdx.x == 0) out[0] = s;
}

}  // namespace

// ------------------------------------------------------------------------
// launchers

void launch_cg_at(const BatchDev& B, const UnitsDev& U, hipStream_t s) {
    if (U.grid > 0) hipLaunchKernelGGL(k_cg_at, dim3(U.grid), dim3(kWG), 0, s, B, U);
}
void launch_cg_init(const BatchDev& B, const UnitsDev& U, hipStream_t s) {
    if (U.grid > 0) hipLaunchKernelGGL(k_cg_init, dim3(U.grid), dim3(kWG), 0, s, B, U);
}
bool cg_small_fits(int a_slices, int at_slices, int a_multi, int at_multi) {
    return std::max(a_slices, at_slices) <= kSmallHeld * (kSmallNT / 64) && std::max(a_multi, at_multi) <= kSmallNT;
}
void launch_cg_small(const BatchDev& B, const int* list, int n, int64_t vec_doubles, hipStream_t s) {
    const size_t lds = sizeof(double) * (size_t)(vec_doubles + 544);
    static_assert(kSmallCgDoubles + 544 <= 160 * 1024 / 8, "one workgroup's LDS");
    if (n > 0) hipLaunchKernelGGL(k_cg_small, dim3(n), dim3(kSmallNT), lds, s, B, list);
}
void set_cg_small_lds_limit() {
    V2H_HIP(hipFuncSetAttribute((const void*)k_cg_small, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
}
void launch_cg_a(const BatchDev& B, const UnitsDev& U, hipStream_t s) {
    if (U.grid > 0) hipLaunchKernelGGL(k_cg_a, dim3(U.grid), dim3(kWG), 0, s, B, U);
}
void launch_pre(const BatchDev& B, const UnitsDev& U, hipStream_t s) {
    // every instance: k_pre_reduce also finishes the bookkeeping of instances
    // outside the plan
    if (U.nwg <= 0) return;
    if (U.grid > 0) hipLaunchKernelGGL(k_pre, dim3(U.grid), dim3(kWG), 0, s, B, U);
    hipLaunchKernelGGL(k_pre_reduce, dim3(U.ninst), dim3(kWG), 0, s, B, U);
}
void launch_post(const BatchDev& B, const UnitsDev& U, hipStream_t s) {
    if (U.grid > 0) hipLaunchKernelGGL(k_post, dim3(U.grid), dim3(kWG), 0, s, B, U);
}
void launch_spmv_plain(const SellDev& S, const int4* units, int wg0, int nwg, const double* in, double* out,
                       hipStream_t s) {
    if (nwg > 0) hipLaunchKernelGGL(k_spmv_plain, dim3(nwg), dim3(kWG), 0, s, S, units, wg0, in, out);
}

static int grid_for(int64_t n) {
    int64_t g = (n + 255) / 256;
    return (int)(g < 1 ? 1 : (g > 4096 ? 4096 : g));
}

void launch_fill(double* p, int64_t n, double v, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_fill, dim3(grid_for(n)), dim3(256), 0, s, p, n, v);
}
void launch_copy(double* dst, const double* src, int64_t n, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_copy, dim3(grid_for(n)), dim3(256), 0, s, dst, src, n);
}
void launch_pack_cost(const int32_t* i1, const int32_t* i2, const double* src, double* c, int64_t n, hipStream_t s) {
    if (n > 0) hipLaunchKernelGGL(k_pack_cost, dim3(grid_for(n)), dim3(256), 0, s, i1, i2, src, c, n);
}
void launch_cost_adjoint(const int32_t* ptr, const int32_t* ent, const double* xbar, double* dsrc, int64_t nsrc,
                         hipStream_t s) {
    if (nsrc > 0) hipLaunchKernelGGL(k_cost_adjoint, dim3(grid_for(nsrc)), dim3(256), 0, s, ptr, ent, xbar, dsrc, nsrc);
}
void launch_dot1(const double* a, const double* b, int64_t n, double* out, hipStream_t s) {
    static_assert(kDotParts == 256, "k_dot_final sums one part per thread");
    hipLaunchKernelGGL(k_dot_part, dim3(kDotParts), dim3(256), 0, s, a, b, n, out);
    hipLaunchKernelGGL(k_dot_final, dim3(1), dim3(256), 0, s, out);
}

}  // namespace v2h
