// refine.hpp -- warm-started PSD projection on the FP64 matrix cores: blocks
// above 64 rows by launches over their tiles (refine.hip), blocks of up to 64
// rows by one launch per size class (refine_small.hip).
//
// Between two outer iterations of BPSDP, U = mu x + A^T y - c changes little,
// so the eigenvectors of the previous iteration almost diagonalise the new U.
// Each outer iteration refines them with the iteration of Ogita and Aishima
// (Japan J. Indust. Appl. Math. 35, 1007 (2018)), whose steps are matrix
// products only:
//     G = X^T X,  S = X^T U X  (X with normalised columns),  r = I - G,
//     l_i = s_ii,  a_ij = s_ij + (l_i + l_j) r_ij / 2,
//     E_ij = r_ij / 2 + 2 a_ij / (l_j - l_i +- sqrt((l_j - l_i)^2 + 4 a_ij^2)),
//     X <- X + X E
// (the second term is their a_ij / (l_j - l_i) for small a_ij, limited like a
// Jacobi rotation), which converges quadratically, restores the orthogonality
// of X in the same step, and then U+ = X diag(l+) X^T.  Pairs inside a cluster
// threshold keep only r_ij / 2 and, beside diag(l+), their coupling a_ij.  A block
// whose correction does not fall below the acceptance threshold within
// max_steps steps, and every block without eigenvectors yet (first iteration,
// after a reset), takes a tridiagonal eigensolver instead (eig_tri.hip, above
// 224 rows eig_big.hip); its eigenvectors seed the next iteration.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "common.hpp"
#include "dbuf.hpp"

namespace v2h {

// One block on the refined path.
struct RefBlock {
    int inst, d, gblock, nt;  // nt: 32-row tiles per side
    int64_t off;              // primal offset of the block inside its instance
    int64_t w;                // work area (doubles): kRefSlots d x d matrices, then d eigenvalues
    int64_t tri;              // the block's tridiagonal work area (reflectors, eigenvectors)
    int64_t part;             // first tile-partial pair (2 doubles per tile)
};
// Matrices of a block's work area, row-major d x d each.
enum RefSlot : int { kSlotV = 0, kSlotU = 1, kSlotXa = 2, kSlotXb = 3, kSlotK = 4, kSlotS = 5, kSlotG = 6 };
constexpr int kRefSlots = 7;

// One 32 x 32 output tile of one block.
struct RefJob {
    int blk, ti, tj, tile;
};

// Per-block state of the refinement.
struct RefState {
    int vvalid;     // slot V holds eigenvector estimates of a recent U
    int phase;      // 0 idle, 1 refining, 2 accepted (at step cstep), 3 rejected, kPhaseFresh
    int cstep;      // step whose correction was accepted
    int xfinal;     // slot of the accepted X
    double max_e;   // largest correction of the last step
    double cpl;     // largest coupling of a cluster across zero, relative
    // accepted with coupled clusters: pairs within om in gap and coupling whose
    // coupling is above keep stay coupled in U+ = X (L+ + C) X^T
    double om, keep;
    int coupled;
    int ticket;     // tiles of the block that finished the current step
    int64_t refined, fallback;  // counts of outer iterations on each path
    // rejections: diverging or non-finite corrections, correction above the
    // acceptance threshold after the last step, clusters left coupled
    int64_t rej_div, rej_e, rej_c;
    // FP64 flops of the block's d x d x d products so far (2 d^3 each: K, G,
    // S and X + XE per step, the final X diag(l+) X^T)
    int64_t flops;
    // After a rejection the block stays on the fallback for `wait` outer
    // iterations (doubling with consecutive rejections, up to kMaxBackoff);
    // its eigenvectors are formed only for the iteration before it tries again.
    int wait, backoff;
    // The instance was running when this iteration's projection began (set
    // by k_ref_state).  The eigenvector formation reads it instead of the
    // instance state, which the next k_pre_reduce on the main stream may
    // change while the formation runs on its side stream.
    int live, pad;
};
constexpr int kMaxBackoff = 64;
constexpr int kPhaseFresh = 4;  // slot V holds eigenvectors of this iteration's U (eig_big.hip)
// Blocks up to kTriMaxRows have a tridiagonal eigensolver in one workgroup, the
// larger ones, up to kBigMaxRows, that of eig_big.hip.
constexpr int kTriMaxRows = 224, kBigMaxRows = 2048;

struct RefDev {
    const RefBlock* blk;
    const RefJob* jobs;
    RefState* rs;
    int* route;         // [global block]: how this iteration projects the block (kRoute*)
    double* work;
    double* part;
    double* tri_work;
    int nblk, njobs;
};

// Route of a block of the refined classes in the current outer iteration:
// the tridiagonal fallback known at its start (no eigenvectors, backoff),
// refining, rejected during the refinement (fallback after it), accepted.
enum Route : int { kRouteFallback = 0, kRouteRefining = 1, kRouteRejected = 2, kRouteAccepted = 3 };

// Thresholds of the refinement.
// A step whose largest correction is eps leaves off-diagonal couplings and an
// orthogonality error of order eps^2 (measured: U+ within 7.5e-11 relative of
// LAPACK at eps = 1e-6 on (16e,16o) blocks, so the default keeps it near
// 3e-12).
struct RefParams {
    double cluster_rel = 1e-8;   // |l_i - l_j| <= cluster_rel max|l|: one cluster
    double accept_e = 2e-7;      // accept a step whose largest correction is below this
    double accept_cpl = 1e-13;   // ... and whose clusters across zero are decoupled to this (relative to max|l|)
    // refinement steps before a block is rejected (1..kMaxSteps): 7 keeps
    // most blocks that converge slowly off the tridiagonal fallback, whose
    // launch after the refinement is on the critical path of the iteration
    // (8 (6e,6o) SDPs with T2: 3.02 / 2.05 / 1.55 / 1.37 ms per outer iteration
    // with 5 / 6 / 7 / 8 steps; a step that finds nothing to do costs 7 us,
    // 1 % of a (16e,16o) iteration)
    int max_steps = 7;
};
constexpr int kMaxSteps = 8;

// Start of an outer iteration: phases, backoff and routes of every block.
void launch_ref_state(const BatchDev& B, const RefDev& R, hipStream_t s);
// sym(U) of the refining blocks.
void launch_ref_sym(const BatchDev& B, const RefDev& R, hipStream_t s);
// One refinement step k (1..max_steps): X_in = V (k = 1), then Xa and Xb in turn.
void launch_ref_step(const BatchDev& B, const RefDev& R, const RefParams& P, int k, hipStream_t s);
// x = X diag(l+) X^T / mu with z, v1, partial sums; the block's projection sums.
void launch_ref_final(const BatchDev& B, const RefDev& R, hipStream_t s);
// Eigenvectors of the blocks that took the tridiagonal path this iteration.
void launch_ref_form_v(const BatchDev& B, const RefDev& R, hipStream_t s);
// x, z and sums of the blocks whose eigenvectors eig_big.hip just computed.
void launch_ref_fresh(const BatchDev& B, const RefDev& R, hipStream_t s);
// eig_big.hip: which of the n blocks list[] need the eigensolver, and the
// eigenvectors of those (max_d: the largest of them); returns its launches.
void launch_big_need(const BatchDev& B, const RefDev& R, const int* list, int n, bool refined, int* need,
                     hipStream_t s);
int launch_big_eig(const BatchDev& B, const RefDev& R, const int* list, const int* need, int n, int max_d,
                   hipStream_t s);
void launch_ref_forget(const RefDev& R, int blk_begin, int blk_end, hipStream_t s);

// Blocks of up to 64 rows (refine_small.hip): one launch does the whole
// refinement; the blocks that it does not accept keep a route other than
// kRouteAccepted and are projected by an eigensolver right after it
// (launch_project_small), which leaves their eigenvectors in the work area and
// sets vvalid.  There is no backoff: a failed attempt costs little.
struct SmallDev {
    const RefBlock* blk;  // blocks of 17..64 rows, then those of up to 16; w: the eigenvectors (d x d) in `work`
    int* vvalid;
    int* route;
    double* work;
};
// n1 blocks of 17..64 rows, n in all, the largest of max_d rows
void launch_ref_small(const BatchDev& B, const SmallDev& R, const RefParams& P, int n1, int n, int max_d,
                      hipStream_t s);
void launch_ref_small_forget(const SmallDev& R, int n, int inst, hipStream_t s);

class Refiner {
  public:
    // items of the tridiagonal classes that take the refined path
    struct Item {
        int inst, d, gblock;
        int64_t off, tri;
    };
    void build(const std::vector<Item>& items, int count, int nblocks_total, hipStream_t s);
    bool empty() const { return blk_.empty(); }
    // One outer iteration: begin() sets every block's route (the fallback
    // launches for kRouteFallback may start right after it); refine() runs
    // the refinement and routes its rejections to kRouteRejected.
    void begin(const BatchDev& B, hipStream_t s) const;
    void refine(const BatchDev& B, hipStream_t s) const;
    // kernel launches of begin() + refine(): state, sym, four per step, middle factor, final product and close
    int launches() const { return 5 + 4 * params_.max_steps; }
    // Projection of the blocks above kTriMaxRows that the refinement has not
    // taken (refined), or of all of them; the former waits for the refinement on
    // the host.  Returns the kernel launches.
    bool has_big() const { return !big_.empty(); }
    int project_big(const BatchDev& B, bool refined, hipStream_t s);
    // After the fallback: eigenvectors of the blocks it projected.
    void seed(const BatchDev& B, hipStream_t s) const;
    void forget(int inst, hipStream_t s) const;
    int* route() const { return route_.p; }
    // [block projections by the refinement, by the fallback, rejections for
    // divergence, for the correction size, for coupled clusters]
    static constexpr int kStats = 6;
    void stats(int64_t* out) const;
    void set_work_base(double* tri_work) { tri_work_ = tri_work; }
    void set_params(const RefParams& p) { params_ = p; }
    const RefParams& params() const { return params_; }

  private:
    RefDev dev() const;
    std::vector<RefBlock> blk_;
    std::vector<int> inst_begin_;  // [count + 1] refine blocks of each instance
    int njobs_ = 0;
    RefParams params_;
    DBuf<RefBlock> d_blk_;
    DBuf<RefJob> d_jobs_;
    DBuf<RefState> d_rs_;
    DBuf<int> route_;
    DBuf<double> work_, part_;
    double* tri_work_ = nullptr;
    std::vector<int> big_, need_host_;  // blocks above kTriMaxRows
    int big_max_ = 0;
    DBuf<int> d_big_, need_;
};

}  // namespace v2h
