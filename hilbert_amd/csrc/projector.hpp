// projector.hpp -- the PSD projection of every block of a batch: blocks
// grouped by size class, one launch per class and outer iteration, and the
// device work areas the classes need.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "common.hpp"
#include "dbuf.hpp"
#include "refine.hpp"

namespace v2h {

class Projector {
  public:
    // d <= 16 / 64 / 128 / 192 / 224 / 256, d > 256
    static constexpr int kClasses = 7;

    // dims[i]: PSD block sizes of instance i in primal order (zeros allowed);
    // fills block_first / nblocks of inst[i].  Blocks are numbered
    // consecutively (the index of a block's partial sums in proj_part()).
    void build(const std::vector<std::vector<int>>& dims, std::vector<InstDev>& inst, hipStream_t s);
    // forget instance i's eigenvalues (the warm start of the tridiagonal path)
    void forget(int i, hipStream_t s);
    // Classes 0 and 1 (up to 64 rows) share their launches: class 0 is
    // launched with class 1 where a batch has both.
    // Classes 5 and 6 are projected by project_big.
    bool has(int k) const { return !cls_[k].items.empty() && !big_class(k) && !(k == 0 && !cls_[1].items.empty()); }
    // The launch of class k.  With the refinement on, a refined class (2..4)
    // is launched twice per outer iteration: route kRouteFallback (blocks known
    // to need the tridiagonal eigensolver when the iteration starts, alongside
    // the refinement) and kRouteRejected (after it); route < 0: every block.
    void launch(int k, const BatchDev& B, hipStream_t s, int route = -1) const;
    int64_t nblocks() const { return nblocks_; }
    double* proj_part() const { return proj_part_.p; }

    // Warm-started refinement (refine.hpp): on by default.  The classes of up
    // to 64 rows refine inside launch(); the others by the calls below.
    static bool small_class(int k) { return k <= 1; }
    static bool refined_class(int k) { return k >= 2 && k <= 4; }
    static bool big_class(int k) { return k >= 5; }
    // Classes 5 and 6: after refine_run where the refinement is on.  Returns the
    // kernel launches.
    bool has_big() const { return refiner_.has_big(); }
    int project_big(const BatchDev& B, hipStream_t s) { return refiner_.project_big(B, refine_on(), s); }
    bool refine_on() const { return refine_on_ && !refiner_.empty(); }
    void set_refine(bool on) { refine_on_ = on; }
    void refine_begin(const BatchDev& B, hipStream_t s) const { refiner_.begin(B, s); }
    void refine_run(const BatchDev& B, hipStream_t s) const { refiner_.refine(B, s); }
    void refine_seed(const BatchDev& B, hipStream_t s) const { refiner_.seed(B, s); }
    void refine_stats(int64_t* out) const { refiner_.stats(out); }
    void set_refine_params(const RefParams& p) { refiner_.set_params(p); }
    const RefParams& refine_params() const { return refiner_.params(); }
    int refine_launches() const { return refiner_.launches(); }
    // kernel launches of launch(k)
    int class_launches(int k) const { return small_class(k) && refine_on_ ? 2 : 1; }

  private:
    struct Class {
        int max_d = 0;
        int tri = -1;  // tridiagonal kernel class of eig_tri.hip, or -1
        std::vector<ProjItem> items;
        DBuf<ProjItem> d_items;
    };
    Class cls_[kClasses];
    SmallDev small_dev() const { return SmallDev{d_small_.p, d_small_valid_.p, refiner_.route(), work_.p}; }
    DBuf<double> proj_part_, work_, lam_;
    std::vector<RefBlock> small_;    // class 1, then class 0, each in the order of its items
    DBuf<RefBlock> d_small_;
    DBuf<ProjItem> d_small_items_;
    DBuf<int> d_small_valid_;
    std::vector<int64_t> lam_begin_;  // [count + 1] eigenvalue-store range of each instance
    int64_t nblocks_ = 0;
    int max_sweeps_ = 24;
    Refiner refiner_;
    bool refine_on_ = true;
};

}  // namespace v2h
