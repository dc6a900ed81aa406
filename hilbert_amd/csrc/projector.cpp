// projector.cpp -- grouping of PSD blocks by size class and their launches.
#include "projector.hpp"

#include <algorithm>
#include <cmath>
#include <stdexcept>

#include "kernels.hpp"

namespace v2h {

namespace {
// Projection classes by block size, with the eigensolver of the blocks that
// are not refined: Jacobi up to 16 rows, the tridiagonal path in one wavefront
// per block up to 64, in register tiles up to 192, in registers and LDS up to
// 224, and spread over the GPU beyond (eig_big.hip).
constexpr int kClassTri[Projector::kClasses] = {-1, 0, 1, 2, 3, -1, -1};
int proj_class(int d) {
    if (d <= 16) return 0;
    if (d <= 64) return 1;
    if (d <= 128) return 2;
    if (d <= 192) return 3;
    if (d <= 224) return 4;
    if (d <= 256) return 5;
    return 6;
}
// work doubles of a block: eigenvectors, and above 16 rows reflectors and LU
// factors (7 d^2 in all), above 224 also a few vectors
int64_t work_size(int k, int64_t d) {
    return k == 0 ? d * d : 7 * d * d + (Projector::big_class(k) ? 8 * d : 0);
}
}  // namespace

void Projector::build(const std::vector<std::vector<int>>& dims, std::vector<InstDev>& inst, hipStream_t s) {
    int gblock = 0;
    int64_t work = 0, lam = 0;
    const int count = (int)dims.size();
    std::vector<Refiner::Item> ritems;
    for (auto& c : cls_) c.items.clear();
    lam_begin_.assign(count + 1, 0);
    for (int i = 0; i < count; i++) {
        inst[i].block_first = gblock;
        lam_begin_[i] = lam;
        int nb = 0;
        int64_t off = 0;
        for (const int dim : dims[i]) {
            const int64_t boff = off;
            off += (int64_t)dim * dim;
            if (dim == 0) continue;
            const int k = proj_class(dim);
            if (dim > kBigMaxRows) throw std::invalid_argument("PSD block larger than 2048 is not supported");
            ProjItem it{};
            it.inst = i;
            it.d = dim;
            it.gblock = gblock++;
            it.off = boff;
            it.work_off = work;
            work += work_size(k, dim);
            if (kClassTri[k] >= 0) {
                it.lam_off = lam;
                lam += dim + 1;
            }
            if (!small_class(k)) ritems.push_back(Refiner::Item{i, dim, it.gblock, boff, it.work_off});
            cls_[k].items.push_back(it);
            nb++;
        }
        inst[i].nblocks = nb;
    }
    lam_begin_[count] = lam;
    nblocks_ = gblock;
    small_.clear();
    for (int k = 0; k < kClasses; k++) {
        auto& c = cls_[k];
        c.tri = kClassTri[k];
        std::stable_sort(c.items.begin(), c.items.end(), [](const ProjItem& a, const ProjItem& b) { return a.d > b.d; });
        c.max_d = c.items.empty() ? 0 : c.items.front().d;
        if (!c.items.empty() && c.tri >= 0 && c.max_d > project_tri_max_d(c.tri))
            throw std::logic_error("projection class table is inconsistent");
        c.d_items.upload(c.items);
    }
    std::vector<ProjItem> sitems;
    for (int k : {1, 0})
        for (ProjItem it : cls_[k].items) {
            it.ref = (int)small_.size();
            RefBlock b{};
            b.inst = it.inst;
            b.d = it.d;
            b.gblock = it.gblock;
            b.off = it.off;
            // eigenvectors: after the reflectors of a tridiagonal block
            b.w = it.work_off + (cls_[k].tri >= 0 ? (int64_t)it.d * it.d : 0);
            small_.push_back(b);
            sitems.push_back(it);
        }
    d_small_.upload(small_);
    d_small_items_.upload(sitems);
    d_small_valid_.upload(std::vector<int>(std::max<size_t>(small_.size(), 1), 0));
    proj_part_.alloc(2 * (size_t)std::max(gblock, 1));
    work_.alloc(std::max<int64_t>(work, 1));
    lam_.alloc(std::max<int64_t>(lam, 1));
    launch_fill(lam_.p, std::max<int64_t>(lam, 1), std::nan(""), s);
    refiner_.build(ritems, count, gblock, s);
    refiner_.set_work_base(work_.p);
}

void Projector::forget(int i, hipStream_t s) {
    if (lam_begin_[i + 1] > lam_begin_[i])
        launch_fill(lam_.p + lam_begin_[i], lam_begin_[i + 1] - lam_begin_[i], std::nan(""), s);
    launch_ref_small_forget(small_dev(), (int)small_.size(), i, s);
    refiner_.forget(i, s);
}

void Projector::launch(int k, const BatchDev& B, hipStream_t s, int route) const {
    const Class& c = cls_[k];
    if (c.items.empty()) return;
    const int n = (int)c.items.size();
    if (small_class(k)) {
        const SmallDev R = small_dev();
        const int n1 = (int)cls_[1].items.size(), all = (int)small_.size();
        if (refine_on_) launch_ref_small(B, R, refiner_.params(), n1, all, c.max_d, s);
        launch_project_small(B, d_small_items_.p, all, work_.p, lam_.p, max_sweeps_, refine_on_ ? R.vvalid : nullptr,
                             R.route, s);
    } else {
        launch_project_tri(c.tri, B, c.d_items.p, n, work_.p, lam_.p,
                           route >= 0 && refined_class(k) && refine_on() ? refiner_.route() : nullptr, route, s);
    }
}

}  // namespace v2h
