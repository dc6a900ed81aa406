// kernels.hpp -- host-side launchers of the HIP kernels (kernels.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "common.hpp"

namespace v2h {

void launch_cg_init(const BatchDev& B, const UnitsDev& U, hipStream_t s);  // U: the units of A
// The CG of the n small instances list[] (those running); vec_doubles: the most
// LDS doubles that one of them needs (n_primal + n_dual + the partial sums of the
// wider operator).  cg_small_fits: whether an operator's pieces fit the registers.
bool cg_small_fits(int a_slices, int at_slices, int a_multi, int at_multi);
void launch_cg_small(const BatchDev& B, const int* list, int n, int64_t vec_doubles, hipStream_t s);
void set_cg_small_lds_limit();
void launch_cg_at(const BatchDev& B, const UnitsDev& U, hipStream_t s);
void launch_cg_a(const BatchDev& B, const UnitsDev& U, hipStream_t s);
void launch_pre(const BatchDev& B, const UnitsDev& U, hipStream_t s);
void launch_post(const BatchDev& B, const UnitsDev& U, hipStream_t s);
void launch_spmv_plain(const SellDev& S, const int4* units, int wg0, int nwg, const double* in, double* out,
                       hipStream_t s);

// Tridiagonal projection (eig_tri.hip), classes 0..3 for blocks up to
// 64 / 128 / 192 / 224.  work: 7 d^2 doubles per block; lam: d + 1 doubles per block, kept between calls
// (NaN = no previous eigenvalues).  route (may be null, classes 1-3): only
// blocks with route[global block] == want are projected.  Each reflector's tau
// is kept on the diagonal of the reflector matrix (row k, column k).
int project_tri_max_d(int cls);
// Blocks of up to 64 rows, one wavefront per block (tridiagonal class 0, Jacobi
// up to 16 rows).  Each block's eigenvectors are left after its reflectors, at
// work + work_off + d^2 (up to 16 rows: at work + work_off).  vvalid (may be
// null): only the blocks whose route is not kRouteAccepted are projected, and
// their vvalid[ref] is set.
void launch_project_small(const BatchDev& B, const ProjItem* items, int nitems, double* work, double* lam,
                          int max_sweeps, int* vvalid, const int* route, hipStream_t s);
void launch_project_tri(int cls, const BatchDev& B, const ProjItem* items, int nitems, double* work, double* lam,
                        const int* route, int want, hipStream_t s);

void launch_fill(double* p, int64_t n, double v, hipStream_t s);
void launch_copy(double* dst, const double* src, int64_t n, hipStream_t s);
void launch_pack_cost(const int32_t* i1, const int32_t* i2, const double* src, double* c, int64_t n,
                      hipStream_t s);
void launch_cost_adjoint(const int32_t* ptr, const int32_t* ent, const double* xbar, double* dsrc, int64_t nsrc,
                         hipStream_t s);
// out[0] = a . b; out[1..256] receive the partial sums
void launch_dot1(const double* a, const double* b, int64_t n, double* out, hipStream_t s);

}  // namespace v2h
