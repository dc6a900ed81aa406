// wave_ops.hpp -- cross-lane exchange and sums of doubles in one wavefront.
#pragma once

#include <hip/hip_runtime.h>

namespace v2h {

namespace {

// ---- cross-lane exchange of doubles (DPP within rows of 16 lanes, ds_swizzle
// within 32).  Every lane of the wavefront must be active.
template <int CTRL>
__device__ __forceinline__ double dpp(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
    return __hiloint2double(hi, lo);
}
template <int PATTERN>
__device__ __forceinline__ double swz(double v) {
    const int lo = __builtin_amdgcn_ds_swizzle(__double2loint(v), PATTERN);
    const int hi = __builtin_amdgcn_ds_swizzle(__double2hiint(v), PATTERN);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_value(double v, int l) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), l),
                            __builtin_amdgcn_readlane(__double2loint(v), l));
}
constexpr int kQuadXor1 = 0xB1;      // quad_perm [1,0,3,2]
constexpr int kQuadXor2 = 0x4E;      // quad_perm [2,3,0,1]
constexpr int kRowHalfMirror = 0x141;
constexpr int kRowMirror = 0x140;
constexpr int kRowRor8 = 0x128;      // rotate by 8 in a row of 16 = lane xor 8
constexpr int kSwzXor4 = (4 << 10) | 0x1F;
constexpr int kSwzXor16 = (16 << 10) | 0x1F;

// Sum over the 64 lanes; every lane receives the same total.
__device__ __forceinline__ double wsum(double v) {
    v += dpp<kQuadXor1>(v);
    v += dpp<kQuadXor2>(v);
    v += dpp<kRowHalfMirror>(v);
    v += dpp<kRowMirror>(v);
    v += swz<kSwzXor16>(v);
    return lane_value(v, 0) + lane_value(v, 32);
}

}  // namespace

}  // namespace v2h
