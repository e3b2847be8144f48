// The sparse model's arguments and the ray / voxel test of its march, shared by
// the two sparse march kernels (SDF::sphereTrace, sol-renderer/SDF.cu:218-472).
#pragma once

#include "trace_common.hpp"

namespace nglod {

struct SolArgs {
    int target, lod, din;
    const int16_t* points;
    int64_t psum_target;  // global index of the first point of level `target`
    const uint32_t* tv;   // [P][8]
    const int32_t* parent;
    const int32_t* cc;    // [Nc][3]
    const float* cf;      // [Nc][32]
    const float* w0;
    const float* b0;
    const float* w1;
    const float* b1;
    // rays
    const float* o;
    const float* d;
    int64_t n;
    const int32_t* offs;  // [n+1] CSR over nuggets
    const int32_t* nug;   // [M][2]
    float* x;
    float* t;
    uint8_t* hit;
    float* normal;
    int32_t* iters;
    uint32_t* queue;
    unsigned long long* evals;
    float r;  // voxel half size at `target`
};

__device__ __forceinline__ float sol_ray_aabb(float qx, float qy, float qz, float dx, float dy, float dz, float ivx,
                                              float ivy, float ivz, float sx_, float sy_, float sz_, float cx, float cy,
                                              float cz, float r) {
    const float ox = qx - cx, oy = qy - cy, oz = qz - cz;
    const float cmax = fmaxf(fmaxf(fabsf(ox), fabsf(oy)), fabsf(oz));
    float winding = cmax < r ? -1.0f : 1.0f;
    winding *= r;
    if (winding < 0) return winding;
    const float d0 = __builtin_fmaf(winding, sx_, -ox) * ivx;
    const float d1 = __builtin_fmaf(winding, sy_, -oy) * ivy;
    const float d2 = __builtin_fmaf(winding, sz_, -oz) * ivz;
    const float ltxy = __builtin_fmaf(dy, d0, oy), ltxz = __builtin_fmaf(dz, d0, oz);
    const float ltyx = __builtin_fmaf(dx, d1, ox), ltyz = __builtin_fmaf(dz, d1, oz);
    const float ltzx = __builtin_fmaf(dx, d2, ox), ltzy = __builtin_fmaf(dy, d2, oy);
    const bool t0 = (d0 >= 0.0f) && (fabsf(ltxy) < r) && (fabsf(ltxz) < r);
    const bool t1 = (d1 >= 0.0f) && (fabsf(ltyx) < r) && (fabsf(ltyz) < r);
    const bool t2 = (d2 >= 0.0f) && (fabsf(ltzx) < r) && (fabsf(ltzy) < r);
    float ssx = 0.0f, ssy = 0.0f, ssz = 0.0f;
    if (t0) ssx = sx_;
    else if (t1) ssy = sy_;
    else if (t2) ssz = sz_;
    float dd = 0.0f;
    if (ssx != 0.0f) dd = d0;
    else if (ssy != 0.0f) dd = d1;
    else if (ssz != 0.0f) dd = d2;
    return dd;
}

// Levels whose corner tables trace_sparse_group_kernel holds in LDS: 2 KB a level,
// 34 KB in all (four blocks share a CU's 160).
constexpr int kSolGroupLevels = 8;

int launch_trace_sparse_group(const SolArgs& a, hipStream_t s);

}  // namespace nglod
