// Batch SDF queries in spatial order: nglod_sdf_fwd_ordered.
//
// Uniformly scattered query points put unrelated grid cells in neighbouring
// lanes, so a wave's corner loads touch as many cache lines as it has lanes.
// Sorting the points by the Morton code of their cell first gives a wave few
// cells: the FP32 kernel then interpolates cell by cell (cell_gather.hpp), the
// mixed one finds its lines in L1 and L2.  The batch kernels evaluate point
// order[t] in thread t and write out[order[t]].
#include <cstring>

#include "api_common.hpp"
#include "radix_sort.hpp"

namespace nglod {

// Spreads the low 10 bits of v to every third bit.
__device__ __forceinline__ uint32_t spread3(uint32_t v) {
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Key of a point: the Morton code of its cell in a grid of resolution r, less
// its low `drop` bits.
__global__ void morton_keys_kernel(const float* __restrict__ x, int64_t n, int r, int drop,
                                   uint32_t* __restrict__ keys) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t qx = (uint32_t)axis_weights(x[3 * i], r).i0, qy = (uint32_t)axis_weights(x[3 * i + 1], r).i0,
                   qz = (uint32_t)axis_weights(x[3 * i + 2], r).i0;
    keys[i] = ((spread3(qz) << 2) | (spread3(qy) << 1) | spread3(qx)) >> drop;
}

// Sorted bits: the finest grid's cells as far as a bin of the order still holds
// about a wave's 64 points (the cells of a wave need not be in runs).  Each 8
// bits are a pass over the pairs: 2^22 points at LOD 4 take two passes instead
// of the four of a 30-bit position code.
static int order_bits(int64_t n, int r, int* drop) {
    int axis = 0, want = 1;
    while ((1 << axis) < r) ++axis;
    while (((int64_t)64 << want) < n) ++want;
    const int all = 3 * axis > 0 ? 3 * axis : 1;
    *drop = all > want ? all - want : 0;
    return all - *drop;
}

// The evaluation order of n points over a grid of resolution r, in a checked
// workspace of sort_workspace_bytes(n).
int launch_cell_order(const float* x, int64_t n, int r, void* workspace, size_t workspace_bytes,
                      const uint32_t** order, hipStream_t s) {
    if (!workspace || workspace_bytes < sort_workspace_bytes(n))
        return fail(NGLOD_ERR_WORKSPACE, "workspace too small");
    if (!aligned16(workspace)) return fail(NGLOD_ERR_ARG, "workspace not 16-byte aligned");
    const SortBuffers sb = sort_buffers(workspace, n);
    int drop = 0;
    const int bits = order_bits(n, r, &drop);
    hipLaunchKernelGGL(morton_keys_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, x, n, r, drop,
                       sb.keys[0]);
    *order = sb.vals[launch_sort(sb, n, bits, s)];
    return check_launch("sort_scatter_kernel");
}

}  // namespace nglod

using namespace nglod;

extern "C" {

size_t nglod_sdf_fwd_ordered_workspace_size(int64_t n) { return sort_workspace_bytes(n < 1 ? 1 : n); }

int nglod_sdf_fwd_ordered(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, int32_t form, float* out,
                          void* workspace, size_t workspace_bytes, void* stream) {
    ModelArgs m;
    int rc = make_model_args(model, lod, form, &m);
    if (rc) return rc;
    if (n < 0 || n > (int64_t)0x7fff0000) return fail(NGLOD_ERR_ARG, "n out of range");
    if (n == 0) return NGLOD_OK;
    if (!x || !out) return fail(NGLOD_ERR_ARG, "NULL pointer");
    hipStream_t s = (hipStream_t)stream;
    const uint32_t* order = nullptr;
    rc = launch_cell_order(x, n, model->res[lod], workspace, workspace_bytes, &order, s);
    if (rc) return rc;
    const int dec = decoder_of(model, lod);
    if (form == NGLOD_MIXED) return launch_sdf_mixed(m, 0, dec, x, n, out, order, s);
    return launch_sdf_ordered_fp32(m, lod, dec, x, n, out, order, s);
}

}  // extern "C"
