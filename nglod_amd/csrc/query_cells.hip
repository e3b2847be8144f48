// Batch query in the FP32 form for spatially sorted points: launch_sdf_ordered_fp32
// (nglod_sdf_fwd_ordered).  A file of its own: it is built with MFMA results in
// ordinary VGPRs, which the selects and the ReLU read.
#include "api_common.hpp"
#include "cell_gather.hpp"

namespace nglod {

// Batch query of a spatially sorted permutation: thread t evaluates point
// order[t], and a wave's points share cells (gather_cells).  The same bits as
// in input order.  Persistent blocks: the decoder is staged once per block.
template <bool POSINV>
__global__ __launch_bounds__(256) void sdf_ordered_fp32_kernel(ModelArgs m, int lod, int dec,
                                                               const float* __restrict__ x, int64_t n,
                                                               float* __restrict__ out,
                                                               const uint32_t* __restrict__ order) {
    __shared__ Fp32Lds lds;
    stage_fp32_lds(m, dec, &lds);
    __syncthreads();
    const uint32_t lane = lane_id();
    const float b1 = m.b1[dec][0];
    const int64_t waves = (int64_t)gridDim.x * 4;
    for (int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); w * 64 < n; w += waves) {
        const int64_t t = w * 64 + lane;
        const bool valid = t < n;
        const int64_t i = order[valid ? t : n - 1];
        const float px = x[3 * i], py = x[3 * i + 1], pz = x[3 * i + 2];
        const bool use1 = w * 64 + 32 < n;
        CellFeatures f = zero_cell_features();
        for (int l = 0; l <= lod; ++l) gather_cells(m.grid[l], m.res[l], px, py, pz, lane, use1, f);
        const float d = decode_cells<POSINV>(f, &lds, b1, lane, px, py, pz);
        if (valid) out[i] = d;
    }
}

int launch_sdf_ordered_fp32(const ModelArgs& m, int lod, int dec, const float* x, int64_t n, float* out,
                            const uint32_t* order, hipStream_t s) {
    const int64_t blocks = (n + 255) / 256, cap = (int64_t)device_cu_count() * 8;
    const dim3 grid((unsigned)(blocks < cap ? blocks : cap));
    if (m.pos_inv)
        hipLaunchKernelGGL(sdf_ordered_fp32_kernel<true>, grid, dim3(256), 0, s, m, lod, dec, x, n, out, order);
    else
        hipLaunchKernelGGL(sdf_ordered_fp32_kernel<false>, grid, dim3(256), 0, s, m, lod, dec, x, n, out, order);
    return check_launch("sdf_ordered_fp32_kernel");
}

}  // namespace nglod
