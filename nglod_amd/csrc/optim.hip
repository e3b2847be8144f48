// The training step's loss and parameter update, a launch or two each.
//   nglod_geometry_loss   sum over levels of sum (pred - gt)^2 / n and its
//                         gradient (Trainer.step_geometry,
//                         sdf-net/lib/trainer.py:325-337)
//   nglod_adam_step       torch.optim.Adam's update of many tensors (:184-185)
#include "api_common.hpp"

namespace nglod {

constexpr int kLossBlocks = 256;

// grad = (1 / n) * (2 (pred - gt)) as autograd forms it; the loss in FP64
// partials per block, in a fixed order.
__global__ __launch_bounds__(256) void loss_kernel(const float* __restrict__ pred, const float* __restrict__ gt,
                                                   int64_t n, int levels, uint32_t mask, float inv,
                                                   float* __restrict__ grad, double* __restrict__ partial) {
    double s = 0.0;
    for (int l = 0; l < levels; ++l) {
        const bool on = (mask >> l) & 1u;
        for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
            const float d = pred[(size_t)l * n + i] - gt[i];
            grad[(size_t)l * n + i] = on ? inv * (2.0f * d) : 0.0f;
            if (on) s += (double)(d * d);
        }
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    __shared__ double ws[4];
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) partial[blockIdx.x] = ((ws[0] + ws[1]) + ws[2]) + ws[3];
}

__global__ __launch_bounds__(64) void loss_final_kernel(const double* __restrict__ partial, int blocks, int64_t n,
                                                        float* __restrict__ loss) {
    double s = 0.0;
    for (int b = threadIdx.x; b < blocks; b += 64) s += partial[b];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (threadIdx.x == 0) loss[0] = (float)(s / (double)n);
}

// Tensors of one launch, by value; block b works on tensor t with
// first[t] <= b < first[t + 1], kAdamChunk elements from (b - first[t]) kAdamChunk.
constexpr int kAdamTensors = 64;
constexpr int kAdamChunk = 4096;

struct AdamArgs {
    float* p[kAdamTensors];
    const float* g[kAdamTensors];
    float* m[kAdamTensors];
    float* v[kAdamTensors];
    int64_t n[kAdamTensors];
    uint32_t first[kAdamTensors + 1];
    int count;
    float w1, w1_rest, beta2, w2, bias2_sqrt, eps, step;
};

// One element, rounding as torch's multi-tensor Adam on this GPU does (checked
// bit for bit): m by an FMA (lerp, which starts from the nearer end: beta1 = 0 gives g
// itself), v = fma(1 - beta2, g g, v beta2), the update p = fma(-lr / bias1, m /
// (sqrt(v) / bias2_sqrt + eps), p).
__device__ __forceinline__ void adam_one(const AdamArgs& a, float& p, float g, float& m, float& v) {
    const float d1 = g - m;
    m = a.w1 < 0.5f ? __builtin_fmaf(a.w1, d1, m) : __builtin_fmaf(-d1, a.w1_rest, g);
    v = __builtin_fmaf(a.w2, g * g, v * a.beta2);
    const float d = sqrtf(v) / a.bias2_sqrt + a.eps;
    p = __builtin_fmaf(a.step, m / d, p);
}

// Every parameter in one pass: p, g, m and v read once, p, m and v written once
// (10.1 M parameters, 284 MB: 47 us, 6.0 TB/s; the eight passes of the multi-tensor
// operators 0.19 ms and eight launches).
__global__ __launch_bounds__(256) void adam_kernel(AdamArgs a) {
    int lo = 0, hi = a.count - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (a.first[mid] <= blockIdx.x) lo = mid;
        else hi = mid - 1;
    }
    const int64_t b0 = (int64_t)(blockIdx.x - a.first[lo]) * kAdamChunk;
    const int64_t n = a.n[lo];
    const int64_t b1 = b0 + kAdamChunk < n ? b0 + kAdamChunk : n;
    float* P = a.p[lo];
    const float* G = a.g[lo];
    float* M = a.m[lo];
    float* V = a.v[lo];
    const bool wide = ((((uintptr_t)P | (uintptr_t)G | (uintptr_t)M | (uintptr_t)V) & 15u) == 0);
    if (wide) {
        for (int64_t i = b0 + 4 * threadIdx.x; i + 3 < b1; i += 1024) {
            float4 p = *reinterpret_cast<float4*>(P + i), m = *reinterpret_cast<float4*>(M + i),
                   v = *reinterpret_cast<float4*>(V + i);
            const float4 g = *reinterpret_cast<const float4*>(G + i);
            adam_one(a, p.x, g.x, m.x, v.x);
            adam_one(a, p.y, g.y, m.y, v.y);
            adam_one(a, p.z, g.z, m.z, v.z);
            adam_one(a, p.w, g.w, m.w, v.w);
            *reinterpret_cast<float4*>(P + i) = p;
            *reinterpret_cast<float4*>(M + i) = m;
            *reinterpret_cast<float4*>(V + i) = v;
        }
    }
    // the last elements of a tensor, or all of a chunk that is not 16-byte aligned
    const int64_t rest = wide ? b0 + (b1 - b0) / 4 * 4 : b0;
    for (int64_t i = rest + threadIdx.x; i < b1; i += 256) {
        float p = P[i], m = M[i], v = V[i];
        adam_one(a, p, G[i], m, v);
        P[i] = p;
        M[i] = m;
        V[i] = v;
    }
}

}  // namespace nglod

using namespace nglod;

extern "C" {

size_t nglod_geometry_loss_workspace_size(void) { return kLossBlocks * sizeof(double); }

int nglod_geometry_loss(const float* pred, const float* gt, int64_t n, int32_t levels, uint32_t level_mask, float* grad,
                        float* loss, void* workspace, size_t workspace_bytes, void* stream) {
    if (n < 1 || levels < 1 || levels > NGLOD_MAX_LODS) return fail(NGLOD_ERR_ARG, "size out of range");
    if (!pred || !gt || !grad || !loss) return fail(NGLOD_ERR_ARG, "NULL pointer");
    if (!workspace || workspace_bytes < nglod_geometry_loss_workspace_size() || ((uintptr_t)workspace & 7))
        return fail(NGLOD_ERR_WORKSPACE, "workspace too small or misaligned");
    hipStream_t s = (hipStream_t)stream;
    const int64_t want = (n + 255) / 256;
    const int blocks = (int)(want < kLossBlocks ? want : kLossBlocks);
    hipLaunchKernelGGL(loss_kernel, dim3(blocks), dim3(256), 0, s, pred, gt, n, levels, level_mask, 1.0f / (float)n,
                       grad, (double*)workspace);
    hipLaunchKernelGGL(loss_final_kernel, dim3(1), dim3(64), 0, s, (const double*)workspace, blocks, n, loss);
    return check_launch("loss_kernel");
}

int nglod_adam_step(float* const* p, const float* const* g, float* const* m, float* const* v, const int64_t* n,
                    int32_t count, double beta1, double beta2, double eps, double lr, int64_t step, void* stream) {
    if (count < 0 || step < 1) return fail(NGLOD_ERR_ARG, "size out of range");
    if (count > 0 && (!p || !g || !m || !v || !n)) return fail(NGLOD_ERR_ARG, "NULL pointer");
    AdamArgs a;
    a.w1 = (float)(1.0 - beta1);
    a.w1_rest = 1.0f - a.w1;
    a.beta2 = (float)beta2;
    a.w2 = (float)(1.0 - beta2);
    a.bias2_sqrt = (float)pow(1.0 - pow(beta2, (double)step), 0.5);
    a.eps = (float)eps;
    a.step = (float)((lr / (1.0 - pow(beta1, (double)step))) * -1.0);
    for (int i = 0; i < count;) {
        uint64_t blocks = 0;
        a.count = 0;
        for (; i < count && a.count < kAdamTensors; ++i) {
            if (n[i] < 0) return fail(NGLOD_ERR_ARG, "negative size");
            if (n[i] == 0) continue;
            if (!p[i] || !g[i] || !m[i] || !v[i]) return fail(NGLOD_ERR_ARG, "NULL pointer");
            const uint64_t more = ((uint64_t)n[i] + kAdamChunk - 1) / kAdamChunk;
            if (more > ((uint64_t)1 << 23)) return fail(NGLOD_ERR_ARG, "tensor too large");
            if (blocks + more > ((uint64_t)1 << 23)) break;  // below the 2^32 threads of a launch
            a.p[a.count] = p[i];
            a.g[a.count] = g[i];
            a.m[a.count] = m[i];
            a.v[a.count] = v[i];
            a.n[a.count] = n[i];
            a.first[a.count++] = (uint32_t)blocks;
            blocks += more;
        }
        if (a.count == 0) continue;
        a.first[a.count] = (uint32_t)blocks;
        hipLaunchKernelGGL(adam_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, a);
        const int rc = check_launch("adam_kernel");
        if (rc) return rc;
    }
    return NGLOD_OK;
}

}  // extern "C"
