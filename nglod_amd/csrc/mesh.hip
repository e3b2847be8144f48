// Samples of the mesh the model is fitted to (the distances: mesh_sdf.hip).
//   nglod_sample_uniform   points uniform in [-1,1]^3      (torchgp/sample_uniform.py)
//   nglod_sample_surface   area-weighted surface points (+ Gaussian offset)
//                          (torchgp/sample_surface.py, sample_near_surface.py)
#include "api_common.hpp"

namespace nglod {

// ---------------------------------------------------------------------------
// Counter-based RNG: SplitMix64 (Steele, Lea, Flood 2014) of (sample, draw).
__device__ __forceinline__ uint64_t splitmix64(uint64_t x) {
    uint64_t z = x + 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

__device__ __forceinline__ double rnd01(uint64_t seed, uint64_t i, uint32_t k) {
    const uint64_t z = splitmix64(seed ^ splitmix64(i * 8ull + k));
    return (double)(z >> 40) * (1.0 / 16777216.0);
}

__global__ void sample_uniform_kernel(uint64_t seed, int64_t n, float* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    for (int k = 0; k < 3; ++k) out[3 * i + k] = (float)(rnd01(seed, (uint64_t)i, (uint32_t)k) * 2.0 - 1.0);
}

// Directions uniform on S^2 (geoutils.sample_unif_sphere, sdf-net/lib/geoutils.py:31-40):
// z = 1 - 2u, phi = 2*pi*v, (sqrt(1 - z^2) cos phi, sqrt(1 - z^2) sin phi, z).
__global__ void sample_directions_kernel(uint64_t seed, int64_t n, float* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double z = 1.0 - 2.0 * rnd01(seed, (uint64_t)i, 0);
    const double r = sqrt(1.0 - z * z);
    const double phi = 2.0 * M_PI * rnd01(seed, (uint64_t)i, 1);
    out[3 * i] = (float)(r * cos(phi));
    out[3 * i + 1] = (float)(r * sin(phi));
    out[3 * i + 2] = (float)z;
}

__global__ void sample_surface_kernel(const float* __restrict__ mesh, const double* __restrict__ cdf, int64_t nf,
                                      uint64_t seed, int64_t n, double sigma, float* __restrict__ out,
                                      int32_t* __restrict__ face) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const double r0 = rnd01(seed, (uint64_t)i, 0);
    int64_t lo = 0, hi = nf - 1;
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (cdf[mid] > r0) hi = mid;
        else lo = mid + 1;
    }
    if (face) face[i] = (int32_t)lo;
    const float* t = mesh + 9 * lo;
    const double u = sqrt(rnd01(seed, (uint64_t)i, 1));
    const double v = rnd01(seed, (uint64_t)i, 2);
    double g[3] = {0.0, 0.0, 0.0};
    if (sigma > 0.0) {  // Box-Muller
        const double u1 = 1.0 - rnd01(seed, (uint64_t)i, 3), u2 = rnd01(seed, (uint64_t)i, 4);
        const double u3 = 1.0 - rnd01(seed, (uint64_t)i, 5), u4 = rnd01(seed, (uint64_t)i, 6);
        const double r1 = sqrt(-2.0 * log(u1)), r2 = sqrt(-2.0 * log(u3));
        g[0] = r1 * cos(2.0 * M_PI * u2);
        g[1] = r1 * sin(2.0 * M_PI * u2);
        g[2] = r2 * cos(2.0 * M_PI * u4);
    }
    for (int k = 0; k < 3; ++k) {
        const double p = (1.0 - u) * t[k] + (u * (1.0 - v)) * t[3 + k] + (u * v) * t[6 + k];
        out[3 * i + k] = (float)(p + sigma * g[k]);
    }
}

}  // namespace nglod

using namespace nglod;

extern "C" {

int nglod_sample_uniform(int64_t n, uint64_t seed, float* out, void* stream) {
    if (n < 0) return fail(NGLOD_ERR_ARG, "n < 0");
    if (n == 0) return NGLOD_OK;
    if (!out) return fail(NGLOD_ERR_ARG, "NULL pointer");
    hipLaunchKernelGGL(sample_uniform_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       seed, n, out);
    return check_launch("sample_uniform_kernel");
}

int nglod_sample_directions(int64_t n, uint64_t seed, float* out, void* stream) {
    if (n < 0) return fail(NGLOD_ERR_ARG, "n < 0");
    if (n == 0) return NGLOD_OK;
    if (!out) return fail(NGLOD_ERR_ARG, "NULL pointer");
    hipLaunchKernelGGL(sample_directions_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       seed, n, out);
    return check_launch("sample_directions_kernel");
}

int nglod_sample_surface(const float* mesh, const double* cdf, int64_t nf, int64_t n, uint64_t seed, double sigma,
                         float* out, int32_t* face, void* stream) {
    if (n < 0 || nf < 0) return fail(NGLOD_ERR_ARG, "negative size");
    if (n == 0) return NGLOD_OK;
    if (nf == 0 || !mesh || !cdf || !out) return fail(NGLOD_ERR_ARG, "NULL pointer or empty mesh");
    hipLaunchKernelGGL(sample_surface_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       mesh, cdf, nf, seed, n, sigma, out, face);
    return check_launch("sample_surface_kernel");
}

}  // extern "C"
