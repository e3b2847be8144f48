// FP32 SDF evaluation for one wavefront (64 queries, one per lane): the FP32
// trilinear gather per lane, then the first decoder layer as FP32 MFMA
// 32x32x2 tiles (v_mfma_f32_32x32x2_f32: exact FP32 products, FP32
// accumulation), then bias, ReLU and the 128 -> 1 layer in FP32 on the MFMA
// output registers.  Twice the FP32 rate of the vector FMA decoder (the two do
// not overlap on a SIMD: 64 cycles per product plus 4.4 per vector FMA, whatever
// the number of waves).
//
// MFMA operand layout (32x32x2, one block): lane l holds A[m = l%32][k = l/32]
// and B[k = l/32][n = l%32]; output: lane l holds C[m][n = l%32] for
// m = 8*(i/4) + 4*(l/32) + i%4, i = 0..15.  A = W0 (hidden x feature
// channels), B = features^T (channel pair x 32 queries).  The 64 queries of
// a wave form two 32-query tiles: tile 0 is lanes 0..31, tile 1 lanes 32..63;
// one v_permlane32_swap per channel pair turns a lane's own two channels into
// both tiles' B operands.
#pragma once

#include "device_common.hpp"

namespace nglod {


// Per-workgroup constants of the FP32 MFMA decoder, staged once in LDS
// (18.5 KB): A fragments [h tile 0..3][channel-pair quad 0..3][lane] (4
// channel pairs each), b0, w1 and the xyz columns of W0.
struct Fp32Lds {
    float4 afrag[4 * 4 * 64];
    float b0[kH];
    float w1[kH];
    float wxyz[kH][4];  // W0 columns 0..2 (xyz input); [3] unused
};

// Stage a decoder (W0 [128][din], din = 32 or 35 with xyz first; b0; w1) into
// LDS.  Every thread of the block must call this, followed by __syncthreads().
__device__ __forceinline__ void stage_fp32_lds_raw(const float* W0, int din, const float* b0, const float* w1,
                                                   Fp32Lds* s) {
    const bool pos_inv = din == kC;
    const int off = pos_inv ? 0 : 3;
    for (int j = threadIdx.x; j < 4 * 4 * 64; j += blockDim.x) {
        const int lane = j & 63;
        const int kq = (j >> 6) & 3;
        const int h = j >> 8;
        const int row = 32 * h + (lane & 31);
        const int col = off + 8 * kq + (lane >> 5);  // channel 2*(4kq+e) + lane/32
        float4 v;
        v.x = W0[row * din + col + 0];
        v.y = W0[row * din + col + 2];
        v.z = W0[row * din + col + 4];
        v.w = W0[row * din + col + 6];
        s->afrag[j] = v;
    }
    for (int j = threadIdx.x; j < kH; j += blockDim.x) {
        s->b0[j] = b0[j];
        s->w1[j] = w1[j];
        if (!pos_inv) {
            s->wxyz[j][0] = W0[j * din + 0];
            s->wxyz[j][1] = W0[j * din + 1];
            s->wxyz[j][2] = W0[j * din + 2];
        } else {
            s->wxyz[j][0] = s->wxyz[j][1] = s->wxyz[j][2] = 0.0f;
        }
        s->wxyz[j][3] = 0.0f;
    }
}

// Stage decoder `dec` of the model.
__device__ __forceinline__ void stage_fp32_lds(const ModelArgs& m, int dec, Fp32Lds* s) {
    stage_fp32_lds_raw(m.w0[dec], m.pos_inv ? kC : kC + 3, m.b0[dec], m.w1[dec], s);
}

// Second layer over one 32x32 output tile held in registers: sum of
// w1[row] * relu(C + b0[row] + wxyz[row] . xyz) over this lane's 16 rows.
template <typename LDS>
__device__ __forceinline__ float layer2_tile(const f32x16_t& c, int h, uint32_t half, const LDS* s, bool xyz,
                                             float px, float py, float pz) {
    f32x16_t v;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const float4 b = *reinterpret_cast<const float4*>(&s->b0[32 * h + 8 * g + 4 * (int)half]);
        v[4 * g + 0] = c[4 * g + 0] + b.x;
        v[4 * g + 1] = c[4 * g + 1] + b.y;
        v[4 * g + 2] = c[4 * g + 2] + b.z;
        v[4 * g + 3] = c[4 * g + 3] + b.w;
    }
    if (xyz) v = add_xyz(v, h, half, s, px, py, pz);
    float acc = 0.0f;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const float4 w = *reinterpret_cast<const float4*>(&s->w1[32 * h + 8 * g + 4 * (int)half]);
        acc = __builtin_fmaf(w.x, fmaxf(v[4 * g + 0], 0.0f), acc);
        acc = __builtin_fmaf(w.y, fmaxf(v[4 * g + 1], 0.0f), acc);
        acc = __builtin_fmaf(w.z, fmaxf(v[4 * g + 2], 0.0f), acc);
        acc = __builtin_fmaf(w.w, fmaxf(v[4 * g + 3], 0.0f), acc);
    }
    return acc;
}

// The decoder on the 64 lanes' feature vectors f (zero on inactive lanes).  Every
// lane of the wave must call this (no divergent branch around it): the MFMAs and
// lane swaps are wave-wide.  A 32-query tile with no active lane skips its MFMAs.
// Each output column depends only on its own query, so a lane's result is the
// same whatever the other lanes hold.
template <bool POSINV>
__device__ __forceinline__ float decode_fp32_wave(const float (&f)[kC], const Fp32Lds* s, float b1, uint32_t lane,
                                                  bool active, float px, float py, float pz) {
    const uint64_t am = __ballot(active);
    const bool use0 = (uint32_t)am != 0u, use1 = (uint32_t)(am >> 32) != 0u;
    const uint32_t half = lane >> 5;
    // B operands of both tiles for channel pair kk: tile 0 takes (own channel
    // 2kk | channel 2kk+1 of lane l-32), tile 1 (channel 2kk of lane l+32 |
    // own channel 2kk+1).
    float B0[kC / 2], B1[kC / 2];
#pragma unroll
    for (int kk = 0; kk < kC / 2; ++kk) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(f[2 * kk]), __float_as_uint(f[2 * kk + 1]),
                                                         false, false);
        B0[kk] = __uint_as_float(sw[0]);
        B1[kk] = __uint_as_float(sw[1]);
    }
    float qx0, qy0, qz0, qx1, qy1, qz1;
    tile_coords(px, py, pz, qx0, qy0, qz0, qx1, qy1, qz1);
    float part0 = 0.0f, part1 = 0.0f;
#pragma unroll 1
    for (int h = 0; h < 4; ++h) {
        // a tile with no active query (a draining wave) skips its MFMAs
        if (use0) {
            f32x16_t c = {};
#pragma unroll
            for (int kq = 0; kq < 4; ++kq) {
                const float4 a = s->afrag[(h * 4 + kq) * 64 + lane];
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, B0[4 * kq + 0], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, B0[4 * kq + 1], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, B0[4 * kq + 2], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, B0[4 * kq + 3], c, 0, 0, 0);
            }
            part0 += layer2_tile(c, h, half, s, !POSINV, qx0, qy0, qz0);
        }
        if (use1) {
            f32x16_t c = {};
#pragma unroll
            for (int kq = 0; kq < 4; ++kq) {
                const float4 a = s->afrag[(h * 4 + kq) * 64 + lane];
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, B1[4 * kq + 0], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, B1[4 * kq + 1], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, B1[4 * kq + 2], c, 0, 0, 0);
                c = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, B1[4 * kq + 3], c, 0, 0, 0);
            }
            part1 += layer2_tile(c, h, half, s, !POSINV, qx1, qy1, qz1);
        }
    }
    return halves_sum(part0, part1) + b1;
}

// A model's level table in LDS, for the cooperative tail gathers: read as vector
// values, its pointers and resolutions add no scalar registers to the persistent
// kernels, which already use nearly all of theirs.
struct SoloLevels {
    const float* grid[NGLOD_MAX_LODS];
    int res[NGLOD_MAX_LODS];
};

}  // namespace nglod
