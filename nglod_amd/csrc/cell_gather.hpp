// The FP32 trilinear gather for waves whose queries are neighbours in space
// (batches in Morton order): the interpolation of one cell is a small matrix
// product, features^T [32 channels][queries] += corners^T [32][8] weights [8][queries],
// so the queries of a tile in one cell take four v_mfma_f32_32x32x2_f32 and read
// the cell's eight rows once, instead of eight rows per query through the
// vector memory path.  A NaN or an infinity in a cell reaches its own queries
// only: the others keep their accumulators by a select.
//
// Bits: the MFMA accumulates like fma(a1, b1, fma(a0, b0, c)) (exact products, k
// = 0 first), so corners 0 .. 7 in k order are gather_fp32's FMA chain, and the
// accumulator carries the chain from level to level.
//
// Layout: the accumulators are kept as the decoder's B operands: tile t (queries
// 32 t .. 32 t + 31 of the wave), register kk of lane (n, half) = channel 2 kk + half
// of query n.  MFMA output register i of half h is row m = 8 (i / 4) + 4 h + i % 4, so
// row m of the A operand is channel 2 i + h.
//
// Which path: a cell costs its tiles four MFMAs and a select each (about 320
// cycles of the SIMD), the per-lane gather of 64 queries about 1000 cycles of the
// CU's vector memory path, which its four SIMDs share: up to kMaxProducts (cell,
// tile) pairs the product is the cheaper one.  2^22 uniform points at LOD 4 (16
// points per finest cell, 19 products a wave where 10 is the least): batch query 1.02
// -> 0.66 ms, of which the matrix cores are busy 0.35 ms (128 of 205 MFMAs a wave
// are the decoder's).
#pragma once

#include "fp32_wave.hpp"

namespace nglod {

constexpr int kMaxProducts = 12;

struct CellFeatures {
    f32x16_t t[2];
};

__device__ __forceinline__ CellFeatures zero_cell_features() { return CellFeatures{{{}, {}}}; }

// Channel of row n of the A operand.
__device__ __forceinline__ uint32_t cell_row(uint32_t n) {
    return 2u * (4u * (n >> 3) + (n & 3u)) + ((n >> 2) & 1u);
}

// One more level onto f.  Every lane of the wave calls this with a position
// (lanes without a query: any position); use1: tile 1 holds a query.
// ONLY: f is this level alone (what it holds is not read).
template <bool ONLY = false>
__device__ __forceinline__ void gather_cells(const float* __restrict__ grid, int r, float px, float py, float pz,
                                             uint32_t lane, bool use1, CellFeatures& f) {
    const int S = r + 1;
    const AxisW ax = axis_weights(px, r);
    const AxisW ay = axis_weights(py, r);
    const AxisW az = axis_weights(pz, r);
    const uint32_t base = (uint32_t)((az.i0 * S + ay.i0) * S + ax.i0);
    const float wxy[4] = {ax.w0 * ay.w0, ax.w1 * ay.w0, ax.w0 * ay.w1, ax.w1 * ay.w1};
    // the wave's cells, counted up to the limit
    const uint64_t all = use1 ? ~0ull : 0xffffffffull;
    int products = 0;
    for (uint64_t m = all; m != 0 && products <= kMaxProducts;) {
        const uint32_t cell = (uint32_t)__builtin_amdgcn_readlane((int)base, __ffsll((unsigned long long)m) - 1);
        const uint64_t same = __ballot(base == cell) & all;
        products += ((uint32_t)same != 0) + ((uint32_t)(same >> 32) != 0);
        m &= ~same;
    }
    if (products > kMaxProducts) {
        // a row per query and corner: back to a lane's own channels and on
        float v[kC];
#pragma unroll
        for (int kk = 0; kk < kC / 2; ++kk) {
            if (ONLY) {
                v[2 * kk] = v[2 * kk + 1] = 0.0f;
                continue;
            }
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(f.t[0][kk]), __float_as_uint(f.t[1][kk]),
                                                             false, false);
            v[2 * kk] = __uint_as_float(sw[0]);
            v[2 * kk + 1] = __uint_as_float(sw[1]);
        }
        const float* b = grid + (size_t)base * kC;
        const size_t sx = kC, sy = (size_t)S * kC, sz = (size_t)S * S * kC;
        corner_fma(v, b, wxy[0] * az.w0);
        corner_fma(v, b + sx, wxy[1] * az.w0);
        corner_fma(v, b + sy, wxy[2] * az.w0);
        corner_fma(v, b + sy + sx, wxy[3] * az.w0);
        corner_fma(v, b + sz, wxy[0] * az.w1);
        corner_fma(v, b + sz + sx, wxy[1] * az.w1);
        corner_fma(v, b + sz + sy, wxy[2] * az.w1);
        corner_fma(v, b + sz + sy + sx, wxy[3] * az.w1);
#pragma unroll
        for (int kk = 0; kk < kC / 2; ++kk) {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[2 * kk]), __float_as_uint(v[2 * kk + 1]),
                                                             false, false);
            f.t[0][kk] = __uint_as_float(sw[0]);
            f.t[1][kk] = __uint_as_float(sw[1]);
        }
        return;
    }
    // B operands of k-steps s: corners 2 s (lanes 0..31) and 2 s + 1 of a tile's queries
    float w[2][4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
        const float wz = s < 2 ? az.w0 : az.w1;
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(wxy[2 * (s & 1)] * wz),
                                                         __float_as_uint(wxy[2 * (s & 1) + 1] * wz), false, false);
        w[0][s] = __uint_as_float(sw[0]);
        w[1][s] = __uint_as_float(sw[1]);
    }
    const uint32_t n = lane & 31u, half = lane >> 5;
    const float* mine = grid + half * kC + cell_row(n);  // corner 2 s + half: x = half
    const size_t sy = (size_t)S * kC, sz = (size_t)S * S * kC;
    uint64_t left = ONLY ? all : 0;  // queries of a tile whose features are not set yet: all or none
    for (uint64_t m = all; m != 0;) {
        const uint32_t cell = (uint32_t)__builtin_amdgcn_readlane((int)base, __ffsll((unsigned long long)m) - 1);
        const uint64_t same = __ballot(base == cell) & all;
        m &= ~same;
        const float* p = mine + (size_t)cell * kC;
        const float a0 = p[0], a1 = p[sy], a2 = p[sz], a3 = p[sz + sy];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const uint32_t here = (uint32_t)(same >> (32 * t));
            if (here == 0) continue;
            f32x16_t d = __builtin_amdgcn_mfma_f32_32x32x2f32(a0, w[t][0], ONLY ? f32x16_t{} : f.t[t], 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_32x32x2f32(a1, w[t][1], d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_32x32x2f32(a2, w[t][2], d, 0, 0, 0);
            d = __builtin_amdgcn_mfma_f32_32x32x2f32(a3, w[t][3], d, 0, 0, 0);
            if (here == 0xffffffffu || (ONLY && (uint32_t)(left >> (32 * t)) != 0u)) {
                left &= ~(0xffffffffull << (32 * t));
                f.t[t] = d;
            } else {
                const bool in = (here >> n) & 1u;
#pragma unroll
                for (int i = 0; i < 16; ++i) f.t[t][i] = in ? d[i] : f.t[t][i];
            }
        }
    }
}

// The decoder on such features (decode_fp32_wave from its B operands on).
template <bool POSINV>
__device__ __forceinline__ float decode_cells(const CellFeatures& f, const Fp32Lds* s, float b1, uint32_t lane,
                                              float px, float py, float pz) {
    const uint32_t half = lane >> 5;
    float qx0, qy0, qz0, qx1, qy1, qz1;
    tile_coords(px, py, pz, qx0, qy0, qz0, qx1, qy1, qz1);
    float part[2] = {0.0f, 0.0f};
#pragma unroll 1
    for (int h = 0; h < 4; ++h) {
        // both tiles whether used or not: one block, so that a tile's ReLU runs beside
        // the other's products
        f32x16_t c[2] = {{}, {}};
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int kq = 0; kq < 4; ++kq) {
                const float4 a = s->afrag[(h * 4 + kq) * 64 + lane];
                c[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, f.t[t][4 * kq + 0], c[t], 0, 0, 0);
                c[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, f.t[t][4 * kq + 1], c[t], 0, 0, 0);
                c[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, f.t[t][4 * kq + 2], c[t], 0, 0, 0);
                c[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, f.t[t][4 * kq + 3], c[t], 0, 0, 0);
            }
        }
        part[0] += layer2_tile(c[0], h, half, s, !POSINV, qx0, qy0, qz0);
        part[1] += layer2_tile(c[1], h, half, s, !POSINV, qx1, qy1, qz1);
    }
    return halves_sum(part[0], part[1]) + b1;
}

}  // namespace nglod
