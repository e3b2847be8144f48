// The SDF of a group of 32 queries by one block of four waves, FP32: every wave
// holds the same 32 queries (lanes n and n + 32: query n) and does a part of each.
//
//  1. A thread per (level, query) computes the cell and the eight corner weights.
//  2. Eight threads per query gather: thread q of a query owns channels 4 q .. 4 q + 3,
//     so the eight threads read a corner's row of 128 bytes in one piece (15 cycles
//     of the vector L1 per load instruction; one query per lane, 64 rows at a time:
//     25).
//  3. Wave h multiplies hidden units 32 h .. 32 h + 31 (its rows of W0 stay in 16
//     registers) by the features of all 32 queries and takes its units' share of the
//     second layer; the four shares are added in the order of h.
//
// The sums have the order of the wave-wide decoder's (fp32_wave.hpp), so the bits
// are the same.  A grid of
// 5^3 corners (level 0) is kept in LDS: one fifth of a 5-level gather leaves the
// L1 (1280x720: 3.82 -> 3.43 ms); with 34 KB of LDS a CU holds four blocks.
// Interpolating the cells that neighbouring rays share on the matrix cores (as
// cell_gather.hpp does for sorted points) cut the L1's traffic to a quarter but
// was slower (5.5 ms; only cells shared by most rays: 5.1): a group's rays lie in
// four cells per level and 16 rays on average, one dependent product each.
#pragma once

#include "fp32_wave.hpp"

namespace nglod {

constexpr int kGroup = 32;            // queries of a block
constexpr int kGroupThreads = 256;
constexpr int kFewQueries = 16;       // group_decode_few's columns
constexpr int kFeatStride = 20;       // floats between queries: 16-byte aligned, spread over the banks

struct alignas(16) GroupDecoder {
    float feat[2][kGroup][kFeatStride];  // [half][query][kk] = channel 2 kk + half
    float part[4][64];
    int col[kGroup];                     // group_decode_few: the query of each column
    float b0[kH];
    float w1[kH];
    float wxyz[kH][4];
};

template <bool COARSE>
struct GroupLds {
    float4 w[NGLOD_MAX_LODS][kGroup][2];  // corner weights, corner = 4 z + 2 y + x
    uint32_t base[NGLOD_MAX_LODS][kGroup];
    float4 coarse[COARSE ? 125 * (kC / 4) : 1];  // level 0's grid when it has at most 5^3 corners
    GroupDecoder dec;
};

struct GroupWeights {
    float a[kC / 2];  // A operands: W0[32 h + n][2 kk + half]
};

// Every thread of the block (W0 [128][din], din = 32, or 35 with xyz first); a
// barrier comes before the first group_decode.
__device__ __forceinline__ GroupWeights stage_group_decoder(const float* W0, int din, const float* b0, const float* w1,
                                                            GroupDecoder* s) {
    const int off = din - kC;
    const int lane = threadIdx.x & 63, h = threadIdx.x >> 6;
    const float* row = W0 + (32 * h + (lane & 31)) * din + off + (lane >> 5);
    GroupWeights g;
#pragma unroll
    for (int kk = 0; kk < kC / 2; ++kk) g.a[kk] = row[2 * kk];
    for (int j = threadIdx.x; j < kH; j += kGroupThreads) {
        s->b0[j] = b0[j];
        s->w1[j] = w1[j];
        for (int k = 0; k < 3; ++k) s->wxyz[j][k] = off == 0 ? 0.0f : W0[j * din + k];
        s->wxyz[j][3] = 0.0f;
    }
    return g;
}

// COARSE: with level 0 in LDS (for blocks of many trips).
template <bool COARSE>
__device__ __forceinline__ GroupWeights stage_group(const ModelArgs& m, int dec, GroupLds<COARSE>* s) {
    if (COARSE && m.res[0] <= 4) {
        const int S = m.res[0] + 1;
        const float4* g4 = reinterpret_cast<const float4*>(m.grid[0]);
        for (int j = threadIdx.x; j < S * S * S * (kC / 4); j += kGroupThreads) s->coarse[j] = g4[j];
    }
    return stage_group_decoder(m.w0[dec], m.pos_inv ? kC : kC + 3, m.b0[dec], m.w1[dec], &s->dec);
}

// Channels 4 q .. 4 q + 3 of a query.
__device__ __forceinline__ void store_features(GroupDecoder* s, uint32_t query, uint32_t q, const float4& f) {
    *reinterpret_cast<float2*>(&s->feat[0][query][2 * q]) = make_float2(f.x, f.z);
    *reinterpret_cast<float2*>(&s->feat[1][query][2 * q]) = make_float2(f.y, f.w);
}

// The decoder on the stored features: every thread, with the position of query
// lane % 32.
template <bool POSINV>
__device__ __forceinline__ float group_decode(GroupDecoder* s, const GroupWeights& gw, float b1, float px, float py,
                                              float pz) {
    const uint32_t lane = lane_id(), n = lane & 31u, half = lane >> 5;
    const int h = (int)(threadIdx.x >> 6);
    __syncthreads();
    f32x16_t c = {};
    const float4* b4 = reinterpret_cast<const float4*>(s->feat[half][n]);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const float4 b = b4[k];
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(gw.a[4 * k + 0], b.x, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(gw.a[4 * k + 1], b.y, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(gw.a[4 * k + 2], b.z, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f32_32x32x2f32(gw.a[4 * k + 3], b.w, c, 0, 0, 0);
    }
    s->part[h][lane] = layer2_tile(c, h, half, s, !POSINV, px, py, pz);
    __syncthreads();
    float p = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) p += s->part[k][lane];
    return halves_sum(p, p) + b1;
}

// From here on this block decodes with group_decode_few: the rows as A operands of
// v_mfma_f32_16x16x4_f32, gw.a[2 k + s] of lane (m, j) = W0[32 h + 16 s + m][4 k + j]
// (m = lane % 16, j = lane / 16).
__device__ __forceinline__ void few_weights(GroupWeights& gw) {
#pragma unroll
    for (int k = 0; k < kC / 4; ++k) {
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(gw.a[2 * k]), __float_as_uint(gw.a[2 * k + 1]),
                                                        false, false);
        const auto q = __builtin_amdgcn_permlane16_swap(p[0], p[1], false, false);
        gw.a[2 * k] = __uint_as_float(q[0]);
        gw.a[2 * k + 1] = __uint_as_float(q[1]);
    }
}

// Column of query n of `act` (the queries of `act` first).  The first 32 threads
// store it before a barrier that comes before group_decode_few.
__device__ __forceinline__ uint32_t few_column(uint32_t act, uint32_t n) {
    const uint32_t rank = (uint32_t)__popc(act & ((1u << n) - 1u));
    return (act >> n) & 1u ? rank : (uint32_t)__popc(act) + n - rank;
}

// group_decode for at most 16 queries `act`: half the matrix work, in two chains
// of eight products instead of one of sixteen of twice the length.  The same sums in
// the same order: a chain of the second layer takes units 0-3, 8-11, 16-19, 24-27 (or
// 4-7, ...), which lie in lanes n, n + 32, n, n + 32 here and pass the sum on.
template <bool POSINV>
__device__ __forceinline__ float group_decode_few(GroupDecoder* s, const GroupWeights& gw, float b1, uint32_t act,
                                                  float px, float py, float pz) {
    typedef float f32x4_t __attribute__((ext_vector_type(4)));
    const uint32_t lane = lane_id(), m = lane & 15u, j = lane >> 4;
    const int h = (int)(threadIdx.x >> 6);
    const int query = s->col[m];
    float pos = 0.0f;
    if (!POSINV) {
        const float x = __shfl(px, query), y = __shfl(py, query), z = __shfl(pz, query);
        pos = j == 0 ? z : j == 1 ? y : j == 2 ? x : 0.0f;
    }
    __syncthreads();
    f32x4_t c[2] = {{}, {}};
    const float* b = &s->feat[j & 1u][query][j >> 1];
#pragma unroll
    for (int k = 0; k < kC / 4; ++k) {
        c[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(gw.a[2 * k], b[2 * k], c[0], 0, 0, 0);
        c[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(gw.a[2 * k + 1], b[2 * k], c[1], 0, 0, 0);
    }
    float4 w[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int unit = 32 * h + 16 * t + 4 * (int)j;
        const float4 bias = *reinterpret_cast<const float4*>(&s->b0[unit]);
        c[t][0] += bias.x;
        c[t][1] += bias.y;
        c[t][2] += bias.z;
        c[t][3] += bias.w;
        if (!POSINV)
            c[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(s->wxyz[32 * h + 16 * t + (int)m][j == 3 ? 3 : 2 - j], pos, c[t],
                                                        0, 0, 0);
        w[t] = *reinterpret_cast<const float4*>(&s->w1[unit]);
    }
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            acc = __builtin_fmaf(w[t].x, fmaxf(c[t][0], 0.0f), acc);
            acc = __builtin_fmaf(w[t].y, fmaxf(c[t][1], 0.0f), acc);
            acc = __builtin_fmaf(w[t].z, fmaxf(c[t][2], 0.0f), acc);
            acc = __builtin_fmaf(w[t].w, fmaxf(c[t][3], 0.0f), acc);
            if (t + u < 2) {
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc), __float_as_uint(acc), false, false);
                acc = __uint_as_float(sw[u]);
            }
        }
    }
    if (j >= 2) s->part[h][m + 32u * (j & 1u)] = acc;
    const uint32_t from = few_column(act, lane & 31u) + (lane & 32u);
    __syncthreads();
    float p = 0.0f;
#pragma unroll
    for (int k = 0; k < 4; ++k) p += s->part[k][from];
    return halves_sum(p, p) + b1;
}

// Eight corner rows' float4 of this thread.
__device__ __forceinline__ void group_rows(const float* __restrict__ grid, int S, uint32_t base, uint32_t q,
                                           float4 (&g)[8]) {
    const float* b = grid + (size_t)base * kC + 4 * q;
    const size_t sy = (size_t)S * kC, sz = (size_t)S * S * kC;
#pragma unroll
    for (int k = 0; k < 8; ++k)
        g[k] = *reinterpret_cast<const float4*>(b + (k & 1) * kC + (k & 2 ? sy : 0) + (k & 4 ? sz : 0));
}

__device__ __forceinline__ void group_corners(const float4 (&g)[8], const float4* w, float4& f) {
    const float4 w0 = w[0], w1 = w[1];
    const float ww[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        f.x = __builtin_fmaf(g[k].x, ww[k], f.x);
        f.y = __builtin_fmaf(g[k].y, ww[k], f.y);
        f.z = __builtin_fmaf(g[k].z, ww[k], f.z);
        f.w = __builtin_fmaf(g[k].w, ww[k], f.w);
    }
}

// The gather for at most eight queries (`act`), as when a march runs out of rays
// and its trips are all latency: 32 threads per query, a channel each, the rows of
// four levels on their way at once instead of one level after the other.  Same
// order of sums.
template <bool COARSE>
__device__ __forceinline__ void group_gather_few(const ModelArgs& m, int lod, GroupLds<COARSE>* s, uint32_t act) {
    const int slot = (int)(threadIdx.x >> 5), c = (int)(threadIdx.x & 31u);
    if (slot >= __popc(act)) return;
    const int ray = nth_set_bit(act, slot);
    float f = 0.0f;
    auto add = [&](int l, const float (&g)[8]) {
        const float4* w = s->w[l][ray];
        const float4 w0 = w[0], w1 = w[1];
        const float ww[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
#pragma unroll
        for (int k = 0; k < 8; ++k) f = __builtin_fmaf(g[k], ww[k], f);
    };
    int l = 0;
    if (COARSE && m.res[0] <= 4) {
        const int S = m.res[0] + 1;
        const float* b = reinterpret_cast<const float*>(s->coarse) + s->base[0][ray] * kC + c;
        float g[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) g[k] = b[((k & 1) + (k & 2 ? S : 0) + (k & 4 ? S * S : 0)) * kC];
        add(0, g);
        l = 1;
    }
#pragma unroll 1
    for (; l <= lod; l += 4) {
        float g[4][8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (l + j <= lod) {
                const int S = m.res[l + j] + 1;
                const float* b = m.grid[l + j] + (size_t)s->base[l + j][ray] * kC + c;
                const size_t sy = (size_t)S * kC, sz = (size_t)S * S * kC;
#pragma unroll
                for (int k = 0; k < 8; ++k) g[j][k] = b[(k & 1) * kC + (k & 2 ? sy : 0) + (k & 4 ? sz : 0)];
            }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (l + j <= lod) add(l + j, g[j]);
    }
    s->dec.feat[c & 1][ray][c >> 1] = f;
}

// Every thread of the block, with the position of query lane % 32 (the same in
// all four waves; any position for queries whose result is not used).  act: the
// queries whose result is used.
// FEW: group_gather_few for at most eight of them.  DECODE_FEW: at most 16 of them, and
// few_weights has run.
template <bool POSINV, bool FEW, bool DECODE_FEW, bool COARSE>
__device__ __forceinline__ float group_sdf(const ModelArgs& m, int lod, GroupLds<COARSE>* s, const GroupWeights& gw, float b1,
                                           uint32_t act, float px, float py, float pz) {
    const uint32_t lane = lane_id(), n = lane & 31u, half = lane >> 5;
    {
        const int l = 2 * (int)(threadIdx.x >> 6) + (int)half;  // NGLOD_MAX_LODS = 8 levels
        if (l <= lod) {
            const int r = m.res[l], S = r + 1;
            const AxisW ax = axis_weights(px, r);
            const AxisW ay = axis_weights(py, r);
            const AxisW az = axis_weights(pz, r);
            const float wxy00 = ax.w0 * ay.w0, wxy10 = ax.w1 * ay.w0;
            const float wxy01 = ax.w0 * ay.w1, wxy11 = ax.w1 * ay.w1;
            s->base[l][n] = (uint32_t)((az.i0 * S + ay.i0) * S + ax.i0);
            s->w[l][n][0] = make_float4(wxy00 * az.w0, wxy10 * az.w0, wxy01 * az.w0, wxy11 * az.w0);
            s->w[l][n][1] = make_float4(wxy00 * az.w1, wxy10 * az.w1, wxy01 * az.w1, wxy11 * az.w1);
        }
    }
    if (DECODE_FEW && threadIdx.x < kGroup) s->dec.col[few_column(act, n)] = (int)n;
    __syncthreads();
    if (FEW && __popc(act) <= 8) {
        group_gather_few(m, lod, s, act);
    } else {
        const uint32_t ray = threadIdx.x >> 3, q = threadIdx.x & 7u;
        float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        float4 g[8];
        int l = 0;
        if (COARSE && m.res[0] <= 4) {
            const int S = m.res[0] + 1;
            const float4* b = s->coarse + s->base[0][ray] * (kC / 4) + q;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                g[k] = b[((k & 1) + (k & 2 ? S : 0) + (k & 4 ? S * S : 0)) * (kC / 4)];
            group_corners(g, s->w[0][ray], f);
            l = 1;
        }
#pragma unroll 1
        for (; l <= lod; ++l) {
            group_rows(m.grid[l], m.res[l] + 1, s->base[l][ray], q, g);
            group_corners(g, s->w[l][ray], f);
        }
        store_features(&s->dec, ray, q, f);
    }
    if (DECODE_FEW) return group_decode_few<POSINV>(&s->dec, gw, b1, act, px, py, pz);
    return group_decode<POSINV>(&s->dec, gw, b1, px, py, pz);
}

}  // namespace nglod
