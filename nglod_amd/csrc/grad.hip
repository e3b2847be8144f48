// Gradients of the SDF with respect to the query position and the
// minimum-tracking sphere trace:
//   nglod_gradient     diffutils.gradient (sdf-net/lib/diffutils.py:29-84):
//                      'finitediff', 'tetrahedron' and 'autodiff', optionally
//                      masked and normalised as the tracers use it
//                      (SphereTracer.py:128-130, :214-215)
//   nglod_trace_min    SphereTracer.get_min (sdf-net/lib/tracer/SphereTracer.py:134-218)
// FP32.  The gradients' features, their derivatives and both directions of the
// first decoder layer are matrix products (grad_cells); the minimum-tracking
// trace has one ray per lane and the decoder on the vector ALU (decode_fp32).
#include "api_common.hpp"
#include "cell_gather.hpp"
#include "trace_common.hpp"

namespace nglod {

// Tetrahedron taps (diffutils.py:38-62): f at x + h k_j for the four corners
// k_j of a tetrahedron, gradient sum_j k_j f(x + h k_j) / (4 h), h = 1/192.
constexpr float kTetraFourH = (float)((1.0 / (64.0 * 3.0)) * 4.0);

// One query's SDF at `lod` and its gradient with respect to the position, on the
// vector ALU (only for decoders with a weight that is not finite), as
// torch autograd of OctreeSDF.sdf (OctreeSDF.py:94-155) gives it:
//  - F.grid_sample's backward with align_corners=True and padding_mode=
//    'border': d u / d p = r / 2 per axis, and 0 where the unclamped u is <= 0
//    or >= r (the border counts as outside, so the clamp passes no gradient);
//    within the cell [floor(u), floor(u) + 1] the derivative of the trilinear
//    weights, (-1, +1) on the axis times the other two axes' weights;
//  - ReLU's backward: hidden unit j contributes where its pre-activation is > 0;
//  - a position-dependent decoder's xyz columns of W0 add their own term.
// The SDF value is computed exactly as decode_fp32 computes it.
template <bool POSINV>
__device__ __forceinline__ float sdf_and_grad_fp32(const ModelArgs& m, int lod, int dec, float px, float py,
                                                   float pz, float& gx, float& gy, float& gz) {
    constexpr int D = POSINV ? kC : kC + 3;
    constexpr int OFF = POSINV ? 0 : 3;
    float f[kC];
    gather_fp32(m, lod, px, py, pz, f);
    const float* W0 = m.w0[dec];
    const float* B0 = m.b0[dec];
    const float* W1 = m.w1[dec];
    float v[kC];
#pragma unroll
    for (int c = 0; c < kC; ++c) v[c] = 0.0f;
    float vx = 0.0f, vy = 0.0f, vz = 0.0f;
    float out = 0.0f;
#pragma unroll 2
    for (int j = 0; j < kH; ++j) {
        float acc = 0.0f;
        if (!POSINV) {
            acc = __builtin_fmaf(ldc(W0, j * D + 0), px, acc);
            acc = __builtin_fmaf(ldc(W0, j * D + 1), py, acc);
            acc = __builtin_fmaf(ldc(W0, j * D + 2), pz, acc);
        }
#pragma unroll
        for (int k = 0; k < kC; ++k) acc = __builtin_fmaf(ldc(W0, j * D + OFF + k), f[k], acc);
        const float pre = acc + ldc(B0, j);
        const float w = ldc(W1, j);
        out = __builtin_fmaf(w, fmaxf(pre, 0.0f), out);
        if (pre > 0.0f) {
#pragma unroll
            for (int k = 0; k < kC; ++k) v[k] = __builtin_fmaf(w, ldc(W0, j * D + OFF + k), v[k]);
            if (!POSINV) {
                vx = __builtin_fmaf(w, ldc(W0, j * D + 0), vx);
                vy = __builtin_fmaf(w, ldc(W0, j * D + 1), vy);
                vz = __builtin_fmaf(w, ldc(W0, j * D + 2), vz);
            }
        }
    }
    gx = vx;
    gy = vy;
    gz = vz;
    for (int l = 0; l <= lod; ++l) {
        const int r = m.res[l];
        const int S = r + 1;
        const float rf = (float)r;
        const AxisW ax = axis_weights(px, r);
        const AxisW ay = axis_weights(py, r);
        const AxisW az = axis_weights(pz, r);
        const float ux = ((px + 1.0f) * 0.5f) * rf, uy = ((py + 1.0f) * 0.5f) * rf, uz = ((pz + 1.0f) * 0.5f) * rf;
        const float sxg = (ux > 0.0f && ux < rf) ? rf * 0.5f : 0.0f;
        const float syg = (uy > 0.0f && uy < rf) ? rf * 0.5f : 0.0f;
        const float szg = (uz > 0.0f && uz < rf) ? rf * 0.5f : 0.0f;
        const float* base = m.grid[l] + ((size_t)((az.i0 * S + ay.i0) * S + ax.i0)) * kC;
        const size_t stride[3] = {(size_t)kC, (size_t)S * kC, (size_t)S * S * kC};
        float dx = 0.0f, dy = 0.0f, dz = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int bx = k & 1, by = (k >> 1) & 1, bz = k >> 2;
            const float4* q = reinterpret_cast<const float4*>(base + bx * stride[0] + by * stride[1] + bz * stride[2]);
            float pk = 0.0f;  // corner k's features projected on d sdf / d feature
#pragma unroll
            for (int c4 = 0; c4 < kC / 4; ++c4) {
                const float4 gq = q[c4];
                pk = __builtin_fmaf(gq.x, v[4 * c4 + 0], pk);
                pk = __builtin_fmaf(gq.y, v[4 * c4 + 1], pk);
                pk = __builtin_fmaf(gq.z, v[4 * c4 + 2], pk);
                pk = __builtin_fmaf(gq.w, v[4 * c4 + 3], pk);
            }
            const float wx = bx ? ax.w1 : ax.w0, wy = by ? ay.w1 : ay.w0, wz = bz ? az.w1 : az.w0;
            dx = __builtin_fmaf(bx ? pk : -pk, wy * wz, dx);
            dy = __builtin_fmaf(by ? pk : -pk, wx * wz, dy);
            dz = __builtin_fmaf(bz ? pk : -pk, wx * wy, dz);
        }
        gx = __builtin_fmaf(sxg, dx, gx);
        gy = __builtin_fmaf(syg, dy, gy);
        gz = __builtin_fmaf(szg, dz, gz);
    }
    return out + ldc(m.b1[dec], 0);
}

// One decoder for the wave-wide evaluations below, its hidden units in the order
// in which MFMA output registers hold them when the A operand's rows are
// permuted: unit 32 h + 2 i + half sits in register i of lanes' half `half`.
// With that order the units of a half-pair (2 i, 2 i + 1) follow each other, so
//  - the second layer's sum runs over the units 0, 1, 2, .. after one
//    v_permlane32_swap per register, and
//  - the ReLU-gated second-layer weights are, as they lie, the B operand of the
//    product with W0^T (the backward), whose k order is again 0, 1, 2, ..:
// both are decode_fp32's chains of FMAs, bit for bit.
struct GradLds {
    float4 fwd[4 * 4 * 64];  // [h][channel quad][lane]: W0[row of lane][channel]
    float4 bwd[4 * 4 * 64];  // [h][i / 4][lane]: W0[32 h + 2 i + half][grad_channel of lane]
    float b0[kH], w1[kH];    // [h][half][i]
    float wxyz[kH][4];       // [h][half][i]: W0's position columns
};

// Channel of row n of the backward's A operand: output register i of half h is
// row m = 8 (i / 4) + 4 h + i % 4, and takes channel 16 h + i.
__device__ __forceinline__ int grad_channel(int n) { return 16 * ((n >> 2) & 1) + 4 * (n >> 3) + (n & 3); }

// Returns whether W0 is finite (the same on every thread); ends with a barrier.
__device__ __forceinline__ bool stage_grad_lds(const ModelArgs& m, int dec, GradLds* s) {
    const int din = m.pos_inv ? kC : kC + 3, off = m.pos_inv ? 0 : 3;
    const float* W0 = m.w0[dec];
    bool finite = true;
    for (int j = threadIdx.x; j < 4 * 4 * 64; j += blockDim.x) {
        const int n = j & 31, half = (j >> 5) & 1, q = (j >> 6) & 3, h = j >> 8;
        const float* a = W0 + (32 * h + (int)cell_row(n)) * din + off + 8 * q + half;  // channels 2 (4 q + e) + half
        s->fwd[j] = make_float4(a[0], a[2], a[4], a[6]);
        const float* b = W0 + (32 * h + 8 * q + half) * din + off + grad_channel(n);  // units 2 (4 q + e) + half
        s->bwd[j] = make_float4(b[0], b[2 * din], b[4 * din], b[6 * din]);
    }
    for (int j = threadIdx.x; j < kH; j += blockDim.x) {
        const int unit = (j & ~31) + 2 * (j & 15) + ((j >> 4) & 1);
        s->b0[j] = m.b0[dec][unit];
        s->w1[j] = m.w1[dec][unit];
        for (int a = 0; a < 3; ++a) s->wxyz[j][a] = m.pos_inv ? 0.0f : W0[unit * din + a];
        s->wxyz[j][3] = 0.0f;
    }
    for (int j = threadIdx.x; j < kH * din; j += blockDim.x) finite = finite && fabsf(W0[j]) <= 3.4028234e38f;
    return __syncthreads_and(finite);
}

// decode_fp32 of the wave's 64 queries.  GRAD: also v, the derivative with
// respect to the features (register i of half h: channel 16 h + i), and vp, with
// respect to the position through W0's own columns (this lane's half of its
// tiles' units).  q: the tiles' positions (tile_coords).
template <bool POSINV, bool GRAD>
__device__ __forceinline__ float decode_ordered(const CellFeatures& f, const GradLds* s, float b1, uint32_t lane,
                                                const float (&q)[2][3], CellFeatures& v, float (&vp)[2][3]) {
    const int half = (int)(lane >> 5);
    float out = 0.0f;
#pragma unroll 1
    for (int h = 0; h < 4; ++h) {
        const int row = (2 * h + half) * 16;
        f32x16_t z[2] = {{}, {}};
        if (!POSINV) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const float4 w = *reinterpret_cast<const float4*>(s->wxyz[row + i]);
#pragma unroll
                for (int t = 0; t < 2; ++t)
                    z[t][i] = __builtin_fmaf(w.z, q[t][2], __builtin_fmaf(w.y, q[t][1], w.x * q[t][0]));
                if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // four rows at a time in registers
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float4 a = s->fwd[(h * 4 + k) * 64 + lane];
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                z[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, f.t[t][4 * k + 0], z[t], 0, 0, 0);
                z[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, f.t[t][4 * k + 1], z[t], 0, 0, 0);
                z[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, f.t[t][4 * k + 2], z[t], 0, 0, 0);
                z[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, f.t[t][4 * k + 3], z[t], 0, 0, 0);
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float4 b4 = *reinterpret_cast<const float4*>(&s->b0[row + 4 * k]);
            const float4 w4 = *reinterpret_cast<const float4*>(&s->w1[row + 4 * k]);
            const float bb[4] = {b4.x, b4.y, b4.z, b4.w}, ww[4] = {w4.x, w4.y, w4.z, w4.w};
            const float4 a4 = GRAD ? s->bwd[(h * 4 + k) * 64 + lane] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            const float aa[4] = {a4.x, a4.y, a4.z, a4.w};
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int i = 4 * k + e;
                const float z0 = z[0][i] + bb[e], z1 = z[1][i] + bb[e];
                // (unit 2 i, unit 2 i + 1) of the lane's own query; its w1 pair
                const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(fmaxf(z0, 0.0f)),
                                                                __float_as_uint(fmaxf(z1, 0.0f)), false, false);
                const float wa = s->w1[2 * h * 16 + i], wb = s->w1[(2 * h + 1) * 16 + i];
                out = __builtin_fmaf(wb, __uint_as_float(r[1]), __builtin_fmaf(wa, __uint_as_float(r[0]), out));
                if (GRAD) {
                    const float g[2] = {z0 > 0.0f ? ww[e] : 0.0f, z1 > 0.0f ? ww[e] : 0.0f};
                    v.t[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(aa[e], g[0], v.t[0], 0, 0, 0);
                    v.t[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(aa[e], g[1], v.t[1], 0, 0, 0);
                    if (!POSINV) {
                        const float4 w = *reinterpret_cast<const float4*>(s->wxyz[row + i]);
#pragma unroll
                        for (int t = 0; t < 2; ++t) {
                            vp[t][0] = __builtin_fmaf(g[t], w.x, vp[t][0]);
                            vp[t][1] = __builtin_fmaf(g[t], w.y, vp[t][1]);
                            vp[t][2] = __builtin_fmaf(g[t], w.z, vp[t][2]);
                        }
                    }
                }
            }
        }
    }
    return out + b1;
}

// The projections pk of v on the features of the eight corners (4 z + 2 y + x) of
// each lane's cell.  Up to four cells' corners onto a tile's 32 queries are one
// product, corners [4 * 8][32 channels] v [32][queries], of 16 MFMAs whose B
// operand v already is; lane (n, half) then holds the z = half corners of its
// tile's query n, in registers 4 slot + 2 y + x.  Four such products take what
// the wave's 64 x 8 corner rows through L1 take: beyond that a lane reads its own
// rows.  Both ways add the channels in the same order (0, 16, 1, 17, ..): the same
// bits, whatever the other queries of the wave.
constexpr int kMaxCellGroups = 4;

__device__ __forceinline__ int tile_cells(uint32_t base, int t) {
    int cells = 0;
    for (uint32_t m = ~0u; m != 0 && cells <= 4 * kMaxCellGroups; ++cells) {
        const uint32_t cell = (uint32_t)__builtin_amdgcn_readlane((int)base, 32 * t + __ffs(m) - 1);
        m &= ~(uint32_t)(__ballot(base == cell) >> (32 * t));
    }
    return cells;
}

__device__ __forceinline__ void project_corners(const float* __restrict__ grid, int S, uint32_t base, uint32_t lane,
                                                bool use1, const CellFeatures& v, float (&pk)[8]) {
    const size_t sy = (size_t)S * kC, sz = (size_t)S * S * kC;
    const int groups = (tile_cells(base, 0) + 3) / 4 + (use1 ? (tile_cells(base, 1) + 3) / 4 : 0);
    if (groups > kMaxCellGroups) {
        float c0[16], c1[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(v.t[0][i]), __float_as_uint(v.t[1][i]),
                                                             false, false);
            c0[i] = __uint_as_float(sw[0]);
            c1[i] = __uint_as_float(sw[1]);
        }
        const float* b = grid + (size_t)base * kC;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float4* row = reinterpret_cast<const float4*>(b + (k & 1) * kC + (k & 2 ? sy : 0) + (k & 4 ? sz : 0));
            float p = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 lo = row[i], hi = row[4 + i];
                p = __builtin_fmaf(hi.x, c1[4 * i + 0], __builtin_fmaf(lo.x, c0[4 * i + 0], p));
                p = __builtin_fmaf(hi.y, c1[4 * i + 1], __builtin_fmaf(lo.y, c0[4 * i + 1], p));
                p = __builtin_fmaf(hi.z, c1[4 * i + 2], __builtin_fmaf(lo.z, c0[4 * i + 2], p));
                p = __builtin_fmaf(hi.w, c1[4 * i + 3], __builtin_fmaf(lo.w, c0[4 * i + 3], p));
            }
            pk[k] = p;
        }
        return;
    }
    const auto tb = __builtin_amdgcn_permlane32_swap(base, base, false, false);  // cells of tiles 0, 1's queries
    const uint32_t n = lane & 31u, slot = n >> 3;
    // A: lane (slot, corner), its half's 16 channels
    const float* mine = grid + (n & 1u) * kC + (n & 2u ? sy : 0) + (n & 4u ? sz : 0) + 16u * (lane >> 5);
    float p[2][4] = {};
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        if (t == 1 && !use1) continue;
        for (uint32_t m = ~0u; m != 0;) {
            uint32_t cell[4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                cell[s] = s == 0 || m != 0 ? (uint32_t)__builtin_amdgcn_readlane((int)tb[t], __ffs(m) - 1) : cell[0];
                m &= ~(uint32_t)__ballot(tb[t] == cell[s]);
            }
            const uint32_t c = slot < 2 ? (slot == 0 ? cell[0] : cell[1]) : (slot == 2 ? cell[2] : cell[3]);
            const float4* row = reinterpret_cast<const float4*>(mine + (size_t)c * kC);
            f32x16_t d = {};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float4 a = row[k];
                d = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, v.t[t][4 * k + 0], d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, v.t[t][4 * k + 1], d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, v.t[t][4 * k + 2], d, 0, 0, 0);
                d = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, v.t[t][4 * k + 3], d, 0, 0, 0);
            }
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const bool in = tb[t] == cell[s];
#pragma unroll
                for (int j = 0; j < 4; ++j) p[t][j] = in ? d[4 * s + j] : p[t][j];
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(p[0][j]), __float_as_uint(p[1][j]), false,
                                                         false);
        pk[j] = __uint_as_float(sw[0]);
        pk[4 + j] = __uint_as_float(sw[1]);
    }
}

// One level's share of the gradient onto g: the corners' projections times the
// derivatives of their weights.
__device__ __forceinline__ void project_level(const float* __restrict__ grid, int r, float px, float py, float pz,
                                              uint32_t lane, bool use1, const CellFeatures& v, float (&g)[3]) {
    const int S = r + 1;
    const float rf = (float)r;
    const AxisW ax = axis_weights(px, r);
    const AxisW ay = axis_weights(py, r);
    const AxisW az = axis_weights(pz, r);
    float pk[8];
    project_corners(grid, S, (uint32_t)((az.i0 * S + ay.i0) * S + ax.i0), lane, use1, v, pk);
    float dx = 0.0f, dy = 0.0f, dz = 0.0f;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float wx = k & 1 ? ax.w1 : ax.w0, wy = k & 2 ? ay.w1 : ay.w0, wz = k & 4 ? az.w1 : az.w0;
        dx = __builtin_fmaf(k & 1 ? pk[k] : -pk[k], wy * wz, dx);
        dy = __builtin_fmaf(k & 2 ? pk[k] : -pk[k], wx * wz, dy);
        dz = __builtin_fmaf(k & 4 ? pk[k] : -pk[k], wx * wy, dz);
    }
    auto slope = [&](float p) {  // d u / d p: 0 on and beyond the box's faces
        const float u = ((p + 1.0f) * 0.5f) * rf;
        return u > 0.0f && u < rf ? rf * 0.5f : 0.0f;
    };
    g[0] = __builtin_fmaf(slope(px), dx, g[0]);
    g[1] = __builtin_fmaf(slope(py), dy, g[1]);
    g[2] = __builtin_fmaf(slope(pz), dz, g[2]);
}

// sdf_fp32 of the wave's 64 queries; GRAD: and sdf_and_grad_fp32's gradient.
template <bool POSINV, bool GRAD>
__device__ __forceinline__ float sdf_cells(const ModelArgs& m, int lod, const GradLds* s, float b1, uint32_t lane,
                                           bool use1, float px, float py, float pz, float (&g)[3]) {
    CellFeatures f = zero_cell_features(), v = zero_cell_features();
    for (int l = 0; l <= lod; ++l) gather_cells(m.grid[l], m.res[l], px, py, pz, lane, use1, f);
    float q[2][3], vp[2][3] = {};
    tile_coords(px, py, pz, q[0][0], q[0][1], q[0][2], q[1][0], q[1][1], q[1][2]);
    const float y = decode_ordered<POSINV, GRAD>(f, s, b1, lane, q, v, vp);
    if (GRAD) {
#pragma unroll
        for (int a = 0; a < 3; ++a) g[a] = halves_sum(vp[0][a], vp[1][a]);
        for (int l = 0; l <= lod; ++l) project_level(m.grid[l], m.res[l], px, py, pz, lane, use1, v, g);
    }
    return y;
}

// Gradients, 64 queries a wave; order (optional): thread t takes point order[t].
// sdf (optional, autodiff): the values too.  Bound: the matrix cores (128 MFMAs a
// tile for both directions of the decoder, 4 and up to 16 per cell and level)
// where neighbouring queries share cells, else the corner rows of the finest
// levels through L1.  Persistent blocks: the decoder is staged once per block
// (three blocks a CU by registers; two: 229 instead of 215 us).  300001 uniform
// points at LOD 4, xyz decoder, with the sort, against one query per lane and
// the decoder on the vector ALU: autodiff 641 -> 215 us, finite differences 1346
// -> 501, tetrahedron 828 -> 390; 1000 points: 120 -> 94, 308 -> 236, 207 -> 167.
template <bool POSINV, int METHOD>
__global__ __launch_bounds__(256, 3) void gradient_fp32_kernel(ModelArgs m, int lod, int dec,
                                                               const float* __restrict__ x,
                                                               const uint8_t* __restrict__ mask, int64_t n,
                                                               int normalize, float* __restrict__ out,
                                                               float* __restrict__ sdf,
                                                               const uint32_t* __restrict__ order) {
    __shared__ GradLds lds;
    const bool finite = stage_grad_lds(m, dec, &lds);
    const uint32_t lane = lane_id();
    const float b1 = m.b1[dec][0];
    const int64_t waves = (int64_t)gridDim.x * 4;
    for (int64_t w = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6); w * 64 < n; w += waves) {
        const int64_t t = w * 64 + lane;
        const bool valid = t < n;
        const int64_t i = order ? order[valid ? t : n - 1] : (valid ? t : n - 1);
        const bool on = valid && (!mask || mask[i]);
        const uint64_t active = __ballot(on);
        float g[3] = {0.0f, 0.0f, 0.0f};
        if (active != 0) {
            // lanes without a query stand on one that has: no cells of their own
            float p0 = x[3 * i], p1 = x[3 * i + 1], p2 = x[3 * i + 2];
            const int some = __ffsll((unsigned long long)active) - 1;
            const float e0 = __shfl(p0, some), e1 = __shfl(p1, some), e2 = __shfl(p2, some);
            if (!on) {
                p0 = e0;
                p1 = e1;
                p2 = e2;
            }
            const bool use1 = (uint32_t)(active >> 32) != 0u;
            if (METHOD == NGLOD_GRAD_FINITEDIFF) {
                // diffutils.py:61-70: (f(x + h e_a) - f(x - h e_a)) / (2h)
#pragma unroll 1
                for (int a = 0; a < 3; ++a) {
                    float d[2];
#pragma unroll 1
                    for (int side = 0; side < 2; ++side) {
                        const float h = side ? -kFdH : kFdH;
                        const float y =
                            sdf_cells<POSINV, false>(m, lod, &lds, b1, lane, use1, a == 0 ? p0 + h : p0 + 0.0f,
                                                     a == 1 ? p1 + h : p1 + 0.0f, a == 2 ? p2 + h : p2 + 0.0f, g);
                        d[1] = side ? y : 0.0f;
                        d[0] = side ? d[0] : y;
                    }
                    const float da = (d[0] - d[1]) / kFdTwoH;
                    g[0] = a == 0 ? da : g[0];
                    g[1] = a == 1 ? da : g[1];
                    g[2] = a == 2 ? da : g[2];
                }
            } else if (METHOD == NGLOD_GRAD_TETRAHEDRON) {
                // k0 = (1,-1,-1), k1 = (-1,-1,1), k2 = (-1,1,-1), k3 = (1,1,1):
                // ((+f0 - f1) - f2) + f3, ((-f0 - f1) + f2) + f3, ((-f0 + f1) - f2) + f3
#pragma unroll 1
                for (int k = 0; k < 4; ++k) {
                    const float s0 = k == 0 || k == 3 ? kFdH : -kFdH, s1 = k >= 2 ? kFdH : -kFdH,
                                s2 = k & 1 ? kFdH : -kFdH;
                    const float y = sdf_cells<POSINV, false>(m, lod, &lds, b1, lane, use1, p0 + s0, p1 + s1,
                                                             p2 + s2, g);
                    g[0] = g[0] + (s0 > 0.0f ? y : -y);
                    g[1] = g[1] + (s1 > 0.0f ? y : -y);
                    g[2] = g[2] + (s2 > 0.0f ? y : -y);
                }
                g[0] = g[0] / kTetraFourH;
                g[1] = g[1] / kTetraFourH;
                g[2] = g[2] / kTetraFourH;
            } else {
                float y;
                if (finite)
                    y = sdf_cells<POSINV, true>(m, lod, &lds, b1, lane, use1, p0, p1, p2, g);
                else
                    y = sdf_and_grad_fp32<POSINV>(m, lod, dec, p0, p1, p2, g[0], g[1], g[2]);
                if (sdf && on) sdf[i] = y;
            }
            if (normalize) normalize_grad(g[0], g[1], g[2], g[0], g[1], g[2]);
        }
        if (valid) {
            out[3 * i] = on ? g[0] : 0.0f;
            out[3 * i + 1] = on ? g[1] : 0.0f;
            out[3 * i + 2] = on ? g[2] : 0.0f;
        }
    }
}

// ---------------------------------------------------------------------------
// SphereTracer.get_min, per ray (SphereTracer.py:134-218).  Differences from
// forward: every ray marches from its box entry (or from its origin, t = 0,
// when there is none: cond does not start from the box test), and the loop
// keeps the smallest distance seen, mind, with minx.  In the loop body the
// comparison d < mind runs after x has moved to o + d t, so minx is the point
// reached by the step of length d, not the point where d was evaluated.  The
// batch loop stops at the first iteration at which no ray is still marching;
// a ray that stops at iteration k < that one still runs the comparison once
// more at k (with x unchanged), a ray that stops at the batch's last
// iteration does not.  The first kernel marches each ray and records k and
// whether that last comparison would move minx; the batch's last iteration is
// the largest k (atomicMax); the second kernel applies the comparison.
struct TraceMinArgs {
    const float* ray_o;
    const float* ray_d;
    int64_t n;
    int num_steps;
    float min_dis, min_dis3, step, far_clip;
    float* x;
    float* t;
    uint8_t* hit;
    float* min_x;
    uint32_t* kinfo;  // [n]: k | (pending comparison << 31)
    uint32_t* kmax;   // [1]: the batch's last iteration
};

__global__ void trace_min_clear_kernel(uint32_t* kmax) {
    if (threadIdx.x == 0 && blockIdx.x == 0) *kmax = 0u;
}

template <bool POSINV>
__global__ __launch_bounds__(256) void trace_min_kernel(ModelArgs m, int lod, int dec, TraceMinArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const float ox = a.ray_o[3 * i], oy = a.ray_o[3 * i + 1], oz = a.ray_o[3 * i + 2];
    const float dx = a.ray_d[3 * i], dy = a.ray_d[3 * i + 1], dz = a.ray_d[3 * i + 2];
    const BoxEntry e = box_entry(ox, oy, oz, dx, dy, dz);
    float x0 = e.x, x1 = e.y, x2 = e.z, t = e.t;
    float D = sdf_fp32<POSINV>(m, lod, dec, x0, x1, x2);
    float Dp = D, mind = D;
    float m0 = x0, m1 = x1, m2 = x2;
    bool hitflag = false;
    int k = 0;
    bool pending = false;
    for (; k < a.num_steps; ++k) {
        hitflag = fabsf(t) < a.far_clip;
        const bool cond = (fabsf(D) > a.min_dis) && (fabsf((D + Dp) * 0.5f) > a.min_dis3) && hitflag;
        if (!cond) {
            pending = D < mind;
            break;
        }
        x0 = ox + dx * t;
        x1 = oy + dy * t;
        x2 = oz + dz * t;
        if (D < mind) {
            mind = D;
            m0 = x0;
            m1 = x1;
            m2 = x2;
        }
        Dp = D;
        D = sdf_fp32<POSINV>(m, lod, dec, x0, x1, x2) * a.step;
        t = t + D;
    }
    const bool outside = (fabsf(x0) > 1.0f) || (fabsf(x1) > 1.0f) || (fabsf(x2) > 1.0f);
    a.x[3 * i] = x0;
    a.x[3 * i + 1] = x1;
    a.x[3 * i + 2] = x2;
    a.t[i] = t;
    a.hit[i] = (hitflag && !outside) ? 1 : 0;
    a.min_x[3 * i] = m0;
    a.min_x[3 * i + 1] = m1;
    a.min_x[3 * i + 2] = m2;
    a.kinfo[i] = (uint32_t)k | (pending ? 0x80000000u : 0u);
    atomicMax(a.kmax, (uint32_t)k);
}

__global__ __launch_bounds__(256) void trace_min_finish_kernel(TraceMinArgs a) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n) return;
    const uint32_t info = a.kinfo[i];
    const uint32_t k = info & 0x7fffffffu;
    if ((info & 0x80000000u) && k < *a.kmax) {
        a.min_x[3 * i] = a.x[3 * i];
        a.min_x[3 * i + 1] = a.x[3 * i + 1];
        a.min_x[3 * i + 2] = a.x[3 * i + 2];
    }
}

template <bool POSINV>
static int launch_gradient(const ModelArgs& m, int lod, int dec, const float* x, const uint8_t* mask, int64_t n,
                           int method, int normalize, float* out, float* sdf, const uint32_t* order, hipStream_t s) {
    const int64_t blocks = (n + 255) / 256, cap = (int64_t)device_cu_count() * 3;
    const dim3 grid((unsigned)(blocks < cap ? blocks : cap));
    if (method == NGLOD_GRAD_FINITEDIFF)
        hipLaunchKernelGGL((gradient_fp32_kernel<POSINV, NGLOD_GRAD_FINITEDIFF>), grid, dim3(256), 0, s, m, lod, dec,
                           x, mask, n, normalize, out, sdf, order);
    else if (method == NGLOD_GRAD_TETRAHEDRON)
        hipLaunchKernelGGL((gradient_fp32_kernel<POSINV, NGLOD_GRAD_TETRAHEDRON>), grid, dim3(256), 0, s, m, lod, dec,
                           x, mask, n, normalize, out, sdf, order);
    else
        hipLaunchKernelGGL((gradient_fp32_kernel<POSINV, NGLOD_GRAD_AUTODIFF>), grid, dim3(256), 0, s, m, lod, dec, x,
                           mask, n, normalize, out, sdf, order);
    return check_launch("gradient_fp32_kernel");
}

// The gradient entries behind their own checks; ordered: points are sorted by
// cell first, in `workspace`.
static int run_gradient(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, int32_t form,
                        int32_t method, const uint8_t* mask, int32_t normalize, float* sdf, float* grad, bool ordered,
                        void* workspace, size_t workspace_bytes, hipStream_t s) {
    ModelArgs m;
    int rc = make_model_args(model, lod, form, &m);
    if (rc) return rc;
    if (n < 0 || n > (int64_t)0x7fff0000) return fail(NGLOD_ERR_ARG, "n out of range");
    if (n == 0) return NGLOD_OK;
    if (!x || !grad) return fail(NGLOD_ERR_ARG, "NULL pointer");
    const uint32_t* order = nullptr;
    if (ordered) {
        rc = launch_cell_order(x, n, model->res[lod], workspace, workspace_bytes, &order, s);
        if (rc) return rc;
    }
    const int dec = decoder_of(model, lod);
    const int gl = gather_lod(form, lod);
    return m.pos_inv ? launch_gradient<true>(m, gl, dec, x, mask, n, method, normalize, grad, sdf, order, s)
                     : launch_gradient<false>(m, gl, dec, x, mask, n, method, normalize, grad, sdf, order, s);
}

}  // namespace nglod

using namespace nglod;

extern "C" {

int nglod_gradient(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, int32_t form, int32_t method,
                   const uint8_t* mask, int32_t normalize, float* grad, void* stream) {
    if (method != NGLOD_GRAD_FINITEDIFF && method != NGLOD_GRAD_TETRAHEDRON && method != NGLOD_GRAD_AUTODIFF)
        return fail(NGLOD_ERR_ARG, "unknown gradient method");
    return run_gradient(model, x, n, lod, form, method, mask, normalize ? 1 : 0, nullptr, grad, false, nullptr, 0,
                        (hipStream_t)stream);
}

int nglod_gradient_ordered(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, int32_t form,
                           int32_t method, const uint8_t* mask, int32_t normalize, float* grad, void* workspace,
                           size_t workspace_bytes, void* stream) {
    if (method != NGLOD_GRAD_FINITEDIFF && method != NGLOD_GRAD_TETRAHEDRON && method != NGLOD_GRAD_AUTODIFF)
        return fail(NGLOD_ERR_ARG, "unknown gradient method");
    return run_gradient(model, x, n, lod, form, method, mask, normalize ? 1 : 0, nullptr, grad, true, workspace,
                        workspace_bytes, (hipStream_t)stream);
}

int nglod_sdf_grad(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, int32_t form, float* sdf,
                   float* grad, void* stream) {
    return run_gradient(model, x, n, lod, form, NGLOD_GRAD_AUTODIFF, nullptr, 0, sdf, grad, false, nullptr, 0,
                        (hipStream_t)stream);
}

size_t nglod_trace_min_workspace_size(int64_t n) {
    if (n < 0) n = 0;
    return 256 + ((size_t)n * 4 + 255) / 256 * 256;
}

int nglod_trace_min(const nglod_model_t* model, const float* ray_o, const float* ray_d, int64_t n, int32_t lod,
                    const nglod_trace_params_t* params, float* x, float* t, uint8_t* hit, float* min_x,
                    void* workspace, size_t workspace_bytes, void* stream) {
    ModelArgs m;
    int rc = make_model_args(model, lod, NGLOD_FP32, &m);
    if (rc) return rc;
    if (!params) return fail(NGLOD_ERR_ARG, "params is NULL");
    if (params->num_steps < 1) return fail(NGLOD_ERR_ARG, "num_steps must be >= 1");
    if (n < 0 || n > (int64_t)0x7fff0000) return fail(NGLOD_ERR_ARG, "n out of range");
    if (n == 0) return NGLOD_OK;
    if (!ray_o || !ray_d || !x || !t || !hit || !min_x) return fail(NGLOD_ERR_ARG, "NULL pointer");
    if (!workspace || workspace_bytes < nglod_trace_min_workspace_size(n) || ((uintptr_t)workspace & 3u))
        return fail(NGLOD_ERR_WORKSPACE, "workspace too small or not 4-byte aligned");
    TraceMinArgs a;
    a.ray_o = ray_o;
    a.ray_d = ray_d;
    a.n = n;
    a.num_steps = params->num_steps;
    a.min_dis = (float)params->min_dis;
    a.min_dis3 = (float)(params->min_dis * 3.0);
    a.step = (float)params->step_size;
    a.far_clip = (float)params->far_clip;
    a.x = x;
    a.t = t;
    a.hit = hit;
    a.min_x = min_x;
    a.kmax = (uint32_t*)workspace;
    a.kinfo = (uint32_t*)((char*)workspace + 256);
    const int dec = decoder_of(model, lod);
    hipStream_t s = (hipStream_t)stream;
    hipLaunchKernelGGL(trace_min_clear_kernel, dim3(1), dim3(64), 0, s, a.kmax);
    rc = check_launch("trace_min_clear_kernel");
    if (rc) return rc;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (m.pos_inv)
        hipLaunchKernelGGL(trace_min_kernel<true>, grid, dim3(256), 0, s, m, lod, dec, a);
    else
        hipLaunchKernelGGL(trace_min_kernel<false>, grid, dim3(256), 0, s, m, lod, dec, a);
    rc = check_launch("trace_min_kernel");
    if (rc) return rc;
    hipLaunchKernelGGL(trace_min_finish_kernel, grid, dim3(256), 0, s, a);
    return check_launch("trace_min_finish_kernel");
}

}  // extern "C"
