// Hand-written backward of the fused query (OctreeSDF.sdf, every level up
// to lod) for training, deterministic by construction (no float atomics):
//
// The training forward (nglod_sdf_fwd_save) runs steps 1 and 2 with the
// predictions and leaves their results for the backward.
//
//   1. the queries are visited in the Morton order of their cell in the
//      finest grid ("positions"), so that neighbouring lanes share corners;
//   2. features: per position and level the running trilinear features E
//      (stored by query) and the signs of the decoder's pre-activations
//      Z = W0 e + b0 (128 bits);
//   3. feature gradients: ds = W0^T dz with dz = g * W1 * [Z > 0], finest level
//      first; dg_l = ds_lod + .. + ds_l (stored by position);
//   4. decoder gradients: each block reduces a fixed chunk of queries in
//      query order into partial dW0 (FP32 MFMA), db0, dW1, db1, with Z computed
//      again from E; a second kernel sums fixed groups of partials in chunk
//      order and a third the group sums in group order (and over levels, in
//      level order, for a joint decoder);
//   5. grid gradients: every (query, corner) contribution w_c * dg gets the
//      corner index as a key; a stable radix sort groups equal corners with
//      queries in ascending order; runs are cut into pieces of kRunPiece
//      contributions summed in order, and the piece sums of a run are added in
//      order (coarse levels have runs of thousands of contributions, so a run
//      is not left to one lane).
//
// Every sum runs in the order of queries, whatever the visiting order, so the
// gradients do not depend on it.  Z and ds are chains of FP32 MFMA 32x32x2,
// which accumulate like FMA chains; Z is the forward's, bit for bit.
//
// Replaces autograd through F.grid_sample and nn.Linear in
// Trainer.step_geometry (sdf-net/lib/trainer.py:317-339).
#include <cstring>

#include <rocprim/rocprim.hpp>

#include "api_common.hpp"
#include "fp32_wave.hpp"
#include "radix_sort.hpp"

namespace nglod {

constexpr int kChunk = 256;    // queries per partial of the decoder-gradient reduction
constexpr int kRunPiece = 64;  // sorted contributions per partial of a corner's gradient

struct BwdArgs {
    ModelArgs m;
    int lod;
    int din;       // decoder input width (32 or 35)
    int off;       // 0 or 3: offset of the features in the decoder input
    int mask;      // bit i: level i has an incoming gradient
    int64_t n;
    const float* x;
    const float* g;         // [lod+1][n]
    const uint32_t* order;  // query of each position
    uint32_t* rank;         // position of each query
    float* xs;              // [n][3] points by position
    float* E;               // [lod+1][n][32] features by query
    uint4* bits;            // [lod+1][n] signs of Z by position: bit r of word h is row 32 h + r
    float* dg;              // [lod+1][n][32] feature gradients by position
};

// Morton code of a cell (10 bits per axis).
__device__ __forceinline__ uint32_t spread_bits(uint32_t v) {
    v &= 0x3FFu;
    v = (v | (v << 16)) & 0x030000FFu;
    v = (v | (v << 8)) & 0x0300F00Fu;
    v = (v | (v << 4)) & 0x030C30C3u;
    v = (v | (v << 2)) & 0x09249249u;
    return v;
}

// Key of each query's cell in a grid of resolution r.
__global__ __launch_bounds__(256) void bwd_cell_keys_kernel(const float* __restrict__ x, int64_t n, int r,
                                                            uint32_t* __restrict__ keys) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    keys[i] = (spread_bits((uint32_t)axis_weights(x[3 * i + 2], r).i0) << 2) |
              (spread_bits((uint32_t)axis_weights(x[3 * i + 1], r).i0) << 1) |
              spread_bits((uint32_t)axis_weights(x[3 * i], r).i0);
}

// One level of a model, as gather_fp32_add takes it.
struct OneLevel {
    int res[1];
    const float* grid[1];
};

// layer2_tile of fp32_wave.hpp, and the signs of its 16 pre-activations: bit
// 8 g + 4 half + j of `bits` is row 32 h + 8 g + 4 half + j.
__device__ __forceinline__ float layer2_tile_bits(const f32x16_t& c, int h, uint32_t half, const Fp32Lds* s, bool xyz,
                                                  float px, float py, float pz, uint32_t& bits) {
    float acc = 0.0f;
    bits = 0;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int row0 = 32 * h + 8 * g + 4 * (int)half;
        const float4 b = *reinterpret_cast<const float4*>(&s->b0[row0]);
        const float4 w = *reinterpret_cast<const float4*>(&s->w1[row0]);
        const float bv[4] = {b.x, b.y, b.z, b.w}, wv[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float v = c[4 * g + j] + bv[j];
            if (xyz) {
                const float4 q = *reinterpret_cast<const float4*>(s->wxyz[row0 + j]);
                v = __builtin_fmaf(q.x, px, __builtin_fmaf(q.y, py, __builtin_fmaf(q.z, pz, v)));
            }
            bits |= v > 0.0f ? 1u << (8 * g + j) : 0u;
            acc = __builtin_fmaf(wv[j], fmaxf(v, 0.0f), acc);
        }
    }
    bits <<= 4 * half;
    return acc;
}

// Features and pre-activation signs of 64 positions per wave, a persistent
// block: the decoders of its levels stay in LDS (dynamic: one Fp32Lds each).
// Block y takes levels l0 .. l1 of the split: all of them, or for few queries
// one (its features still start at level 0).  decode_fp32_wave's arithmetic;
// PRED: the levels' predictions too (the training forward), out [lod+1][n].
//
// 2^19 queries, 5 levels: the forward in query order 0.50 ms and the features
// again in the backward 0.30 ms -> 0.34 ms for both.
template <bool POSINV, bool PRED>
__global__ __launch_bounds__(512) void train_features_kernel(BwdArgs a, int split, float* __restrict__ out) {
    extern __shared__ __align__(16) char dyn[];
    Fp32Lds* lds = reinterpret_cast<Fp32Lds*>(dyn);
    const int l0 = split ? (int)blockIdx.y : 0, l1 = split ? (int)blockIdx.y : a.lod;
    const bool joint = a.m.num_dec == 1;
    for (int l = l0; l <= (joint ? l0 : l1); ++l) stage_fp32_lds(a.m, joint ? 0 : l, &lds[l - l0]);
    __syncthreads();
    const uint32_t lane = lane_id(), half = lane >> 5;
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t t = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); t * 64 < a.n; t += waves) {
        const int64_t pos = t * 64 + lane;
        const bool valid = pos < a.n;
        const int64_t q = valid ? (int64_t)a.order[pos] : 0;
        const float px = valid ? a.x[3 * q] : 0.0f, py = valid ? a.x[3 * q + 1] : 0.0f,
                    pz = valid ? a.x[3 * q + 2] : 0.0f;
        if (valid && l1 == a.lod) {
            a.rank[q] = (uint32_t)pos;
            a.xs[3 * pos] = px;
            a.xs[3 * pos + 1] = py;
            a.xs[3 * pos + 2] = pz;
        }
        const uint64_t am = __ballot(valid);
        const bool use1 = (uint32_t)(am >> 32) != 0u;  // tile 0 holds a position, or the loop had ended
        float qx0, qy0, qz0, qx1, qy1, qz1;
        tile_coords(px, py, pz, qx0, qy0, qz0, qx1, qy1, qz1);
        float f[kC];
#pragma unroll
        for (int c = 0; c < kC; ++c) f[c] = 0.0f;
        for (int l = 0; l <= l1; ++l) {
            if (valid) {
                const OneLevel one = {{a.m.res[l]}, {a.m.grid[l]}};
                gather_fp32_add<1>(one, 0, px, py, pz, f);
            }
            if (l < l0 || !((a.mask >> l) & 1)) continue;
            if (valid) {
                float4* E4 = reinterpret_cast<float4*>(a.E + ((size_t)l * a.n + q) * kC);
#pragma unroll
                for (int c = 0; c < kC / 4; ++c) E4[c] = make_float4(f[4 * c], f[4 * c + 1], f[4 * c + 2], f[4 * c + 3]);
            }
            const Fp32Lds* s = &lds[joint ? 0 : l - l0];
            float B0[kC / 2], B1[kC / 2];
#pragma unroll
            for (int kk = 0; kk < kC / 2; ++kk) {
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(f[2 * kk]),
                                                                 __float_as_uint(f[2 * kk + 1]), false, false);
                B0[kk] = __uint_as_float(sw[0]);
                B1[kk] = __uint_as_float(sw[1]);
            }
            uint32_t* word = reinterpret_cast<uint32_t*>(a.bits + (size_t)l * a.n + (valid ? pos : 0));
            float part[2] = {0.0f, 0.0f};
#pragma unroll 1
            for (int h = 0; h < 4; ++h) {
                uint32_t b[2] = {0u, 0u};
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    if (u == 1 && !use1) continue;
                    f32x16_t c = {};
#pragma unroll
                    for (int kq = 0; kq < 4; ++kq) {
                        const float4 w = s->afrag[(h * 4 + kq) * 64 + lane];
                        const float* B = u == 0 ? B0 : B1;
                        c = __builtin_amdgcn_mfma_f32_32x32x2f32(w.x, B[4 * kq + 0], c, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_32x32x2f32(w.y, B[4 * kq + 1], c, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_32x32x2f32(w.z, B[4 * kq + 2], c, 0, 0, 0);
                        c = __builtin_amdgcn_mfma_f32_32x32x2f32(w.w, B[4 * kq + 3], c, 0, 0, 0);
                    }
                    const float sum = layer2_tile_bits(c, h, half, s, !POSINV, u == 0 ? qx0 : qx1,
                                                       u == 0 ? qy0 : qy1, u == 0 ? qz0 : qz1, b[u]);
                    if (PRED) part[u] += sum;
                }
                const auto sw = __builtin_amdgcn_permlane32_swap(b[0], b[1], false, false);
                if (valid) word[h] = sw[0] | sw[1];
            }
            if (PRED) {
                const float d = halves_sum(part[0], part[1]) + a.m.b1[joint ? 0 : l][0];
                if (valid) out[(size_t)l * a.n + q] = d;
            }
        }
    }
}

// W0^T of one level's decoder as A operands: frag[(4 h + g) 64 + lane] holds, for
// j = 0 .. 3, W0[32 h + 8 g + 4 (lane / 32) + j][off + lane % 32]: k-step (h, g, j)
// pairs hidden rows 8 g + j and 8 g + 4 + j.
struct BwdLds {
    float4 frag[16 * 64];
    float w1[kH];
};

__device__ __forceinline__ void stage_bwd_lds(const ModelArgs& m, int dec, int din, int off, BwdLds* s) {
    const float* W0 = m.w0[dec];
    for (int t = threadIdx.x; t < 16 * 64; t += blockDim.x) {
        const int lane = t & 63, g = (t >> 6) & 3, h = t >> 8;
        const float* p = W0 + (size_t)(32 * h + 8 * g + 4 * (lane >> 5)) * din + off + (lane & 31);
        s->frag[t] = make_float4(p[0], p[din], p[2 * din], p[3 * din]);
    }
    for (int t = threadIdx.x; t < kH; t += blockDim.x) s->w1[t] = m.w1[dec][t];
}

// Feature gradients of 32 positions per wave: ds^T = W0^T dz by FP32 MFMA, dz
// from the signs and g * W1 on the fly (lane (n, half): the rows 8 g + 4 half + j
// of query n), the levels from the finest down with their running sum in
// registers.  split: block y takes one level and stores its ds
// (bwd_suffix_kernel then adds the levels up).
__global__ __launch_bounds__(512) void bwd_ds_kernel(BwdArgs a, int split) {
    extern __shared__ __align__(16) char dyn[];
    BwdLds* lds = reinterpret_cast<BwdLds*>(dyn);
    const int l0 = split ? (int)blockIdx.y : 0, l1 = split ? (int)blockIdx.y : a.lod;
    const bool joint = a.m.num_dec == 1;
    for (int l = l0; l <= (joint ? l0 : l1); ++l) stage_bwd_lds(a.m, joint ? 0 : l, a.din, a.off, &lds[l - l0]);
    __syncthreads();
    const uint32_t lane = lane_id();
    const int col = lane & 31, half = lane >> 5;
    const int64_t waves = (int64_t)gridDim.x * (blockDim.x >> 6);
    for (int64_t t = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); t * 32 < a.n; t += waves) {
        const bool in = t * 32 + col < a.n;
        const int64_t pos = in ? t * 32 + col : a.n - 1;
        const int64_t q = a.order[pos];
        float sum[16];
        for (int l = l1; l >= l0; --l) {
            f32x16_t d = {};
            if ((a.mask >> l) & 1) {
                const BwdLds* s = &lds[joint ? 0 : l - l0];
                const float gq = a.g[(size_t)l * a.n + q];
                const uint4 bw = a.bits[(size_t)l * a.n + pos];
                const uint32_t word[4] = {bw.x >> (4 * half), bw.y >> (4 * half), bw.z >> (4 * half), bw.w >> (4 * half)};
#pragma unroll
                for (int h = 0; h < 4; ++h)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const float4 w = *reinterpret_cast<const float4*>(&s->w1[32 * h + 8 * g + 4 * half]);
                        const float4 f = s->frag[(4 * h + g) * 64 + lane];
                        const uint32_t b = word[h] >> (8 * g);
                        d = __builtin_amdgcn_mfma_f32_32x32x2f32(f.x, (b & 1u) ? gq * w.x : 0.0f, d, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_32x32x2f32(f.y, (b & 2u) ? gq * w.y : 0.0f, d, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_32x32x2f32(f.z, (b & 4u) ? gq * w.z : 0.0f, d, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_f32_32x32x2f32(f.w, (b & 8u) ? gq * w.w : 0.0f, d, 0, 0, 0);
                    }
            }
#pragma unroll
            for (int i = 0; i < 16; ++i) sum[i] = l == l1 ? d[i] : sum[i] + d[i];
            if (!in) continue;
            // lane (n, half) holds channels 8 i + 4 half + (0..3) of query n
            float* out = a.dg + ((size_t)l * a.n + pos) * kC + 4 * half;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<float4*>(out + 8 * i) =
                    make_float4(sum[4 * i], sum[4 * i + 1], sum[4 * i + 2], sum[4 * i + 3]);
        }
    }
}

// Partial decoder gradients of level blockIdx.y over one chunk of kChunk
// queries.  Output layout per (level, chunk): dW0 [128][din], db0 [128], dW1
// [128], db1 [1].  Wave w owns hidden rows 32w..32w+31, a lane one row and every
// other query: Z = E W0^T as FP32 MFMA 32x32x2 (A = E: row m of a 32-query tile
// is query 2 (4 (m / 8) + m % 4) + m / 4 % 2, so that register i of half hf holds
// query 2 i + hf; B = the wave's rows of W0, in registers), which leaves dz where
// dW0 = dZ^T E needs it: step i takes queries 2i and 2i + 1, A[m][k] = dz of query
// 2i + k at row m, B[k][n] = E of that query at channel n.  The products are exact
// and accumulate in FP32 in query order, so a partial is the same every run.
// db0, dW1 and db1 accumulate in the lanes beside it (each half-wave over its
// query of every pair, the two halves added at the end), and so do the xyz
// columns of dW0, each lane over both queries.
//
// Z again instead of read back (268 MB per level at 2^19 queries) makes the
// matrix cores the bound: 2^19 queries, 5 levels:
// 0.91 -> 0.53 ms, and Z is not written either.
template <bool POSINV>
__global__ __launch_bounds__(256) void bwd_decoder_partial_kernel(BwdArgs a, float* __restrict__ part,
                                                                  int64_t nchunks) {
    const int level = blockIdx.y;
    if (!((a.mask >> level) & 1)) return;
    __shared__ float4 qs[kChunk];  // x, y, z, g of the chunk's queries; 0 past the end
    const int64_t chunk = blockIdx.x;
    const int64_t q0 = chunk * kChunk;
    const int cnt = (int)(a.n - q0 < kChunk ? a.n - q0 : kChunk);
    {
        const int i = threadIdx.x;
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (i < cnt) {
            if (!POSINV) {
                v.x = a.x[3 * (q0 + i)];
                v.y = a.x[3 * (q0 + i) + 1];
                v.z = a.x[3 * (q0 + i) + 2];
            }
            v.w = a.g[(size_t)level * a.n + q0 + i];
        }
        qs[i] = v;
    }
    const int wave = threadIdx.x >> 6;
    const int lane = threadIdx.x & 63;
    const int col = lane & 31;
    const int half = lane >> 5;
    const int j = 32 * wave + col;
    const int dec = a.m.num_dec == 1 ? 0 : level;
    const float* W0 = a.m.w0[dec] + (size_t)j * a.din;
    const float w1 = a.m.w1[dec][j], b0 = a.m.b0[dec][j];
    const float wx = POSINV ? 0.0f : W0[0], wy = POSINV ? 0.0f : W0[1], wz = POSINV ? 0.0f : W0[2];
    float Bw[kC / 2];
#pragma unroll
    for (int kk = 0; kk < kC / 2; ++kk) Bw[kk] = W0[a.off + 2 * kk + half];
    const float* El = a.E + ((size_t)level * a.n + q0) * kC;
    const int am = 2 * (4 * (col >> 3) + (col & 3)) + ((col >> 2) & 1);  // A row -> query of the tile
    float4 ra[4];
    float re[16];
    auto load = [&](int t) {  // tile t's rows, both ways round
        const int qa = min(t + am, cnt - 1);
        const float4* e4 = reinterpret_cast<const float4*>(El + (size_t)qa * kC + 16 * half);
#pragma unroll
        for (int i = 0; i < 4; ++i) ra[i] = e4[i];
#pragma unroll
        for (int i = 0; i < 16; ++i) re[i] = El[(size_t)min(t + 2 * i + half, cnt - 1) * kC + col];
    };
    load(0);
    __syncthreads();
    f32x16_t c0 = {};
    float cx = 0.0f, cy = 0.0f, cz = 0.0f;
    float acc_b0 = 0.0f, acc_w1 = 0.0f, acc_b1 = 0.0f;
    for (int t = 0; t < cnt; t += 32) {
        float A[kC / 2], e[16];
        {
            const float r[16] = {ra[0].x, ra[0].y, ra[0].z, ra[0].w, ra[1].x, ra[1].y, ra[1].z, ra[1].w,
                                 ra[2].x, ra[2].y, ra[2].z, ra[2].w, ra[3].x, ra[3].y, ra[3].z, ra[3].w};
            // lane (m, half) holds channels 16 half ..: a swap per pair puts channel 2 kk + half in A[kk]
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(r[2 * k]),
                                                                 __float_as_uint(r[2 * k + 1]), false, false);
                A[k] = __uint_as_float(sw[0]);
                A[8 + k] = __uint_as_float(sw[1]);
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) e[i] = t + 2 * i + half < cnt ? re[i] : 0.0f;
        if (t + 32 < cnt) load(t + 32);  // in flight during this tile's products
        f32x16_t z = {};
#pragma unroll
        for (int kk = 0; kk < kC / 2; ++kk) z = __builtin_amdgcn_mfma_f32_32x32x2f32(A[kk], Bw[kk], z, 0, 0, 0);
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const bool valid = t + 2 * i + half < cnt;
            const float4 own = qs[t + 2 * i + half];
            float v = z[i] + b0;
            if (!POSINV) v = __builtin_fmaf(wx, own.x, __builtin_fmaf(wy, own.y, __builtin_fmaf(wz, own.z, v)));
            const float dz = valid && v > 0.0f ? own.w * w1 : 0.0f;
            acc_b0 = valid ? acc_b0 + dz : acc_b0;
            acc_w1 = valid ? __builtin_fmaf(own.w, v > 0.0f ? v : 0.0f, acc_w1) : acc_w1;
            acc_b1 = valid ? acc_b1 + own.w : acc_b1;
            c0 = __builtin_amdgcn_mfma_f32_32x32x2f32(dz, e[i], c0, 0, 0, 0);
            if (!POSINV) {
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(dz), __float_as_uint(dz), false, false);
                const float d0 = __uint_as_float(sw[0]), d1 = __uint_as_float(sw[1]);
                const float4 p0 = qs[t + 2 * i], p1 = qs[t + 2 * i + 1];
                cx = __builtin_fmaf(d1, p1.x, __builtin_fmaf(d0, p0.x, cx));
                cy = __builtin_fmaf(d1, p1.y, __builtin_fmaf(d0, p0.y, cy));
                cz = __builtin_fmaf(d1, p1.z, __builtin_fmaf(d0, p0.z, cz));
            }
        }
    }
    const int outs = kH * a.din + 2 * kH + 1;
    float* P = part + ((size_t)level * nchunks + chunk) * outs;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int row = 32 * wave + 8 * (i >> 2) + 4 * half + (i & 3);
        P[row * a.din + a.off + col] = c0[i];
    }
    acc_b0 += __shfl_xor(acc_b0, 32);
    acc_w1 += __shfl_xor(acc_w1, 32);
    acc_b1 += __shfl_xor(acc_b1, 32);
    if (half == 0) {
        if (!POSINV) {
            P[j * a.din + 0] = cx;
            P[j * a.din + 1] = cy;
            P[j * a.din + 2] = cz;
        }
        P[kH * a.din + j] = acc_b0;
        P[kH * a.din + kH + j] = acc_w1;
    }
    if (threadIdx.x == 0) P[kH * a.din + 2 * kH] = acc_b1;
}

// First stage of the partials' sum: group g of level l (grid z) adds chunks
// g*kGroup .. g*kGroup+kGroup-1 in order for every output.
constexpr int kGroup = 32;

__global__ void bwd_decoder_group_kernel(BwdArgs a, const float* __restrict__ part, int64_t nchunks,
                                         float* __restrict__ gpart, int64_t ngroups) {
    const int outs = kH * a.din + 2 * kH + 1;
    const int o = blockIdx.x * blockDim.x + threadIdx.x;
    const int l = blockIdx.z;
    const int64_t g = blockIdx.y;
    if (o >= outs || !((a.mask >> l) & 1)) return;
    const int64_t c0 = g * kGroup;
    const int64_t c1 = c0 + kGroup < nchunks ? c0 + kGroup : nchunks;
    const float* P = part + (size_t)l * nchunks * outs + o;
    float s = 0.0f;
    for (int64_t c = c0; c < c1; ++c) s += P[c * outs];
    gpart[((size_t)l * ngroups + g) * outs + o] = s;
}

// Sums the group sums of decoder blockIdx.y over its levels (ascending) and
// groups (ascending) and writes dW0, db0, dW1, db1 (0 for a decoder that no level
// with a gradient uses).
__global__ void bwd_decoder_final_kernel(BwdArgs a, const float* __restrict__ gpart, int64_t ngroups,
                                         nglod_model_grads_t grads) {
    const int outs = kH * a.din + 2 * kH + 1;
    const int o = blockIdx.x * blockDim.x + threadIdx.x;
    const int dec = blockIdx.y;
    if (o >= outs) return;
    float s = 0.0f;
    for (int l = 0; l <= a.lod; ++l) {
        const int d = a.m.num_dec == 1 ? 0 : l;
        if (d != dec || !((a.mask >> l) & 1)) continue;
        const float* P = gpart + (size_t)l * ngroups * outs + o;
        for (int64_t g = 0; g < ngroups; ++g) s += P[g * outs];
    }
    if (o < kH * a.din) grads.w0[dec][o] = s;
    else if (o < kH * a.din + kH) grads.b0[dec][o - kH * a.din] = s;
    else if (o < kH * a.din + 2 * kH) grads.w1[dec][o - kH * a.din - kH] = s;
    else grads.b1[dec][0] = s;
}

// ds_l(q) -> dg_l(q) = sum_{i >= l} ds_i(q) in place, added from the finest
// level down (((ds_lod + ds_lod-1) + ...) + ds_l): one thread per query and
// group of 4 channels.  (Where bwd_ds_kernel ran a level per block.)
__global__ void bwd_suffix_kernel(BwdArgs a) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= a.n * (kC / 4)) return;
    const int64_t q = t / (kC / 4);
    const int c4 = (int)(t % (kC / 4));
    float4 acc = reinterpret_cast<const float4*>(a.dg + ((size_t)a.lod * a.n + q) * kC)[c4];
    for (int l = a.lod - 1; l >= 0; --l) {
        float4* d = reinterpret_cast<float4*>(a.dg + ((size_t)l * a.n + q) * kC) + c4;
        const float4 v = *d;
        acc.x += v.x;
        acc.y += v.y;
        acc.z += v.z;
        acc.w += v.w;
        *d = acc;
    }
}

// The levels of one sort: the corners of level i have keys base[i] .. base[i+1] - 1.
struct CornerLevels {
    int count;
    int level[NGLOD_MAX_LODS];
    int res[NGLOD_MAX_LODS];
    uint32_t base[NGLOD_MAX_LODS + 1];
    float* grad[NGLOD_MAX_LODS];
    uint32_t strided;  // bit i: many pieces per corner, added by bwd_run_strided_kernel
};

__device__ __forceinline__ int level_of(const CornerLevels& L, uint32_t key) {
    int i = 0;
    while (i + 1 < L.count && key >= L.base[i + 1]) ++i;
    return i;
}

// Keys (corner) and values (position * 8 + corner slot) in query order.
__global__ __launch_bounds__(256) void bwd_corner_keys_kernel(BwdArgs a, CornerLevels L, uint32_t* __restrict__ keys,
                                                              uint32_t* __restrict__ vals) {
    const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (q >= a.n) return;
    const int i = blockIdx.y;
    const int r = L.res[i];
    const int S = r + 1;
    const AxisW ax = axis_weights(a.x[3 * q], r);
    const AxisW ay = axis_weights(a.x[3 * q + 1], r);
    const AxisW az = axis_weights(a.x[3 * q + 2], r);
    const uint32_t k = L.base[i] + (uint32_t)((az.i0 * S + ay.i0) * S + ax.i0);
    const uint32_t v = a.rank[q] * 8u;
    uint4* ko = reinterpret_cast<uint4*>(keys + ((size_t)i * a.n + q) * 8);
    uint4* vo = reinterpret_cast<uint4*>(vals + ((size_t)i * a.n + q) * 8);
    const uint32_t sy = (uint32_t)S, sz = (uint32_t)(S * S);
    ko[0] = make_uint4(k, k + 1, k + sy, k + sy + 1);
    ko[1] = make_uint4(k + sz, k + sz + 1, k + sz + sy, k + sz + sy + 1);
    vo[0] = make_uint4(v, v + 1, v + 2, v + 3);
    vo[1] = make_uint4(v + 4, v + 5, v + 6, v + 7);
}

// runs[key] = {first sorted entry, past the last} of each key that occurs.
__global__ __launch_bounds__(256) void bwd_runs_kernel(const uint32_t* __restrict__ keys, uint32_t m,
                                                       uint2* __restrict__ runs) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= m) return;
    const uint32_t k = keys[i];
    if (i == 0 || keys[i - 1] != k) runs[k].x = i;
    if (i == m - 1 || keys[i + 1] != k) runs[k].y = i + 1;
}

// Sums of the pieces that start in a window of `size` sorted entries: piece p
// of a run covers its entries 64 p .. 64 p + 63, each contribution
// w_c(x) * dg one FMA per channel, in order.  8 lanes take a piece (a float4 of
// channels each, so a row of dg is one coalesced 128-byte access); their
// entries' rows and weights are worked out 8 at a time, one per lane, and
// passed round.  A run's first piece goes to its gradient (the whole of it for
// most fine-level runs), the others to row (first entry) / 64 of `partial`:
// later pieces of all runs start at least 64 entries apart.
//
// 2^19 queries, 5 levels: 1.13 ms with a lane per piece and the rows in query
// order -> 0.45 ms.
// A window is smaller where the entries would not fill the GPU (512 queries, 10
// windows of 2048: 123 us, 80 of 256: 18 us).
constexpr int kWindow = 2048;

__global__ __launch_bounds__(256) void bwd_pieces_kernel(BwdArgs a, CornerLevels L, const uint32_t* __restrict__ keys,
                                                         const uint32_t* __restrict__ vals, uint32_t m, uint32_t size,
                                                         const uint2* __restrict__ runs, float* __restrict__ partial) {
    __shared__ uint32_t starts[kWindow];
    __shared__ uint32_t count;
    if (threadIdx.x == 0) count = 0;
    __syncthreads();
    // consecutive windows on one XCD (blocks go to the XCDs in turn): their rows share its L2
    const uint32_t per = (gridDim.x + 7) / 8;
    const uint32_t window = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    const uint64_t w0 = (uint64_t)window * size;
    const uint32_t lane = lane_id();
    for (uint32_t r = 0; r < size / 256; ++r) {
        const uint64_t i = w0 + r * 256 + threadIdx.x;
        const bool first = i < m && (((uint32_t)i - runs[keys[i]].x) & (kRunPiece - 1)) == 0;
        const uint64_t mask = __ballot(first);
        uint32_t at = 0;
        if (lane == 0 && mask) at = atomicAdd(&count, (uint32_t)__popcll(mask));
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
        if (first) starts[at + mask_rank(mask)] = (uint32_t)i;
    }
    __syncthreads();
    const uint32_t total = count;
    const uint32_t c = threadIdx.x & 7u;
    // every lane of a wave takes part in the exchanges until the wave's last piece is done
    for (uint32_t p = threadIdx.x >> 3; __ballot(p < total) != 0; p += 32) {
        const bool on = p < total;
        const uint32_t i0 = on ? starts[p] : 0u;
        const uint32_t key = on ? keys[i0] : 0u;
        const uint2 run = on ? runs[key] : make_uint2(0u, 0u);
        const uint32_t end = on ? min(run.y, i0 + kRunPiece) : 0u;
        const int li = level_of(L, key);
        const int res = L.res[li];
        const float* dg = a.dg + (size_t)L.level[li] * a.n * kC + 4 * c;
        float4 acc = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        for (uint32_t i = i0; __ballot(i < end) != 0; i += 8) {
            uint32_t row = 0;
            float w = 0.0f;
            if (i + c < end) {
                const uint32_t v = vals[i + c];
                row = v >> 3;
                const AxisW ax = axis_weights(a.xs[3 * (size_t)row], res);
                const AxisW ay = axis_weights(a.xs[3 * (size_t)row + 1], res);
                const AxisW az = axis_weights(a.xs[3 * (size_t)row + 2], res);
                w = (((v & 1) ? ax.w1 : ax.w0) * ((v & 2) ? ay.w1 : ay.w0)) * ((v & 4) ? az.w1 : az.w0);
            }
            float4 d[8];
            float wk[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint32_t rk = (uint32_t)__shfl((int)row, (int)((lane & 56u) + k));
                wk[k] = __shfl(w, (int)((lane & 56u) + k));
                d[k] = i + k < end ? *reinterpret_cast<const float4*>(dg + (size_t)rk * kC)
                                   : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (i + k < end) {
                    acc.x = __builtin_fmaf(wk[k], d[k].x, acc.x);
                    acc.y = __builtin_fmaf(wk[k], d[k].y, acc.y);
                    acc.z = __builtin_fmaf(wk[k], d[k].z, acc.z);
                    acc.w = __builtin_fmaf(wk[k], d[k].w, acc.w);
                }
            }
        }
        if (!on) continue;
        float4* grad = reinterpret_cast<float4*>(L.grad[li] + (size_t)(key - L.base[li]) * kC) + c;
        if (run.y - run.x <= (uint32_t)kRunPiece) {  // the sum of one piece, added to 0 as the others are
            *grad = make_float4(0.0f + acc.x, 0.0f + acc.y, 0.0f + acc.z, 0.0f + acc.w);
        } else if (i0 == run.x) {
            *grad = acc;
        } else {
            reinterpret_cast<float4*>(partial + (size_t)(i0 / kRunPiece) * kC)[c] = acc;
        }
    }
}

// Piece p of a run with several: the first lies in the run's gradient.
__device__ __forceinline__ float piece_of(const float* grad, const float* partial, uint32_t first, uint32_t p, int c) {
    return p == 0 ? grad[c] : partial[(size_t)((first + p * kRunPiece) / kRunPiece) * kC + c];
}

// A thread per (corner, channel) and turn: sums the run's pieces in order.  The
// grid is capped: 8 levels of up to 512^3 cells are 4.9e9 (corner, channel) pairs,
// and a launch holds fewer than 2^32 threads.
constexpr uint32_t kFinalBlocks = 1u << 20;
static_assert((uint64_t)kFinalBlocks * 256 < ((uint64_t)1 << 32), "threads of a launch");

__global__ __launch_bounds__(256) void bwd_run_final_kernel(CornerLevels L, const uint2* __restrict__ runs,
                                                            const float* __restrict__ partial) {
    const uint64_t end = (uint64_t)L.base[L.count] * kC;
    for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < end; t += (uint64_t)gridDim.x * 256) {
        const uint32_t k = (uint32_t)(t / kC);
        const int c = (int)(t % kC);
        const uint2 run = runs[k];
        const uint32_t cnt = run.y - run.x;
        if (cnt <= (uint32_t)kRunPiece) continue;
        const int li = level_of(L, k);
        if ((L.strided >> li) & 1u) continue;
        float* grad = L.grad[li] + (size_t)(k - L.base[li]) * kC;
        const uint32_t np = (cnt + kRunPiece - 1) / kRunPiece;
        float s = 0.0f;
        for (uint32_t p = 0; p < np; ++p) s += piece_of(grad, partial, run.x, p, c);
        grad[c] = s;
    }
}

// The same sums for levels whose runs hold many pieces (the coarse grids:
// 2^19 queries put ~500 pieces in each of LOD 0's 125 corners): one block of
// kRunGroups x kC threads per run; thread (g, c) sums pieces g, g + kRunGroups,
// ... of channel c in order (a row of kC partials is one coalesced load for
// the block's 32 channels), then thread (0, c) adds the kRunGroups group sums
// in group order.  A fixed order, so the result is the same every run.  A
// strided level has at most n / 64 corners, so all of them below 2^22 blocks.
constexpr int kRunGroups = 8;

__global__ __launch_bounds__(kRunGroups * kC) void bwd_run_strided_kernel(CornerLevels L, const uint2* __restrict__ runs,
                                                                          const float* __restrict__ partial) {
    __shared__ float gs[kRunGroups][kC];
    // block b: corner b of the strided levels, counted through them alone
    uint32_t k = blockIdx.x;
    int li = 0;
    for (;; ++li) {
        if (!((L.strided >> li) & 1u)) continue;
        const uint32_t corners = L.base[li + 1] - L.base[li];
        if (k < corners) break;
        k -= corners;
    }
    k += L.base[li];
    const uint2 run = runs[k];
    const uint32_t cnt = run.y - run.x;
    if (cnt == 0) return;
    float* grad = L.grad[li] + (size_t)(k - L.base[li]) * kC;
    const int c = threadIdx.x % kC;
    const int g = threadIdx.x / kC;
    const uint32_t np = (cnt + kRunPiece - 1) / kRunPiece;
    float s = 0.0f;
    for (uint32_t p = g; p < np; p += kRunGroups) s += piece_of(grad, partial, run.x, p, c);
    gs[g][c] = s;
    __syncthreads();
    if (g == 0) {
        float t = gs[0][c];
#pragma unroll
        for (int i = 1; i < kRunGroups; ++i) t += gs[i][c];
        grad[c] = t;
    }
}

__global__ void fill_f32_kernel(float* p, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0f;
}

// Zeroes every gradient of a call and the run table.
struct FillList {
    float* p[5 * NGLOD_MAX_LODS + 1];
    int64_t n[5 * NGLOD_MAX_LODS + 1];
};
__global__ __launch_bounds__(256) void bwd_fill_kernel(FillList l) {
    float* p = l.p[blockIdx.y];
    const int64_t n = l.n[blockIdx.y];
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) p[i] = 0.0f;
}

// What the training forward leaves for the backward.
struct SavedLayout {
    size_t order, rank, xs, E, bits, total;
};

struct BwdLayout {
    size_t saved, order_ws, dg, part, gpart, keys_in, keys_out, vals_in, vals_out, sort_tmp, runs, partial, total;
    size_t sort_bytes;
    int64_t nchunks, ngroups;
    bool together;  // the contributions of all levels in one sort
};

static int bits_for(uint64_t keys) {
    int b = 1;
    while ((1ull << b) < keys) ++b;
    return b;
}
static int cell_bits(int r) {  // of the Morton codes of a grid's cells
    int b = 1;
    while ((1 << b) < r) ++b;
    return 3 * b;
}
static uint64_t corners_of(int r) { return (uint64_t)(r + 1) * (r + 1) * (r + 1); }

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

// One sort of all levels' contributions up to this many, else a sort per level:
// fewer launches against more sorting passes over a level's contributions (and
// buffers of one level's size).  Steps in us, together / per level: 3 levels 774 / 867 with
// 2^18 queries, 1353 / 1398 with 2^19, 2647 / 2628 with 2^20 (3 << 23 contributions), 10870 /
// 10520 with 2^22; 5 levels 1381 / 1509, 2384 / 2388, 4614 / 4428, 18740 / 17190.
constexpr int64_t kTogether = (int64_t)3 << 23;

static void saved_layout(int64_t n, int lod, SavedLayout* L) {
    const size_t levels = (size_t)lod + 1;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off += align256(bytes);
        return at;
    };
    L->order = take((size_t)n * 4);
    L->rank = take((size_t)n * 4);
    L->xs = take((size_t)n * 3 * sizeof(float));
    L->bits = take(levels * n * sizeof(uint4));
    L->E = take(levels * n * kC * sizeof(float));
    L->total = off;
}

// saved: the features come from a training forward, else the call computes them.
static int bwd_layout(int64_t n, int lod, int din, const int32_t* res, bool saved, BwdLayout* L) {
    const size_t levels = (size_t)lod + 1;
    L->nchunks = (n + kChunk - 1) / kChunk;
    L->ngroups = (L->nchunks + kGroup - 1) / kGroup;
    const size_t outs = (size_t)kH * din + 2 * kH + 1;
    size_t off = 0;
    auto take = [&](size_t bytes) {
        const size_t at = off;
        off += align256(bytes);
        return at;
    };
    uint64_t corners = 0, most = 0;
    for (int l = 0; l <= lod; ++l) {
        corners += corners_of(res[l]);
        most = corners_of(res[l]) > most ? corners_of(res[l]) : most;
    }
    L->together = (int64_t)levels * n * 8 < kTogether && corners < ((uint64_t)1 << 31);
    const size_t m = (size_t)n * 8 * (L->together ? levels : 1);
    SavedLayout S;
    saved_layout(n, lod, &S);
    L->saved = saved ? 0 : take(S.total);
    L->order_ws = saved ? 0 : take(sort_workspace_bytes(n));
    L->dg = take(levels * n * kC * sizeof(float));
    L->part = take(levels * L->nchunks * outs * sizeof(float));
    L->gpart = take(levels * L->ngroups * outs * sizeof(float));
    L->keys_in = take(m * 4);
    L->keys_out = take(m * 4);
    L->vals_in = take(m * 4);
    L->vals_out = take(m * 4);
    size_t tmp = 0;
    for (int j = 0; j <= lod; ++j) {
        size_t t = 0;
        if (rocprim::radix_sort_pairs((void*)nullptr, t, (uint32_t*)nullptr, (uint32_t*)nullptr, (uint32_t*)nullptr,
                                      (uint32_t*)nullptr, m, 0, bits_for(L->together ? corners : corners_of(res[j])),
                                      (hipStream_t)0) != hipSuccess)
            return fail(NGLOD_ERR_HIP, "radix sort size query failed");
        tmp = t > tmp ? t : tmp;
        if (L->together) break;
    }
    L->sort_bytes = tmp;
    L->sort_tmp = take(tmp);
    L->runs = take((size_t)(L->together ? corners : most) * sizeof(uint2));
    L->partial = take((m / kRunPiece + 1) * kC * sizeof(float));
    L->total = off;
    return NGLOD_OK;
}

static BwdArgs bwd_args(const ModelArgs& m, const float* x, int64_t n, int lod, int mask, const float* g, void* saved) {
    SavedLayout S;
    saved_layout(n, lod, &S);
    char* w = (char*)saved;
    BwdArgs a;
    a.m = m;
    a.lod = lod;
    a.din = m.pos_inv ? kC : kC + 3;
    a.off = m.pos_inv ? 0 : 3;
    a.mask = mask;
    a.n = n;
    a.x = x;
    a.g = g;
    a.order = (const uint32_t*)(w + S.order);
    a.rank = (uint32_t*)(w + S.rank);
    a.xs = (float*)(w + S.xs);
    a.bits = (uint4*)(w + S.bits);
    a.E = (float*)(w + S.E);
    a.dg = nullptr;
    return a;
}

// Fewer 64-query tiles than CUs: a level per block, so that the levels'
// latencies run side by side (512 queries: 92 -> 41 us for the features); else
// a block per CU with every level's decoder in LDS.
struct Split {
    int on, held, threads, cus;
    Split(int64_t n, const ModelArgs& m, int lod) {
        cus = device_cu_count();
        on = (n + 63) / 64 < (int64_t)cus ? 1 : 0;
        held = on || m.num_dec == 1 ? 1 : lod + 1;
        threads = on ? 256 : 512;
    }
    dim3 grid(int64_t waves, int lod) const {
        const int64_t want = (waves + threads / 64 - 1) / (threads / 64);
        return dim3((unsigned)(on || want < cus ? want : cus), on ? lod + 1 : 1);
    }
};

// Positions, features and signs of the levels in a.mask, and the predictions
// into `out` unless NULL.
static int launch_features(const BwdArgs& a, float* out, void* sort_ws, hipStream_t s) {
    SortBuffers sb = sort_buffers(sort_ws, a.n);
    const int bits = cell_bits(a.m.res[a.lod]);
    sb.vals[sort_result(bits)] = const_cast<uint32_t*>(a.order);
    hipLaunchKernelGGL(bwd_cell_keys_kernel, dim3((unsigned)((a.n + 255) / 256)), dim3(256), 0, s, a.x, a.n,
                       a.m.res[a.lod], sb.keys[0]);
    launch_sort(sb, a.n, bits, s);
    const Split sp(a.n, a.m, a.lod);
    auto k = a.m.pos_inv ? (out ? train_features_kernel<true, true> : train_features_kernel<true, false>)
                         : (out ? train_features_kernel<false, true> : train_features_kernel<false, false>);
    hipLaunchKernelGGL(k, sp.grid((a.n + 63) / 64, a.lod), dim3(sp.threads), sp.held * sizeof(Fp32Lds), s, a, sp.on, out);
    return check_launch("train_features_kernel");
}

static bool bwd_sizes_ok(const nglod_model_t* model, int64_t n, int32_t lod) {
    return model && n >= 0 && lod >= 0 && lod < model->num_lods && lod < NGLOD_MAX_LODS;
}

static size_t bwd_workspace(const nglod_model_t* model, int64_t n, int32_t lod, bool saved) {
    if (!bwd_sizes_ok(model, n, lod)) return 0;
    BwdLayout L;
    return bwd_layout(n, lod, model->pos_invariant ? kC : kC + 3, model->res, saved, &L) ? 0 : L.total;
}

constexpr int64_t kMaxQueries = (int64_t)1 << 28;

// The backward; saved NULL: the features are computed here.
static int backward(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, const float* grad_out,
                    int32_t level_mask, const nglod_model_grads_t* grads, void* saved, size_t saved_bytes,
                    void* workspace, size_t workspace_bytes, void* stream) {
    ModelArgs m;
    int rc = make_model_args(model, lod, NGLOD_FP32, &m);
    if (rc) return rc;
    if (n < 0) return fail(NGLOD_ERR_ARG, "n < 0");
    if (n > kMaxQueries) return fail(NGLOD_ERR_ARG, "n too large for 32-bit sort values");
    if (!grads) return fail(NGLOD_ERR_ARG, "grads is NULL");
    const int din = m.pos_inv ? kC : kC + 3;
    hipStream_t s = (hipStream_t)stream;
    level_mask &= (1 << (lod + 1)) - 1;
    const bool work = n > 0 && level_mask != 0;
    // zero every gradient this call owns (the decoders' are all written where there is work)
    FillList fl;
    int fills = 0;
    int64_t largest = 0;
    auto zero = [&](float* p, int64_t cnt) {
        fl.p[fills] = p;
        fl.n[fills++] = cnt;
        largest = cnt > largest ? cnt : largest;
    };
    for (int l = 0; l <= lod; ++l) {
        if (!grads->grid[l] || !aligned16(grads->grid[l])) return fail(NGLOD_ERR_ARG, "grid grad NULL or misaligned");
        zero(grads->grid[l], (int64_t)corners_of(m.res[l]) * kC);
    }
    for (int d = 0; d < m.num_dec; ++d) {
        if (!grads->w0[d] || !grads->b0[d] || !grads->w1[d] || !grads->b1[d])
            return fail(NGLOD_ERR_ARG, "decoder grad NULL");
        if (work) continue;
        zero(grads->w0[d], (int64_t)kH * din);
        zero(grads->b0[d], kH);
        zero(grads->w1[d], kH);
        zero(grads->b1[d], 1);
    }
    auto fill = [&]() {
        const int64_t blocks = (largest + 1023) / 1024;
        hipLaunchKernelGGL(bwd_fill_kernel, dim3((unsigned)(blocks < 4096 ? blocks : 4096), fills), dim3(256), 0, s, fl);
        return check_launch("bwd_fill_kernel");
    };
    if (!work) return fill();
    if (!x || !grad_out) return fail(NGLOD_ERR_ARG, "NULL pointer");
    BwdLayout L;
    rc = bwd_layout(n, lod, din, model->res, saved != nullptr, &L);
    if (rc) return rc;
    if (!workspace || workspace_bytes < L.total || !aligned16(workspace))
        return fail(NGLOD_ERR_WORKSPACE, "workspace too small or misaligned");
    SavedLayout S;
    saved_layout(n, lod, &S);
    if (saved && (saved_bytes < S.total || !aligned16(saved)))
        return fail(NGLOD_ERR_WORKSPACE, "saved features too small or misaligned");
    char* ws = (char*)workspace;
    uint2* runs = (uint2*)(ws + L.runs);
    if (L.together) {
        uint64_t corners = 0;
        for (int l = 0; l <= lod; ++l) corners += corners_of(m.res[l]);
        zero((float*)runs, (int64_t)corners * 2);
    }
    rc = fill();
    if (rc) return rc;
    const unsigned qblocks = (unsigned)((n + 255) / 256);
    BwdArgs a = bwd_args(m, x, n, lod, level_mask, grad_out, saved ? saved : ws + L.saved);
    a.dg = (float*)(ws + L.dg);
    float* part = (float*)(ws + L.part);
    if (!saved) {
        rc = launch_features(a, nullptr, ws + L.order_ws, s);
        if (rc) return rc;
    }
    const Split sp(n, m, lod);
    const int cus = sp.cus;
    hipLaunchKernelGGL(bwd_ds_kernel, sp.grid((n + 31) / 32, lod), dim3(sp.threads), sp.held * sizeof(BwdLds), s, a,
                       sp.on);
    rc = check_launch("bwd_ds_kernel");
    if (rc) return rc;
    if (sp.on && lod > 0)
        hipLaunchKernelGGL(bwd_suffix_kernel, dim3((unsigned)((n * (kC / 4) + 255) / 256)), dim3(256), 0, s, a);
    // decoder gradients
    auto pk = m.pos_inv ? bwd_decoder_partial_kernel<true> : bwd_decoder_partial_kernel<false>;
    hipLaunchKernelGGL(pk, dim3((unsigned)L.nchunks, (unsigned)(lod + 1)), dim3(256), 0, s, a, part, L.nchunks);
    rc = check_launch("bwd_decoder_partial_kernel");
    if (rc) return rc;
    const int outs = kH * din + 2 * kH + 1;
    float* gpart = (float*)(ws + L.gpart);
    hipLaunchKernelGGL(bwd_decoder_group_kernel, dim3((outs + 255) / 256, (unsigned)L.ngroups, (unsigned)(lod + 1)),
                       dim3(256), 0, s, a, part, L.nchunks, gpart, L.ngroups);
    hipLaunchKernelGGL(bwd_decoder_final_kernel, dim3((outs + 255) / 256, m.num_dec), dim3(256), 0, s, a, gpart,
                       L.ngroups, *grads);
    rc = check_launch("bwd_decoder_final_kernel");
    if (rc) return rc;
    // grid gradients: levels that receive gradient from some level i >= j
    uint32_t* kin = (uint32_t*)(ws + L.keys_in);
    uint32_t* kout = (uint32_t*)(ws + L.keys_out);
    uint32_t* vin = (uint32_t*)(ws + L.vals_in);
    uint32_t* vout = (uint32_t*)(ws + L.vals_out);
    float* partial = (float*)(ws + L.partial);
    auto corner_gradients = [&](int j0, int j1) {
        CornerLevels C;
        memset(&C, 0, sizeof(C));
        for (int j = j0; j <= j1; ++j) {
            if ((level_mask >> j) == 0) continue;  // no level >= j carries gradient
            const int i = C.count++;
            C.level[i] = j;
            C.res[i] = m.res[j];
            C.base[i + 1] = C.base[i] + (uint32_t)corners_of(m.res[j]);
            C.grad[i] = grads->grid[j];
            // levels averaging 8 or more pieces per corner: a block per run
            if (n * 8 >= (int64_t)corners_of(m.res[j]) * 8 * kRunPiece) C.strided |= 1u << i;
        }
        if (C.count == 0) return (int)NGLOD_OK;
        const uint32_t corners = C.base[C.count];
        const uint32_t mm = (uint32_t)(n * 8 * C.count);
        if (!L.together)
            hipLaunchKernelGGL(fill_f32_kernel, dim3((2 * corners + 255) / 256), dim3(256), 0, s, (float*)runs,
                               (int64_t)corners * 2);
        hipLaunchKernelGGL(bwd_corner_keys_kernel, dim3(qblocks, C.count), dim3(256), 0, s, a, C, kin, vin);
        const int bits = bits_for(corners);
        size_t tmp = 0;
        if (rocprim::radix_sort_pairs((void*)nullptr, tmp, kin, kout, vin, vout, (size_t)mm, 0, bits, s) != hipSuccess ||
            tmp > L.sort_bytes)
            return fail(NGLOD_ERR_HIP, "radix sort temp size");
        tmp = L.sort_bytes;
        if (rocprim::radix_sort_pairs((void*)(ws + L.sort_tmp), tmp, kin, kout, vin, vout, (size_t)mm, 0, bits, s) !=
            hipSuccess)
            return fail(NGLOD_ERR_HIP, "radix sort failed");
        hipLaunchKernelGGL(bwd_runs_kernel, dim3((mm + 255) / 256), dim3(256), 0, s, kout, mm, runs);
        uint32_t size = kWindow;
        while (size > 256 && mm / size < 4u * (uint32_t)cus) size /= 2;
        const uint32_t windows = (mm + size - 1) / size;
        hipLaunchKernelGGL(bwd_pieces_kernel, dim3((windows + 7) / 8 * 8), dim3(256), 0, s, a, C, kout, vout, mm, size,
                           runs, partial);
        if (C.strided != (1u << C.count) - 1u) {
            const uint64_t blocks = ((uint64_t)corners * kC + 255) / 256;
            hipLaunchKernelGGL(bwd_run_final_kernel, dim3((unsigned)(blocks < kFinalBlocks ? blocks : kFinalBlocks)),
                               dim3(256), 0, s, C, runs, partial);
        }
        if (C.strided) {
            uint32_t blocks = 0;
            for (int i = 0; i < C.count; ++i) blocks += (C.strided >> i) & 1u ? C.base[i + 1] - C.base[i] : 0u;
            hipLaunchKernelGGL(bwd_run_strided_kernel, dim3(blocks), dim3(kRunGroups * kC), 0, s, C, runs, partial);
        }
        return check_launch("bwd_pieces_kernel");
    };
    if (L.together) return corner_gradients(0, lod);
    for (int j = 0; j <= lod; ++j) {
        rc = corner_gradients(j, j);
        if (rc) return rc;
    }
    return NGLOD_OK;
}

}  // namespace nglod

using namespace nglod;

extern "C" {

size_t nglod_sdf_bwd_workspace_size(const nglod_model_t* model, int64_t n, int32_t lod) {
    return bwd_workspace(model, n, lod, false);
}

size_t nglod_sdf_bwd_saved_workspace_size(const nglod_model_t* model, int64_t n, int32_t lod) {
    return bwd_workspace(model, n, lod, true);
}

size_t nglod_sdf_fwd_save_bytes(const nglod_model_t* model, int64_t n, int32_t lod) {
    if (!bwd_sizes_ok(model, n, lod)) return 0;
    SavedLayout S;
    saved_layout(n, lod, &S);
    return S.total;
}

size_t nglod_sdf_fwd_save_workspace_size(int64_t n) { return n > 0 ? sort_workspace_bytes(n) : 0; }

int nglod_sdf_fwd_save(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, float* out, void* saved,
                       size_t saved_bytes, void* workspace, size_t workspace_bytes, void* stream) {
    ModelArgs m;
    int rc = make_model_args(model, lod, NGLOD_FP32, &m);
    if (rc) return rc;
    if (n < 0 || n > kMaxQueries) return fail(NGLOD_ERR_ARG, "n out of range");
    if (n == 0) return NGLOD_OK;
    if (!x || !out || !saved) return fail(NGLOD_ERR_ARG, "NULL pointer");
    if (saved_bytes < nglod_sdf_fwd_save_bytes(model, n, lod) || !aligned16(saved))
        return fail(NGLOD_ERR_WORKSPACE, "saved features too small or misaligned");
    if (!workspace || workspace_bytes < sort_workspace_bytes(n) || !aligned16(workspace))
        return fail(NGLOD_ERR_WORKSPACE, "workspace too small or misaligned");
    const BwdArgs a = bwd_args(m, x, n, lod, (1 << (lod + 1)) - 1, nullptr, saved);
    return launch_features(a, out, workspace, (hipStream_t)stream);
}

int nglod_sdf_bwd(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, const float* grad_out,
                  int32_t level_mask, const nglod_model_grads_t* grads, void* workspace, size_t workspace_bytes,
                  void* stream) {
    return backward(model, x, n, lod, grad_out, level_mask, grads, nullptr, 0, workspace, workspace_bytes, stream);
}

int nglod_sdf_bwd_saved(const nglod_model_t* model, const float* x, int64_t n, int32_t lod, const float* grad_out,
                        int32_t level_mask, const nglod_model_grads_t* grads, void* saved, size_t saved_bytes,
                        void* workspace, size_t workspace_bytes, void* stream) {
    if (n > 0 && !saved) return fail(NGLOD_ERR_ARG, "NULL pointer");
    return backward(model, x, n, lod, grad_out, level_mask, grads, saved, saved_bytes, workspace, workspace_bytes,
                    stream);
}

}  // extern "C"
