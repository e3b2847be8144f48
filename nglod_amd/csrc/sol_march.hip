// The sparse march by groups of 32 rays: launch_trace_sparse_group
// (nglod_trace_sparse; SDF::sphereTrace + getNormal, sol-renderer/SDF.cu:218-472).
// A file of its own: it is built with MFMA results in ordinary VGPRs.
#include "api_common.hpp"
#include "group_eval.hpp"
#include "sol_common.hpp"

namespace nglod {

enum : int { SG_IDLE = -1, SG_EVAL = 0, SG_N0 = 1, SG_WALK = 8 };

struct alignas(16) SolGroupLds {
    float w[kSolGroupLevels][kGroup][8];        // corner weights, corner = 4 z + 2 y + x
    uint32_t vert[kSolGroupLevels][kGroup][8];  // the corners' rows, in float4s
    float x[kGroup][3], iv[kGroup][3];          // for the voxel walk
    float o[kGroup][3], d[kGroup][3];
    int32_t nb[kGroup], ne[kGroup];
    int2 near[kGroup][16];    // the first voxels of a ray's list: coordinates
    int32_t near_id[kGroup][16];  // and ids
    int32_t queue[64];  // claimed rays that have voxels, not yet started
    int32_t queued, drained;
    int32_t found[kGroup];  // the voxel the walk ended in; -1: none
    float ahead[kGroup];    // and the distance to it
    GroupDecoder dec;
};

// A ray's state: lanes n and n + 32 of every wave hold ray n of the group.
struct SolGroupRay {
    int32_t ray;
    int phase, it;
    bool hitf, writes;
    int32_t pidx;
    float x0, x1, x2, t, dprev;
    float qx, qy, qz, fplus, g0, g1, g2;

    __device__ __forceinline__ void retire(const SolArgs& a, float n0, float n1, float n2) {
        if (writes) {
            const int64_t r = ray;
            a.x[3 * r] = x0;
            a.x[3 * r + 1] = x1;
            a.x[3 * r + 2] = x2;
            a.t[r] = t;
            a.hit[r] = hitf ? 1 : 0;
            a.normal[3 * r] = n0;
            a.normal[3 * r + 1] = n1;
            a.normal[3 * r + 2] = n2;
            if (a.iters) a.iters[r] = it;
        }
        phase = SG_IDLE;
        ray = -1;
    }

    __device__ __forceinline__ void finish(const SolArgs& a) {
        if (hitf) {
            phase = SG_N0;
            qx = x0 + 0.001f;
            qy = x1 + 0.0f;
            qz = x2 + 0.0f;
        } else {
            retire(a, 1.0f, 1.0f, 1.0f);
        }
    }

    __device__ __forceinline__ void move(float to, const SolGroupLds* s, uint32_t n) {
        t = to;
        x0 = __builtin_fmaf(s->d[n][0], t, s->o[n][0]);
        x1 = __builtin_fmaf(s->d[n][1], t, s->o[n][1]);
        x2 = __builtin_fmaf(s->d[n][2], t, s->o[n][2]);
    }

    __device__ __forceinline__ void start(const SolArgs& a, int64_t r, SolGroupLds* s, uint32_t n) {
        ray = (int32_t)r;
        x0 = a.o[3 * r];
        x1 = a.o[3 * r + 1];
        x2 = a.o[3 * r + 2];
        t = 0.0f;
        dprev = 0.0f;
        it = 0;
        hitf = false;
        pidx = -1;
        phase = SG_WALK;
        if (writes) {
            const float dx = a.d[3 * r], dy = a.d[3 * r + 1], dz = a.d[3 * r + 2];
            s->o[n][0] = x0;
            s->o[n][1] = x1;
            s->o[n][2] = x2;
            s->d[n][0] = dx;
            s->d[n][1] = dy;
            s->d[n][2] = dz;
            s->iv[n][0] = 1.0f / dx;
            s->iv[n][1] = 1.0f / dy;
            s->iv[n][2] = 1.0f / dz;
            s->nb[n] = a.offs[r];
            s->ne[n] = a.offs[r + 1];
        }
    }

    // The walk's result; a ray without a voxel left is a miss.
    __device__ __forceinline__ void walked(const SolArgs& a, const SolGroupLds* s, uint32_t n) {
        const int32_t voxel = s->found[n];
        if (voxel >= 0) {
            const float dist = s->ahead[n];
            pidx = voxel;
            if (dist > 0.0f) move(t + dist, s, n);
            if (it < 50) {
                phase = SG_EVAL;
                qx = x0;
                qy = x1;
                qz = x2;
                return;
            }
        } else {
            move(100.0f, s, n);
        }
        finish(a);
    }

    __device__ __forceinline__ void consume(const SolArgs& a, float d, const SolGroupLds* s, uint32_t n) {
        if (phase == SG_EVAL) {
            ++it;
            hitf = ((double)fabsf(d) < 0.0003) || (((double)fabsf(d + dprev) * 0.5) < 0.0015);
            move(t + d, s, n);
            dprev = d;
            if (((double)t < 5.0) && !hitf)
                phase = SG_WALK;
            else
                finish(a);
            return;
        }
        const int k = phase - SG_N0;  // 0..5
        const int axis = k >> 1;
        if ((k & 1) == 0) {
            fplus = d;
            qx = axis == 0 ? x0 - 0.001f : x0 - 0.0f;
            qy = axis == 1 ? x1 - 0.001f : x1 - 0.0f;
            qz = axis == 2 ? x2 - 0.001f : x2 - 0.0f;
            ++phase;
            return;
        }
        const float g = fplus - d;
        g0 = axis == 0 ? g : g0;
        g1 = axis == 1 ? g : g1;
        g2 = axis == 2 ? g : g2;
        if (axis == 2) {
            const float len = sqrtf(g0 * g0 + g1 * g1 + g2 * g2);
            retire(a, g0 / len, g1 / len, g2 / len);
        } else {
            const int na = axis + 1;
            qx = na == 0 ? x0 + 0.001f : x0 + 0.0f;
            qy = na == 1 ? x1 + 0.001f : x1 + 0.0f;
            qz = na == 2 ? x2 + 0.001f : x2 + 0.0f;
            ++phase;
        }
    }
};

// The first voxel of each walking ray's nugget list that contains its point or
// lies ahead of it: eight threads per ray test eight voxels at a time, the first
// sixteen (cached: the ray whose list begins at this index) from LDS; each thread
// reads back what it put there itself.
__device__ __forceinline__ void group_walk(const SolArgs& a, SolGroupLds* s, uint32_t walking, int32_t& cached) {
    const uint32_t ray = threadIdx.x >> 3, q = threadIdx.x & 7u, lane = lane_id();
    bool look = (walking >> ray) & 1u;
    const int32_t nb = look ? s->nb[ray] : 0, ne = look ? s->ne[ray] : 0;
    auto voxel = [&](int32_t i, int2& p) {
        const int32_t pl = a.nug[2 * (int64_t)i + 1];
        p = *reinterpret_cast<const int2*>(a.points + 4 * (a.psum_target + pl));
        return pl;
    };
    if (look && nb != cached) {
        cached = nb;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            if (nb + 8 * j + (int32_t)q < ne) {
                int2 p;
                s->near_id[ray][8 * j + q] = voxel(nb + 8 * j + (int32_t)q, p);
                s->near[ray][8 * j + q] = p;
            }
        }
    }
    const float x0 = s->x[ray][0], x1 = s->x[ray][1], x2 = s->x[ray][2];
    const float dx = s->d[ray][0], dy = s->d[ray][1], dz = s->d[ray][2];
    const float ivx = s->iv[ray][0], ivy = s->iv[ray][1], ivz = s->iv[ray][2];
    const float sgx = __builtin_signbit(dx) ? 1.0f : -1.0f, sgy = __builtin_signbit(dy) ? 1.0f : -1.0f,
                sgz = __builtin_signbit(dz) ? 1.0f : -1.0f;
    int32_t i = nb;
    while (__ballot(look) != 0) {
        float dd = 0.0f;
        int32_t pl = -1;
        if (look && i + (int32_t)q < ne) {
            int2 p;
            const int32_t j = i - nb + (int32_t)q;
            if (j < 16) {
                p = s->near[ray][j];
                pl = s->near_id[ray][j];
            } else {
                pl = voxel(i + (int32_t)q, p);
            }
            const float cx = __builtin_fmaf(a.r, __builtin_fmaf(2.0f, (float)(int16_t)(p.x & 0xffff), 1.0f), -1.0f);
            const float cy = __builtin_fmaf(a.r, __builtin_fmaf(2.0f, (float)(int16_t)(p.x >> 16), 1.0f), -1.0f);
            const float cz = __builtin_fmaf(a.r, __builtin_fmaf(2.0f, (float)(int16_t)(p.y & 0xffff), 1.0f), -1.0f);
            dd = sol_ray_aabb(x0, x1, x2, dx, dy, dz, ivx, ivy, ivz, sgx, sgy, sgz, cx, cy, cz, a.r);
        }
        const uint32_t any = (uint32_t)(__ballot(dd != 0.0f) >> (lane & 56u)) & 0xffu;
        if (look) {
            if (any != 0) {
                if (q == (uint32_t)__ffs(any) - 1u) {
                    s->found[ray] = pl;
                    s->ahead[ray] = dd;
                }
                look = false;
            } else {
                i += 8;
                if (i >= ne) {
                    if (q == 0) s->found[ray] = -1;
                    look = false;
                }
            }
        }
    }
}

// Wave 0 claims rays until some have voxels (or none are left): those are queued,
// the others are written out as misses at once, a lane each.
__device__ __forceinline__ void group_claim(const SolArgs& a, SolGroupLds* s, RayFeed& feed, uint32_t lane) {
    uint32_t got = 0;
    while (got == 0 && !feed.drained) {
        if (!feed.claim<true>(a.queue, lane, 0, 64)) continue;
        const int64_t r = feed.cb + lane;
        const bool have = r < feed.ce;
        feed.cb = feed.ce;
        const bool march = have && a.offs[r + 1] > a.offs[r];
        const uint64_t m = __ballot(march);
        if (march) s->queue[mask_rank(m)] = (int32_t)r;
        got = (uint32_t)__popcll(m);
        if (have && !march) {
            SolGroupRay miss = {};
            miss.ray = (int32_t)r;
            miss.writes = true;
            miss.hitf = false;
            miss.it = 0;
            miss.t = 0.0f;
            miss.x0 = a.o[3 * r];
            miss.x1 = a.o[3 * r + 1];
            miss.x2 = a.o[3 * r + 2];
            miss.retire(a, 1.0f, 1.0f, 1.0f);
        }
    }
    if (lane == 0) {
        s->queued = (int32_t)got;
        s->drained = feed.drained ? 1 : 0;
    }
}

// A block of four waves marches 32 rays (group_eval.hpp): the voxel walk and the
// corner tables take eight threads per ray, the decoder a quarter of the hidden
// units per wave.  The rows of a ray's corners are looked up only when its voxel
// changes, those of the coarser levels only when its parent does (most
// evaluations, the six normal taps among them, stay in theirs), and a corner's
// coordinates come from its voxel's.  Bound: the vector memory path (TA busy 56%, TD
// 68% of the cycles) and the vector ALU (47%), in trips of dependent loads and
// barriers (waves wait for memory 28% of theirs); four blocks a CU by registers.
// 1280x720, LOD 4, 5.4 M evaluations: one ray per lane 2.71 ms; by groups, corners
// and voxels looked up in every trip 2.60; this 1.84.
template <bool POSINV>
__global__ __launch_bounds__(kGroupThreads, 4) void trace_sparse_group_kernel(SolArgs a) {
    __shared__ SolGroupLds lds;
    const GroupWeights gw = stage_group_decoder(a.w0, a.din, a.b0, a.w1, &lds.dec);
    const float b1 = a.b1[0];
    const uint32_t lane = lane_id(), n = lane & 31u;
    const uint32_t mine = threadIdx.x >> 3, corner = threadIdx.x & 7u;  // of the gather
    const bool first = threadIdx.x < 64;
    RayFeed feed;
    feed.init(a.n, kQueueStride);
    SolGroupRay s = {};
    s.ray = -1;
    s.phase = SG_IDLE;
    s.writes = threadIdx.x < kGroup;
    int32_t cached = -1;  // group_walk
    int32_t voxel = -1;   // the voxel of ray `mine` whose corner rows vert holds,
    int2 at = make_int2(0, 0);  // its coordinates,
    int32_t parent = -1;  // and its parent
    int32_t next = 0, queued = 0;  // of lds.queue
    bool drained = false;
    uint32_t nevals = 0;
    for (;;) {
        // One refill and one walk a trip (a lane whose ray ends in the walk waits for
        // the next trip's).  Block-uniform: every wave sees the same phases.
        const uint32_t need = (uint32_t)__ballot(s.phase == SG_IDLE);
        if (need != 0 && !(drained && next >= queued)) {
            const bool claims = next >= queued;
            if (claims && first) group_claim(a, &lds, feed, lane);
            // Wave 0 starts a ray by writing its origin, direction and list; until this
            // barrier another wave may still be moving the lane's last ray by the old ones
            // (consume in the last trip, walked in a trip that ended without an evaluation).
            __syncthreads();
            if (claims) {
                next = 0;
                queued = lds.queued;
                drained = lds.drained != 0;
            }
            const int32_t i = next + __popc(need & ((1u << n) - 1u)), end = next + __popc(need);
            next = end < queued ? end : queued;
            if (s.phase == SG_IDLE && i < queued) s.start(a, lds.queue[i], &lds, n);
        }
        const uint32_t walking = (uint32_t)__ballot(s.phase == SG_WALK);
        if (walking != 0) {
            if (s.writes) {
                lds.x[n][0] = s.x0;
                lds.x[n][1] = s.x1;
                lds.x[n][2] = s.x2;
            }
            __syncthreads();
            group_walk(a, &lds, walking, cached);
            __syncthreads();
            if (s.phase == SG_WALK) s.walked(a, &lds, n);
        }
        const bool busy = s.phase != SG_IDLE;
        const uint32_t act = (uint32_t)__ballot(busy);
        if (act == 0) {
            if (drained && next >= queued) break;
            continue;
        }
        // the gather's threads take over their ray's point and voxel
        const int src = (int)mine;  // lane `mine` of this wave holds ray `mine`
        const float px = __shfl(s.qx, src), py = __shfl(s.qy, src), pz = __shfl(s.qz, src);
        const int32_t v = __shfl(s.pidx, src);
        const bool on = (act >> mine) & 1u;
        if (on && v != voxel) {
            voxel = v;
            const int64_t leaf = (int64_t)v + a.psum_target;
            at = *reinterpret_cast<const int2*>(a.points + 4 * leaf);
            const uint32_t slot = ((corner & 1u) << 2) | (corner & 2u) | (corner >> 2);  // tv's order: z + 2 y + 4 x
            lds.vert[0][mine][corner] = a.tv[8 * leaf + slot] * (kC / 4);
            // the coarser levels' rows change with the parent only
            const int32_t up = a.lod > 0 ? a.parent[leaf] : -1;
            if (up != parent) {
                parent = up;
                int32_t c = up;
                for (int j = 1; j <= a.lod; ++j) {
                    lds.vert[j][mine][corner] = a.tv[8 * (int64_t)c + slot] * (kC / 4);
                    if (j < a.lod) c = a.parent[c];
                }
            }
        }
        if (on) {
            // this thread's corner is the far one of corner 7 - corner, whose weight it computes
            const float nx = __builtin_fmaf(px, 0.5f, 0.5f), ny = __builtin_fmaf(py, 0.5f, 0.5f),
                        nz = __builtin_fmaf(pz, 0.5f, 0.5f);
            const uint32_t k = 7u - corner;
            const int vx = (int16_t)(at.x & 0xffff), vy = (int16_t)(at.x >> 16), vz = (int16_t)(at.y & 0xffff);
            for (int j = 0; j <= a.lod; ++j) {
                const float res = (float)(4u << (a.lod - j));
                const float iz = nx * res, iy = ny * res, ix = nz * res;
                const float cx = (float)((vx >> j) + (int)(corner & 1u)), cy = (float)((vy >> j) + (int)((corner >> 1) & 1u)),
                            cz = (float)((vz >> j) + (int)(corner >> 2));
                const float fa = k & 4u ? ix - cz : cz - ix, fb = k & 2u ? iy - cy : cy - iy,
                            fc = k & 1u ? iz - cx : cx - iz;
                lds.w[j][mine][k] = (fa * fb) * fc;
            }
        }
        // a ray's eight threads are of one wave: its tables need no block barrier
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        float4 f = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const float4* cf4 = reinterpret_cast<const float4*>(a.cf) + corner;
        if (on) {
#pragma unroll 1
            for (int j = 0; j <= a.lod; ++j) {
                const uint4* vp = reinterpret_cast<const uint4*>(lds.vert[j][mine]);
                const uint4 va = vp[0], vb = vp[1];
                const uint32_t row[8] = {va.x, va.y, va.z, va.w, vb.x, vb.y, vb.z, vb.w};
                float4 g[8];
#pragma unroll
                for (int k = 0; k < 8; ++k) g[k] = cf4[row[k]];
                group_corners(g, reinterpret_cast<const float4*>(lds.w[j][mine]), f);
            }
        }
        store_features(&lds.dec, mine, corner, f);
        const float d = group_decode<POSINV>(&lds.dec, gw, b1, s.qx, s.qy, s.qz);
        if (busy) {
            ++nevals;
            s.consume(a, d, &lds, n);
        }
    }
    if (a.evals && first) {
        unsigned long long tot = lane < kGroup ? nevals : 0;
        for (int off = 32; off > 0; off >>= 1) tot += __shfl_xor(tot, off);
        if (lane == 0 && tot) atomicAdd(a.evals, tot);
    }
}

int launch_trace_sparse_group(const SolArgs& a, hipStream_t s) {
    const int64_t blocks = (a.n + kGroup - 1) / kGroup, cap = (int64_t)device_cu_count() * 4;
    const dim3 grid((unsigned)(blocks < cap ? blocks : cap));
    if (a.din == kC)
        hipLaunchKernelGGL(trace_sparse_group_kernel<true>, grid, dim3(kGroupThreads), 0, s, a);
    else
        hipLaunchKernelGGL(trace_sparse_group_kernel<false>, grid, dim3(kGroupThreads), 0, s, a);
    return check_launch("trace_sparse_group_kernel");
}

}  // namespace nglod
