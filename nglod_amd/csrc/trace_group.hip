// The FP32 dense sphere trace, launch_trace_fp32 (nglod_trace_dense), and the FP32
// query in input order, launch_sdf_group_fp32 (nglod_sdf_fwd).  A file of its own:
// it is built with MFMA results in ordinary VGPRs, which the ReLU reads.
#include "api_common.hpp"
#include "group_eval.hpp"
#include "trace_common.hpp"

namespace nglod {

// A block of four waves marches 32 rays, one evaluation of all of them a trip
// (group_sdf).  Every wave keeps the state of all 32 rays (lanes n and n + 32: ray
// n) and steps it by the same results, so the state is never exchanged; the first
// 32 threads write the rays out.  Persistent: a block claims 32 consecutive rays
// at a time and hands them to its idle lanes in order.
//
// Bound: small frames by the length of the longest ray times a trip's latency
// (about 2 us: the dependent loads, three barriers, 16 MFMAs in a row), large ones
// by the corner rows through the vector L1 (TA busy 59%, TD 67% of the cycles at
// 1280x720), the FP32 units (vector ALU 47%, matrix cores 27%: not beside each other on a
// SIMD) and by the four blocks a CU that the registers
// allow: three measured a quarter slower, also with a second level's rows in
// flight.  A whole frame, 5 LODs, against one ray per lane and 64 rays a wave:
// 64x48 1339 -> 365 us, 128x96 1367 -> 430, 320x180 1445 -> 677, 1280x720 4091 ->
// 3430.
//
// FEW: trips of at most eight rays read four levels at once.  TAIL: once no rays are
// left to claim, trips of at most 16 rays run in a loop of their own, where
// group_decode_few takes half the matrix work (0.2 us) and at most eight rays read
// four levels at once, too.  A frame ends with rays of up to 128 steps, a few per
// block, whose trips are pure latency.  A whole frame at LOD 1 / 2 / 4, us: 64x48
// without the loop 275 / 322 / 325 (FEW; 348 without), with it 261 / 279 / 290; 128x96 302 /
// 385 / 395, 283 / 322 / 346; 320x180 451 / 516 / 593, 415 / 450 / 535; 640x360 800 / 975 / 1165,
// 816 / 915 / 1135; 960x540 1390 / 1705 / 2096 (2182 without FEW), 1435 / 1685 / 2104; 1280x720
// 2230 / 2704 / 3382, 2346 / 2761 / 3427: the second loop costs the first one up to 5%,
// hence the line at kTailRays.  Above it FEW from LOD 3 on: below, its instructions
// cost 2-5% and there are too few levels to gain by it.
constexpr int64_t kTailRays = 1 << 18;

template <bool POSINV, bool TAIL, bool FEW>
__global__ __launch_bounds__(kGroupThreads, 4) void trace_dense_fp32_kernel(TraceArgs a) {
    __shared__ GroupLds<true> lds;
    __shared__ int64_t claimed[2];
    __shared__ int claims_left;
    GroupWeights gw = stage_group(a.m, a.dec, &lds);
    const float b1 = a.m.b1[a.dec][0];
    const uint32_t lane = lane_id();
    const bool first = threadIdx.x < 64;
    RayFeed feed;
    feed.init(a.nrays, a.queue_stride);
    RayState s;
    s.ray = -1;
    s.phase = PH_IDLE;
    s.writes = threadIdx.x < kGroup;
    uint32_t nevals = 0;
    for (;;) {
        // refill: block-uniform, every wave sees the same idle lanes
        for (;;) {
            const uint32_t need = (uint32_t)__ballot(s.phase == PH_IDLE);
            if (need == 0 || feed.empty()) break;
            if (feed.cb >= feed.ce) {
                if (first) {
                    feed.claim<true>(a.queue, lane, 0, kGroup);
                    if (lane == 0) {
                        claimed[0] = feed.cb;
                        claimed[1] = feed.ce;
                        claims_left = feed.drained ? 0 : 1;
                    }
                }
                __syncthreads();
                feed.cb = claimed[0];
                feed.ce = claimed[1];
                feed.drained = claims_left == 0;
                __syncthreads();
                continue;
            }
            const int64_t id = feed.cb + __popc(need & ((1u << (lane & 31u)) - 1u));
            const int64_t end = feed.cb + __popc(need);
            if (s.phase == PH_IDLE && id < feed.ce) s.start(a, id);
            feed.cb = end < feed.ce ? end : feed.ce;
        }
        const bool busy = s.phase != PH_IDLE;
        const uint32_t act = (uint32_t)__ballot(busy);
        if (TAIL ? feed.empty() && __popc(act) <= kFewQueries : act == 0) break;
        const float d = group_sdf<POSINV, FEW, false>(a.m, a.lod, &lds, gw, b1, act, busy ? s.qx : 0.0f, busy ? s.qy : 0.0f,
                                                      busy ? s.qz : 0.0f);
        if (busy) {
            ++nevals;
            s.consume(a, d);
        }
    }
    if (TAIL) few_weights(gw);
    while (TAIL) {
        const bool busy = s.phase != PH_IDLE;
        const uint32_t act = (uint32_t)__ballot(busy);
        if (act == 0) break;
        const float d = group_sdf<POSINV, true, true>(a.m, a.lod, &lds, gw, b1, act, busy ? s.qx : 0.0f, busy ? s.qy : 0.0f,
                                                      busy ? s.qz : 0.0f);
        if (busy) {
            ++nevals;
            s.consume(a, d);
        }
    }
    if (a.evals && first) {
        unsigned long long tot = lane < kGroup ? nevals : 0;
        for (int off = 32; off > 0; off >>= 1) tot += __shfl_xor(tot, off);
        if (lane == 0) atomicAdd(a.evals, tot);
    }
}

template <bool POSINV>
static void launch_dense(const TraceArgs& a, int64_t n, dim3 grid, hipStream_t s) {
    if (n <= kTailRays)
        hipLaunchKernelGGL((trace_dense_fp32_kernel<POSINV, true, false>), grid, dim3(kGroupThreads), 0, s, a);
    else if (a.lod >= 3)
        hipLaunchKernelGGL((trace_dense_fp32_kernel<POSINV, false, true>), grid, dim3(kGroupThreads), 0, s, a);
    else
        hipLaunchKernelGGL((trace_dense_fp32_kernel<POSINV, false, false>), grid, dim3(kGroupThreads), 0, s, a);
}

int launch_trace_fp32(const TraceArgs& a, int64_t n, hipStream_t s) {
    const int64_t blocks = (n + kGroup - 1) / kGroup, cap = (int64_t)device_cu_count() * 4;
    const dim3 grid((unsigned)(blocks < cap ? blocks : cap));
    if (a.m.pos_inv)
        launch_dense<true>(a, n, grid, s);
    else
        launch_dense<false>(a, n, grid, s);
    return check_launch("trace_dense_fp32_kernel");
}

// Batch query in input order, 32 points a block and trip.  A thousand points are
// one short trip each on 32 CUs; large batches of scattered points are bound by
// the corner rows through L1 and L2 (six blocks a CU).  Against a point per lane
// and 64 a wave, LOD 4: 1000 points 44 -> 6.5 us, 2^16 49 -> 30, 2^18 164 -> 81, 2^22
// 2460 -> 1060; LOD 0: 16 -> 5.5, 17 -> 17, 48 -> 36.
template <bool POSINV>
__global__ __launch_bounds__(kGroupThreads, 6) void sdf_group_fp32_kernel(ModelArgs m, int lod, int dec,
                                                                       const float* __restrict__ x, int64_t n,
                                                                       float* __restrict__ out) {
    __shared__ GroupLds<false> lds;
    const GroupWeights gw = stage_group(m, dec, &lds);
    const float b1 = m.b1[dec][0];
    const int64_t stride = (int64_t)gridDim.x * kGroup;
    for (int64_t first = (int64_t)blockIdx.x * kGroup; first < n; first += stride) {
        const int64_t i = first + (threadIdx.x & 31u), j = i < n ? i : n - 1;
        const float d = group_sdf<POSINV, false, false>(m, lod, &lds, gw, b1, ~0u, x[3 * j], x[3 * j + 1], x[3 * j + 2]);
        if (threadIdx.x < kGroup && i < n) out[i] = d;
    }
}

int launch_sdf_group_fp32(const ModelArgs& m, int lod, int dec, const float* x, int64_t n, float* out, hipStream_t s) {
    const int64_t blocks = (n + kGroup - 1) / kGroup, cap = (int64_t)device_cu_count() * 6;
    const dim3 grid((unsigned)(blocks < cap ? blocks : cap));
    if (m.pos_inv)
        hipLaunchKernelGGL(sdf_group_fp32_kernel<true>, grid, dim3(kGroupThreads), 0, s, m, lod, dec, x, n, out);
    else
        hipLaunchKernelGGL(sdf_group_fp32_kernel<false>, grid, dim3(kGroupThreads), 0, s, m, lod, dec, x, n, out);
    return check_launch("sdf_group_fp32_kernel");
}

}  // namespace nglod
