// Stable radix sort of (key, index) pairs by the low bits of 32-bit keys, the
// indices those of the keys' input order.  It orders query points and
// triangles along a Morton curve (2^22 points: 38 us per digit; 2^18: 13).
//
// Per 8-bit digit three launches: a histogram per tile of kSortTile keys, an
// exclusive scan of every digit's tile counts, and the scatter, which ranks
// the tile's keys with ballots (wave w ranks keys 1024 w .. 1024 w + 1023, 64
// at a time, in order), puts the tile in order in LDS and writes each digit's
// keys as one run.  No memory is cleared and no host value is read, so a
// captured call replays, and no block waits for another.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device_common.hpp"

namespace nglod {

constexpr int kSortBlock = 256, kSortRounds = 16;
constexpr int kSortTile = kSortBlock * kSortRounds;  // 4096
constexpr int kSortDigits = 256;
static_assert(kSortBlock == kSortDigits, "a thread per digit");

static __global__ __launch_bounds__(kSortBlock) void sort_hist_kernel(const uint32_t* __restrict__ keys, uint32_t n,
                                                                      int shift, uint32_t tiles,
                                                                      uint32_t* __restrict__ hist) {
    __shared__ uint32_t cnt[kSortDigits];
    cnt[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * kSortTile;
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const uint64_t i = base + r * kSortBlock + threadIdx.x;
        if (i < n) atomicAdd(&cnt[(keys[i] >> shift) & 255u], 1u);
    }
    __syncthreads();
    hist[(size_t)threadIdx.x * tiles + blockIdx.x] = cnt[threadIdx.x];
}

// Exclusive prefix of one value per thread over the block (256 threads); the
// block's sum in `total`.
static __device__ __forceinline__ uint32_t sort_block_scan(uint32_t v, uint32_t& total) {
    __shared__ uint32_t ws[kSortBlock / 64];
    const uint32_t lane = lane_id(), wave = threadIdx.x >> 6;
    uint32_t x = v;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, o);
        if (lane >= (uint32_t)o) x += y;
    }
    __syncthreads();
    if (lane == 63) ws[wave] = x;
    __syncthreads();
    uint32_t before = 0;
    total = 0;
#pragma unroll
    for (uint32_t w = 0; w < kSortBlock / 64; ++w) {
        if (w < wave) before += ws[w];
        total += ws[w];
    }
    return before + x - v;
}

// Block d: hist[d][*] becomes its exclusive scan, totals[d] its sum.
static __global__ __launch_bounds__(kSortBlock) void sort_scan_kernel(uint32_t* __restrict__ hist, uint32_t tiles,
                                                                      uint32_t* __restrict__ totals) {
    uint32_t* h = hist + (size_t)blockIdx.x * tiles;
    uint32_t carry = 0;
    for (uint32_t t0 = 0; t0 < tiles; t0 += kSortBlock) {
        const uint32_t t = t0 + threadIdx.x;
        const uint32_t v = t < tiles ? h[t] : 0u;
        uint32_t total;
        const uint32_t before = sort_block_scan(v, total);
        if (t < tiles) h[t] = carry + before;
        carry += total;
    }
    if (threadIdx.x == 0) totals[blockIdx.x] = carry;
}

// vals_in == NULL: the values are the keys' positions.
static __global__ __launch_bounds__(kSortBlock) void sort_scatter_kernel(
    const uint32_t* __restrict__ keys_in, const uint32_t* __restrict__ vals_in, uint32_t* __restrict__ keys_out,
    uint32_t* __restrict__ vals_out, uint32_t n, int shift, uint32_t tiles, const uint32_t* __restrict__ hist,
    const uint32_t* __restrict__ totals) {
    __shared__ uint32_t cnt[kSortBlock / 64][kSortDigits];  // keys of a digit in each wave's part, then its start
    __shared__ uint32_t gofs[kSortDigits];                  // global position of local position 0 of a digit's run
    __shared__ uint32_t sk[kSortTile], sv[kSortTile];
    const uint32_t lane = lane_id(), wave = threadIdx.x >> 6, d = threadIdx.x;
    const uint64_t base = (uint64_t)blockIdx.x * kSortTile;
    const uint32_t m = n - base < kSortTile ? (uint32_t)(n - base) : (uint32_t)kSortTile;
    volatile uint32_t* mine = cnt[wave];
#pragma unroll
    for (int k = 0; k < kSortDigits / 64; ++k) mine[64 * k + lane] = 0;
    uint32_t key[kSortRounds], rank[kSortRounds];
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t j = wave * 64 * kSortRounds + r * 64 + lane;
        key[r] = j < m ? keys_in[base + j] : 0u;
    }
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t j = wave * 64 * kSortRounds + r * 64 + lane;
        const uint32_t digit = (key[r] >> shift) & 255u;
        uint64_t same = __ballot(j < m);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t bit = __ballot((digit >> b) & 1u);
            same &= ((digit >> b) & 1u) ? bit : ~bit;
        }
        if (j < m) {
            const uint32_t before = mask_rank(same), seen = mine[digit];
            rank[r] = seen + before;
            if (before == 0) mine[digit] = seen + (uint32_t)__popcll(same);
        }
    }
    __syncthreads();
    // thread d: digit d's run in the tile
    uint32_t c[kSortBlock / 64], sum = 0, total;
#pragma unroll
    for (int w = 0; w < kSortBlock / 64; ++w) {
        c[w] = cnt[w][d];
        sum += c[w];
    }
    const uint32_t gstart = sort_block_scan(totals[d], total) + hist[(size_t)d * tiles + blockIdx.x];
    uint32_t local = sort_block_scan(sum, total);
    gofs[d] = gstart - local;
#pragma unroll
    for (int w = 0; w < kSortBlock / 64; ++w) {
        cnt[w][d] = local;
        local += c[w];
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t j = wave * 64 * kSortRounds + r * 64 + lane;
        if (j < m) {
            const uint32_t at = cnt[wave][(key[r] >> shift) & 255u] + rank[r];
            sk[at] = key[r];
            sv[at] = vals_in ? vals_in[base + j] : (uint32_t)(base + j);
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < kSortRounds; ++r) {
        const uint32_t j = r * kSortBlock + threadIdx.x;
        if (j < m) {
            const uint32_t k = sk[j], at = gofs[(k >> shift) & 255u] + j;
            keys_out[at] = k;
            vals_out[at] = sv[j];
        }
    }
}

// All digits of up to kSortTile keys by one block, in LDS (512 keys of 18 bits:
// 9 launches, 37 us -> one, 9 us).  keys / vals out: the sorted keys and their
// positions.
static __global__ __launch_bounds__(kSortBlock) void sort_small_kernel(const uint32_t* __restrict__ keys_in, uint32_t m,
                                                                       int bits, uint32_t* __restrict__ keys_out,
                                                                       uint32_t* __restrict__ vals_out) {
    __shared__ uint32_t cnt[kSortBlock / 64][kSortDigits];
    __shared__ uint32_t sk[kSortTile], sv[kSortTile];
    const uint32_t lane = lane_id(), wave = threadIdx.x >> 6, d = threadIdx.x;
    const uint32_t rounds = (m + kSortBlock - 1) / kSortBlock;
    volatile uint32_t* mine = cnt[wave];
    uint32_t key[kSortRounds], val[kSortRounds], rank[kSortRounds];
#pragma unroll
    for (uint32_t r = 0; r < kSortRounds; ++r) {
        const uint32_t j = (wave * rounds + r) * 64 + lane;
        val[r] = j;
        key[r] = r < rounds && j < m ? keys_in[j] : 0u;
    }
    for (int shift = 0; shift < bits; shift += 8) {
#pragma unroll
        for (int k = 0; k < kSortDigits / 64; ++k) mine[64 * k + lane] = 0;
#pragma unroll
        for (uint32_t r = 0; r < kSortRounds; ++r) {
            if (r >= rounds) continue;
            const bool in = (wave * rounds + r) * 64 + lane < m;
            const uint32_t digit = (key[r] >> shift) & 255u;
            uint64_t same = __ballot(in);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const uint64_t bit = __ballot((digit >> b) & 1u);
                same &= ((digit >> b) & 1u) ? bit : ~bit;
            }
            if (in) {
                const uint32_t before = mask_rank(same), seen = mine[digit];
                rank[r] = seen + before;
                if (before == 0) mine[digit] = seen + (uint32_t)__popcll(same);
            }
        }
        __syncthreads();
        uint32_t c[kSortBlock / 64], sum = 0, total;
#pragma unroll
        for (int w = 0; w < kSortBlock / 64; ++w) {
            c[w] = cnt[w][d];
            sum += c[w];
        }
        uint32_t local = sort_block_scan(sum, total);
#pragma unroll
        for (int w = 0; w < kSortBlock / 64; ++w) {
            cnt[w][d] = local;
            local += c[w];
        }
        __syncthreads();
#pragma unroll
        for (uint32_t r = 0; r < kSortRounds; ++r) {
            if (r < rounds && (wave * rounds + r) * 64 + lane < m) {
                const uint32_t at = cnt[wave][(key[r] >> shift) & 255u] + rank[r];
                sk[at] = key[r];
                sv[at] = val[r];
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t r = 0; r < kSortRounds; ++r) {
            const uint32_t j = (wave * rounds + r) * 64 + lane;
            if (r < rounds && j < m) {
                key[r] = sk[j];
                val[r] = sv[j];
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (uint32_t r = 0; r < kSortRounds; ++r) {
        const uint32_t j = (wave * rounds + r) * 64 + lane;
        if (r < rounds && j < m) {
            keys_out[j] = key[r];
            vals_out[j] = val[r];
        }
    }
}

inline uint32_t sort_tiles(int64_t n) { return (uint32_t)((n + kSortTile - 1) / kSortTile); }

// Bytes of the two key buffers, the two index buffers and the histograms.
inline size_t sort_workspace_bytes(int64_t n) {
    return ((size_t)n * 4 + 255) / 256 * 256 * 4 + ((size_t)sort_tiles(n) + 1) * kSortDigits * 4;
}

struct SortBuffers {
    uint32_t* keys[2];
    uint32_t* vals[2];
    uint32_t* hist;
    uint32_t* totals;
};

inline SortBuffers sort_buffers(void* workspace, int64_t n) {
    const size_t seg = ((size_t)n * 4 + 255) / 256 * 256;
    char* w = (char*)workspace;
    SortBuffers b;
    for (int k = 0; k < 2; ++k) {
        b.keys[k] = (uint32_t*)(w + k * seg);
        b.vals[k] = (uint32_t*)(w + (2 + k) * seg);
    }
    b.totals = (uint32_t*)(w + 4 * seg);
    b.hist = b.totals + kSortDigits;
    return b;
}

// Which of the two buffers launch_sort leaves its result in.
inline int sort_result(int bits) { return ((bits + 7) / 8) & 1; }

// Sorts keys[0] (n < 2^32 of them) by their low `bits` bits; the returned 0 or
// 1 (sort_result) says which keys / vals hold the sorted keys and their input
// positions.
inline int launch_sort(const SortBuffers& b, int64_t n, int bits, hipStream_t s) {
    const uint32_t tiles = sort_tiles(n);
    if (tiles == 1) {
        const int to = sort_result(bits);
        hipLaunchKernelGGL(sort_small_kernel, dim3(1), dim3(kSortBlock), 0, s, b.keys[0], (uint32_t)n, bits, b.keys[to],
                           b.vals[to]);
        return to;
    }
    int from = 0;
    for (int shift = 0; shift < bits; shift += 8) {
        hipLaunchKernelGGL(sort_hist_kernel, dim3(tiles), dim3(kSortBlock), 0, s, b.keys[from], (uint32_t)n, shift,
                           tiles, b.hist);
        hipLaunchKernelGGL(sort_scan_kernel, dim3(kSortDigits), dim3(kSortBlock), 0, s, b.hist, tiles, b.totals);
        hipLaunchKernelGGL(sort_scatter_kernel, dim3(tiles), dim3(kSortBlock), 0, s, b.keys[from],
                           shift == 0 ? (const uint32_t*)nullptr : b.vals[from], b.keys[1 - from], b.vals[1 - from],
                           (uint32_t)n, shift, tiles, b.hist, b.totals);
        from = 1 - from;
    }
    return from;
}

}  // namespace nglod
