// tl_partition.hpp -- pieces of the splitter partitions (tl_tile.hip: queries to
// the ranges of an array, tl_sort.hip: keys to buckets): heap order, tiles of a
// one- or two-pass partition, and the kernels that turn the tiles' counts into
// places.  `queries` below are the items of either.
#pragma once

#include "tl_internal.hpp"
#include "tl_slots.hpp"

namespace tl {

constexpr uint32_t PART_LG = 10;        // log2 of the ranges of one pass, at most
constexpr uint32_t PART_BINS = 1u << PART_LG;
constexpr uint32_t PART_NT = 1024;
constexpr uint32_t PART_GROUP = 32;     // tiles of one column sum

// first rank of range j of 2^lg
__device__ inline uint32_t range_first(uint32_t j, uint32_t n, uint32_t lg) {
    return (uint32_t)(((uint64_t)j * n) >> lg);
}

// in-order place (1 .. 2^lg - 1) of node i of a complete tree of lg levels
__device__ inline uint32_t heap_order(uint32_t i, uint32_t lg) {
    const uint32_t t = 31u - (uint32_t)__clz((int)i);
    return (2 * (i - (1u << t)) + 1) << (lg - 1 - t);
}

// its inverse: the node at place y of a complete tree of lg levels
__device__ inline uint32_t heap_node(uint32_t y, uint32_t lg) {
    return (y | (1u << lg)) >> ((uint32_t)__clz((int)__brev(y)) + 1);
}

// where place y of a range's keys lies (range_fill)
__device__ inline uint32_t heap_at(uint32_t y, uint32_t lg) {
    return y ? heap_node(y, lg) : 0u;
}

// what a tile of a pass is: queries [lo, hi) of the input, to be split at the
// bounds first + step, first + 2 * step, ..
struct PartTile {
    uint64_t lo, hi;
    uint32_t first;
};

// the tile's bucket tables: tile t of the first pass is queries t * T ..; of
// the second pass, a piece of one first-pass bucket (tstart: tiles before each
// bucket, bstart: queries before each bucket)
template <bool SECOND>
__device__ inline PartTile part_tile(uint32_t t, uint64_t nq, uint32_t T, uint32_t lg1,
                                     uint32_t lg2, const uint32_t *__restrict__ bstart,
                                     const uint32_t *__restrict__ tstart) {
    PartTile p;
    if constexpr (SECOND) {
        uint32_t lo = 0, hi = 1u << lg1;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (tstart[mid] <= t) lo = mid;
            else hi = mid;
        }
        p.lo = bstart[lo] + (uint64_t)(t - tstart[lo]) * T;
        p.hi = min((uint64_t)bstart[lo + 1], p.lo + T);
        p.first = lo << lg2;
    } else {
        p.lo = (uint64_t)t * T;
        p.hi = min(nq, p.lo + T);
        p.first = 0;
    }
    return p;
}

// first pass: sums of each bucket over groups of PART_GROUP tiles
static __global__ __launch_bounds__(PART_NT) void k_part_sums(const uint32_t *__restrict__ counts,
                                                       uint32_t B, uint32_t tiles,
                                                       uint32_t *__restrict__ gsum) {
    const uint32_t t0 = blockIdx.x * PART_GROUP, t1 = min(tiles, t0 + PART_GROUP);
    if (threadIdx.x >= B) return;
    uint32_t x = 0;
#pragma unroll 8
    for (uint32_t t = t0; t < t1; t++) x += counts[(uint64_t)t * B + threadIdx.x];
    gsum[(uint64_t)blockIdx.x * B + threadIdx.x] = x;
}

// exclusive scan of one value a lane over the whole workgroup; the total in
// *total
__device__ inline uint32_t block_scan(uint32_t v, uint32_t *wsum, uint32_t *total) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t x = v;
    for (int o = 1; o < 64; o <<= 1) {
        const uint32_t y = (uint32_t)__shfl_up((int)x, (unsigned)o);
        if (lane >= (uint32_t)o) x += y;
    }
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t w = 0; w < blockDim.x / 64; w++) {
        if (w < wave) before += wsum[w];
        all += wsum[w];
    }
    __syncthreads();
    *total = all;
    return before + x - v;
}

// first pass, one workgroup: the groups' sums become the queries of the
// bucket in earlier groups; bstart[] the queries of earlier buckets; tstart[]
// the second pass's tiles of T queries of earlier buckets (bcount, where not
// null: the queries of each)
static __global__ __launch_bounds__(PART_NT) void k_part_starts(uint32_t *__restrict__ gsum, uint32_t B,
                                                         uint32_t groups, uint32_t T,
                                                         uint32_t *__restrict__ bstart,
                                                         uint32_t *__restrict__ tstart,
                                                         uint32_t *__restrict__ bcount) {
    __shared__ uint32_t wsum[PART_NT / 64];
    const uint32_t bin = threadIdx.x;
    uint32_t run = 0;
    if (bin < B) {
#pragma unroll 8
        for (uint32_t g = 0; g < groups; g++) {
            const uint32_t v = gsum[(uint64_t)g * B + bin];
            gsum[(uint64_t)g * B + bin] = run;
            run += v;
        }
    }
    uint32_t total, tiles;
    const uint32_t at = block_scan(run, wsum, &total);
    const uint32_t tl = block_scan((run + T - 1) / T, wsum, &tiles);
    if (bin < B) {
        bstart[bin] = at;
        tstart[bin] = tl;
        if (bcount) bcount[bin] = run;
    }
    if (bin == 0) {
        bstart[B] = total;
        tstart[B] = tiles;
    }
}

// first pass: places[t][bucket], the place of the tile's first query of the
// bucket
static __global__ __launch_bounds__(PART_NT) void k_part_places(const uint32_t *__restrict__ counts,
                                                         uint32_t B, uint32_t tiles,
                                                         const uint32_t *__restrict__ gsum,
                                                         const uint32_t *__restrict__ bstart,
                                                         uint32_t *__restrict__ places) {
    const uint32_t t0 = blockIdx.x * PART_GROUP, t1 = min(tiles, t0 + PART_GROUP);
    const uint32_t bin = threadIdx.x;
    if (bin >= B) return;
    uint32_t run = bstart[bin] + gsum[(uint64_t)blockIdx.x * B + bin];
#pragma unroll 8
    for (uint32_t t = t0; t < t1; t++) {
        places[(uint64_t)t * B + bin] = run;
        run += counts[(uint64_t)t * B + bin];
    }
}

// second pass, a workgroup per first-pass bucket: the same for its tiles, and
// the start of each of its ranges (rstart; rcount, where not null: its queries,
// fewer than up to the next start where the second pass leaves some out)
static __global__ __launch_bounds__(PART_NT) void k_part_places2(const uint32_t *__restrict__ counts,
                                                          uint32_t lg1, uint32_t lg2,
                                                          const uint32_t *__restrict__ bstart,
                                                          const uint32_t *__restrict__ tstart,
                                                          uint32_t *__restrict__ places,
                                                          uint32_t *__restrict__ rstart,
                                                          uint32_t *__restrict__ rcount) {
    __shared__ uint32_t wsum[PART_NT / 64];
    const uint32_t B = 1u << lg2, bin = threadIdx.x, k = blockIdx.x;
    const uint32_t t0 = tstart[k], t1 = tstart[k + 1];
    uint32_t sum = 0;
    if (bin < B) {
#pragma unroll 8
        for (uint32_t t = t0; t < t1; t++) sum += counts[(uint64_t)t * B + bin];
    }
    uint32_t total;
    uint32_t run = bstart[k] + block_scan(sum, wsum, &total);
    if (bin < B) {
        rstart[((uint64_t)k << lg2) + bin] = run;
        if (rcount) rcount[((uint64_t)k << lg2) + bin] = sum;
#pragma unroll 8
        for (uint32_t t = t0; t < t1; t++) {
            places[(uint64_t)t * B + bin] = run;
            run += counts[(uint64_t)t * B + bin];
        }
    }
    if (k + 1 == gridDim.x && bin == 0) rstart[(uint64_t)gridDim.x << lg2] = bstart[k + 1];
}

}   // namespace tl
