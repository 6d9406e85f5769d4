// tl_sort.hip -- the step before the layouts: sort raw keys and drop
// duplicates on the device, so that an unsorted key set with repeats becomes
// the sorted, distinct input every layout assumes (the reference's drivers
// build such input themselves, cpu/src/common.h:33-40).
//
// Splitter sort.  The keys are partitioned into buckets of 768 to 1536 on
// average by splitters from samples, in one pass (1024 buckets) or two, each a
// count and a scatter whose tile leaves LDS in bucket order; a bucket is then
// sorted in LDS by one workgroup and its repeats dropped, and one pass closes the
// gaps.  Whatever the key width and range, every key moves four times (the digits
// of a radix sort move it once per 8 bits that vary: 100 million 40-bit keys took
// five passes at 1.0 ms and 6.2 ms in all; now 3.1 ms, as many of 62 bits).  A key
// equal to a splitter is not partitioned but noted with it, so a key that repeats
// often costs nothing, however often.
//
// Bucket sizes are the samples' luck: with m samples to a splitter, a bucket is
// its average times a Gamma(m) / m of each pass.  For distinct keys in random
// order 4096 are passed by 0.7 buckets of 2*10^8 keys and by 1.6 of 4*10^8 (32 and
// 32 samples, an average of 1530), by 0.01 of 10^8 and by fewer below; those few
// are sorted by larger workgroups.  16384 are passed by fewer than 10^-27.  Inputs
// made to (or whose repeats lie where no sample does) still can: nothing has been
// lost then, the partitioned keys and the noted splitters are the input's distinct
// keys and some repeats, and the radix sort below takes over from them.  It also
// serves the largest arrays.
//
// LSD radix sort, 8-bit digits, stable, ping-ponging between the caller's
// array and one library-owned buffer of n keys.  Signed keys sort by their
// bits with the sign bit flipped.  A pass whose digit is the same for every
// key (found by one AND/OR reduction over all keys) is skipped: keys built
// from small gaps leave their top bytes constant.  Per pass:
//   k_radix_hist     per tile of 8192 keys, a 256-bucket histogram, stored
//                    digit-major (counts[d * tiles + tile]);
//   scan             exclusive scan of those counts (the global offset of
//                    every (digit, tile) bucket);
//   k_radix_scatter  every tile again: each wave ranks its keys by digit with
//                    8 ballots per key slot (lanes with equal digits find each
//                    other), waves are offset by the earlier waves' counts,
//                    and every key goes to its bucket's next slot.
// Keys are processed in (wave, slot, lane) order, which is their order in
// memory, so equal digits keep their order (the sort is stable).
// Duplicates: every sorted key that differs from its predecessor is kept;
// a count per tile, a scan, and a compaction into the other buffer.
#include <stdlib.h>

#include <algorithm>
#include <type_traits>
#include <vector>

#include "tl_internal.hpp"
#include "tl_partition.hpp"
#include "tl_plan.hpp"

namespace tl {

constexpr uint32_t SORT_THREADS = 256;
constexpr uint32_t SORT_ITEMS = 32;
constexpr uint32_t SORT_TILE = SORT_THREADS * SORT_ITEMS;   // keys per tile
constexpr uint32_t SORT_WAVES = SORT_THREADS / 64;
constexpr uint32_t SCAN_CHUNK = 4096;                        // counts per scan workgroup

// AND and OR of every key's order bits (bits ^ flip)
template <typename U>
__global__ __launch_bounds__(256) void k_and_or(const U *__restrict__ a, uint64_t n, U flip,
                                                unsigned long long *andor) {
    U va = ~(U)0, vo = 0;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x) {
        const U u = a[i] ^ flip;
        va &= u;
        vo |= u;
    }
    __shared__ unsigned long long sa[256], so[256];
    sa[threadIdx.x] = (unsigned long long)va | (sizeof(U) == 4 ? 0xFFFFFFFF00000000ull : 0ull);
    so[threadIdx.x] = (unsigned long long)vo;
    __syncthreads();
    for (uint32_t s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            sa[threadIdx.x] &= sa[threadIdx.x + s];
            so[threadIdx.x] |= so[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        atomicAnd(&andor[0], sa[0]);
        atomicOr(&andor[1], so[0]);
    }
}

template <typename U>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_hist(const U *__restrict__ a, uint64_t n,
                                                             uint32_t shift, U flip,
                                                             uint32_t *__restrict__ counts,
                                                             uint32_t tiles) {
    __shared__ uint32_t h[256];
    h[threadIdx.x] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * SORT_TILE;
    const uint64_t end = min(n, base + SORT_TILE);
    for (uint64_t i = base + threadIdx.x; i < end; i += SORT_THREADS)
        atomicAdd(&h[(uint32_t)(((a[i] ^ flip) >> shift) & 0xFF)], 1u);
    __syncthreads();
    counts[(uint64_t)threadIdx.x * tiles + blockIdx.x] = h[threadIdx.x];
}

// exclusive scan of v[0..len) in chunks of SCAN_CHUNK: local scan, chunk sums
__global__ __launch_bounds__(256) void k_scan_chunks(uint32_t *__restrict__ v, uint64_t len,
                                                     uint32_t *__restrict__ sums) {
    constexpr uint32_t PER = SCAN_CHUNK / 256;
    __shared__ uint32_t part[256];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_CHUNK + (uint64_t)threadIdx.x * PER;
    uint32_t x[PER], t = 0;
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
        x[k] = base + k < len ? v[base + k] : 0u;
        const uint32_t y = x[k];
        x[k] = t;
        t += y;
    }
    part[threadIdx.x] = t;
    __syncthreads();
    // Hillis-Steele inclusive scan of the 256 thread totals
    for (uint32_t s = 1; s < 256; s <<= 1) {
        const uint32_t y = threadIdx.x >= s ? part[threadIdx.x - s] : 0u;
        __syncthreads();
        part[threadIdx.x] += y;
        __syncthreads();
    }
    const uint32_t off = threadIdx.x ? part[threadIdx.x - 1] : 0u;
#pragma unroll
    for (uint32_t k = 0; k < PER; k++)
        if (base + k < len) v[base + k] = x[k] + off;
    if (threadIdx.x == 255) sums[blockIdx.x] = part[255];
}

// exclusive scan of the chunk sums in one workgroup (any count), then the
// grand total at sums[len]
__global__ __launch_bounds__(1024) void k_scan_sums(uint32_t *__restrict__ sums, uint64_t len) {
    __shared__ uint32_t part[1024];
    __shared__ uint32_t carry;
    if (threadIdx.x == 0) carry = 0;
    __syncthreads();
    for (uint64_t base = 0; base < len; base += 1024) {
        const uint64_t i = base + threadIdx.x;
        const uint32_t x = i < len ? sums[i] : 0u;
        part[threadIdx.x] = x;
        __syncthreads();
        for (uint32_t s = 1; s < 1024; s <<= 1) {
            const uint32_t y = threadIdx.x >= s ? part[threadIdx.x - s] : 0u;
            __syncthreads();
            part[threadIdx.x] += y;
            __syncthreads();
        }
        if (i < len) sums[i] = carry + part[threadIdx.x] - x;
        __syncthreads();
        if (threadIdx.x == 1023) carry += part[1023];
        __syncthreads();
    }
    if (threadIdx.x == 0) sums[len] = carry;
}

__global__ __launch_bounds__(256) void k_scan_add(uint32_t *__restrict__ v, uint64_t len,
                                                  const uint32_t *__restrict__ sums) {
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_CHUNK;
    const uint32_t add = sums[blockIdx.x];
    for (uint64_t i = base + threadIdx.x; i < min(len, base + SCAN_CHUNK); i += 256) v[i] += add;
}

// (wave, slot, lane) order of a tile: element e of wave w, slot k, lane l
__device__ inline uint64_t tile_elem(uint64_t base, uint32_t w, uint32_t k, uint32_t lane) {
    return base + (uint64_t)w * (64 * SORT_ITEMS) + (uint64_t)k * 64 + lane;
}

template <typename U>
__global__ __launch_bounds__(SORT_THREADS) void k_radix_scatter(const U *__restrict__ a,
                                                                U *__restrict__ out, uint64_t n,
                                                                uint32_t shift, U flip,
                                                                const uint32_t *__restrict__ offs,
                                                                uint32_t tiles) {
    __shared__ uint32_t cnt[SORT_WAVES][256];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (uint32_t i = threadIdx.x; i < SORT_WAVES * 256; i += SORT_THREADS) (&cnt[0][0])[i] = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * SORT_TILE;
    const uint64_t lt = (1ull << lane) - 1;
    U key[SORT_ITEMS];
    uint32_t rank[SORT_ITEMS];
#pragma unroll
    for (uint32_t k = 0; k < SORT_ITEMS; k++) {
        const uint64_t e = tile_elem(base, w, k, lane);
        const bool valid = e < n;
        key[k] = valid ? a[e] : (U)0;
        const uint32_t d = (uint32_t)(((key[k] ^ flip) >> shift) & 0xFF);
        // lanes whose digit equals mine: 8 ballots, one per digit bit
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (uint32_t bit = 0; bit < 8; bit++) {
            const bool on = (d >> bit) & 1u;
            const uint64_t m = __ballot(on);
            peers &= on ? m : ~m;
        }
        uint32_t r = 0;
        if (valid) {
            // every peer reads the bucket before the lowest peer advances it
            // (one wave: the reads of this slot issue before its write)
            r = cnt[w][d] + (uint32_t)__popcll(peers & lt);
        }
        __builtin_amdgcn_wave_barrier();
        if (valid && (peers & lt) == 0) cnt[w][d] += (uint32_t)__popcll(peers);
        __builtin_amdgcn_wave_barrier();
        rank[k] = r;
    }
    __syncthreads();
    // bucket d of wave w starts at the tile's global offset of d plus the
    // counts of d in the earlier waves
    {
        const uint32_t d = threadIdx.x;   // SORT_THREADS == 256 digits
        uint32_t run = offs[(uint64_t)d * tiles + blockIdx.x];
        for (uint32_t ww = 0; ww < SORT_WAVES; ww++) {
            const uint32_t c = cnt[ww][d];
            cnt[ww][d] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < SORT_ITEMS; k++) {
        const uint64_t e = tile_elem(base, w, k, lane);
        if (e < n) {
            const uint32_t d = (uint32_t)(((key[k] ^ flip) >> shift) & 0xFF);
            out[cnt[w][d] + rank[k]] = key[k];
        }
    }
}

// keys of a sorted tile that differ from their predecessor: count per tile
template <typename U>
__global__ __launch_bounds__(SORT_THREADS) void k_unique_count(const U *__restrict__ a, uint64_t n,
                                                               uint32_t *__restrict__ counts) {
    __shared__ uint32_t c;
    if (threadIdx.x == 0) c = 0;
    __syncthreads();
    const uint64_t base = (uint64_t)blockIdx.x * SORT_TILE;
    const uint64_t end = min(n, base + SORT_TILE);
    uint32_t mine = 0;
    for (uint64_t i = base + threadIdx.x; i < end; i += SORT_THREADS)
        mine += (i == 0 || a[i] != a[i - 1]) ? 1u : 0u;
    atomicAdd(&c, mine);
    __syncthreads();
    if (threadIdx.x == 0) counts[blockIdx.x] = c;
}

template <typename U>
__global__ __launch_bounds__(SORT_THREADS) void k_unique_scatter(const U *__restrict__ a,
                                                                 U *__restrict__ out, uint64_t n,
                                                                 const uint32_t *__restrict__ offs) {
    __shared__ uint32_t wsum[SORT_WAVES];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint64_t base = (uint64_t)blockIdx.x * SORT_TILE;
    const uint64_t lt = (1ull << lane) - 1;
    uint32_t before = 0;   // kept keys of this wave in earlier slots
    uint32_t pos[SORT_ITEMS];
    bool keep[SORT_ITEMS];
    U key[SORT_ITEMS];
#pragma unroll
    for (uint32_t k = 0; k < SORT_ITEMS; k++) {
        const uint64_t e = tile_elem(base, w, k, lane);
        keep[k] = false;
        key[k] = 0;
        if (e < n) {
            key[k] = a[e];
            keep[k] = (e == 0 || key[k] != a[e - 1]);
        }
        const uint64_t m = __ballot(keep[k]);
        pos[k] = before + (uint32_t)__popcll(m & lt);
        before += (uint32_t)__popcll(m);
    }
    if (lane == 0) wsum[w] = before;
    __syncthreads();
    uint32_t woff = offs[blockIdx.x];
    for (uint32_t ww = 0; ww < w; ww++) woff += wsum[ww];
#pragma unroll
    for (uint32_t k = 0; k < SORT_ITEMS; k++)
        if (keep[k]) out[woff + pos[k]] = key[k];
}

// exclusive scan of v[0..len) in place; the total lands in *total_dev
// (sums needs len / SCAN_CHUNK + 2 words)
static tl_status scan_u32(uint32_t *v, uint64_t len, uint32_t *sums, hipStream_t s) {
    const uint64_t chunks = (len + SCAN_CHUNK - 1) / SCAN_CHUNK;
    hipLaunchKernelGGL(k_scan_chunks, dim3((uint32_t)chunks), dim3(256), 0, s, v, len, sums);
    TL_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(1024), 0, s, sums, chunks);
    TL_LAUNCH_CHECK();
    hipLaunchKernelGGL(k_scan_add, dim3((uint32_t)chunks), dim3(256), 0, s, v, len,
                       (const uint32_t *)sums);
    TL_LAUNCH_CHECK();
    return TL_OK;
}

// ---------------------------------------------------------------------------
// the splitter sort

constexpr uint32_t RANGE_NT = 512, RANGE_IT = 8;
constexpr uint32_t RANGE_CAP = RANGE_NT * RANGE_IT;   // keys of a bucket, mostly
constexpr uint32_t LARGE_NT = 1024, LARGE_IT = 16;
constexpr uint32_t LARGE_CAP = LARGE_NT * LARGE_IT;   // ... at most
constexpr uint32_t RANGE_GOAL = 1536;                 // ... on average, fewer than
constexpr uint32_t RANGE_BINS = 2048;
constexpr uint32_t SORT_LG1 = 8;   // log2 of the first of two passes' buckets
constexpr uint64_t SPLIT_MAX_KEYS = 1ull << 29;       // 2^10 and 2^9 buckets

template <typename K>
using Bits = typename std::conditional<sizeof(K) == 4, uint32_t, uint64_t>::type;
// the key's bits in its own order, and back
template <typename K>
__device__ inline Bits<K> to_bits(K k) {
    const Bits<K> top = (K)-1 < (K)0 ? (Bits<K>)1 << (8 * sizeof(K) - 1) : 0;
    return (Bits<K>)k ^ top;
}
template <typename K>
__device__ inline K from_bits(Bits<K> u) {
    const Bits<K> top = (K)-1 < (K)0 ? (Bits<K>)1 << (8 * sizeof(K) - 1) : 0;
    return (K)(u ^ top);
}

// sorts buf[0 .. cnt) in LDS, cnt <= NT * IT: LSD radix over the 8-bit digits
// that vary.  hist: NT / 64 * 256 words
template <typename U, uint32_t NT, uint32_t IT>
__device__ inline void lds_sort(U *buf, uint32_t cnt, uint32_t *hist, uint32_t *wsum) {
    __shared__ uint32_t vary_lo, vary_hi;
    constexpr uint32_t NW = NT / 64;
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint64_t lt = (1ull << lane) - 1;
    if (tid == 0) vary_lo = vary_hi = 0;
    __syncthreads();
    uint64_t vary = 0;
    for (uint32_t i = tid; i < cnt; i += NT) vary |= (uint64_t)(buf[i] ^ buf[0]);
    if ((uint32_t)vary) atomicOr(&vary_lo, (uint32_t)vary);
    if (vary >> 32) atomicOr(&vary_hi, (uint32_t)(vary >> 32));
    __syncthreads();
    vary = (uint64_t)vary_hi << 32 | vary_lo;
    const uint32_t items = (cnt + NT - 1) / NT;   // slots of a lane, in memory order
    for (uint32_t shift = 0; shift < 8 * sizeof(U); shift += 8) {
        if (((vary >> shift) & 0xFF) == 0) continue;
        for (uint32_t i = tid; i < NW * 256; i += NT) hist[i] = 0;
        __syncthreads();
        U x[IT];
        uint32_t rank[IT];
#pragma unroll
        for (uint32_t k = 0; k < IT; k++) {
            if (k >= items) continue;
            const uint32_t i = (w * items + k) * 64 + lane;
            const bool valid = i < cnt;
            x[k] = valid ? buf[i] : (U)0;
            const uint32_t d = (uint32_t)(x[k] >> shift) & 0xFF;
            uint64_t peers = __ballot(valid);
#pragma unroll
            for (uint32_t bit = 0; bit < 8; bit++) {
                const bool on = (d >> bit) & 1u;
                const uint64_t m = __ballot(on);
                peers &= on ? m : ~m;
            }
            rank[k] = valid ? hist[w * 256 + d] + (uint32_t)__popcll(peers & lt) : 0u;
            __builtin_amdgcn_wave_barrier();
            if (valid && (peers & lt) == 0) hist[w * 256 + d] += (uint32_t)__popcll(peers);
            __builtin_amdgcn_wave_barrier();
        }
        __syncthreads();
        // starts of (digit, wave) in digit order, then wave order
        uint32_t sum = 0;
        if (tid < 256)
            for (uint32_t ww = 0; ww < NW; ww++) sum += hist[ww * 256 + tid];
        uint32_t total;
        uint32_t run = block_scan(sum, wsum, &total);
        if (tid < 256)
            for (uint32_t ww = 0; ww < NW; ww++) {
                const uint32_t c = hist[ww * 256 + tid];
                hist[ww * 256 + tid] = run;
                run += c;
            }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < IT; k++) {
            const uint32_t i = (w * items + k) * 64 + lane;
            if (k < items && i < cnt)
                buf[hist[w * 256 + ((uint32_t)(x[k] >> shift) & 0xFF)] + rank[k]] = x[k];
        }
        __syncthreads();
    }
}

// place of sample i of `samples` among count items: one of each equal share, at
// a place that does not follow a stride of the data
__device__ inline uint64_t sample_at(uint32_t i, uint32_t samples, uint64_t count) {
    const uint64_t lo = (uint64_t)i * count / samples, hi = (uint64_t)(i + 1) * count / samples;
    return hi > lo ? lo + (uint64_t)(i * 2654435761u) % (hi - lo) : lo;
}

// bound[j << lg2], j < 2^lg1: the first pass's splitters (one workgroup), or
// with SECOND bound[k << lg2 | o], 0 < o < 2^lg2: those of bucket k, a
// workgroup each
template <typename K, bool SECOND, uint32_t IT>
__global__ __launch_bounds__(1024) void k_sort_sample(const K *__restrict__ keys, uint64_t n,
                                                      uint32_t lg1, uint32_t lg2,
                                                      const uint32_t *__restrict__ bstart,
                                                      K *__restrict__ bound) {
    constexpr uint32_t SAMPLES = 1024 * IT;
    __shared__ Bits<K> buf[SAMPLES];
    __shared__ uint32_t hist[16 * 256], wsum[16];
    const uint64_t lo = SECOND ? bstart[blockIdx.x] : 0;
    const uint64_t count = SECOND ? bstart[blockIdx.x + 1] - lo : n;
    if (SECOND && count == 0) {   // no key meets these
        for (uint32_t o = threadIdx.x + 1; o < (1u << lg2); o += 1024)
            bound[((uint64_t)blockIdx.x << lg2) + o] = bound[(uint64_t)blockIdx.x << lg2];
        return;
    }
    for (uint32_t i = threadIdx.x; i < SAMPLES; i += 1024)
        buf[i] = to_bits<K>(keys[lo + sample_at(i, SAMPLES, count)]);
    __syncthreads();
    lds_sort<Bits<K>, 1024, IT>(buf, SAMPLES, hist, wsum);
    if (SECOND) {
        for (uint32_t o = threadIdx.x + 1; o < (1u << lg2); o += 1024)
            bound[((uint64_t)blockIdx.x << lg2) + o] =
                from_bits<K>(buf[(uint64_t)o * SAMPLES >> lg2]);
    } else {
        for (uint32_t j = threadIdx.x; j < (1u << lg1); j += 1024)
            bound[(uint64_t)j << lg2] = from_bits<K>(buf[(uint64_t)j * SAMPLES >> lg1]);
    }
}

// the tile's splitters in heap order (node 0 unused), and bucket by bucket
template <typename K, bool SECOND>
__device__ inline void sort_splitters(const K *__restrict__ bound, const PartTile &p, uint32_t lg1,
                                      uint32_t lg2, K *spl, K *low) {
    const uint32_t lg = SECOND ? lg2 : lg1, step = SECOND ? 1u : 1u << lg2;
    if (threadIdx.x < (1u << lg)) {
        low[threadIdx.x] = bound[p.first + (uint64_t)threadIdx.x * step];
        if (threadIdx.x)
            spl[threadIdx.x] = bound[p.first + (uint64_t)heap_order(threadIdx.x, lg) * step];
    }
}

// bucket of each key, and whether the key equals the bucket's splitter (the
// first bucket of all has none)
template <typename K, int IT>
__device__ inline void sort_buckets(const K (&q)[IT], const K *spl, const K *low, uint32_t first,
                                    uint32_t lg, uint32_t (&bin)[IT], bool (&eq)[IT]) {
#pragma unroll
    for (int k = 0; k < IT; k++) bin[k] = 1;
    for (uint32_t l = 0; l < lg; l++) {
#pragma unroll
        for (int k = 0; k < IT; k++) bin[k] = 2 * bin[k] + (q[k] >= spl[bin[k]] ? 1u : 0u);
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {
        bin[k] -= 1u << lg;
        eq[k] = q[k] == low[bin[k]] && (first + bin[k]) != 0;
    }
}

template <typename K, bool SECOND, int IT>
__global__ __launch_bounds__(PART_NT) void k_sort_count(
    const K *__restrict__ keys, uint64_t n, const K *__restrict__ bound, uint32_t lg1,
    uint32_t lg2, const uint32_t *__restrict__ bstart, const uint32_t *__restrict__ tstart,
    uint32_t tiles, uint32_t *__restrict__ counts, uint32_t *__restrict__ present) {
    __shared__ K spl[PART_BINS], low[PART_BINS];
    __shared__ uint32_t cnt[PART_BINS];
    const uint32_t lg = SECOND ? lg2 : lg1, B = 1u << lg, t = xcd_tile(tiles);
    if (t >= (SECOND ? tstart[1u << lg1] : tiles)) return;
    const PartTile p = part_tile<SECOND>(t, n, PART_NT * IT, lg1, lg2, bstart, tstart);
    K q[IT];
    uint32_t bin[IT];
    bool eq[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + threadIdx.x;
        q[k] = i < p.hi ? keys[i] : K{};
    }
    if (threadIdx.x < B) cnt[threadIdx.x] = 0;
    sort_splitters<K, SECOND>(bound, p, lg1, lg2, spl, low);
    __syncthreads();
    sort_buckets<K, IT>(q, spl, low, p.first, lg, bin, eq);
#pragma unroll
    for (int k = 0; k < IT; k++) {
        if (p.lo + k * PART_NT + threadIdx.x < p.hi) {
            if (eq[k])
                present[SECOND ? p.first + bin[k] : bin[k] << lg2] = 1;
            else
                atomicAdd(&cnt[bin[k]], 1u);
        }
    }
    __syncthreads();
    if (threadIdx.x < B) counts[(uint64_t)t * B + threadIdx.x] = cnt[threadIdx.x];
}

// every key that equals no splitter to its bucket, the tile in bucket order in
// LDS first (the places, then the keys), so that it is written in runs
template <typename K, bool SECOND, int IT>
__global__ __launch_bounds__(PART_NT) void k_sort_scatter(
    const K *__restrict__ keys, uint64_t n, const K *__restrict__ bound, uint32_t lg1,
    uint32_t lg2, const uint32_t *__restrict__ bstart, const uint32_t *__restrict__ tstart,
    uint32_t tiles, const uint32_t *__restrict__ places, const uint32_t *__restrict__ counts,
    K *__restrict__ out) {
    __shared__ K stage[PART_NT * IT];
    __shared__ uint32_t at[PART_BINS], local[PART_BINS];
    __shared__ uint32_t wsum[PART_NT / 64];
    K *spl = stage, *low = stage + PART_BINS;   // read before the stage is written
    uint32_t *stage_to = reinterpret_cast<uint32_t *>(stage);
    const uint32_t lg = SECOND ? lg2 : lg1, B = 1u << lg, tid = threadIdx.x, t = xcd_tile(tiles);
    if (t >= (SECOND ? tstart[1u << lg1] : tiles)) return;
    const PartTile p = part_tile<SECOND>(t, n, PART_NT * IT, lg1, lg2, bstart, tstart);
    K q[IT];
    uint32_t bin[IT], to[IT];
    bool eq[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        q[k] = i < p.hi ? keys[i] : K{};
    }
    sort_splitters<K, SECOND>(bound, p, lg1, lg2, spl, low);
    const uint32_t mine = tid < B ? counts[(uint64_t)t * B + tid] : 0u;
    uint32_t total;
    const uint32_t before = block_scan(mine, wsum, &total);
    if (tid < B) {
        local[tid] = before;
        at[tid] = places[(uint64_t)t * B + tid] - before;
    }
    __syncthreads();
    sort_buckets<K, IT>(q, spl, low, p.first, lg, bin, eq);
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        eq[k] |= p.lo + k * PART_NT + tid >= p.hi;   // not moved
        if (!eq[k]) {
            const uint32_t x = atomicAdd(&local[bin[k]], 1u);
            stage_to[x] = at[bin[k]] + x;
            bin[k] = x;
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t x = k * PART_NT + tid;
        to[k] = x < total ? stage_to[x] : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++)
        if (!eq[k]) stage[bin[k]] = q[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t x = k * PART_NT + tid;
        if (x < total) out[to[k]] = stage[x];
    }
}

// smallest / largest value of a wave, in every lane
template <typename U, bool LARGEST>
__device__ inline U wave_extreme(U v) {
    for (int o = 1; o < 64; o <<= 1) {
        U other = (U)(uint32_t)__shfl_xor((int)(uint32_t)v, o);
        if constexpr (sizeof(U) == 8)
            other |= (U)(uint32_t)__shfl_xor((int)(uint32_t)((uint64_t)v >> 32), o) << 32;
        v = LARGEST ? max(v, other) : min(v, other);
    }
    return v;
}

// Bucket j (rcount[j] keys at S[rstart[j]]) sorted in LDS, its distinct keys to
// the same place of out (which may be S), their number plus the splitter's
// presence to kept[j].  One counting pass over 2048 equal parts of the bucket's
// span leaves a key or two in each, which find their order by comparing.
// Buckets whose keys crowd are left (kept[j] = CROWDED) to a second launch,
// which sorts all their digits (and needs the registers for it), and those of more
// than RANGE_CAP keys (noted in large[]) to a third.
constexpr uint32_t CROWDED = ~0u;
template <typename K, bool CROWD_PASS>
__global__ __launch_bounds__(RANGE_NT) void k_sort_range(const K *S,
                                                         const uint32_t *__restrict__ rstart,
                                                         const uint32_t *__restrict__ rcount,
                                                         const uint32_t *__restrict__ present,
                                                         K *out, uint32_t *__restrict__ kept,
                                                         uint32_t *__restrict__ overflow,
                                                         uint32_t *__restrict__ nlarge,
                                                         uint32_t *__restrict__ large) {
    using U = Bits<K>;
    constexpr uint32_t CROWD = 32, NW = RANGE_NT / 64;
    __shared__ U buf[RANGE_CAP];
    __shared__ uint32_t bins[RANGE_BINS + 1], wsum[NW], wcount[RANGE_IT * NW];
    __shared__ U span[2 * NW];
    __shared__ uint32_t crowded;
    if (CROWD_PASS && kept[blockIdx.x] != CROWDED) return;
    const uint32_t j = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const uint32_t lo = rstart[j], cnt = rcount[j];
    if (cnt == 0 || cnt > RANGE_CAP) {
        if (tid == 0) {
            kept[j] = present[j];
            if (cnt > LARGE_CAP) *overflow = 1;
            else if (cnt) large[atomicAdd(nlarge, 1u)] = j;
        }
        return;
    }
    U x[RANGE_IT];
    uint32_t place[RANGE_IT];
    if (tid == 0) crowded = 0;
    for (uint32_t i = tid; i <= RANGE_BINS; i += RANGE_NT) bins[i] = 0;
    U least = ~(U)0, most = 0;
#pragma unroll
    for (uint32_t k = 0; k < RANGE_IT; k++) {
        if (k * RANGE_NT >= cnt) continue;   // the whole workgroup's, here and below
        const uint32_t i = k * RANGE_NT + tid;
        if (i < cnt) {
            x[k] = to_bits<K>(S[lo + i]);
            least = min(least, x[k]);
            most = max(most, x[k]);
        }
    }
    least = wave_extreme<U, false>(least);
    most = wave_extreme<U, true>(most);
    if (lane == 0) {
        span[w] = least;
        span[NW + w] = most;
    }
    __syncthreads();
    for (uint32_t ww = 0; ww < NW; ww++) {
        least = min(least, span[ww]);
        most = max(most, span[NW + ww]);
    }
    const U first = least;
    const uint64_t width = most - least;
    const uint32_t bits = width ? 64u - (uint32_t)__clzll((long long)width) : 0u;
    const uint32_t shift = bits > 11 ? bits - 11 : 0u;
#pragma unroll
    for (uint32_t k = 0; k < RANGE_IT; k++) {
        if (k * RANGE_NT >= cnt) continue;
        if (k * RANGE_NT + tid < cnt)
            place[k] = atomicAdd(&bins[(uint32_t)((U)(x[k] - first) >> shift)], 1u);
    }
    __syncthreads();
    {
        constexpr uint32_t PER = RANGE_BINS / RANGE_NT;
        uint32_t c[PER], sum = 0, top = 0;
#pragma unroll
        for (uint32_t k = 0; k < PER; k++) {
            c[k] = bins[tid * PER + k];
            sum += c[k];
            top = max(top, c[k]);
        }
        if (top > CROWD && shift) crowded = 1;
        uint32_t total;
        uint32_t run = block_scan(sum, wsum, &total);
#pragma unroll
        for (uint32_t k = 0; k < PER; k++) {
            bins[tid * PER + k] = run;
            run += c[k];
        }
        if (tid == 0) bins[RANGE_BINS] = cnt;
    }
    __syncthreads();
    if (!CROWD_PASS && crowded) {
        if (tid == 0) kept[j] = CROWDED;
        return;
    }
    if constexpr (CROWD_PASS) {
#pragma unroll
        for (uint32_t k = 0; k < RANGE_IT; k++) {
            const uint32_t i = k * RANGE_NT + tid;
            if (i < cnt) buf[i] = x[k];
        }
        __syncthreads();
        lds_sort<U, RANGE_NT, RANGE_IT>(buf, cnt, bins, wsum);
    } else {
#pragma unroll
        for (uint32_t k = 0; k < RANGE_IT; k++) {
            if (k * RANGE_NT >= cnt) continue;
            if (k * RANGE_NT + tid < cnt) {
                place[k] += bins[(uint32_t)((U)(x[k] - first) >> shift)];
                buf[place[k]] = x[k];
            }
        }
        __syncthreads();
    }
    if (!CROWD_PASS && shift) {   // a part holds keys that differ
#pragma unroll
        for (uint32_t k = 0; k < RANGE_IT; k++) {
            if (k * RANGE_NT >= cnt) continue;
            if (k * RANGE_NT + tid < cnt) {
                const uint32_t b = (uint32_t)((U)(x[k] - first) >> shift);
                const uint32_t s0 = bins[b], s1 = bins[b + 1];
                uint32_t at = s0;
                for (uint32_t i = s0; i < s1; i++) {
                    const U y = buf[i];
                    at += y < x[k] || (y == x[k] && i < place[k]) ? 1u : 0u;
                }
                place[k] = at;
            }
        }
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < RANGE_IT; k++) {
            if (k * RANGE_NT >= cnt) continue;
            if (k * RANGE_NT + tid < cnt) buf[place[k]] = x[k];
        }
        __syncthreads();
    }
    // distinct keys in order: 64 at a time, (k, wave) after (k, wave)
    bool keep[RANGE_IT];
#pragma unroll
    for (uint32_t k = 0; k < RANGE_IT; k++) {
        keep[k] = false;
        if (k * RANGE_NT >= cnt) {
            if (lane == 0) wcount[k * NW + w] = 0;
            continue;
        }
        const uint32_t i = k * RANGE_NT + tid;
        keep[k] = i < cnt;
        if (keep[k]) {
            x[k] = buf[i];
            keep[k] = i == 0 || x[k] != buf[i - 1];
        }
        const uint64_t m = __ballot(keep[k]);
        place[k] = (uint32_t)__popcll(m & ((1ull << lane) - 1));
        if (lane == 0) wcount[k * NW + w] = (uint32_t)__popcll(m);
    }
    __syncthreads();
    static_assert(RANGE_IT * NW <= 64, "one count a lane of a wave");
    uint32_t total;
    const uint32_t mine = tid < RANGE_IT * NW ? wcount[tid] : 0u;
    const uint32_t before = block_scan(mine, wsum, &total);
    if (tid < RANGE_IT * NW) wcount[tid] = before;
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < RANGE_IT; k++) {
        if (k * RANGE_NT >= cnt) continue;
        if (keep[k]) out[lo + wcount[k * NW + w] + place[k]] = from_bits<K>(x[k]);
    }
    if (tid == 0) kept[j] = total + present[j];
}

// The buckets of more than RANGE_CAP keys, LARGE_CAP at most: all their digits in
// the LDS of a whole compute unit.  Launched once the host knows that there are any.  A bucket or two of inputs whose average is
// near the goal: five of eight sets of 2*10^8 8-byte keys had one, and took 24.3 ms
// by the radix sort of everything where the others took 6.1; now 6.2 against 6.05.
template <typename K>
__global__ __launch_bounds__(LARGE_NT) void k_sort_large(const K *__restrict__ S,
                                                         const uint32_t *__restrict__ rstart,
                                                         const uint32_t *__restrict__ rcount,
                                                         const uint32_t *__restrict__ present,
                                                         K *__restrict__ out,
                                                         uint32_t *__restrict__ kept,
                                                         const uint32_t *__restrict__ nlarge,
                                                         const uint32_t *__restrict__ large) {
    using U = Bits<K>;
    constexpr uint32_t NW = LARGE_NT / 64;
    __shared__ U buf[LARGE_CAP];
    __shared__ uint32_t hist[NW * 256], wsum[NW], wcount[LARGE_IT * NW];
    const uint32_t tid = threadIdx.x, lane = tid & 63, w = tid >> 6, m = *nlarge;
    for (uint32_t l = blockIdx.x; l < m; l += gridDim.x) {
        const uint32_t j = large[l], lo = rstart[j], cnt = rcount[j];
        for (uint32_t i = tid; i < cnt; i += LARGE_NT) buf[i] = to_bits<K>(S[lo + i]);
        __syncthreads();
        lds_sort<U, LARGE_NT, LARGE_IT>(buf, cnt, hist, wsum);
        // distinct keys in order: 64 at a time, (k, wave) after (k, wave)
        uint32_t place[LARGE_IT];
        uint32_t keep = 0;
#pragma unroll
        for (uint32_t k = 0; k < LARGE_IT; k++) {
            const uint32_t i = k * LARGE_NT + tid;
            const bool first = i < cnt && (i == 0 || buf[i] != buf[i - 1]);
            const uint64_t peers = __ballot(first);
            place[k] = (uint32_t)__popcll(peers & ((1ull << lane) - 1));
            keep |= first ? 1u << k : 0u;
            if (lane == 0) wcount[k * NW + w] = (uint32_t)__popcll(peers);
        }
        __syncthreads();
        static_assert(LARGE_IT * NW <= LARGE_NT, "one count a lane");
        uint32_t total;
        const uint32_t mine = tid < LARGE_IT * NW ? wcount[tid] : 0u;
        const uint32_t before = block_scan(mine, wsum, &total);
        if (tid < LARGE_IT * NW) wcount[tid] = before;
        __syncthreads();
#pragma unroll
        for (uint32_t k = 0; k < LARGE_IT; k++)
            if (keep >> k & 1)
                out[lo + wcount[k * NW + w] + place[k]] = from_bits<K>(buf[k * LARGE_NT + tid]);
        if (tid == 0) kept[j] = total + present[j];
        __syncthreads();   // buf and wcount are the next bucket's
    }
}

// counts[j]: what became off[j] when it was scanned
__global__ __launch_bounds__(256) void k_sort_counts(const uint32_t *__restrict__ off,
                                                     uint32_t ranges, const uint32_t *sum,
                                                     uint32_t *__restrict__ counts) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < ranges) counts[j] = (j + 1 < ranges ? off[j + 1] : *sum) - off[j];
}

// the distinct keys of bucket j, behind its splitter where present, to
// off[j] .. of the result, unless buckets are yet to be sorted
template <typename K>
__global__ __launch_bounds__(256) void k_sort_close(const K *__restrict__ T,
                                                    const uint32_t *__restrict__ rstart,
                                                    const uint32_t *__restrict__ present,
                                                    const K *__restrict__ bound,
                                                    const uint32_t *__restrict__ off,
                                                    uint32_t ranges, const uint32_t *sum,
                                                    const uint32_t *__restrict__ overflow,
                                                    const uint32_t *__restrict__ nlarge,
                                                    K *__restrict__ keys) {
    if (*overflow || (nlarge && *nlarge)) return;
    const uint32_t j = blockIdx.x, o = off[j], lo = rstart[j], pre = present[j];
    const uint32_t c = (j + 1 < ranges ? off[j + 1] : *sum) - o - pre;
    if (pre && threadIdx.x == 0) keys[o] = bound[j];
    for (uint32_t i = threadIdx.x; i < c; i += 256) keys[o + pre + i] = T[lo + i];
}

// After an overflow: the splitters present back among the keys.  The first
// pass's go behind the *count partitioned keys; the second pass's into the gap
// that their keys left at the end of their bucket (what else the gap holds is
// still keys of the input).
template <typename K>
__global__ __launch_bounds__(1024) void k_sort_append(const uint32_t *__restrict__ present,
                                                      const K *__restrict__ bound, uint32_t lg1,
                                                      uint32_t lg2,
                                                      const uint32_t *__restrict__ rstart,
                                                      const uint32_t *__restrict__ rcount, K *dst,
                                                      uint32_t *count) {
    const uint32_t k = threadIdx.x, B2 = 1u << lg2;
    if (k >= (1u << lg1)) return;
    const uint32_t j0 = k << lg2, last = j0 + B2 - 1;
    if (present[j0]) dst[atomicAdd(count, 1u)] = bound[j0];
    uint32_t at = rstart[last] + rcount[last];
    for (uint32_t j = j0 + 1; j <= last; j++)
        if (present[j]) dst[at++] = bound[j];
}

__global__ void k_sort_range_of(uint32_t *rstart, uint32_t n, uint32_t *rcount,
                                uint32_t *present) {
    *rstart = 0;
    *rcount = n;
    *present = 0;
}

template <typename K, bool SECOND, int IT>
static void sort_pass(const K *in, K *out, uint64_t n, uint32_t lg1, uint32_t lg2, uint32_t tiles,
                      uint32_t groups, const K *bound, uint32_t *bstart, uint32_t *tstart,
                      uint32_t *rstart, uint32_t *rcount, uint32_t *gsum, uint32_t *counts,
                      uint32_t *places, uint32_t *present, hipStream_t s) {
    const dim3 grid((tiles + 7) / 8 * 8), block(PART_NT);
    hipLaunchKernelGGL((k_sort_count<K, SECOND, IT>), grid, block, 0, s, in, n, bound, lg1, lg2,
                       (const uint32_t *)bstart, (const uint32_t *)tstart, tiles, counts, present);
    if (SECOND) {
        hipLaunchKernelGGL(k_part_places2, dim3(1u << lg1), block, 0, s, (const uint32_t *)counts,
                           lg1, lg2, (const uint32_t *)bstart, (const uint32_t *)tstart, places,
                           rstart, rcount);
    } else {
        hipLaunchKernelGGL(k_part_sums, dim3(groups), block, 0, s, (const uint32_t *)counts,
                           1u << lg1, tiles, gsum);
        hipLaunchKernelGGL(k_part_starts, dim3(1), block, 0, s, gsum, 1u << lg1, groups,
                           (uint32_t)(PART_NT * IT), bstart, tstart,
                           lg2 ? (uint32_t *)nullptr : rcount);
        hipLaunchKernelGGL(k_part_places, dim3(groups), block, 0, s, (const uint32_t *)counts,
                           1u << lg1, tiles, (const uint32_t *)gsum, (const uint32_t *)bstart,
                           places);
    }
    hipLaunchKernelGGL((k_sort_scatter<K, SECOND, IT>), grid, block, 0, s, in, n, bound, lg1, lg2,
                       (const uint32_t *)bstart, (const uint32_t *)tstart, tiles,
                       (const uint32_t *)places, (const uint32_t *)counts, out);
}

template <typename K>
static void sort_ranges(const K *S, const uint32_t *rstart, const uint32_t *rcount,
                        const uint32_t *present, K *out, uint32_t *kept, uint32_t *overflow,
                        uint32_t *nlarge, uint32_t *large, uint32_t ranges, hipStream_t s) {
    hipLaunchKernelGGL((k_sort_range<K, false>), dim3(ranges), dim3(RANGE_NT), 0, s, S, rstart,
                       rcount, present, out, kept, overflow, nlarge, large);
    hipLaunchKernelGGL((k_sort_range<K, true>), dim3(ranges), dim3(RANGE_NT), 0, s, S, rstart,
                       rcount, present, out, kept, overflow, nlarge, large);
}

template <typename U>
static tl_status sort_dedupe_t(Ctx *c, U *keys, uint64_t n, U flip, uint64_t *n_out, hipStream_t s);

// sorts and drops repeats; n <= SPLIT_MAX_KEYS
template <typename K>
static tl_status split_sort(Ctx *c, K *keys, uint64_t n, uint64_t *n_out, hipStream_t s) {
    if (n <= 1) {
        *n_out = n;
        return TL_OK;
    }
    uint32_t lg = 1;
    while ((n >> lg) >= RANGE_GOAL) lg++;
    // few enough splitters a pass for their samples: 16 (2^10 of them) or 32 and
    // more each in the first, 32 (2^9) or more in the second
    const uint32_t lg1 = lg <= PART_LG ? lg : lg > SORT_LG1 + 9 ? lg - 9 : SORT_LG1;
    const uint32_t lg2 = lg - lg1, ranges = 1u << lg;
    const bool wide = n >= (1u << 22);   // queries per lane of a tile: 16, else 4
    const uint64_t T = (uint64_t)PART_NT * (wide ? 16 : 4);
    const uint32_t tiles1 = (uint32_t)((n + T - 1) / T), tiles2 = lg2 ? tiles1 + (1u << lg1) : 0;
    const uint32_t groups = (tiles1 + PART_GROUP - 1) / PART_GROUP;
    const uint64_t cells = std::max((uint64_t)tiles1 << lg1, (uint64_t)tiles2 << lg2);
    // scratch slot 5, each from a cache line on: overflow, a count and the number of
    // large buckets; bstart, tstart, rstart, rcount, present, kept and the sums of its
    // scan, the large buckets, gsum, counts, places; then the splitters
    const uint64_t B1 = (1ull << lg1) + 1, sums = ranges / SCAN_CHUNK + 3;
    const uint32_t most_large = (uint32_t)(n / RANGE_CAP);
    uint64_t words = 64;
    auto take = [&](uint64_t count) {
        const uint64_t at = words;
        words += (count + 63) & ~63ull;
        return at;
    };
    const uint64_t at_b = take(B1), at_t = take(B1), at_r = take(ranges + 1ull);
    const uint64_t at_rc = take(ranges), at_p = take(ranges), at_k = take(ranges);
    const uint64_t at_ks = take(sums), at_l = take(most_large);
    const uint64_t at_g = take((uint64_t)groups << lg1), at_c = take(cells), at_pl = take(cells);
    uint32_t *m = nullptr;
    TL_TRY(scratch(c, 5, words * 4 + (size_t)ranges * sizeof(K), (void **)&m));
    uint32_t *overflow = m, *count = m + 1, *nlarge = m + 2;
    uint32_t *bstart = m + at_b, *tstart = m + at_t, *rstart = lg2 ? m + at_r : bstart;
    uint32_t *rcount = m + at_rc, *present = m + at_p, *kept = m + at_k, *ksum = m + at_ks;
    uint32_t *large = m + at_l, *gsum = m + at_g, *counts = m + at_c, *places = m + at_pl;
    K *bound = (K *)(m + words);
    if (n <= RANGE_CAP) {   // one bucket, sorted where it is
        hipLaunchKernelGGL(k_sort_range_of, dim3(1), dim3(1), 0, s, bstart, (uint32_t)n, rcount,
                           present);
        sort_ranges<K>(keys, bstart, rcount, present, keys, kept, overflow, nlarge, large, 1, s);
        TL_LAUNCH_CHECK();
        uint32_t u = 0;
        TL_HIP(hipMemcpyAsync(&u, kept, 4, hipMemcpyDeviceToHost, s));
        TL_HIP(hipStreamSynchronize(s));
        *n_out = u;
        return TL_OK;
    }
    K *tmp = nullptr;
    TL_TRY(scratch(c, 4, n * sizeof(K), (void **)&tmp));
    TL_TRY(fill_u32_launch(m, 3, 0, s));
    TL_TRY(fill_u32_launch(present, ranges, 0, s));
    if (lg1 <= 8)
        hipLaunchKernelGGL((k_sort_sample<K, false, 8>), dim3(1), dim3(1024), 0, s,
                           (const K *)keys, n, lg1, lg2, (const uint32_t *)nullptr, bound);
    else
        hipLaunchKernelGGL((k_sort_sample<K, false, 16>), dim3(1), dim3(1024), 0, s,
                           (const K *)keys, n, lg1, lg2, (const uint32_t *)nullptr, bound);
    TL_LAUNCH_CHECK();
    K *sorted = tmp, *other = keys;   // the partitioned keys, and the other buffer
#define TL_SORT_PASS(SECOND, IT, in, out, tiles)                                                   \
    sort_pass<K, SECOND, IT>(in, out, n, lg1, lg2, tiles, groups, bound, bstart, tstart, rstart,   \
                             rcount, gsum, counts, places, present, s)
    if (wide) TL_SORT_PASS(false, 16, keys, tmp, tiles1);
    else TL_SORT_PASS(false, 4, keys, tmp, tiles1);
    TL_LAUNCH_CHECK();
    if (lg2) {
        if (lg2 <= 6)
            hipLaunchKernelGGL((k_sort_sample<K, true, 4>), dim3(1u << lg1), dim3(1024), 0, s,
                               (const K *)tmp, n, lg1, lg2, (const uint32_t *)bstart, bound);
        else
            hipLaunchKernelGGL((k_sort_sample<K, true, 16>), dim3(1u << lg1), dim3(1024), 0, s,
                               (const K *)tmp, n, lg1, lg2, (const uint32_t *)bstart, bound);
        if (wide) TL_SORT_PASS(true, 16, tmp, keys, tiles2);
        else TL_SORT_PASS(true, 4, tmp, keys, tiles2);
        TL_LAUNCH_CHECK();
        std::swap(sorted, other);
    }
#undef TL_SORT_PASS
    sort_ranges<K>(sorted, rstart, rcount, present, other, kept, overflow, nlarge, large, ranges,
                   s);
    TL_LAUNCH_CHECK();
    const uint32_t *sum = ksum + (ranges + SCAN_CHUNK - 1) / SCAN_CHUNK;
    // close the gaps into the buffer that held the partitioned keys
    auto close = [&](uint32_t *off, const uint32_t *unsorted) -> tl_status {
        TL_TRY(scan_u32(off, ranges, ksum, s));
        hipLaunchKernelGGL(k_sort_close<K>, dim3(ranges), dim3(256), 0, s, (const K *)other,
                           (const uint32_t *)rstart, (const uint32_t *)present, (const K *)bound,
                           (const uint32_t *)off, ranges, sum, (const uint32_t *)overflow,
                           unsorted, sorted);
        TL_LAUNCH_CHECK();
        return TL_OK;
    };
    TL_TRY(close(kept, nlarge));
    // overflow, a count, large buckets; keys partitioned (and the second pass's
    // gaps); distinct keys
    uint32_t w[3], h[3];
    TL_HIP(hipMemcpyAsync(w, overflow, 12, hipMemcpyDeviceToHost, s));
    TL_HIP(hipMemcpyAsync(&h[1], bstart + (1u << lg1), 4, hipMemcpyDeviceToHost, s));
    TL_HIP(hipMemcpyAsync(&h[2], sum, 4, hipMemcpyDeviceToHost, s));
    TL_HIP(hipStreamSynchronize(s));
    h[0] = w[0];
    if (!h[0] && w[2]) {
        hipLaunchKernelGGL(k_sort_counts, dim3((ranges + 255) / 256), dim3(256), 0, s,
                           (const uint32_t *)kept, ranges, sum, counts);
        hipLaunchKernelGGL(k_sort_large<K>, dim3(std::min<uint32_t>(w[2], c->num_cus)),
                           dim3(LARGE_NT), 0, s, (const K *)sorted, (const uint32_t *)rstart,
                           (const uint32_t *)rcount, (const uint32_t *)present, other, counts,
                           (const uint32_t *)nlarge, (const uint32_t *)large);
        TL_LAUNCH_CHECK();
        TL_TRY(close(counts, nullptr));
        TL_HIP(hipMemcpyAsync(&h[2], sum, 4, hipMemcpyDeviceToHost, s));
        TL_HIP(hipStreamSynchronize(s));
    }
    const uint64_t have = h[0] ? h[1] : h[2];
    if (sorted != keys && have)
        TL_HIP(hipMemcpyAsync(keys, sorted, have * sizeof(K), hipMemcpyDeviceToDevice, s));
    if (!h[0]) {
        *n_out = h[2];
        return TL_OK;
    }
    // a bucket was too large: the partitioned keys and the splitters present
    // hold every distinct key
    TL_TRY(fill_u32_launch(count, 1, h[1], s));
    hipLaunchKernelGGL(k_sort_append<K>, dim3(1), dim3(1024), 0, s, (const uint32_t *)present,
                       (const K *)bound, lg1, lg2, (const uint32_t *)rstart,
                       (const uint32_t *)rcount, keys, count);
    TL_LAUNCH_CHECK();
    uint32_t left = 0;
    TL_HIP(hipMemcpyAsync(&left, count, 4, hipMemcpyDeviceToHost, s));
    TL_HIP(hipStreamSynchronize(s));
    const Bits<K> flip = (K)-1 < (K)0 ? (Bits<K>)1 << (8 * sizeof(K) - 1) : 0;
    return sort_dedupe_t<Bits<K>>(c, (Bits<K> *)keys, left, flip, n_out, s);
}

template <typename U>
static tl_status sort_dedupe_t(Ctx *c, U *keys, uint64_t n, U flip, uint64_t *n_out,
                               hipStream_t s) {
    if (n <= 1) {
        *n_out = n;
        return TL_OK;
    }
    const uint64_t tiles = (n + SORT_TILE - 1) / SORT_TILE;
    const uint64_t clen = 256 * tiles;
    const uint64_t csums = (clen + SCAN_CHUNK - 1) / SCAN_CHUNK + 2;
    U *tmp = nullptr;
    TL_TRY(scratch(c, 4, n * sizeof(U), (void **)&tmp));
    uint32_t *counts = nullptr;
    // counts, scan sums, and the AND/OR words (16-byte aligned at the end)
    const size_t cbytes = (clen + csums) * 4;
    TL_TRY(scratch(c, 5, cbytes + 64, (void **)&counts));
    uint32_t *sums = counts + clen;
    unsigned long long *andor =
        (unsigned long long *)(((uintptr_t)(counts + clen + csums) + 15) & ~(uintptr_t)15);
    const unsigned long long init[2] = {~0ull, 0ull};
    TL_HIP(hipMemcpyAsync(andor, init, sizeof(init), hipMemcpyHostToDevice, s));
    const uint32_t g = (uint32_t)std::min<uint64_t>((n + 255) / 256, (uint64_t)c->num_cus * 8);
    hipLaunchKernelGGL(k_and_or<U>, dim3(g), dim3(256), 0, s, (const U *)keys, n, flip, andor);
    TL_LAUNCH_CHECK();
    unsigned long long ao[2];
    TL_HIP(hipMemcpyAsync(ao, andor, sizeof(ao), hipMemcpyDeviceToHost, s));
    TL_HIP(hipStreamSynchronize(s));
    const uint64_t varies = (uint64_t)(ao[0] ^ ao[1]);   // bits not equal across all keys
    U *src = keys, *dst = tmp;
    for (uint32_t shift = 0; shift < 8 * sizeof(U); shift += 8) {
        if (((varies >> shift) & 0xFF) == 0) continue;   // one digit value: nothing to move
        hipLaunchKernelGGL(k_radix_hist<U>, dim3((uint32_t)tiles), dim3(SORT_THREADS), 0, s,
                           (const U *)src, n, shift, flip, counts, (uint32_t)tiles);
        TL_LAUNCH_CHECK();
        TL_TRY(scan_u32(counts, clen, sums, s));
        hipLaunchKernelGGL(k_radix_scatter<U>, dim3((uint32_t)tiles), dim3(SORT_THREADS), 0, s,
                           (const U *)src, dst, n, shift, flip, (const uint32_t *)counts,
                           (uint32_t)tiles);
        TL_LAUNCH_CHECK();
        std::swap(src, dst);
    }
    // drop repeats: sorted src -> dst
    hipLaunchKernelGGL(k_unique_count<U>, dim3((uint32_t)tiles), dim3(SORT_THREADS), 0, s,
                       (const U *)src, n, counts);
    TL_LAUNCH_CHECK();
    TL_TRY(scan_u32(counts, tiles, sums, s));
    hipLaunchKernelGGL(k_unique_scatter<U>, dim3((uint32_t)tiles), dim3(SORT_THREADS), 0, s,
                       (const U *)src, dst, n, (const uint32_t *)counts);
    TL_LAUNCH_CHECK();
    uint32_t m = 0;
    const uint64_t chunks = (tiles + SCAN_CHUNK - 1) / SCAN_CHUNK;
    TL_HIP(hipMemcpyAsync(&m, sums + chunks, 4, hipMemcpyDeviceToHost, s));
    TL_HIP(hipStreamSynchronize(s));
    if (dst != keys && m)
        TL_HIP(hipMemcpyAsync(keys, dst, (size_t)m * sizeof(U), hipMemcpyDeviceToDevice, s));
    *n_out = m;
    return TL_OK;
}

}   // namespace tl

extern "C" tl_status tl_sort_dedupe(void *dev_keys, uint64_t n, tl_dtype dtype, uint64_t *n_out,
                                    void *stream, float *ms) {
    using namespace tl;
    uint32_t W;
    if (!width_of(dtype, W)) {
        set_error("unknown dtype");
        return TL_EINVAL;
    }
    if (!n_out || (n > 1 && !dev_keys)) {
        set_error("tl_sort_dedupe: null pointer");
        return TL_EINVAL;
    }
    if (n >= (1ull << 32)) {
        set_error("tl_sort_dedupe: n must be below 2^32");
        return TL_EINVAL;
    }
    Ctx *c;
    TL_TRY(get_ctx(&c));
    hipStream_t s = (hipStream_t)stream;
    Timer tm;
    TL_TRY(tm.start(s, ms));
    tl_status st = TL_ENOMEM;
    if (n <= SPLIT_MAX_KEYS && !(getenv("TL_SORT_RADIX") && atoi(getenv("TL_SORT_RADIX")) == 1)) {
        switch (dtype) {
        case TL_U32: st = split_sort<uint32_t>(c, (uint32_t *)dev_keys, n, n_out, s); break;
        case TL_U64: st = split_sort<uint64_t>(c, (uint64_t *)dev_keys, n, n_out, s); break;
        case TL_I32: st = split_sort<int32_t>(c, (int32_t *)dev_keys, n, n_out, s); break;
        default: st = split_sort<int64_t>(c, (int64_t *)dev_keys, n, n_out, s); break;
        }
    }
    // the radix sort's tables are a quarter of the splitters' at 2^29 keys
    if (st == TL_ENOMEM && W == 4) {
        const uint32_t flip = dtype == TL_I32 ? 0x80000000u : 0u;
        st = sort_dedupe_t<uint32_t>(c, (uint32_t *)dev_keys, n, flip, n_out, s);
    } else if (st == TL_ENOMEM) {
        const uint64_t flip = dtype == TL_I64 ? 0x8000000000000000ull : 0ull;
        st = sort_dedupe_t<uint64_t>(c, (uint64_t *)dev_keys, n, flip, n_out, s);
    }
    if (st != TL_OK) return st;
    TL_TRY(tm.stop());
    return TL_OK;
}
