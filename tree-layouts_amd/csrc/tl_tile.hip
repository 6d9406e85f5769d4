// tl_tile.hip -- lookups of large query batches, for gfx950.
//
// One lane per query, a tile of queries per workgroup.  What bounds such a
// descent is not the bytes: every load of an unsorted wave touches 64
// different cache lines, which the vector cache takes one a clock, and every
// step costs its vector instructions.  So a workgroup first puts its tile in
// approximate key order (1024 buckets split at equal ranks of the array, one
// counting sort in LDS), after which the lanes of a wave walk neighbouring
// paths: their loads fall into few lines on all but the last levels.  The
// descents then run level by level in lock step, with 32-bit positions and
// nothing per lane but the compare, the step and the hit.
//
// The path taken through the layout, and so the answer, is the one of the
// one-array kernels in tl_query.hip for every query: the first key equal to q
// on the descent, also where keys repeat.
//
// Arrays well past the caches are served by the partitioned form below: there
// every unsorted descent waits for lines from memory, however its tile is
// ordered.  Measured (queries of keys that are there, before -> now):
//   BST 2^20 4-byte keys, 2^20 queries          41 -> 28 us (tile)
//   B-tree b=16, 2^30 8-byte keys, 2^27         10.5 -> 4.84 ms (partition)
//   BST, the same                               28.5 -> 5.3 ms (partition)
//   mvEB 3*10^8 8-byte keys, 2^26, Zipf(1.1)    5.58 -> 3.08 ms (partition)
#include <math.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include <algorithm>
#include <type_traits>

#include "tl_descent.hpp"
#include "tl_internal.hpp"
#include "tl_partition.hpp"
#include "tl_slots.hpp"
#include "tl_tile.hpp"

namespace tl {

constexpr uint32_t TILE_BINS = 1024;
constexpr uint32_t TILE_TABLES = 256;   // vEB table entries kept in LDS

constexpr uint32_t RANGE_KEYS = 4096;   // keys of a range, at most (partitioned lookups)

struct TileShape : SlotShape {
    uint32_t nodes;         // TILE_BTREE
    uint32_t levels;        // full levels: of the binary tree, or of nodes
    uint32_t table_size, ntables;
    const tl_veb_table *tables;
    const uint64_t *idx;
    const uint32_t *tidx;
    uint32_t small_mul, small_shift;   // x / (b + 1) = x * mul >> shift, x < 2 RANGE_KEYS
};

struct VebEntry {
    uint32_t L, R, D;
};

// ---- the descents of QN queries of a lane.  res[k]: the slot, or n.

// level-order BST, 1-based node m at A[m - 1]
template <typename K, int QN>
__device__ inline void tile_bst(const K *__restrict__ A, const TileShape &s, const K (&q)[QN],
                                uint32_t (&res)[QN]) {
    uint32_t m[QN], hit[QN];
#pragma unroll
    for (int k = 0; k < QN; k++) {
        m[k] = 1;
        hit[k] = ~0u;
    }
    for (uint32_t t = 0; t < s.levels; t++) {
        K v[QN];
#pragma unroll
        for (int k = 0; k < QN; k++) v[k] = A[m[k] - 1];
#pragma unroll
        for (int k = 0; k < QN; k++) {
            // node numbers grow along the path: the smallest equal one is the first
            if (v[k] == q[k]) hit[k] = min(hit[k], m[k]);
            m[k] = 2 * m[k] + (q[k] > v[k] ? 1u : 0u);
        }
    }
    K v[QN];
#pragma unroll
    for (int k = 0; k < QN; k++)
        if (m[k] <= s.n) v[k] = A[m[k] - 1];
#pragma unroll
    for (int k = 0; k < QN; k++) {
        if (m[k] <= s.n && v[k] == q[k]) hit[k] = min(hit[k], m[k]);
        res[k] = hit[k] == ~0u ? s.n : hit[k] - 1;
    }
}

// level-order B-tree: a branch-free lower bound in every node.  The key at
// the lower bound is the last one compared that was not smaller, so its
// equality needs no load of its own.
template <typename K, int QN>
__device__ inline void tile_btree(const K *__restrict__ A, const TileShape &s, const K (&q)[QN],
                                  uint32_t (&res)[QN]) {
    const uint32_t b = s.b, n = s.n;
    uint32_t node[QN];
#pragma unroll
    for (int k = 0; k < QN; k++) {
        node[k] = 0;
        res[k] = n;
    }
    // the nodes of the full levels are whole; of the last level a node may
    // be short (slots at or past n count as larger than every key) or absent
    for (uint32_t t = 0; t <= s.levels; t++) {
        const bool last = t == s.levels;
        uint32_t at[QN];
        bool eq[QN], in[QN];
#pragma unroll
        for (int k = 0; k < QN; k++) {
            in[k] = !last || node[k] < s.nodes;
            at[k] = in[k] ? node[k] * b : 0u;
            eq[k] = false;
        }
        for (uint32_t len = b; len > 0;) {
            const uint32_t half = (len + 1) >> 1;
            K v[QN];
#pragma unroll
            for (int k = 0; k < QN; k++) v[k] = A[min(at[k] + half, n) - 1];
#pragma unroll
            for (int k = 0; k < QN; k++) {
                const bool less = v[k] < q[k] && (!last || at[k] + half <= n);
                const bool same = v[k] == q[k] && (!last || at[k] + half <= n);
                eq[k] = less ? eq[k] : same;
                at[k] += less ? half : 0u;
            }
            len -= half;
        }
#pragma unroll
        for (int k = 0; k < QN; k++) {
            const uint32_t js = at[k] - node[k] * b;
            if (in[k] && eq[k] && res[k] == n) res[k] = at[k];
            node[k] = node[k] * (b + 1) + 1 + js;
        }
    }
}

// vEB (tables of either split): structure after structure, every lane at the
// same depth, so the table entries are the wave's.  The position at depth t
// is 1 + the sum of R + (bfs & R) * L over t, D[t], D[D[t]], .. (bfs shifted
// to that depth): no per-lane position stack.
template <typename K, int QN>
__device__ inline void tile_veb(const K *__restrict__ A, const TileShape &s, const VebEntry *tb,
                                const uint32_t *s_end, const uint16_t *s_tidx, const K (&q)[QN],
                                uint32_t (&res)[QN]) {
    const uint32_t n = s.n;
    bool pend[QN];
#pragma unroll
    for (int k = 0; k < QN; k++) {
        pend[k] = true;
        res[k] = n;
    }
    uint32_t off = 0;
    for (uint32_t j = 0; j < s.ntables; j++) {
        const uint32_t end = s_end[j];
        if (off >= end) continue;
        const uint32_t d = 32u - (uint32_t)__clz((int)(n - off));
        const VebEntry *e = tb + s_tidx[j];
        bool act[QN], any = false;
        uint32_t bfs[QN], at[QN];
#pragma unroll
        for (int k = 0; k < QN; k++) {
            act[k] = pend[k];
            pend[k] = false;
            any |= act[k];
            bfs[k] = 1;
            at[k] = off;
        }
        if (!__any(any)) break;
        for (uint32_t t = 1;; t++) {
            K v[QN];
#pragma unroll
            for (int k = 0; k < QN; k++)
                if (act[k]) v[k] = A[at[k]];
#pragma unroll
            for (int k = 0; k < QN; k++) {
                if (act[k] && v[k] == q[k]) {
                    res[k] = at[k];
                    act[k] = false;
                }
                bfs[k] = 2 * bfs[k] + (act[k] && q[k] > v[k] ? 1u : 0u);
                at[k] = off;
            }
            if (t >= d) break;
            for (uint32_t x = t; x != 0;) {
                const uint32_t L = e[x].L, R = e[x].R, D = e[x].D;
#pragma unroll
                for (int k = 0; k < QN; k++) at[k] += R + ((bfs[k] >> (t - x)) & R) * L;
                x = D < x ? D : 0u;
            }
            any = false;
#pragma unroll
            for (int k = 0; k < QN; k++) {
                if (act[k] && at[k] >= end) {   // in a later structure
                    act[k] = false;
                    pend[k] = true;
                }
                any |= act[k];
            }
            if (!__any(any)) break;
        }
        off = end;
    }
}

// binary search of the sorted array: the last key <= q (tl_query.hip's
// window steps), or n where every key is larger
template <typename K, int QN>
__device__ inline void tile_sorted(const K *__restrict__ A, const TileShape &s, const K (&q)[QN],
                                   uint32_t (&res)[QN]) {
    const K first = A[0];
#pragma unroll
    for (int k = 0; k < QN; k++) res[k] = 0;
    for (uint32_t len = s.n; len > 1;) {
        const uint32_t half = len >> 1;
        K v[QN];
#pragma unroll
        for (int k = 0; k < QN; k++) v[k] = A[res[k] + half];
#pragma unroll
        for (int k = 0; k < QN; k++) res[k] += v[k] <= q[k] ? half : 0u;
        len -= half;
    }
#pragma unroll
    for (int k = 0; k < QN; k++)
        if (res[k] == 0 && !(first <= q[k])) res[k] = s.n;
}

// ---- the kernel

template <typename K, int LAYOUT, int QN>
__device__ inline void tile_descend(const K *__restrict__ A, const TileShape &s,
                                    const VebEntry *tb, const uint32_t *s_end,
                                    const uint16_t *s_tidx, const K (&q)[QN],
                                    uint32_t (&res)[QN]) {
    if constexpr (LAYOUT == TILE_BST)
        tile_bst<K, QN>(A, s, q, res);
    else if constexpr (LAYOUT == TILE_BTREE)
        tile_btree<K, QN>(A, s, q, res);
    else if constexpr (LAYOUT == TILE_VEB)
        tile_veb<K, QN>(A, s, tb, s_end, s_tidx, q, res);
    else
        tile_sorted<K, QN>(A, s, q, res);
}

constexpr int TILE_NT = 512;   // lanes per workgroup
constexpr int TILE_QN = 4;     // descents of a lane in flight

// IT queries per lane, tiles of NT * IT.  Workgroups go round robin to the 8
// XCDs; each XCD takes one run of consecutive tiles (neighbouring tiles of a
// batch in key order share their cache lines in one L2).
template <typename K, int LAYOUT, int IT>
__global__ __launch_bounds__(TILE_NT) void k_query_tile(const K *__restrict__ A, TileShape s,
                                                        const K *__restrict__ Q, uint64_t nq,
                                                        uint64_t *__restrict__ ans,
                                                        uint32_t tiles) {
    constexpr uint32_t T = TILE_NT * IT;
    __shared__ K spl[TILE_BINS];               // heap order, node 1 the root
    __shared__ uint32_t bins[TILE_BINS];
    __shared__ uint32_t wsum[TILE_NT / 64];
    __shared__ K keys[T];                      // the tile in bucket order; then its answers
    __shared__ uint16_t from[T];               // place in the tile of each sorted query
    __shared__ VebEntry tb[LAYOUT == TILE_VEB ? TILE_TABLES : 1];
    __shared__ uint32_t s_end[64];
    __shared__ uint16_t s_tidx[64];
    uint32_t *answers = reinterpret_cast<uint32_t *>(keys);
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    __shared__ SlotMap<LAYOUT> map;
    slot_map<LAYOUT>(s, map);
    {
        for (uint32_t i = tid; i < TILE_BINS; i += TILE_NT) {
            if (i == 0) continue;
            spl[i] = A[slot_of<LAYOUT>(range_first(heap_order(i, 10), s.n, 10), s, map)];
        }
        if constexpr (LAYOUT == TILE_VEB) {
            for (uint32_t i = tid; i < s.table_size; i += TILE_NT)
                tb[i] = {(uint32_t)s.tables[i].L, (uint32_t)s.tables[i].R, s.tables[i].D};
            if (tid < s.ntables) {
                s_end[tid] = s.idx ? (uint32_t)s.idx[tid] : s.n;
                s_tidx[tid] = s.tidx ? (uint16_t)s.tidx[tid] : (uint16_t)0;
            }
        }
    }
    const uint32_t per = (tiles + 7) >> 3, step = gridDim.x >> 3;
    for (uint32_t loc = blockIdx.x >> 3; loc < per; loc += step) {
        const uint32_t tile = (blockIdx.x & 7) * per + loc;
        if (tile >= tiles) break;
        const uint64_t base = (uint64_t)tile * T;
        const uint32_t cnt = (uint32_t)min((uint64_t)T, nq - base);
        for (uint32_t i = tid; i < TILE_BINS; i += TILE_NT) bins[i] = 0;
        __syncthreads();
        K qv[IT];
        uint32_t place[IT];   // bucket, then rank within it above bit 10
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const uint32_t i = k * TILE_NT + tid;
            qv[k] = i < cnt ? Q[base + i] : K{};
        }
#pragma unroll
        for (int k = 0; k < IT; k++) place[k] = 1;
        for (int t = 0; t < 10; t++) {
#pragma unroll
            for (int k = 0; k < IT; k++)
                place[k] = 2 * place[k] + (qv[k] >= spl[place[k]] ? 1u : 0u);
        }
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const uint32_t bin = place[k] - TILE_BINS;
            const uint32_t i = k * TILE_NT + tid;
            if (i < cnt) place[k] = bin | (atomicAdd(&bins[bin], 1u) << 10);
        }
        __syncthreads();
        {   // exclusive scan of the bucket counts, two a lane
            const uint32_t a = bins[2 * tid], c = bins[2 * tid + 1];
            uint32_t x = a + c;
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t y = (uint32_t)__shfl_up((int)x, (unsigned)o);
                if (lane >= (uint32_t)o) x += y;
            }
            if (lane == 63) wsum[wave] = x;
            __syncthreads();
            uint32_t before = x - a - c;
            for (uint32_t w = 0; w < wave; w++) before += wsum[w];
            bins[2 * tid] = before;
            bins[2 * tid + 1] = before + a;
        }
        __syncthreads();
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const uint32_t i = k * TILE_NT + tid;
            if (i < cnt) {
                const uint32_t p = bins[place[k] & (TILE_BINS - 1)] + (place[k] >> 10);
                keys[p] = qv[k];
                from[p] = (uint16_t)i;
            }
        }
        __syncthreads();
        // a wave takes 64 * IT consecutive queries of the order
        uint32_t src[IT];
#pragma unroll
        for (int k = 0; k < IT; k++) {
            const uint32_t p = min((wave * IT + k) * 64 + lane, cnt - 1);
            qv[k] = keys[p];
            src[k] = from[p];
        }
        __syncthreads();   // keys[] becomes the answers
#pragma unroll
        for (int k0 = 0; k0 < IT; k0 += TILE_QN) {
            K q[TILE_QN];
            uint32_t res[TILE_QN];
#pragma unroll
            for (int k = 0; k < TILE_QN; k++) q[k] = qv[k0 + k];
            tile_descend<K, LAYOUT, TILE_QN>(A, s, tb, s_end, s_tidx, q, res);
#pragma unroll
            for (int k = 0; k < TILE_QN; k++)
                if ((wave * IT + k0 + k) * 64 + lane < cnt) answers[src[k0 + k]] = res[k];
        }
        __syncthreads();
        for (uint32_t i = tid; i < cnt; i += TILE_NT) ans[base + i] = answers[i];
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// partitioned lookups: batches of at least a few queries per array line.
//
// (2^27 queries of 2^30 8-byte keys move 10 GB in the answering kernel, 2.4 ms;
// the first pass of the queries takes 0.5 ms to count, 0.6 to scatter and 0.55
// for the way back, the last 0.6 and 0.25.)
//
// The array is cut into 2^lg ranges of equal rank count, each small enough
// for LDS.  The queries are put in range order tile by tile (where there are
// more ranges than a tile has counters, they are partitioned into 2^lg1 buckets
// first, whole), each workgroup then reads a range's keys once, coalesced, and
// answers the range's queries of many tiles from LDS, and the answers go back to
// the order of the queries.  So the array is read once where the descents of
// unsorted queries miss the caches on every level past the top ones.  A tile
// keeps its own order to itself: no counts over all tiles, no second read of the
// queries, contiguous reads on the way back.

constexpr uint32_t RANGE_NT = 512;

// whether the caller's vEB table set is the one of this layout (the whole
// workgroup calls it): of every structure, a wave each, the end and, level by
// level, the L, R and D that the splits give
__device__ inline bool veb_tables_match(const TileShape &s) {
    __shared__ uint32_t differs;
    if (threadIdx.x == 0) differs = 0;
    __syncthreads();
    bool same = true;
    auto keys_of = [&](uint32_t j) {   // of structure j, up to the next
        const VebLevel e = s.chain[j];
        return (1u << e.rd) - 1 + e.nf * ((1u << e.ld) - 1);
    };
    uint32_t off = 0, i = 0;
    for (uint32_t j = threadIdx.x >> 6; j < s.ntables; j += blockDim.x >> 6) {
        for (; i < j; i++) off += keys_of(i);
        const uint32_t end = j + 1 < s.ntables ? off + keys_of(j) : s.n;
        const uint32_t d = 32u - (uint32_t)__clz((int)(s.n - off));
        const uint32_t at = s.tidx ? s.tidx[j] : 0u;
        if (off >= end || (s.idx ? s.idx[j] : s.n) != end || (uint64_t)at + d > s.table_size) {
            same = false;
            break;
        }
        const uint32_t t = threadIdx.x & 63;
        if (t >= 1 && t < d) {
            uint32_t base = 0, levels = d, rd, ld;
            for (;;) {   // down to the tree whose bottom trees start at level t
                veb_split(levels, rd, ld, s.classic != 0);
                if (t == base + rd) break;
                levels = t < base + rd ? rd : ld;
                base += t < base + rd ? 0u : rd;
            }
            const tl_veb_table e = s.tables[at + t];
            same = same && e.L == (1ull << ld) - 1 && e.R == (1ull << rd) - 1 && e.D == base;
        }
    }
    if (!same) differs = 1;
    __syncthreads();
    return !differs;
}

// bound[j]: the smallest key of range j; the queue is empty.  queued[1]: a vEB's
// table set is another layout's than the call's (the answers then follow the
// tables, as those of every other path do); the last workgroup finds that out.
template <typename W, int LAYOUT>
__global__ __launch_bounds__(256) void k_part_bounds(const W *__restrict__ A, TileShape s,
                                                     uint32_t lg, W *__restrict__ bound,
                                                     uint32_t *queued) {
    __shared__ SlotMap<LAYOUT> map;
    if (blockIdx.x + 1 == gridDim.x) {
        bool same = true;
        if constexpr (LAYOUT == TILE_VEB) same = veb_tables_match(s);
        if (threadIdx.x == 0) {
            queued[0] = 0;
            queued[1] = same ? 0u : 1u;
        }
        return;
    }
    slot_map<LAYOUT>(s, map);
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < (1u << lg)) bound[j] = A[slot_of<LAYOUT>(range_first(j, s.n, lg), s, map)];
}

// Counts of a tile's queries per bucket (counts[t][bucket]); every query's
// bucket and rank among the tile's queries of it go to pack[].
template <typename K, int IT>
__global__ __launch_bounds__(PART_NT) void k_part_count(
    const K *__restrict__ Q, uint64_t nq, const K *__restrict__ bound, uint32_t lg1, uint32_t lg2,
    uint32_t tiles, uint32_t *__restrict__ pack, uint32_t *__restrict__ counts) {
    __shared__ K spl[PART_BINS];
    __shared__ uint32_t cnt[PART_BINS];
    const uint32_t lg = lg1, B = 1u << lg, step = 1u << lg2;
    const uint32_t t = xcd_tile(tiles);
    if (t >= tiles) return;
    const PartTile p = part_tile<false>(t, nq, PART_NT * IT, 0, 0, nullptr, nullptr);
    K q[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + threadIdx.x;
        q[k] = i < p.hi ? Q[i] : K{};
    }
    if (threadIdx.x < B) {
        cnt[threadIdx.x] = 0;
        if (threadIdx.x)
            spl[threadIdx.x] = bound[(uint64_t)heap_order(threadIdx.x, lg) * step];
    }
    __syncthreads();
    uint32_t node[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) node[k] = 1;
    for (uint32_t l = 0; l < lg; l++) {
#pragma unroll
        for (int k = 0; k < IT; k++) node[k] = 2 * node[k] + (q[k] >= spl[node[k]] ? 1u : 0u);
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + threadIdx.x;
        if (i < p.hi) {
            const uint32_t bin = node[k] - B;
            pack[i] = bin | (atomicAdd(&cnt[bin], 1u) << PART_LG);
        }
    }
    __syncthreads();
    if (threadIdx.x < B) counts[(uint64_t)t * B + threadIdx.x] = cnt[threadIdx.x];
}

// Every query to its place.  The tile is put in bucket order in LDS first (the
// places, then the queries, through one buffer), so that a bucket's queries leave
// as one run: written from where they were read, single queries filled cache
// lines so slowly that most were written back several times (5.8 GB for 2^27 8-byte queries, where 1.6 GB
// are written now).
template <typename K, int IT>
__global__ __launch_bounds__(PART_NT) void k_part_scatter(
    const K *__restrict__ Q, uint64_t nq, uint32_t lg1, uint32_t tiles,
    const uint32_t *__restrict__ places, const uint32_t *__restrict__ counts,
    const uint32_t *__restrict__ pack, K *__restrict__ out) {
    __shared__ K stage[PART_NT * IT];
    __shared__ uint32_t at[PART_BINS], local[PART_BINS];
    __shared__ uint32_t wsum[PART_NT / 64];
    uint32_t *stage_to = reinterpret_cast<uint32_t *>(stage);
    const uint32_t B = 1u << lg1, tid = threadIdx.x;
    const uint32_t t = xcd_tile(tiles);
    if (t >= tiles) return;
    const PartTile p = part_tile<false>(t, nq, PART_NT * IT, 0, 0, nullptr, nullptr);
    const uint32_t cnt = (uint32_t)(p.hi - p.lo);
    K q[IT];
    uint32_t pk[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        q[k] = i < p.hi ? Q[i] : K{};
        pk[k] = i < p.hi ? pack[i] : 0u;
    }
    const uint32_t mine = tid < B ? counts[(uint64_t)t * B + tid] : 0u;
    uint32_t total;
    const uint32_t before = block_scan(mine, wsum, &total);
    if (tid < B) {
        local[tid] = before;
        at[tid] = places[(uint64_t)t * B + tid] - before;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        if (i < p.hi) {
            const uint32_t bin = pk[k] & (PART_BINS - 1);
            const uint32_t x = local[bin] + (pk[k] >> PART_LG);   // place in the tile
            pk[k] = x;
            stage_to[x] = at[bin] + x;
        }
    }
    __syncthreads();
    uint32_t to[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t x = k * PART_NT + tid;
        to[k] = x < cnt ? stage_to[x] : 0u;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++)
        if (p.lo + k * PART_NT + tid < p.hi) stage[pk[k]] = q[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t x = k * PART_NT + tid;
        if (x < cnt) out[to[k]] = stage[x];
    }
}

// The way back: dst[i] = src[place of query i], tile by tile as they were
// scattered, the runs read into LDS whole (read one by one from there, 2^27
// answers took 0.72 ms; the vector cache passes on one line a lane).
template <int IT>
__global__ __launch_bounds__(PART_NT) void k_part_return(
    const uint32_t *__restrict__ src, uint64_t nq, uint32_t lg1, uint32_t tiles,
    const uint32_t *__restrict__ places, const uint32_t *__restrict__ counts,
    const uint32_t *pack, uint64_t *dst) {
    __shared__ uint32_t stage[PART_NT * IT];
    __shared__ uint32_t at[PART_BINS], local[PART_BINS];
    __shared__ uint32_t wsum[PART_NT / 64];
    const uint32_t B = 1u << lg1, tid = threadIdx.x;
    const uint32_t t = xcd_tile(tiles);
    if (t >= tiles) return;
    const PartTile p = part_tile<false>(t, nq, PART_NT * IT, 0, 0, nullptr, nullptr);
    const uint32_t cnt = (uint32_t)(p.hi - p.lo);
    uint32_t pk[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        pk[k] = i < p.hi ? pack[i] : 0u;
    }
    const uint32_t mine = tid < B ? counts[(uint64_t)t * B + tid] : 0u;
    uint32_t total;
    const uint32_t before = block_scan(mine, wsum, &total);
    if (tid < B) {
        local[tid] = before;
        at[tid] = places[(uint64_t)t * B + tid] - before;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t bin = pk[k] & (PART_BINS - 1);
        const uint32_t x = local[bin] + (pk[k] >> PART_LG);
        if (p.lo + k * PART_NT + tid < p.hi) stage[x] = at[bin] + x;
        pk[k] = x;
    }
    __syncthreads();
    uint32_t v[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t x = k * PART_NT + tid;
        v[k] = x < cnt ? src[stage[x]] : 0u;
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {   // a lane's own places
        const uint32_t x = k * PART_NT + tid;
        if (x < cnt) stage[x] = v[k];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        if (i < p.hi) dst[i] = stage[pk[k]];
    }
}

template <typename K>
__device__ inline K key_max() {
    const K half = (K)1 << (8 * sizeof(K) - 2);
    return (K)-1 > (K)0 ? (K)-1 : (K)(half - 1 + half);
}

// The last pass (the only one of lg1 buckets where !SECOND): a tile's queries in
// range order to the tile's own place, each query's place in the tile to
// place[], and the places of the ranges' first ones to loc[t][range].
template <typename K, bool SECOND, int IT>
__global__ __launch_bounds__(PART_NT) void k_part_tile(
    const K *__restrict__ Q, uint64_t nq, const K *__restrict__ bound, uint32_t lg1, uint32_t lg2,
    const uint32_t *__restrict__ bstart, const uint32_t *__restrict__ tstart, uint32_t tiles,
    uint16_t *__restrict__ place, uint16_t *__restrict__ loc, K *__restrict__ out) {
    __shared__ K stage[PART_NT * IT];
    __shared__ uint32_t cnt[PART_BINS];
    __shared__ uint32_t wsum[PART_NT / 64];
    K *spl = stage;   // read before the stage is written
    const uint32_t lg = SECOND ? lg2 : lg1, B = 1u << lg, tid = threadIdx.x;
    const uint32_t t = xcd_tile(tiles);
    if (t >= (SECOND ? tstart[1u << lg1] : tiles)) return;
    const PartTile p = part_tile<SECOND>(t, nq, PART_NT * IT, lg1, lg2, bstart, tstart);
    K q[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        q[k] = i < p.hi ? Q[i] : K{};
    }
    if (tid < B) {
        cnt[tid] = 0;
        if (tid) spl[tid] = bound[p.first + heap_order(tid, lg)];
    }
    __syncthreads();
    uint32_t node[IT];   // then the range, and the rank among the tile's queries of it
#pragma unroll
    for (int k = 0; k < IT; k++) node[k] = 1;
    for (uint32_t l = 0; l < lg; l++) {
#pragma unroll
        for (int k = 0; k < IT; k++) node[k] = 2 * node[k] + (q[k] >= spl[node[k]] ? 1u : 0u);
    }
#pragma unroll
    for (int k = 0; k < IT; k++) {
        if (p.lo + k * PART_NT + tid < p.hi) {
            const uint32_t bin = node[k] - B;
            node[k] = bin | (atomicAdd(&cnt[bin], 1u) << PART_LG);
        }
    }
    __syncthreads();
    uint32_t total;
    const uint32_t before = block_scan(tid < B ? cnt[tid] : 0u, wsum, &total);
    if (tid < B) {
        cnt[tid] = before;
        loc[(uint64_t)t * B + tid] = (uint16_t)before;
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        if (i < p.hi) {
            const uint32_t x = cnt[node[k] & (PART_BINS - 1)] + (node[k] >> PART_LG);
            place[i] = (uint16_t)x;
            stage[x] = q[k];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint32_t x = k * PART_NT + tid;
        if (x < total) out[p.lo + x] = stage[x];
    }
}

// the answers of a tile from its own order to that of its input
template <bool SECOND, int IT, typename AT>
__global__ __launch_bounds__(PART_NT) void k_part_back(
    const uint32_t *__restrict__ found, uint64_t nq, uint32_t lg1, uint32_t lg2,
    const uint32_t *__restrict__ bstart, const uint32_t *__restrict__ tstart, uint32_t tiles,
    const uint16_t *__restrict__ place, AT *__restrict__ dst) {
    __shared__ uint32_t stage[PART_NT * IT];
    const uint32_t tid = threadIdx.x, t = xcd_tile(tiles);
    if (t >= (SECOND ? tstart[1u << lg1] : tiles)) return;
    const PartTile p = part_tile<SECOND>(t, nq, PART_NT * IT, lg1, lg2, bstart, tstart);
    uint32_t v[IT], x[IT];
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        v[k] = i < p.hi ? found[i] : 0u;
        x[k] = i < p.hi ? place[i] : 0u;
    }
#pragma unroll
    for (int k = 0; k < IT; k++) stage[k * PART_NT + tid] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < IT; k++) {
        const uint64_t i = p.lo + k * PART_NT + tid;
        if (i < p.hi) dst[i] = (AT)stage[x[k]];
    }
}

// slots of a range on one level of a B-tree, where `level`: place y is at
// first + y - row, row the places' c0 + y in rows of b + 1, or, for a row's
// last, at sep_slot[row] (tabled for the first SEP_SLOTS)
constexpr uint32_t SEP_SLOTS = 1024;
struct RangeSlots {
    bool level;
    uint32_t first, c0;
};

// The m keys of ranks r0 .. : the first in heap[0], rank r0 + y at place y of
// the heap of 2^depth - 1 nodes, the places past them the largest key.  All of
// a lane's loads are issued before the first is stored.  The ranks' slots are
// what this costs (with slot_of() for every key the vector unit was busy for
// three quarters of the time of a B-tree's ranges and all of a vEB's), so they
// are found by what neighbours share:
//   B-tree: all keys of a range on the leaf level (or the one above it) lie at
//     rank - row + a constant, and rows follow from the place in the range by
//     a 24-bit product; the separators between them take slot_of().
//   vEB: 64 consecutive ranks share a bottom tree of 64 or more, which one
//     lane finds for them; the root behind it takes slot_of().
template <typename K, int LAYOUT>
__device__ inline RangeSlots range_fill(const K *__restrict__ A, const TileShape &s,
                                        const SlotMap<LAYOUT> &map, uint32_t r0, uint32_t m,
                                        uint32_t depth, K *heap, uint32_t *sep_slot) {
    constexpr uint32_t PER = RANGE_KEYS / RANGE_NT;
    const uint32_t tid = threadIdx.x;
    // heap_at(k * RANGE_NT + tid): the trailing zeros are the lane's, but lane 0's
    const uint32_t up = tid ? (uint32_t)__clz((int)__brev(tid)) + 1 : 0u;
    auto lane_node = [&](uint32_t k, uint32_t lg) {
        const uint32_t y = k * RANGE_NT + tid;
        return tid ? (y | (1u << lg)) >> up : heap_at(y, lg);
    };
    if constexpr (LAYOUT == TILE_BTREE) {
        const uint32_t k1 = s.b + 1, past = s.span + s.rem;
        const bool leaf = r0 + m <= s.span;
        if (leaf || r0 >= past) {
            const uint32_t x0 = leaf ? r0 : r0 - past + s.nsep;   // rank on its level
            const uint32_t row0 = (uint32_t)__umul64hi(x0, s.recip), c0 = x0 - row0 * k1;
            const uint32_t first = (leaf ? s.nint : map.level[0]) + (x0 - row0);
            const K *at = A + first;
            // separators: the ends of rows row0 ..
            const uint32_t seps = ((c0 + m) * s.small_mul) >> s.small_shift;
            const uint32_t per = (seps + RANGE_NT - 1) / RANGE_NT;
            constexpr uint32_t SEP = 2;   // kept in registers, more where b < 3
            K v[PER], w[SEP];
            auto sep_at = [&](uint32_t i) { return (i + 1) * k1 - 1 - c0; };   // its place
#pragma unroll
            for (uint32_t k = 0; k < PER; k++) {
                const uint32_t y = k * RANGE_NT + tid;
                const uint32_t t = c0 + y, q = (t * s.small_mul) >> s.small_shift;
                v[k] = y < m && t - q * k1 != s.b ? at[y - q] : key_max<K>();
            }
#pragma unroll
            for (uint32_t k = 0; k < SEP; k++) {
                const uint32_t i = k * RANGE_NT + tid;
                if (i < seps) {
                    const uint32_t slot = slot_of<LAYOUT>(r0 + sep_at(i), s, map);
                    w[k] = A[slot];
                    if (i < SEP_SLOTS) sep_slot[i] = slot;
                }
            }
#pragma unroll
            for (uint32_t k = 0; k < PER; k++) {
                const uint32_t y = k * RANGE_NT + tid;
                const uint32_t t = c0 + y, q = (t * s.small_mul) >> s.small_shift;
                if (y < (1u << depth) && (t - q * k1 != s.b || y >= m))
                    heap[lane_node(k, depth)] = v[k];
            }
#pragma unroll
            for (uint32_t k = 0; k < SEP; k++) {
                const uint32_t i = k * RANGE_NT + tid;
                if (i < seps) heap[heap_at(sep_at(i), depth)] = w[k];
            }
            for (uint32_t k = SEP; k < per; k++) {
                const uint32_t i = k * RANGE_NT + tid;
                if (i < seps)
                    heap[heap_at(sep_at(i), depth)] =
                        A[slot_of<LAYOUT>(r0 + sep_at(i), s, map)];
            }
            return {true, first, c0};
        }
    }
    if constexpr (LAYOUT == TILE_VEB) {
        // groups of 64 ranks starting at multiples of 64, PER + 1 a wave: lane k
        // finds the bottom tree of group k (d levels, first slot base, the
        // group's first rank u in it) and whether its last rank is a root
        const uint32_t lane = tid & 63, g0 = (r0 & ~63u) + (tid & ~63u);
        uint32_t base = 0, mine;
        bool root_here = false;
        {
            uint32_t u = g0 + lane * RANGE_NT, d = s.chain_d;
            bool whole = lane <= PER, tail = false;
            for (uint32_t j = 0; j < s.nchain; j++) {
                const VebLevel e = s.chain[j];
                const uint32_t span = e.nf << e.ld, l = (1u << e.ld) - 1;
                if (u < span) {
                    whole = whole && e.ld >= 6;
                    base += (1u << e.rd) - 1 + (u >> e.ld) * l;
                    u &= l;
                    tail = u + 63 == l;
                    d = e.ld;
                    break;
                }
                if (e.ld < 6 || u + 64 > span + e.inc) {
                    whole = false;
                    break;
                }
                base += (1u << e.rd) - 1 + e.nf * l;
                u -= span;
            }
            while (whole && d > SMALL_LEVELS) {
                const uint32_t rd = s.split[d], ld = d - rd, l = (1u << ld) - 1;
                whole = ld >= 6 && u + 64 <= (1u << d) - (tail ? 0u : 1u);
                base += (1u << rd) - 1 + (u >> ld) * l;
                u &= l;
                tail = u + 63 == l;
                d = ld;
            }
            whole = whole && d >= 6 && u + 64 <= (1u << d) - (tail ? 0u : 1u);
            root_here = whole && tail;
            // u < 2^d <= 2^SMALL_LEVELS where whole
            mine = whole ? ((1u << d) + u) | (tail ? 1u << 30 : 0u) | 1u << 31 : 0u;
        }
        K v[PER + 1], root{};
#pragma unroll
        for (uint32_t k = 0; k <= PER; k++) {
            const uint32_t x = g0 + k * RANGE_NT + lane;
            const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)k);
            const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)base, (int)k);
            if (x >= r0 && x < r0 + m && !(lane == 63 && (at >> 30) == 3))
                v[k] = A[at ? first + map.small[(at & 0xFFFF) + lane] : veb_slot(x, s, map)];
        }
        const uint32_t my_root = g0 + lane * RANGE_NT + 63;
        root_here = root_here && my_root >= r0 && my_root < r0 + m;
        if (root_here) root = A[veb_slot(my_root, s, map)];
#pragma unroll
        for (uint32_t k = 0; k <= PER; k++) {
            const uint32_t x = g0 + k * RANGE_NT + lane;
            const uint32_t at = (uint32_t)__builtin_amdgcn_readlane((int)mine, (int)k);
            if (x >= r0 && x < r0 + m && !(lane == 63 && (at >> 30) == 3))
                heap[heap_at(x - r0, depth)] = v[k];
        }
        if (root_here) heap[heap_at(my_root - r0, depth)] = root;
        for (uint32_t y = m + tid; y < (1u << depth); y += RANGE_NT)
            heap[heap_at(y, depth)] = key_max<K>();
        return {false, 0, 0};
    }
    K v[PER];
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
        const uint32_t y = k * RANGE_NT + tid;
        v[k] = y < m ? A[slot_of<LAYOUT>(r0 + y, s, map)] : key_max<K>();
    }
#pragma unroll
    for (uint32_t k = 0; k < PER; k++) {
        const uint32_t y = k * RANGE_NT + tid;
        if (y < (1u << depth)) heap[lane_node(k, depth)] = v[k];
    }
    return {false, 0, 0};
}

// The queries of range j in the tiles [ta, te), at most PART_SPAN of them, from
// the range's keys in LDS: of those in tile order, [skip, skip + PART_SHARE).
struct PartShare {
    uint32_t j, ta, te, skip;
};
template <bool SECOND>
constexpr uint32_t PART_SPAN = SECOND ? 64 : 256;
constexpr uint32_t PART_SHARE = 8192;
// consecutive ranges of a workgroup.  After two passes a range has few queries
// (512 of 2^27 in 2^30 keys), and with one the look-ups that lead to them took a
// fifth of the time.
template <bool SECOND>
constexpr uint32_t PART_RANGES = SECOND ? 8 : 1;

// where the tiles and their queries of each range are
struct PartLoc {
    uint32_t lg1, lg2, T, nq, tiles, span;   // span: tiles of a share, at most
    const uint32_t *bstart, *tstart;         // of two passes
    const uint16_t *loc;
};

// The queries of PART_RANGES ranges from their keys in LDS.  S holds the queries,
// each tile's in range order.  A workgroup takes a range's first share of `span`
// tiles (SECOND: of the ranges' bucket); whatever is more, where queries crowd,
// it puts on the queue, whose shares the second launch (REST) takes.  A key that
// occurs more than once is answered by the descent itself, whose first equal key
// it has to be, and so is every query where queued[1] says that the ranks' slots
// are not those of the caller's vEB tables (a classic table set given to an mvEB
// query, say): the partition then only orders the queries.
// Registers: at most 64 for a vEB, so that four workgroups share a compute unit
// (3.25 -> 3.08 ms); the others are faster with what they ask for (5.16 -> 4.85).
template <typename K, int LAYOUT, bool SECOND, bool REST>
__global__ __launch_bounds__(RANGE_NT, LAYOUT == TILE_VEB ? 8 : 1) void k_part_answer(
    const K *__restrict__ A, TileShape s, PartLoc pl, uint32_t units, const K *__restrict__ S,
    uint32_t *queued, PartShare *queue, uint32_t *__restrict__ out) {
    constexpr uint32_t SPAN = PART_SPAN<SECOND>, RANGES = REST ? 1 : PART_RANGES<SECOND>;
    __shared__ K heap[RANGE_KEYS];
    __shared__ uint32_t sep_slot[LAYOUT == TILE_BTREE ? SEP_SLOTS : 1];
    __shared__ uint32_t pre[SPAN], base[SPAN];   // queries before a tile's, the first's place
    __shared__ uint16_t locs_of[RANGES > 1 ? SPAN : 1][RANGES + 1];
    // one range's are read before its keys come
    uint16_t(*locs)[RANGES + 1] =
        RANGES > 1 ? locs_of : reinterpret_cast<uint16_t(*)[RANGES + 1]>(heap);
    __shared__ uint32_t wsum[RANGE_NT / 64];
    __shared__ VebEntry tb[LAYOUT == TILE_VEB ? TILE_TABLES : 1];
    __shared__ uint32_t s_end[64];
    __shared__ uint16_t s_tidx[64];
    __shared__ SlotMap<LAYOUT> map;
    const uint32_t tid = threadIdx.x, n = s.n, lg = pl.lg1 + (SECOND ? pl.lg2 : 0u);
    const uint32_t B = 1u << (SECOND ? pl.lg2 : pl.lg1);
    uint32_t unit = REST ? blockIdx.x : xcd_tile(units);
    const uint32_t shares = REST ? *queued : units;
    if (unit >= shares) return;
    const bool by_tables = LAYOUT == TILE_VEB && queued[1] != 0;
    if constexpr (LAYOUT == TILE_VEB) {
        for (uint32_t i = tid; i < s.table_size; i += RANGE_NT)
            tb[i] = {(uint32_t)s.tables[i].L, (uint32_t)s.tables[i].R, s.tables[i].D};
        if (tid < s.ntables) {
            s_end[tid] = s.idx ? (uint32_t)s.idx[tid] : n;
            s_tidx[tid] = s.tidx ? (uint16_t)s.tidx[tid] : (uint16_t)0;
        }
    }
    slot_map<LAYOUT>(s, map);
    for (; unit < shares; unit += gridDim.x) {
        PartShare sh;
        uint32_t bucket_end = 0, t_first = 0, q_first = 0, q_end = pl.nq;
        if constexpr (REST) {
            sh = queue[unit];
        } else {
            sh.j = SECOND ? unit * RANGES : unit & (B - 1);
            sh.skip = 0;
        }
        if constexpr (SECOND) {   // the ranges' bucket
            const uint32_t k = sh.j >> pl.lg2;
            t_first = pl.tstart[k];
            bucket_end = pl.tstart[k + 1];
            q_first = pl.bstart[k];
            q_end = pl.bstart[k + 1];
        }
        if constexpr (!REST) {
            sh.ta = SECOND ? t_first : (unit >> pl.lg1) * pl.span;
            sh.te = min(sh.ta + pl.span, SECOND ? bucket_end : pl.tiles);
        }
        auto lo_of = [&](uint32_t t) { return q_first + (t - t_first) * pl.T; };
        // place in tile t of the first query of range r of the bucket
        auto loc_of = [&](uint32_t t, uint32_t r) -> uint32_t {
            return r < B ? pl.loc[(uint64_t)t * B + r] : min(pl.T, q_end - lo_of(t));
        };
        const uint32_t r_first = sh.j & (B - 1);
        for (uint32_t i = tid; i < (sh.te - sh.ta) * (RANGES + 1); i += RANGE_NT) {
            const uint32_t t = i / (RANGES + 1), k = i - t * (RANGES + 1);
            locs[t][k] = (uint16_t)loc_of(sh.ta + t, r_first + k);
        }
        __syncthreads();
        for (uint32_t rr = 0; rr < RANGES; rr++) {
            const uint32_t j = sh.j + rr;
            uint32_t total;
            if constexpr (!REST && SECOND) {
                for (uint32_t ta = sh.te; ta < bucket_end; ta += pl.span) {
                    const uint32_t te = min(ta + pl.span, bucket_end);
                    const uint32_t c = ta + tid < te ? loc_of(ta + tid, r_first + rr + 1) -
                                                           loc_of(ta + tid, r_first + rr)
                                                     : 0u;
                    (void)block_scan(c, wsum, &total);
                    if (tid == 0)
                        for (uint32_t skip = 0; skip < total; skip += PART_SHARE)
                            queue[atomicAdd(queued, 1u)] = {j, ta, te, skip};
                }
            }
            const bool tile = sh.ta + tid < sh.te;
            const uint32_t before =
                block_scan(tile ? locs[tid][rr + 1] - locs[tid][rr] : 0u, wsum, &total);
            if (tid < SPAN) {
                pre[tid] = before;
                base[tid] = tile ? lo_of(sh.ta + tid) + locs[tid][rr] : 0u;
            }
            if (!REST && tid == 0)
                for (uint32_t skip = PART_SHARE; skip < total; skip += PART_SHARE)
                    queue[atomicAdd(queued, 1u)] = {j, sh.ta, sh.te, skip};
            __syncthreads();
            const uint32_t end = min(total, sh.skip + PART_SHARE);
            if (sh.skip >= end) continue;   // the whole workgroup's
            // where query i of the share is
            auto place = [&](uint32_t i) {
                uint32_t t = 0;
                for (uint32_t h = pl.span >> 1; h > 0; h >>= 1) t += pre[t + h] <= i ? h : 0u;
                return base[t] + (i - pre[t]);
            };
            const uint32_t r0 = range_first(j, n, lg), m = range_first(j + 1, n, lg) - r0;
            const uint32_t depth = 32u - (uint32_t)__clz((int)(m - 1));   // 2^depth >= m
            // two queries a lane and turn: 512 queries in 512 lanes would take a
            // second turn for the few of half the ranges that have more (a vEB
            // has no registers for it: 3.1 -> 3.4 ms at 3*10^8 keys)
            constexpr int QN = LAYOUT == TILE_VEB ? 1 : 2;
            uint32_t here[QN];
            K q[QN];
            auto fetch = [&](uint32_t q0) {
#pragma unroll
                for (int k = 0; k < QN; k++) {
                    const uint32_t i = q0 + k * RANGE_NT + tid;
                    here[k] = i < end ? place(i) : ~0u;
                    q[k] = i < end ? S[here[k]] : K{};
                }
            };
            fetch(sh.skip);
            const RangeSlots rs = range_fill<K, LAYOUT>(A, s, map, r0, m, depth, heap, sep_slot);
            __syncthreads();
            for (uint32_t q0 = sh.skip; q0 < end; q0 += QN * RANGE_NT) {
                if (q0 != sh.skip) fetch(q0);
                // the keys after the first that are smaller than q
                // (TILE_SORTED: not larger)
                uint32_t node[QN];
#pragma unroll
                for (int k = 0; k < QN; k++) node[k] = 1;
                for (uint32_t l = 0; l < depth; l++) {
#pragma unroll
                    for (int k = 0; k < QN; k++) {
                        const K key = heap[node[k]];
                        const bool right = LAYOUT == TILE_SORTED ? key <= q[k] : key < q[k];
                        node[k] = 2 * node[k] + (right ? 1u : 0u);
                    }
                }
#pragma unroll
                for (int k = 0; k < QN; k++) {
                    const uint32_t below = min(node[k] - (1u << depth), m - 1);
                    uint32_t ans = n;
                    if constexpr (LAYOUT == TILE_SORTED) {
                        if (heap[0] <= q[k]) ans = r0 + below;
                    } else {
                        bool again = by_tables && here[k] != ~0u;
                        const uint32_t x = q[k] <= heap[0] ? 0u : below + 1;
                        if (x < m && here[k] != ~0u && heap[heap_at(x, depth)] == q[k]) {
                            const uint32_t t = rs.c0 + x, row = (t * s.small_mul) >> s.small_shift;
                            if (LAYOUT == TILE_BTREE && rs.level && row < SEP_SLOTS)
                                ans = t - row * (s.b + 1) != s.b ? rs.first + x - row
                                                                 : sep_slot[row];
                            else
                                ans = slot_of<LAYOUT>(r0 + x, s, map);
                            if (x == 0 && r0 > 0)
                                again |= A[slot_of<LAYOUT>(r0 - 1, s, map)] == q[k];
                            if (x + 1 < m) again |= heap[heap_at(x + 1, depth)] == q[k];
                        }
                        if (__any(again)) {
                            const K qq[1] = {q[k]};
                            uint32_t res[1];
                            tile_descend<K, LAYOUT, 1>(A, s, tb, s_end, s_tidx, qq, res);
                            if (again) ans = res[0];
                        }
                    }
                    if (here[k] != ~0u) out[here[k]] = ans;
                }
            }
            __syncthreads();   // the range's queries are answered
        }
        __syncthreads();   // the last ranges' locs are read
    }
}

// ---- host side

static TileShape tile_shape(const TileArray &a) {
    TileShape s{};
    static_cast<SlotShape &>(s) = slot_shape(a.layout, a.n, a.b, a.classic);
    if (a.layout == TILE_BST || a.layout == TILE_BTREE) {
        s.nodes = (uint32_t)((a.n + s.b - 1) / s.b);
        s.levels = ilog_base(a.n + 1, s.b + 1ull);   // levels whose every node is whole
        // exact below 2 RANGE_KEYS: 2^shift > 2 RANGE_KEYS (b + 1)
        s.small_shift = floor_log2_64(2ull * RANGE_KEYS * (s.b + 1)) + 1;
        s.small_mul = (uint32_t)(((1ull << s.small_shift) + s.b) / (s.b + 1));
    }
    s.table_size = a.table_size;
    s.ntables = a.ntables;
    s.tables = a.tables;
    s.idx = a.idx;
    s.tidx = a.tidx;
    return s;
}

template <typename K, int LAYOUT, int IT>
static void tile_launch(Ctx *c, const TileArray &a, const void *q, uint64_t nq, uint64_t *ans,
                        hipStream_t s) {
    constexpr uint32_t T = TILE_NT * IT;
    const uint32_t tiles = (uint32_t)((nq + T - 1) / T);
    const uint32_t per_cu = 4;
    const uint32_t grid = std::min<uint32_t>((tiles + 7) / 8, c->num_cus * per_cu / 8) * 8;
    hipLaunchKernelGGL((k_query_tile<K, LAYOUT, IT>), dim3(grid), dim3(TILE_NT), 0, s,
                       (const K *)a.A, tile_shape(a), (const K *)q, nq, ans, tiles);
}

template <typename K, int IT>
static void tile_layout(Ctx *c, const TileArray &a, const void *q, uint64_t nq, uint64_t *ans,
                        hipStream_t s) {
    switch (a.layout) {
    case TILE_BST: tile_launch<K, TILE_BST, IT>(c, a, q, nq, ans, s); break;
    case TILE_BTREE: tile_launch<K, TILE_BTREE, IT>(c, a, q, nq, ans, s); break;
    case TILE_VEB: tile_launch<K, TILE_VEB, IT>(c, a, q, nq, ans, s); break;
    default: tile_launch<K, TILE_SORTED, IT>(c, a, q, nq, ans, s); break;
    }
}

tl_status tile_query(Ctx *c, const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
                     uint64_t *ans, hipStream_t s) {
    switch (dtype) {
    case TL_U32: tile_layout<uint32_t, 8>(c, a, q, nq, ans, s); break;
    case TL_U64: tile_layout<uint64_t, 8>(c, a, q, nq, ans, s); break;
    case TL_I32: tile_layout<int32_t, 8>(c, a, q, nq, ans, s); break;
    default: tile_layout<int64_t, 8>(c, a, q, nq, ans, s); break;
    }
    TL_LAUNCH_CHECK();
    return TL_OK;
}

// ---- partitioned lookups

// where everything of one partitioned batch lies in its workspace
struct PartPlan {
    uint32_t lg1, lg2, it, tiles1, tiles2, groups, span;
    uint64_t bound, bstart, tstart, gsum, counts, places, loc, pack, place, found, queued, queue;
    uint64_t second, most, bytes;   // most: shares on the queue
};

static PartPlan part_plan(uint64_t n, uint32_t w, uint64_t nq) {
    PartPlan p{};
    uint32_t lg = 1;
    while (((n + (1ull << lg) - 1) >> lg) > RANGE_KEYS) lg++;
    p.lg1 = std::min(lg, PART_LG);
    p.lg2 = lg - p.lg1;
    if (p.lg2 && p.lg2 < 3) {   // a bucket has the ranges of a workgroup at least
        p.lg1 -= 3 - p.lg2;
        p.lg2 = 3;
    }
    p.it = nq >= (1u << 22) ? 16 : 4;
    const uint64_t T = (uint64_t)PART_NT * p.it;
    p.tiles1 = (uint32_t)((nq + T - 1) / T);
    p.tiles2 = p.lg2 ? p.tiles1 + (1u << p.lg1) : 0;
    p.groups = (p.tiles1 + PART_GROUP - 1) / PART_GROUP;
    // a share is of about as many queries as a range has keys
    const uint64_t tiles = p.lg2 ? p.tiles2 : p.tiles1, ranges = 1ull << (p.lg2 ? p.lg2 : p.lg1);
    const uint32_t most = p.lg2 ? PART_SPAN<true> : PART_SPAN<false>;
    p.span = 1;
    while (p.span < most && p.span * T < RANGE_KEYS * ranges) p.span *= 2;
    uint64_t at = 0;
    auto take = [&](uint64_t bytes) {
        const uint64_t o = at;
        at += (bytes + 255) & ~255ull;
        return o;
    };
    p.bound = take((uint64_t)w << lg);
    if (p.lg2) {
        p.bstart = take(((1ull << p.lg1) + 1) * 4);
        p.tstart = take(((1ull << p.lg1) + 1) * 4);
        p.gsum = take(((uint64_t)p.groups << p.lg1) * 4);
        p.counts = take(((uint64_t)p.tiles1 << p.lg1) * 4);
        p.places = take(((uint64_t)p.tiles1 << p.lg1) * 4);
        p.pack = take(nq * 4);
    }
    p.loc = take(tiles * ranges * 2);
    p.place = take(nq * 2);
    p.found = take(nq * 4);   // of two passes: in the first pass's order
    p.queued = take(8);
    // shares past their workgroups' own: of crowded ranges, and of buckets past
    // their first `span` tiles
    p.most = nq / PART_SHARE + (p.lg2 ? tiles / p.span * ranges : 0) + 1;
    p.queue = take(p.most * sizeof(PartShare));
    // the queries after the second pass: behind those after the first in the
    // answer array, which has room for both when keys have 4 bytes
    p.second = p.lg2 && w == 8 ? take(nq * 8) : 0;
    p.bytes = at;
    return p;
}

constexpr uint64_t PART_MAX_QUERIES = 1ull << 27;   // of one segment of a batch

uint64_t part_bytes(const TileArray &a, uint32_t dtype, uint64_t nq) {
    const uint32_t w = (dtype == TL_U32 || dtype == TL_I32) ? 4 : 8;
    return part_plan(a.n, w, std::min(nq, PART_MAX_QUERIES)).bytes;
}

// the first pass of two: q in bucket order to out
template <typename K, int IT>
static void part_pass(const PartPlan &p, const K *q, uint64_t nq, char *ws, K *out,
                      hipStream_t s) {
    uint32_t *bstart = (uint32_t *)(ws + p.bstart), *tstart = (uint32_t *)(ws + p.tstart);
    uint32_t *counts = (uint32_t *)(ws + p.counts), *places = (uint32_t *)(ws + p.places);
    uint32_t *pack = (uint32_t *)(ws + p.pack), *gsum = (uint32_t *)(ws + p.gsum);
    const uint32_t B1 = 1u << p.lg1;
    const dim3 grid((p.tiles1 + 7) / 8 * 8), block(PART_NT);
    hipLaunchKernelGGL((k_part_count<K, IT>), grid, block, 0, s, q, nq, (const K *)(ws + p.bound),
                       p.lg1, p.lg2, p.tiles1, pack, counts);
    hipLaunchKernelGGL(k_part_sums, dim3(p.groups), block, 0, s, (const uint32_t *)counts, B1,
                       p.tiles1, gsum);
    hipLaunchKernelGGL(k_part_starts, dim3(1), block, 0, s, gsum, B1, p.groups,
                       (uint32_t)(PART_NT * IT), bstart, tstart, (uint32_t *)nullptr);
    hipLaunchKernelGGL(k_part_places, dim3(p.groups), block, 0, s, (const uint32_t *)counts, B1,
                       p.tiles1, (const uint32_t *)gsum, (const uint32_t *)bstart, places);
    hipLaunchKernelGGL((k_part_scatter<K, IT>), grid, block, 0, s, q, nq, p.lg1, p.tiles1,
                       (const uint32_t *)places, (const uint32_t *)counts, (const uint32_t *)pack,
                       out);
}

// the last pass: the queries in, tile by tile, to `tiled`, and their answers to
// dst in the order of in
template <typename K, int LAYOUT, bool SECOND, int IT, typename AT>
static void part_answer(const PartPlan &p, const TileArray &a, const TileShape &sh, const K *in,
                        uint64_t nq, char *ws, K *tiled, uint32_t *found, AT *dst, hipStream_t s) {
    const uint32_t *bstart = (const uint32_t *)(ws + p.bstart);
    const uint32_t *tstart = (const uint32_t *)(ws + p.tstart);
    uint16_t *place = (uint16_t *)(ws + p.place), *loc = (uint16_t *)(ws + p.loc);
    uint32_t *queued = (uint32_t *)(ws + p.queued);
    PartShare *queue = (PartShare *)(ws + p.queue);
    const uint32_t tiles = SECOND ? p.tiles2 : p.tiles1;
    const dim3 grid((tiles + 7) / 8 * 8), block(PART_NT);
    hipLaunchKernelGGL((k_part_tile<K, SECOND, IT>), grid, block, 0, s, in, nq,
                       (const K *)(ws + p.bound), p.lg1, p.lg2, bstart, tstart, tiles, place, loc,
                       tiled);
    const PartLoc pl{p.lg1, p.lg2, (uint32_t)(PART_NT * IT), (uint32_t)nq, tiles, p.span,
                     bstart, tstart, loc};
    const uint32_t units = SECOND ? (1u << (p.lg1 + p.lg2)) / PART_RANGES<true>
                                  : ((tiles + p.span - 1) / p.span) << p.lg1;
    hipLaunchKernelGGL((k_part_answer<K, LAYOUT, SECOND, false>), dim3((units + 7) / 8 * 8),
                       dim3(RANGE_NT), 0, s, (const K *)a.A, sh, pl, units, (const K *)tiled,
                       queued, queue, found);
    hipLaunchKernelGGL((k_part_answer<K, LAYOUT, SECOND, true>),
                       dim3((uint32_t)std::min<uint64_t>(p.most, 1024)), dim3(RANGE_NT), 0, s,
                       (const K *)a.A, sh, pl, units, (const K *)tiled, queued, queue, found);
    hipLaunchKernelGGL((k_part_back<SECOND, IT, AT>), grid, block, 0, s, (const uint32_t *)found,
                       nq, p.lg1, p.lg2, bstart, tstart, tiles, (const uint16_t *)place, dst);
}

template <typename K, int LAYOUT, int IT>
static void part_segment(const PartPlan &p, const TileArray &a, const K *q, uint64_t nq,
                         uint64_t *ans, char *ws, hipStream_t s) {
    using W = typename std::conditional<sizeof(K) == 4, uint32_t, uint64_t>::type;
    const TileShape sh = tile_shape(a);
    const uint32_t lg = p.lg1 + p.lg2;
    hipLaunchKernelGGL((k_part_bounds<W, LAYOUT>), dim3(((1u << lg) + 255) / 256 + 1), dim3(256),
                       0, s, (const W *)a.A, sh, lg, (W *)(ws + p.bound),
                       (uint32_t *)(ws + p.queued));
    uint32_t *found = (uint32_t *)(ws + p.found);
    K *first = (K *)ans;   // the answer array holds queries meanwhile
    if (!p.lg2) {
        part_answer<K, LAYOUT, false, IT>(p, a, sh, q, nq, ws, first, found, ans, s);
        return;
    }
    part_pass<K, IT>(p, q, nq, ws, first, s);
    K *tiled = sizeof(K) == 4 ? first + nq : (K *)(ws + p.second);
    part_answer<K, LAYOUT, true, IT>(p, a, sh, first, nq, ws, tiled, (uint32_t *)ans, found, s);
    hipLaunchKernelGGL((k_part_return<IT>), dim3((p.tiles1 + 7) / 8 * 8), dim3(PART_NT), 0, s,
                       (const uint32_t *)found, nq, p.lg1, p.tiles1,
                       (const uint32_t *)(ws + p.places), (const uint32_t *)(ws + p.counts),
                       (const uint32_t *)(ws + p.pack), ans);
}

template <typename K, int LAYOUT>
static void part_segment(const TileArray &a, const K *q, uint64_t nq, uint64_t *ans, char *ws,
                         hipStream_t s) {
    const PartPlan p = part_plan(a.n, sizeof(K), nq);
    if (p.it == 16)
        part_segment<K, LAYOUT, 16>(p, a, q, nq, ans, ws, s);
    else
        part_segment<K, LAYOUT, 4>(p, a, q, nq, ans, ws, s);
}

template <typename K>
static void part_layout(const TileArray &a, const K *q, uint64_t nq, uint64_t *ans, char *ws,
                        hipStream_t s) {
    for (uint64_t at = 0; at < nq; at += PART_MAX_QUERIES) {
        const uint64_t m = std::min(PART_MAX_QUERIES, nq - at);
        switch (a.layout) {
        case TILE_BST: part_segment<K, TILE_BST>(a, q + at, m, ans + at, ws, s); break;
        case TILE_BTREE: part_segment<K, TILE_BTREE>(a, q + at, m, ans + at, ws, s); break;
        case TILE_VEB: part_segment<K, TILE_VEB>(a, q + at, m, ans + at, ws, s); break;
        default: part_segment<K, TILE_SORTED>(a, q + at, m, ans + at, ws, s); break;
        }
    }
}

tl_status part_query(const TileArray &a, uint32_t dtype, const void *q, uint64_t nq, uint64_t *ans,
                     void *ws, hipStream_t s) {
    switch (dtype) {
    case TL_U32: part_layout<uint32_t>(a, (const uint32_t *)q, nq, ans, (char *)ws, s); break;
    case TL_U64: part_layout<uint64_t>(a, (const uint64_t *)q, nq, ans, (char *)ws, s); break;
    case TL_I32: part_layout<int32_t>(a, (const int32_t *)q, nq, ans, (char *)ws, s); break;
    default: part_layout<int64_t>(a, (const int64_t *)q, nq, ans, (char *)ws, s); break;
    }
    TL_LAUNCH_CHECK();
    return TL_OK;
}

// ---- which of them answers a batch

static uint32_t key_width(uint32_t dtype) { return (dtype == TL_U32 || dtype == TL_I32) ? 4 : 8; }

bool tile_can(const TileArray &a, uint32_t dtype, uint64_t nq) {
    if (dtype > TL_I64 || a.n < 4096 || a.n >= (1ull << 32) - 1 || nq < (1u << 16) ||
        nq >= (1ull << 40))
        return false;
    // every node number of a descent fits 32 bits
    if (a.layout == TILE_BTREE &&
        (a.b < 1 || a.b > 1024 || (a.n + a.b - 1) / a.b >= (1ull << 32) / (a.b + 1) - 1))
        return false;
    // conceptual positions (below twice the structure's keys) fit 32 bits
    if (a.layout == TILE_VEB &&
        (a.table_size > TILE_TABLES || a.ntables > 64 || a.n >= (1ull << 31)))
        return false;
    return true;
}

bool part_can(const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
              const uint64_t *ans) {
    if (!tile_can(a, dtype, nq)) return false;
    // the answer array holds the queries in range order meanwhile
    const char *q0 = (const char *)q, *a0 = (const char *)ans;
    if (q0 < a0 + nq * 8 && a0 < q0 + nq * key_width(dtype)) return false;
    // ranges are of the whole layout: its tables have to be those of all of it
    if (a.layout == TILE_VEB) {
        const TileShape s = tile_shape(a);
        uint32_t structures = 1;
        for (uint32_t j = 0; j < s.nchain; j++) structures += s.chain[j].inc != 0;
        if (structures != a.ntables) return false;
    }
    return true;
}

// Time of a batch in picoseconds by each path, from lookups of uniform keys
// measured on arrays of 2^12 .. 2^28 keys of both widths, nodes of 1 to 33 keys
// and 2^19 .. 2^26 queries: a start-up, and per query a figure that grows with
// the array's bytes (2^16, 2^18 .. 2^32).
struct PathCost {
    double start;
    uint16_t query[9];
};
static double path_ps(const PathCost &c, uint64_t n, uint32_t w, uint64_t nq) {
    const double l = std::min(16.0, std::max(0.0, log2((double)n * w) - 16)) / 2;
    const int i = std::min(7, (int)l);
    return c.start + (double)nq * (c.query[i] + (c.query[i + 1] - c.query[i]) * (l - i));
}

// the kernels of tl_query.hip but the B-trees' (entry TILE_BTREE is not used)
static const PathCost COST_OLD[] = {{8e6, {13, 15, 20, 28, 45, 75, 112, 152, 190}},
                                    {0, {0, 0, 0, 0, 0, 0, 0, 0, 0}},
                                    {8e6, {27, 33, 39, 45, 58, 71, 90, 129, 160}},
                                    {14e6, {9, 19, 31, 41, 115, 192, 245, 285, 310}}};
// the tile-sorted descents, 2^20 queries at least: fewer don't fill the device
static const PathCost COST_TILE[] = {{12e6, {7, 8, 11, 17, 33, 73, 110, 148, 185}},
                                     {14e6, {16, 18, 24, 33, 50, 84, 126, 165, 210}},
                                     {24e6, {21, 25, 27, 38, 50, 74, 103, 144, 180}},
                                     {8e6, {6, 10, 22, 36, 85, 155, 205, 255, 290}}};

static double tile_ps(const TileArray &a, uint32_t w, uint64_t nq) {
    return path_ps(COST_TILE[a.layout], a.n, w, std::max<uint64_t>(nq, 1u << 20));
}

// A B-tree's descent costs its lanes' instructions on every level (wide: 1.3 ps
// a lane of 8-byte keys, 1.9 of 4-byte keys; else about one), or, where that is
// more, the lines of the levels past one L2's 4 MB, 19 ps each.
static double old_ps(const TileArray &a, uint32_t w, uint64_t nq) {
    if (a.layout != TILE_BTREE) return path_ps(COST_OLD[a.layout], a.n, w, nq);
    if (a.b > 64) return 5e6 + (double)nq * 4.0 * a.b;   // one lane scans the nodes
    if (a.b == 1) return path_ps(COST_OLD[TILE_BST], a.n, w, nq);
    uint32_t group = 2;
    while (group < a.b) group *= 2;
    const double level =
        wide_ok(a.A, a.b, w) ? wide_group(a.b, w) * (w == 8 ? 1.3 : 1.9) : group * 0.95;
    const double per_level = log2((double)a.b + 1);
    const double lanes = 1 + level * ceil(log2((double)a.n + 1) / per_level);
    const double lines = 8 + 19 * (log2((double)a.n * w) - 22) / per_level;
    return 6e6 + (double)nq * std::max(lanes, lines);
}

// the partitioned batch, whatever the layout: each query's moves, and every
// range read (with two passes mostly slots and latency)
static double part_ps(const TileArray &a, uint32_t w, uint64_t nq) {
    const bool two = part_plan(a.n, w, std::min(nq, PART_MAX_QUERIES)).lg2 != 0;
    const uint64_t segments = (nq + PART_MAX_QUERIES - 1) / PART_MAX_QUERIES;
    return segments * (two ? 55e6 + 2.6 * a.n : 30e6 + 1.0 * a.n) + (double)nq * (two ? 25 : 12.5);
}

Workspace &query_workspace() {
    static thread_local Workspace w;
    return w;
}

// $TL_QUERY_PATH: plain, tile or part picks that path wherever it can run.  Without
// it, a variable that shapes the plain descents keeps those for batches of any size.
static int forced_path() {
    static const char *const knobs[] = {"TL_BTREE_WIDE=", "TL_BTREE_IDX64=", "TL_BTREE_QPG=",
                                        "TL_LEARNED_FUSED=", "TL_VEB_QPL=", "TL_VEB_TOP="};
    const char *e = getenv("TL_QUERY_PATH");
    if (e && !strcmp(e, "plain")) return 0;
    if (e && !strcmp(e, "tile")) return 1;
    if (e && !strcmp(e, "part")) return 2;
    for (char **v = environ; *v; v++)
        if (!strncmp(*v, "TL_", 3))
            for (const char *k : knobs)
                if (!strncmp(*v, k, strlen(k))) return 0;
    return -1;
}

bool part_wanted(const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
                 const uint64_t *ans, double other) {
    if (!part_can(a, dtype, q, nq, ans)) return false;
    const int f = forced_path();
    if (f >= 0) return f == 2;
    const uint32_t w = key_width(dtype);
    // (the figures are good to a tenth; near a draw the plain path stays)
    return part_ps(a, w, nq) < other * std::min(0.9 * old_ps(a, w, nq), 0.95 * tile_ps(a, w, nq));
}

tl_status part_try(Ctx *c, const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
                   uint64_t *ans, hipStream_t s, double other, bool *taken) {
    *taken = false;
    if (!part_wanted(a, dtype, q, nq, ans, other)) return TL_OK;
    const uint64_t need = part_bytes(a, dtype, nq);
    const Workspace &w = query_workspace();
    if (w.mem) {
        if (w.bytes < need) return TL_OK;
        *taken = true;
        return part_query(a, dtype, q, nq, ans, w.mem, s);
    }
    Lease *l = lease_take(c, need, s);
    if (!l) return TL_OK;
    *taken = true;
    const tl_status st = part_query(a, dtype, q, nq, ans, l->mem, s);
    lease_give(l, s);
    return st;
}

tl_status large_query(Ctx *c, const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
                      uint64_t *ans, hipStream_t s, bool *taken) {
    TL_TRY(part_try(c, a, dtype, q, nq, ans, s, 1.0, taken));
    if (*taken || !tile_can(a, dtype, nq)) return TL_OK;
    const int f = forced_path();
    const uint32_t w = key_width(dtype);
    if (f == 0 || (f < 0 && tile_ps(a, w, nq) >= 0.9 * old_ps(a, w, nq)))
        return TL_OK;
    *taken = true;
    return tile_query(c, a, dtype, q, nq, ans, s);
}

}   // namespace tl
