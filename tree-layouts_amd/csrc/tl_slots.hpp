// tl_slots.hpp -- rank -> slot of every layout for kernels that work from
// global memory: host constants (SlotShape), small tables in LDS (SlotMap) and
// one function per layout without divisions.  Arrays of less than 2^32 - 1
// keys (vEB layouts: 2^31).
#pragma once

#include "tl_internal.hpp"

namespace tl {

enum TileLayout : uint32_t { TILE_BST, TILE_BTREE, TILE_VEB, TILE_SORTED };

// an incomplete vEB tree: top and bottom levels, full bottom trees, keys of the
// incomplete one
constexpr uint32_t VEB_CHAIN = 8;
struct VebLevel {
    uint32_t rd, ld, nf, inc;
};

struct SlotShape {
    uint32_t n, b, classic;
    // a BST or B-tree (BtreeShape's); 2^64 / (b + 1) rounded up
    uint32_t nint, span, rem, nsep, depth;
    uint64_t recip;
    // a vEB: the incomplete trees from the whole one down (the incomplete
    // bottom tree of one is the next), then a perfect tree of chain_d levels
    // (0: none); split[d]: top levels of a perfect tree of d
    VebLevel chain[VEB_CHAIN];
    uint32_t nchain, chain_d;
    uint8_t split[36];
};

inline SlotShape slot_shape(uint32_t layout, uint64_t n, uint64_t b, bool classic) {
    SlotShape s{};
    s.n = (uint32_t)n;
    s.b = layout == TILE_BTREE ? (uint32_t)b : 1u;
    s.classic = classic;
    if (layout == TILE_BST || layout == TILE_BTREE) {
        const BtreeShape bs = btree_shape(s.n, s.b);
        s.nint = bs.nint;
        s.span = bs.span;
        s.rem = bs.rem;
        s.nsep = bs.nsep;
        s.depth = ilog_base((uint64_t)bs.nint + 1, s.b + 1ull);
        s.recip = ~0ull / (s.b + 1ull) + 1;
    }
    if (layout == TILE_VEB) {
        for (uint32_t d = 2; d <= 32; d++) {
            uint32_t rd, ld;
            veb_split(d, rd, ld, classic);
            s.split[d] = (uint8_t)rd;
        }
        while (n & (n + 1)) {
            VebLevel &e = s.chain[s.nchain++];
            veb_split(floor_log2_64(n) + 1, e.rd, e.ld, classic);
            const uint64_t r = (1ull << e.rd) - 1, l = (1ull << e.ld) - 1;
            e.nf = (uint32_t)((n - r) / l);
            e.inc = (uint32_t)(n - r - e.nf * l);
            n = e.inc;
        }
        s.chain_d = n ? floor_log2_64(n) + 1 : 0;
    }
    return s;
}

// What slot_of() looks up in LDS.  TILE_BTREE: level[z].  TILE_VEB: the
// slots of the perfect trees of at most 8 levels, tree d's rank x at
// small[2^d + x]: a rank of a tree of 2^16 keys takes one split and one
// look-up instead of up to four splits.
constexpr uint32_t SMALL_LEVELS = 8;
template <int LAYOUT>
struct SlotMap {
    uint32_t level[32];
};
template <>
struct SlotMap<TILE_VEB> {
    uint8_t small[2u << SMALL_LEVELS];
};

// slot of rank x in the vEB (mveb_pos32 with the tables)
__device__ inline uint32_t veb_slot(uint32_t x, const SlotShape &s, const SlotMap<TILE_VEB> &m) {
    uint32_t base = 0, d = s.chain_d;
    for (uint32_t j = 0; j < s.nchain; j++) {
        const VebLevel e = s.chain[j];
        const uint32_t r = (1u << e.rd) - 1, l = (1u << e.ld) - 1, span = e.nf << e.ld;
        if (x < span) {
            const uint32_t k = x >> e.ld, c = x & l;
            d = c == l ? e.rd : e.ld;
            base += c == l ? 0u : r + k * l;
            x = c == l ? k : c;
            break;
        }
        if (x >= span + e.inc) {
            x = e.nf + (x - span - e.inc);
            d = e.rd;
            break;
        }
        base += r + e.nf * l;
        x -= span;
    }
    while (d > SMALL_LEVELS) {
        const uint32_t rd = s.split[d], ld = d - rd, l = (1u << ld) - 1;
        const uint32_t k = x >> ld, c = x & l;
        base += c == l ? 0u : (1u << rd) - 1 + k * l;
        d = c == l ? rd : ld;
        x = c == l ? k : c;
    }
    return base + m.small[(1u << d) + x];
}

// slot of internal rank x of a BST or B-tree; m.level[z]: first slot of the
// level whose keys' internal ranks + 1 are divisible by (b + 1)^z and no more
// (TILE_BTREE)
template <int LAYOUT>
__device__ inline uint32_t internal_slot(uint32_t x, const SlotShape &s,
                                         const SlotMap<LAYOUT> &m) {
    if constexpr (LAYOUT == TILE_BST) {
        const uint32_t y = x + 1, z = (uint32_t)__clz((int)__brev(y));
        return ((y | (1u << s.depth)) >> (z + 1)) - 1;
    } else {
        auto div = [&](uint32_t v) { return (uint32_t)__umul64hi(v, s.recip); };
        const uint32_t k1 = s.b + 1;
        uint32_t r = x + 1, z = 0, q = div(r);
        while (r == q * k1) {
            r = q;
            q = div(r);
            z++;
        }
        return m.level[z] + r - q - 1;
    }
}

// slot of rank x in the layout
template <int LAYOUT>
__device__ inline uint32_t slot_of(uint32_t x, const SlotShape &s, const SlotMap<LAYOUT> &m) {
    if constexpr (LAYOUT == TILE_SORTED) {
        return x;
    } else if constexpr (LAYOUT == TILE_VEB) {
        return veb_slot(x, s, m);
    } else if constexpr (LAYOUT == TILE_BST) {
        if (x < s.span) {
            if (!(x & 1)) return s.nint + (x >> 1);
            x >>= 1;
        } else {
            x -= s.nsep;
        }
        return internal_slot<LAYOUT>(x, s, m);
    } else {
        if (x < s.span) {
            const uint32_t row = (uint32_t)__umul64hi(x, s.recip);
            if (x - row * (s.b + 1) < s.b) return s.nint + x - row;
            x = row;
        } else if (x < s.span + s.rem) {
            return s.nint + x - s.nsep;
        } else {
            x -= s.span + s.rem - s.nsep;
        }
        return internal_slot<LAYOUT>(x, s, m);
    }
}

// fills the map (a workgroup of at least 64 lanes), ends with a barrier
template <int LAYOUT>
__device__ inline void slot_map(const SlotShape &s, SlotMap<LAYOUT> &m) {
    const uint32_t tid = threadIdx.x;
    if constexpr (LAYOUT == TILE_BTREE) {
        if (tid < s.depth) m.level[tid] = (uint32_t)(ipow64(s.b + 1, s.depth - 1 - tid) - 1);
    }
    if constexpr (LAYOUT == TILE_VEB) {
        for (uint32_t i = tid + 2; i < (2u << SMALL_LEVELS); i += blockDim.x) {
            const uint32_t d = 31u - (uint32_t)__clz((int)i), x = i - (1u << d);
            m.small[i] = x < (1u << d) - 1
                             ? (uint8_t)mveb_pos32(x, (1u << d) - 1, s.classic != 0)
                             : (uint8_t)0;
        }
    }
    __syncthreads();
}

// workgroup b's tile of `tiles` in a grid of 8 * ceil(tiles / 8): workgroups go
// round robin to the 8 XCDs, and each takes one run of consecutive tiles, so
// that lines shared by neighbouring tiles are filled in one L2
__device__ inline uint32_t xcd_tile(uint32_t tiles) {
    const uint32_t per = (tiles + 7) >> 3;
    return (blockIdx.x & 7) * per + (blockIdx.x >> 3);
}

}   // namespace tl
