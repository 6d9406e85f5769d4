// The order between the tiles of the one-pass slides: tl_permute.hip's kernel on
// the CPU with a key type that notes from which slots of the array every tile
// loads and to which it stores, and with the tiles it waits for noted beside.  A
// slot that one tile stores to and another loads from has to be among those that
// the storing tile waits for, or the other may find it overwritten.  (Run serially
// the tiles cannot show that: each is read before the next.)  Arguments: layout
// (bst, btree), keys per node, then sizes.
#include "src/tl_slide_order.cpp"
#include <algorithm>
#include <cstdio>
#include <string>
#include <vector>

static uint64_t g_a0, g_n, g_tile;   // the array's address and keys; the tile at work
static size_t g_width;
static std::vector<uint32_t> g_loads, g_stores;      // tile of each slot, ~0u: none
static std::vector<std::vector<uint32_t>> g_waits;   // of each tile
static uint64_t g_twice;

namespace tl {
void emu_tile(uint32_t tile) { g_tile = tile; }
void emu_wait(uint32_t g) { g_waits[g_tile].push_back(g); }
}   // namespace tl

static void note(const void *p, std::vector<uint32_t> &of) {
    const uint64_t at = ((uint64_t)p - g_a0) / g_width;
    if ((uint64_t)p < g_a0 || at >= g_n) return;
    g_twice += of[at] != ~0u;
    of[at] = (uint32_t)g_tile;
}
template <typename T>
struct Key {
    T v;
    Key() : v(0) {}
    Key(const Key &o) : v(o.v) { note(&o, g_loads); }
    Key &operator=(const Key &o) {
        note(&o, g_loads);
        note(this, g_stores);
        v = o.v;
        return *this;
    }
};

using namespace tl;

template <typename T, int LAYOUT, bool INV>
static uint64_t run(uint64_t n, uint64_t b) {
    using K = Key<T>;
    const SlideShape s = slide_shape(LAYOUT, n, b, SLIDE_KEYS<K, INV>);
    std::vector<K> A(n), stash(s.nint - s.gap);
    std::vector<uint32_t> flags(s.tiles + 1, 0), err(1, 0);
    g_a0 = (uint64_t)A.data();
    g_n = n;
    g_width = sizeof(K);
    g_loads.assign(n, ~0u);
    g_stores.assign(n, ~0u);
    g_waits.assign(s.tiles, {});
    g_twice = 0;
    hipLaunchKernelGGL((k_level_slide<K, LAYOUT, INV>), dim3(1), dim3(SLIDE_NT), 0, nullptr,
                       A.data(), stash.data(), s, flags.data(), err.data(), (uint64_t)1 << 40);
    uint64_t bad = g_twice + err[0], pairs = 0;
    for (auto &w : g_waits) std::sort(w.begin(), w.end());
    for (uint64_t x = 0; x < n; x++) {
        if (g_stores[x] == ~0u || g_loads[x] == ~0u || g_stores[x] == g_loads[x]) continue;
        pairs++;
        const auto &w = g_waits[g_stores[x]];
        bad += !std::binary_search(w.begin(), w.end(), g_loads[x]);
        // tickets: from the right, the inverse from the left
        bad += INV ? g_loads[x] >= g_stores[x] : g_loads[x] <= g_stores[x];
    }
    fprintf(stderr, "[emu-order] %s b=%llu n=%llu %zu bytes%s: %u tiles, %llu slots of another, %llu wrong\n",
            LAYOUT == TILE_BST ? "bst" : "btree", (unsigned long long)b, (unsigned long long)n,
            sizeof(K), INV ? " inverse" : "", s.tiles, (unsigned long long)pairs,
            (unsigned long long)bad);
    return bad;
}

int main(int argc, char **argv) {
    if (argc < 4) return 2;
    const bool bst = std::string(argv[1]) == "bst";
    const uint64_t b = strtoull(argv[2], nullptr, 10);
    uint64_t bad = 0;
    for (int k = 3; k < argc; k++) {
        const uint64_t n = strtoull(argv[k], nullptr, 10);
        if (bst) {
            bad += run<uint64_t, TILE_BST, false>(n, 1) + run<uint64_t, TILE_BST, true>(n, 1);
            bad += run<uint32_t, TILE_BST, false>(n, 1) + run<uint32_t, TILE_BST, true>(n, 1);
        } else {
            bad += run<uint64_t, TILE_BTREE, false>(n, b) + run<uint64_t, TILE_BTREE, true>(n, b);
            bad += run<uint32_t, TILE_BTREE, false>(n, b) + run<uint32_t, TILE_BTREE, true>(n, b);
        }
    }
    return bad ? 1 : 0;
}
