// CPU emulation of the tile-sorted lookups: tl_tile.hip built for the host
// over the HIP shim, one workgroup at a time with every lane a fiber, on
// exactly sized buffers under AddressSanitizer.  Every answer is compared with
// the CPU oracle's search (the reference's visiting order), with distinct
// keys and with keys that repeat.  Arguments: layout (bst, btree, mveb, veb,
// binary; veb-as-mveb, mveb-as-veb: a layout and its tables, given to the other
// one's query), key type (u32, u64, i32, i64), b, queries, then array sizes.
#include "hip/hip_runtime.h"
#include "src/tl_tile.hpp"
#include "tl_oracle.h"
#include <algorithm>
#include <random>
#include <stdio.h>
#include <stdlib.h>
#include <string>
#include <unistd.h>
#include <vector>

using namespace tl;


template <typename T, typename F1, typename FB>
static uint64_t check(const std::string &lay, uint32_t dtype, uint64_t n, uint64_t b, uint64_t nq,
                      bool repeats, F1 search, FB search_b) {
    std::mt19937_64 rng(n * 31 + nq);
    T *A = (T *)malloc(n * sizeof(T)), *Q = (T *)malloc(nq * sizeof(T));
    std::vector<T> keys(n);
    T v = (T)0 - (T)(n * 2);   // signed types start below zero
    if ((T)-1 > 0) v = 5;
    for (uint64_t i = 0; i < n; i++) {
        v = (T)(v + (repeats ? rng() % 2 : 1 + rng() % 7));
        keys[i] = A[i] = v;
    }
    for (uint64_t i = 0; i < nq; i++) {
        const uint64_t r = rng() % 16;
        Q[i] = r == 0   ? (T)rng()
               : r == 1 ? keys[0]
               : r == 2 ? keys[n - 1]
               : r < 9  ? keys[rng() % n]
                        : (T)(keys[rng() % n] + 1);
    }
    Q[0] = (T)(keys[0] - 1);   // smaller than every key
    TileArray a{A, n, TILE_SORTED, b, nullptr, nullptr, nullptr, 0, 0, false};
    std::vector<or_veb_table> tables(4096);
    uint64_t idx[64];
    uint32_t tidx[64], d = 0;
    if (lay == "bst") {
        a.layout = TILE_BST;
        if (sizeof(T) == 4) or_permute_bst_u32((uint32_t *)A, n, 1);
        else or_permute_bst_u64((uint64_t *)A, n, 1);
    } else if (lay == "btree") {
        a.layout = TILE_BTREE;
        if (sizeof(T) == 4) or_permute_btree_u32((uint32_t *)A, n, b, 1);
        else or_permute_btree_u64((uint64_t *)A, n, b, 1);
    } else if (lay != "binary") {
        a.layout = TILE_VEB;
        a.classic = lay.substr(0, 3) == "veb";
        if (a.classic) {
            if (sizeof(T) == 4) or_permute_classic_u32((uint32_t *)A, n, 1);
            else or_permute_classic_u64((uint64_t *)A, n, 1);
            or_classic_tableset(n, &d, &a.ntables, &a.table_size, tables.data(), idx, tidx);
        } else {
            if (sizeof(T) == 4) or_permute_mveb_u32((uint32_t *)A, n);
            else or_permute_mveb_u64((uint64_t *)A, n);
            or_veb_tableset(n, &d, &a.ntables, &a.table_size, tables.data(), idx, tidx);
        }
        a.tables = (const tl_veb_table *)tables.data();
        a.idx = idx;
        a.tidx = tidx;
        if (lay.find("-as-") != std::string::npos) a.classic = !a.classic;
    }
    uint64_t *got = (uint64_t *)malloc(nq * 8), *want = (uint64_t *)malloc(nq * 8);
    uint64_t bad = 0;
#ifdef EMU_PART
    const bool taken = part_can(a, dtype, Q, nq, got);
#else
    const bool taken = tile_can(a, dtype, nq);
#endif
    if (!taken) {
        fprintf(stderr, "[emu-tile] not taken\n");
        bad = 1;
    } else {
        Ctx c;
        c.num_cus = 4;
#ifdef EMU_PART
        void *ws = malloc(part_bytes(a, dtype, nq));
        part_query(a, dtype, Q, nq, got, ws, nullptr);
        free(ws);
#else
        tile_query(&c, a, dtype, Q, nq, got, nullptr);
#endif
        if (lay == "btree") search_b(A, n, b, Q, nq, want, 1);
        else if (lay == "binary" && repeats)   // the last key <= q, or n
            for (uint64_t i = 0; i < nq; i++) {
                const uint64_t le = std::upper_bound(A, A + n, Q[i]) - A;
                want[i] = le ? le - 1 : n;
            }
        else search(A, n, Q, nq, want, 1);
        for (uint64_t i = 0; i < nq; i++) bad += got[i] != want[i];
    }
    fprintf(stderr, "[emu-tile] %s dtype %u b=%llu n=%llu nq=%llu%s: %llu wrong\n", lay.c_str(),
            dtype, (unsigned long long)b, (unsigned long long)n, (unsigned long long)nq,
            repeats ? " repeats" : "", (unsigned long long)bad);
    free(A);
    free(Q);
    free(got);
    free(want);
    return bad;
}

int main(int argc, char **argv) {
    if (argc < 6) _exit(2);
    const std::string lay = argv[1], kind = argv[2];
    const uint64_t b = strtoull(argv[3], nullptr, 10), nq = strtoull(argv[4], nullptr, 10);
    uint64_t bad = 0;
    for (int k = 5; k < argc; k++)
        for (int repeats = 0; repeats < 2; repeats++) {
            const uint64_t n = strtoull(argv[k], nullptr, 10);
#define RUN(KIND, T, DT)                                                                         \
    if (kind == #KIND)                                                                           \
        bad += check<T>(lay, DT, n, b, nq, repeats,                                              \
                        lay == "bst"    ? or_search_bst_##KIND                                   \
                        : lay[0] == 'm' ? or_search_mveb_##KIND                                  \
                        : lay[0] == 'v' ? or_search_classic_##KIND                               \
                                        : or_search_binary_##KIND,                               \
                        or_search_btree_##KIND);
            RUN(u32, uint32_t, TL_U32)
            RUN(u64, uint64_t, TL_U64)
            RUN(i32, int32_t, TL_I32)
            RUN(i64, int64_t, TL_I64)
        }
    fflush(stderr);
    _exit(bad ? 1 : 0);
}
