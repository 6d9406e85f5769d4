// tl_tile.hpp -- lookups of large query batches (tl_tile.hip), shared by the
// one-array entry points, the learned lookups and the uneven batch.
#pragma once

#include "tl_internal.hpp"
#include "tl_slots.hpp"

namespace tl {

// one array as a lookup sees it.  tables / idx / tidx: the vEB query table
// set (idx and tidx null for a perfect tree of one table)
struct TileArray {
    const void *A;
    uint64_t n;
    uint32_t layout;   // TileLayout
    uint64_t b;        // keys per node (TILE_BTREE)
    const tl_veb_table *tables;
    const uint64_t *idx;
    const uint32_t *tidx;
    uint32_t table_size, ntables;
    bool classic;      // the table set is the classic vEB's
};

// answers q[0..nq) into ans[0..nq) on stream s by the faster of the two forms
// below, where one of them can and beats the kernels of tl_query.hip; else
// *taken = false and nothing is enqueued
tl_status large_query(Ctx *c, const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
                      uint64_t *ans, hipStream_t s, bool *taken);

// the tile-sorted form
bool tile_can(const TileArray &a, uint32_t dtype, uint64_t nq);
tl_status tile_query(Ctx *c, const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
                     uint64_t *ans, hipStream_t s);

// the partitioned form.  part_query() needs device memory ws of part_bytes()
// bytes, the stream's until its launches have run; part_wanted() says whether
// it is expected to take less than `other` times the other paths' time, and
// part_try() then runs it with a workspace of the library's.
bool part_can(const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
              const uint64_t *ans);
bool part_wanted(const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
                 const uint64_t *ans, double other);
uint64_t part_bytes(const TileArray &a, uint32_t dtype, uint64_t nq);
tl_status part_query(const TileArray &a, uint32_t dtype, const void *q, uint64_t nq, uint64_t *ans,
                     void *ws, hipStream_t s);
tl_status part_try(Ctx *c, const TileArray &a, uint32_t dtype, const void *q, uint64_t nq,
                   uint64_t *ans, hipStream_t s, double other, bool *taken);

// a caller on this host thread may lend its own workspace for the lookups it
// enqueues (the batch engine, one per branch of its graph); null: the library's
struct Workspace {
    void *mem = nullptr;
    uint64_t bytes = 0;
};
Workspace &query_workspace();

}   // namespace tl
