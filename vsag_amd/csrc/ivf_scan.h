// The streaming kernel over posting lists (ivf_scan.hip) as ivf.hip launches it.
#pragma once

#include "distance.h"
#include "store.h"

namespace vsag_amd {

// Chunks a list of `tiles` tiles is cut into: about tiles_per_item tiles each, at most chunks_max chunks
// (longer lists get longer chunks); 0xFFFFFFFF = never cut.
__device__ inline uint32_t
list_chunks(uint32_t tiles, uint32_t tiles_per_item, uint32_t chunks_max) {
    if (tiles_per_item == 0xFFFFFFFFU) {
        return tiles != 0 ? 1U : 0U;
    }
    uint32_t chunks = (tiles + tiles_per_item - 1) / tiles_per_item;
    return chunks < chunks_max ? chunks : chunks_max;
}

struct IvfArgs {
    const uint32_t* ids;         // inner id per tile slot
    const uint32_t* list_tile;   // 2 nlist: first tile and end of the used tiles of every list
    const uint32_t* pair_off;    // nlist+1
    const uint32_t* item_off;    // nlist+1
    const uint32_t* sorted_pair; // pair index (q * nprobe + p) grouped by list
    uint32_t nlist;
    uint32_t nprobe;
    uint32_t dummy_query;        // index of an all-zero query row
    uint32_t k;
    uint32_t S;
    const uint32_t* deny;        // filtered-out inner ids as a bit mask, or null
    uint32_t tiles_per_item;     // 0xFFFFFFFF: whole lists
    uint32_t chunks_max;         // partial lists per pair
    uint32_t* bound;             // per query: ordered distance no final candidate can exceed
    uint32_t* seed;              // nq x k first-tile minima by work-item class, or null (flat scan's cold start)
    uint64_t* partial;           // npairs_total x chunks_max x k keys
    uint32_t* partial_cnt;       // npairs_total x chunks_max
    const uint32_t* gate;        // per query, or null: only queries with a raised gate are served
    // Direct mode (non-null `direct`): the work is a short array of pairs instead of the per-list grouping;
    // direct_count[0] of them, each worth chunks_max consecutive items.  More than direct_cap pairs are left to a
    // launch over the grouping (which in turn stands back when direct mode can take them).
    const uint32_t* direct;
    const uint32_t* direct_count;
    uint32_t direct_cap;
    const int32_t* buckets;      // direct mode: list of a pair
    // Residual lists (bucket_datacell.h:553-566): the codes hold x - c of their list's centroid c, and a distance is
    // put right by taking off the slot's bias (l2: -2 <c, decoded> - |c|^2) and the pair's term (<q, c>, twice for l2).
    const float* res_bias;       // per slot, or null
    const float* res_term;       // per pair (q * nprobe + p), or null: no residual
};

// One launch of the kernel with T queries per wave (1, 2 or 4).
int launch_ivf(const vsag_amd_store* s, int T, dim3 grid, dim3 block, size_t lds, hipStream_t st, const ScanArgs& a,
               const IvfArgs& v);

}  // namespace vsag_amd
