// The streaming kernel of the flat scan (scan_flat.hip) as scan.hip launches it.
#pragma once

#include "distance.h"
#include "store.h"

namespace vsag_amd {

struct FlatArgs {
    uint64_t n;
    uint64_t tile0;         // the launch covers tiles [tile0, tile_end)
    uint64_t tile_end;
    uint64_t tiles_per_chunk;
    uint64_t nq;
    uint32_t k;
    uint32_t S;
    uint32_t nslots;        // partial lists per query (all launches of the call)
    uint32_t slot0;         // first list of this launch
    const uint32_t* gate;   // per query: 0 = this launch leaves the query alone; null = every query
    uint32_t* bound;        // per query: ordered distance that k candidates are known to reach
    uint64_t* partial;      // nq x nslots x k keys
    uint32_t* partial_cnt;  // nq x nslots
    uint32_t* seed;         // nq x k smallest first-tile distances by wave class, or null (see kSeedTiles)
    const uint32_t* deny;   // filtered-out inner ids as a bit mask, or null
};

// One launch of the kernel with T queries per wave (1, 2, 4 or 8).
int launch_flat(const vsag_amd_store* s, int T, dim3 grid, dim3 block, size_t lds, const ScanArgs& a, const FlatArgs& f,
                hipStream_t st);

}  // namespace vsag_amd
