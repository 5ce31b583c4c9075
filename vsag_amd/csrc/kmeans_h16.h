// The fp16 pre-selection of the k-means assignment (kmeans_h16.hip), as kmeans.hip calls it.
#pragma once

#include "common.h"

namespace vsag_amd {

// What the kernels of a call tell each other.  Lengths are squared and as float bits, but `missed`.
struct KmeansH16State {
    uint32_t centred;      // largest |c - centre|^2 of the centroids that are not far
    uint32_t raw;          // largest |c|^2 of them
    uint32_t missed;       // largest length that fp16 misses of one of them
    uint32_t any_open;     // whether any row is left open
    uint32_t far_from;     // centroids with |c - centre|^2 above this are far: only their distance from the centre is used
    uint32_t nearest_far;  // least |c - centre|^2 of the far ones (infinity: none that any row could choose)
    uint32_t open_groups;  // of every sixteenth group of 64 rows: those in which the last probe left one open
};

struct KmeansH16Buffers {
    uint16_t* x16;      // [slab rows][dpad] rows of the slab, less the centre, in fp16
    uint16_t* c16;      // [k][dpad] centroids, less the centre, in fp16
    float2* xinfo;      // per row of the slab: length of what fp16 misses, length of what it holds
    float* xscale;      // per row of the slab: 1 / scale of the row
    float* group_min;   // [group of 64 centroids][3][slab rows]: the three least approximate distances
    float* centre;      // [dim]
    float* cnorm;       // [k] |c - centre|^2
    KmeansH16State* state;
    uint8_t* row_open;  // [n] rows the fp32 matrix cores still have to do
    uint32_t* open64;   // [n / 64] whether there is one among 64
};

bool kmeans_h16_takes(uint64_t n, uint32_t dim, uint32_t k);
void carve_kmeans_h16(Carver& c, uint64_t n, uint32_t dim, uint32_t k, KmeansH16Buffers* b);
// Fills best[] (keys of (|c|^2 - 2 <c, x>, centroid)) of every row but those marked in row_open / open64, whose keys are
// left at ~0.  cnorm_raw = |c|^2 per centroid; xnorm = |x|^2 per row, written in iteration 0.  From iteration 1 on the rows
// are those of the call before, so where one slab holds all of them their fp16 form is still there.
int launch_kmeans_h16(const float* x, uint64_t n, uint32_t dim, const float* cent, uint32_t k, const float* cnorm_raw,
                      float* xnorm, int iteration, unsigned long long* best, const KmeansH16Buffers& b, hipStream_t st);

}  // namespace vsag_amd
