// Batched IVF search: exact routing, posting-list scan with a fused per-(query, list) top-k, per-query
// merge, fp32 rerank (IVF::search<KNN_SEARCH>, src/algorithm/ivf/ivf.cpp:1693-1828; BucketDataCell::
// ScanBucketById, src/datacell/bucket_datacell.h:527-572; FlatBucketSearcher::Search,
// src/algorithm/ivf/flat_bucket_searcher.cpp:26-138; FlattenReorder::Reorder,
// src/impl/reorder/flatten_reorder.cpp:52-114).
//
// The reference walks "for each query, for each probed list".  Here the (query, list) pairs of the whole
// batch are regrouped by list on the device, so that one wave streams a posting list once for up to T
// queries that probe it.  A pair keeps its own LDS selector; what it cannot beat is cut off early by a
// per-query bound shared through global memory: the first probed list of every query is scanned in a
// first launch and its kcand-th distance seeds the bound for the remaining lists.  The bound only ever
// drops candidates that cannot be in the final kcand, so the result does not depend on scheduling.
//
// Few queries make few (query, list) pairs, and a wave per pair would leave the machine idle while each
// wave walks a whole list.  Then lists are cut into chunks of a few tiles, a work item is (list, query
// group, chunk), all probe columns go in one launch, and the cold waves learn a bound from each other's
// first tiles as in the flat scan.
#include "distance.h"
#include "ivf_scan.h"
#include "store.h"
#include "topk.h"

namespace vsag_amd {

struct ScanPlanIvf {
    int T;
    uint32_t S;
    QueryLayout ql;
    size_t qcode_bytes;
    uint64_t npairs;
    uint32_t tiles_per_item;  // 0xFFFFFFFF: a work item walks its whole list
    uint32_t chunks_max;      // partial lists per (query, list) pair
    bool chunked;             // lists cut into chunks, and seeds for a cold start
    bool nearest_first;       // chunked: the nearest list of every query ahead of the others, as the whole-list plan does
    bool seeded;
    bool mfma;                // probe columns behind the first go through the int8 matrix cores (ivf_i8.hip)
    bool planes;              // ... with sq8 codes: two int8 planes per query, records rescored (prefilter_i8.hip)
    bool bits1;               // ... with rabitq codes: expanded bits, records rescored (prefilter_rb.hip)
    bool pq;                  // ... with pqfs codes: one-hot centroid indices against the byte tables (ivf_pq.hip)
    bool h16;                 // ... sq8 codes beyond 128 dimensions: the fp16 matrix cores, records rescored
    bool f32;                 // ... with fp32 codes (sq8 beyond 128 dimensions): the fp32 matrix cores, records rescored
                              // (prefilter.hip)
    bool b16;                 // ... fp32 codes on the bf16 matrix cores instead, two bf16 values per operand
                              // (prefilter_b16.hip)
};

uint64_t rabitq_query_code_size(uint32_t dim, int metric, int query_bits);
int scan_contraction_mode(const vsag_amd_store* s);
void note_last_scan(int query_tile, uint64_t passes, uint64_t bytes_per_pass);
bool ivf_i8_supports(const vsag_amd_store* s);
uint32_t ivf_i8_lists_per_pair();
// sq8 lists: the two-plane test of prefilter_i8.hip over the same work split, records rescored by prefilter.hip.
bool ivf_sq8_i8_supports(const vsag_amd_store* s);
size_t ivf_sq8_i8_query_bytes(uint64_t nq);
size_t ivf_sq8_i8_scalar_floats(uint64_t nq);
size_t ivf_sq8_i8_tau_words(uint64_t nq);
uint32_t ivf_rescore_capacity();
int launch_ivf_sq8_i8(const vsag_amd_store* s, const float* qtab, uint32_t qstride, const float* qmeta, uint32_t qmeta_stride,
                      uint64_t nq, uint32_t nprobe, uint32_t p0, const uint32_t* pair_off, const uint32_t* item_off,
                      const uint32_t* sorted_pair, const uint32_t* bound, uint32_t kcand, uint8_t* q8, float* u, uint32_t* tau,
                      uint64_t* partial, uint32_t* partial_cnt, uint32_t* gate, hipStream_t st);
// rabitq lists (1-bit codes, 4-bit queries): the expanded-bits contraction of prefilter_rb.hip over 128 pairs per item.
bool ivf_pq_supports(const vsag_amd_store* s);
uint32_t ivf_pq_pairs_per_item();
int launch_ivf_pq(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t kcand,
                  const uint32_t* pair_off, const uint32_t* item_off, const uint32_t* sorted_pair, const uint32_t* bound,
                  int32_t* tq, uint64_t* partial, uint32_t* partial_cnt, uint32_t* gate, const int32_t* buckets,
                  uint32_t* gpairs, uint32_t gpairs_cap, hipStream_t st);
bool ivf_rb_supports(const vsag_amd_store* s);
uint32_t ivf_rb_pairs_per_item();
uint32_t ivf_rb_chunk_tiles();
size_t ivf_rb_scratch_bytes(const vsag_amd_store* s, uint64_t nq);
int launch_ivf_rb(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t nprobe, uint32_t p0, const uint32_t* pair_off,
                  const uint32_t* item_off, const uint32_t* sorted_pair, const uint32_t* bound, uint32_t kcand, uint8_t* scratch,
                  uint64_t* partial, uint32_t* partial_cnt, uint32_t* gate, hipStream_t st);
int launch_ivf_clear_gated(uint32_t* gate, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t* partial_cnt,
                           const int32_t* buckets, uint32_t* gpairs, uint32_t gpairs_cap, uint32_t k, hipStream_t st);
bool ivf_h16_supports(const vsag_amd_store* s);
uint32_t ivf_h16_pairs_per_item();
size_t ivf_h16_scratch_bytes(const vsag_amd_store* s, uint64_t nq);
int launch_ivf_h16(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t nprobe, uint32_t p0, const uint32_t* pair_off,
                   const uint32_t* item_off, const uint32_t* sorted_pair, const uint32_t* bound, uint32_t kcand, float* tau,
                   uint8_t* scratch, uint64_t* partial, uint32_t* partial_cnt, uint32_t* gate, hipStream_t st);
bool ivf_b16_supports(const vsag_amd_store* s);
uint32_t ivf_b16_pairs_per_item();
size_t ivf_b16_scratch_bytes(const vsag_amd_store* s, uint64_t nq);
int launch_ivf_b16(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t nprobe, uint32_t p0, const uint32_t* pair_off,
                   const uint32_t* item_off, const uint32_t* sorted_pair, const uint32_t* bound, uint32_t kcand, float* tau,
                   uint8_t* scratch, uint64_t* partial, uint32_t* partial_cnt, uint32_t* gate, const float* res_term,
                   hipStream_t st);
bool ivf_f32_supports(const vsag_amd_store* s);
uint32_t ivf_f32_pairs_per_item();
int launch_ivf_f32(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t nprobe, uint32_t p0, const uint32_t* pair_off,
                   const uint32_t* item_off, const uint32_t* sorted_pair, const uint32_t* bound, uint32_t kcand, float* tau,
                   uint64_t* partial, uint32_t* partial_cnt, uint32_t* gate, const float* res_term, hipStream_t st);
int launch_ivf_rescore(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t kcand,
                       uint32_t per_pair, uint64_t* partial, uint32_t* partial_cnt, const uint32_t* bound,
                       const float* res_term, hipStream_t st);
int launch_ivf_i8(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t kcand,
                  const uint32_t* pair_off, const uint32_t* item_off, const uint32_t* sorted_pair, const uint32_t* bound,
                  int32_t* tq, uint64_t* partial, uint32_t* partial_cnt, uint32_t* gate, const int32_t* buckets,
                  uint32_t* gpairs, uint32_t gpairs_cap, hipStream_t st);
int prepare_queries(const vsag_amd_store* s, const float* queries, uint64_t nq, uint64_t nq_pad, const QueryLayout& ql,
                    uint32_t* qtab, float* qmeta, uint8_t* qcodes, const FillJob* job, hipStream_t st);
ScanArgs make_scan_args(const vsag_amd_store* s, const QueryLayout& ql, const uint32_t* qtab, const float* qmeta);
void timing_begin(hipStream_t st);
void timing_end(hipStream_t st);
int launch_residual_terms(const vsag_amd_store* s, const float* queries, uint64_t nq, const int32_t* buckets, uint32_t nprobe,
                          float* terms, hipStream_t st);
int launch_merge_partials(const uint64_t* partial, const uint32_t* partial_cnt, const uint32_t* bound, uint32_t nslots,
                          uint32_t stride, uint32_t k, uint32_t S, uint64_t nq, uint32_t* ids, float* dists,
                          hipStream_t st);

// Pairs of probe columns [p0, p1): how many queries probe each list.
__global__ void
count_pairs_kernel(const int32_t* buckets, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t p1, uint32_t nlist,
                   uint32_t* counts) {
    uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    uint32_t w = p1 - p0;
    if (i >= nq * w) {
        return;
    }
    uint64_t q = i / w;
    uint32_t p = p0 + static_cast<uint32_t>(i % w);
    int32_t b = buckets[q * nprobe + p];
    if (b >= 0 && static_cast<uint32_t>(b) < nlist) {
        atomicAdd(&counts[b], 1U);
    }
}

// The same grouping for many pairs without an atomic per pair in global memory (hundreds of thousands of them on a
// few thousand counters take 0.1 ms per launch): a counting sort in three launches.  kRegroupGroups workgroups each
// take a run of the pairs; regroup_hist_kernel counts a run's pairs per list in LDS, regroup_prefix_kernel turns
// the counts of a list into the offsets of the runs inside the list (and their sum into counts[]), and
// regroup_scatter_kernel hands out the places of a run with a cursor per list in LDS.
constexpr uint32_t kRegroupGroups = 128;
constexpr uint32_t kRegroupLists = 8192;  // lists a workgroup's LDS holds a counter for

__global__ void __launch_bounds__(1024)
regroup_hist_kernel(const int32_t* buckets, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t p1, uint32_t nlist,
                    uint32_t* hist) {
    __shared__ uint32_t h[kRegroupLists];
    for (uint32_t b = threadIdx.x; b < nlist; b += blockDim.x) {
        h[b] = 0;
    }
    __syncthreads();
    const uint32_t w = p1 - p0;
    const uint64_t total = nq * w, per = (total + gridDim.x - 1) / gridDim.x;
    const uint64_t begin = blockIdx.x * per, end = begin + per < total ? begin + per : total;
    for (uint64_t i = begin + threadIdx.x; i < end; i += blockDim.x) {
        const uint64_t q = i / w;
        const int32_t b = buckets[q * nprobe + p0 + static_cast<uint32_t>(i - q * w)];
        if (b >= 0 && static_cast<uint32_t>(b) < nlist) {
            atomicAdd(&h[b], 1U);
        }
    }
    __syncthreads();
    for (uint32_t b = threadIdx.x; b < nlist; b += blockDim.x) {
        hist[static_cast<uint64_t>(blockIdx.x) * nlist + b] = h[b];
    }
}

__global__ void __launch_bounds__(256)
regroup_prefix_kernel(uint32_t* hist, uint32_t groups, uint32_t nlist, uint32_t* counts) {
    const uint32_t b = blockIdx.x * blockDim.x + threadIdx.x;
    if (b >= nlist) {
        return;
    }
    uint32_t running = 0;
    // Sixteen loads in flight at a time (the stores into the same array would otherwise keep them apart).
    for (uint32_t g0 = 0; g0 < groups; g0 += 16) {
        uint32_t c[16];
#pragma unroll
        for (uint32_t u = 0; u < 16; ++u) {
            c[u] = g0 + u < groups ? hist[static_cast<uint64_t>(g0 + u) * nlist + b] : 0U;
        }
#pragma unroll
        for (uint32_t u = 0; u < 16; ++u) {
            if (g0 + u < groups) {
                hist[static_cast<uint64_t>(g0 + u) * nlist + b] = running;
                running += c[u];
            }
        }
    }
    counts[b] = running;
}

__global__ void __launch_bounds__(1024)
regroup_scatter_kernel(const int32_t* buckets, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t p1, uint32_t nlist,
                       const uint32_t* pair_off, const uint32_t* hist, uint32_t* sorted_pair) {
    __shared__ uint32_t cursor[kRegroupLists];
    for (uint32_t b = threadIdx.x; b < nlist; b += blockDim.x) {
        cursor[b] = 0;
    }
    __syncthreads();
    const uint32_t w = p1 - p0;
    const uint64_t total = nq * w, per = (total + gridDim.x - 1) / gridDim.x;
    const uint64_t begin = blockIdx.x * per, end = begin + per < total ? begin + per : total;
    for (uint64_t i = begin + threadIdx.x; i < end; i += blockDim.x) {
        const uint64_t q = i / w;
        const uint32_t p = p0 + static_cast<uint32_t>(i - q * w);
        const int32_t b = buckets[q * nprobe + p];
        if (b >= 0 && static_cast<uint32_t>(b) < nlist) {
            const uint32_t pos = pair_off[b] + hist[static_cast<uint64_t>(blockIdx.x) * nlist + b] + atomicAdd(&cursor[b], 1U);
            sorted_pair[pos] = static_cast<uint32_t>(q * nprobe + p);
        }
    }
}

// Work items of a list: query groups x tile chunks.
__device__ inline uint32_t
list_items(uint32_t pairs, uint32_t T, uint32_t tiles, uint32_t tiles_per_item, uint32_t chunks_max) {
    return ((pairs + T - 1) / T) * list_chunks(tiles, tiles_per_item, chunks_max);
}

// Exclusive prefix sums of two per-thread values over a workgroup of up to 1024 threads; wave totals go
// through `wave_sums` (2 x 16 words of LDS).  Returns the grand totals.
__device__ inline void
block_exclusive_scan2(uint32_t& a, uint32_t& b, uint32_t (*wave_sums)[16], uint32_t& total_a, uint32_t& total_b) {
    const uint32_t lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6, nwaves = (blockDim.x + kWave - 1) >> 6;
    uint32_t ia = a, ib = b;
    for (int off = 1; off < kWave; off <<= 1) {
        uint32_t oa = __shfl_up(ia, off), ob = __shfl_up(ib, off);
        if (static_cast<int>(lane) >= off) {
            ia += oa;
            ib += ob;
        }
    }
    if (lane == kWave - 1) {
        wave_sums[0][wave] = ia;
        wave_sums[1][wave] = ib;
    }
    __syncthreads();
    uint32_t ba = 0, bb = 0;
    total_a = 0;
    total_b = 0;
    for (uint32_t w = 0; w < nwaves; ++w) {
        uint32_t sa = wave_sums[0][w], sb = wave_sums[1][w];
        if (w < wave) {
            ba += sa;
            bb += sb;
        }
        total_a += sa;
        total_b += sb;
    }
    a = ba + ia - a;
    b = bb + ib - b;
}

// One workgroup: exclusive prefix sums of the pair counts and of the work items.
__global__ void __launch_bounds__(1024)
offsets_kernel(const uint32_t* counts, const uint32_t* list_tile, uint32_t nlist, uint32_t T, uint32_t tiles_per_item,
               uint32_t chunks_max, uint32_t* pair_off, uint32_t* item_off) {
    __shared__ uint32_t wave_sums[2][16];
    uint32_t per = (nlist + blockDim.x - 1) / blockDim.x;
    uint32_t begin = threadIdx.x * per;
    uint32_t end = begin + per < nlist ? begin + per : nlist;
    uint32_t sp = 0, si = 0;
    for (uint32_t i = begin; i < end; ++i) {
        sp += counts[i];
        si += list_items(counts[i], T, list_tile[2 * i + 1] - list_tile[2 * i], tiles_per_item, chunks_max);
    }
    uint32_t rp = sp, ri = si, all_pairs, all_items;
    block_exclusive_scan2(rp, ri, wave_sums, all_pairs, all_items);
    if (threadIdx.x == 0) {
        pair_off[nlist] = all_pairs;
        item_off[nlist] = all_items;
    }
    for (uint32_t i = begin; i < end; ++i) {
        pair_off[i] = rp;
        item_off[i] = ri;
        rp += counts[i];
        ri += list_items(counts[i], T, list_tile[2 * i + 1] - list_tile[2 * i], tiles_per_item, chunks_max);
    }
}

__global__ void
scatter_pairs_kernel(const int32_t* buckets, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t p1, uint32_t nlist,
                     const uint32_t* pair_off, uint32_t* cursor, uint32_t* sorted_pair) {
    uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    uint32_t w = p1 - p0;
    if (i >= nq * w) {
        return;
    }
    uint64_t q = i / w;
    uint32_t p = p0 + static_cast<uint32_t>(i % w);
    int32_t b = buckets[q * nprobe + p];
    if (b >= 0 && static_cast<uint32_t>(b) < nlist) {
        uint32_t pos = pair_off[b] + atomicAdd(&cursor[b], 1U);
        sorted_pair[pos] = static_cast<uint32_t>(q * nprobe + p);
    }
}

// The three regrouping steps above for a small batch (probe columns [p0, p1); ALL: they are all) in one workgroup.  A chain of
// latencies bounds it: a bucket is loaded, its counter raised, its place written.  With the counters in LDS (LDS: lists up to
// kRegroupLists; more lists count in memory) and kRegroupInFlight buckets of a thread loaded together, 24 000 pairs of 512 lists
// take 17 us (one bucket at a time, counters in memory: 81; the call 651 -> 589), 32 pairs of 1024 lists 5 (the call 127 -> 122).
constexpr uint32_t kRegroupInFlight = 8;

template <bool LDS, bool ALL>
__global__ void __launch_bounds__(1024)
regroup_small_kernel(const int32_t* buckets, uint64_t nq, uint32_t nprobe, uint32_t p0, uint32_t p1,
                     const uint32_t* list_tile, uint32_t nlist, uint32_t T, uint32_t tiles_per_item, uint32_t chunks_max, uint32_t* counts, uint32_t* cursor,
                     uint32_t* pair_off, uint32_t* item_off, uint32_t* sorted_pair) {
    __shared__ uint32_t wave_sums[2][16];
    __shared__ uint32_t place[LDS ? kRegroupLists : 1];  // of a list: its pairs, then the place of its next one
    const uint32_t cols = p1 - p0;
    const uint64_t npairs = nq * cols;
    // (a pair of all columns, from its place among these; both fit 32 bits)
    auto pair_of = [&](uint64_t i) {
        const uint32_t at = static_cast<uint32_t>(i);
        return ALL ? at : at / cols * nprobe + p0 + at % cols;
    };
    for (uint32_t i = threadIdx.x; i < nlist; i += blockDim.x) {
        if (LDS) {
            place[i] = 0;
        } else {
            counts[i] = 0;
            cursor[i] = 0;
        }
    }
    __syncthreads();
    auto each_pair = [&](auto&& visit) {
        for (uint64_t i0 = threadIdx.x; i0 < npairs; i0 += static_cast<uint64_t>(blockDim.x) * kRegroupInFlight) {
            int32_t b[kRegroupInFlight];
#pragma unroll
            for (uint32_t u = 0; u < kRegroupInFlight; ++u) {
                const uint64_t i = i0 + static_cast<uint64_t>(u) * blockDim.x;
                b[u] = i < npairs ? buckets[pair_of(i)] : -1;
            }
#pragma unroll
            for (uint32_t u = 0; u < kRegroupInFlight; ++u) {
                if (b[u] >= 0 && static_cast<uint32_t>(b[u]) < nlist) {
                    visit(static_cast<uint32_t>(b[u]), pair_of(i0 + static_cast<uint64_t>(u) * blockDim.x));
                }
            }
        }
    };
    each_pair([&](uint32_t b, uint32_t) { atomicAdd(LDS ? &place[b] : &counts[b], 1U); });
    if (!LDS) {
        // The counts were made by atomics in L2; the fences keep the plain loads below from an older cached line.
        __threadfence();
    }
    __syncthreads();
    if (!LDS) {
        __threadfence();
    }
    uint32_t per = (nlist + blockDim.x - 1) / blockDim.x;
    uint32_t begin = threadIdx.x * per;
    uint32_t end = begin + per < nlist ? begin + per : nlist;
    uint32_t sp = 0, si = 0;
    for (uint32_t i = begin; i < end; ++i) {
        const uint32_t n = LDS ? place[i] : counts[i];
        sp += n;
        si += list_items(n, T, list_tile[2 * i + 1] - list_tile[2 * i], tiles_per_item, chunks_max);
    }
    uint32_t rp = sp, ri = si, all_pairs, all_items;
    block_exclusive_scan2(rp, ri, wave_sums, all_pairs, all_items);
    if (threadIdx.x == 0) {
        pair_off[nlist] = all_pairs;
        item_off[nlist] = all_items;
    }
    for (uint32_t i = begin; i < end; ++i) {
        const uint32_t n = LDS ? place[i] : counts[i];
        pair_off[i] = rp;
        item_off[i] = ri;
        if (LDS) {
            place[i] = rp;
        }
        rp += n;
        ri += list_items(n, T, list_tile[2 * i + 1] - list_tile[2 * i], tiles_per_item, chunks_max);
    }
    __syncthreads();
    each_pair([&](uint32_t b, uint32_t i) {
        const uint32_t pos = LDS ? atomicAdd(&place[b], 1U) : pair_off[b] + atomicAdd(&cursor[b], 1U);
        sorted_pair[pos] = i;
    });
}

// Exact fp32 distances of the candidates of one query, best k kept.  One workgroup of four waves per query;
// sixteen lanes share a candidate, so a workgroup has sixteen gathered rows in flight.
constexpr uint32_t kRerankThreads = 256;

__global__ void __launch_bounds__(kRerankThreads)
rerank_kernel(const float* raw, uint64_t n, uint32_t dim, int metric, const float* queries, const uint32_t* cand,
              uint32_t kcand, uint32_t k, uint32_t S, uint32_t* ids, float* dists) {
    extern __shared__ uint64_t lds[];
    const uint32_t tid = threadIdx.x;
    const uint32_t sub = tid >> 4, l = tid & 15;  // candidate slot of this step, lane within it
    const uint64_t q = blockIdx.x;
    const float* qv = queries + q * dim;
    for (uint32_t i = tid; i < S; i += kRerankThreads) {
        lds[i] = kInfKey;
    }
    float inv_norm = 1.0F;
    if (metric == VSAG_AMD_METRIC_COSINE) {
        float s = 0.0F;
        for (uint32_t d = l; d < dim; d += 16) {
            s = fmaf(qv[d], qv[d], s);
        }
        for (int off = 8; off > 0; off >>= 1) {
            s += __shfl_xor(s, off);
        }
        inv_norm = s > 0.0F ? 1.0F / sqrtf(s) : 1.0F;
    }
    __syncthreads();
    const bool vec4 = (dim & 3) == 0;
    for (uint32_t j0 = 0; j0 < kcand; j0 += kRerankThreads / 16) {
        const uint32_t j = j0 + sub;
        uint32_t id = j < kcand ? as_const(cand)[q * kcand + j] : VSAG_AMD_INVALID_ID;
        const bool live = id != VSAG_AMD_INVALID_ID && id < n;
        const float* x = raw + static_cast<uint64_t>(live ? id : 0) * dim;
        float s = 0.0F, xx = 0.0F;
        if (live) {
            if (vec4) {
                for (uint32_t d = l * 4; d < dim; d += 64) {
                    float4 xv = *reinterpret_cast<const float4*>(x + d);
                    float4 qq = *reinterpret_cast<const float4*>(qv + d);
                    if (metric == VSAG_AMD_METRIC_L2) {
                        float t0 = qq.x - xv.x, t1 = qq.y - xv.y, t2 = qq.z - xv.z, t3 = qq.w - xv.w;
                        s = fmaf(t0, t0, s);
                        s = fmaf(t1, t1, s);
                        s = fmaf(t2, t2, s);
                        s = fmaf(t3, t3, s);
                    } else {
                        s = fmaf(qq.x, xv.x, s);
                        s = fmaf(qq.y, xv.y, s);
                        s = fmaf(qq.z, xv.z, s);
                        s = fmaf(qq.w, xv.w, s);
                        xx = fmaf(xv.x, xv.x, xx);
                        xx = fmaf(xv.y, xv.y, xx);
                        xx = fmaf(xv.z, xv.z, xx);
                        xx = fmaf(xv.w, xv.w, xx);
                    }
                }
            } else {
                for (uint32_t d = l; d < dim; d += 16) {
                    float xv = x[d];
                    if (metric == VSAG_AMD_METRIC_L2) {
                        float t = qv[d] - xv;
                        s = fmaf(t, t, s);
                    } else {
                        s = fmaf(qv[d], xv, s);
                        xx = fmaf(xv, xv, xx);
                    }
                }
            }
        }
        for (int off = 8; off > 0; off >>= 1) {
            s += __shfl_xor(s, off);
            xx += __shfl_xor(xx, off);
        }
        if (live && l == 0) {
            float dist;
            if (metric == VSAG_AMD_METRIC_L2) {
                dist = s;
            } else if (metric == VSAG_AMD_METRIC_IP) {
                dist = 1.0F - s;
            } else {
                float xn = xx > 0.0F ? 1.0F / sqrtf(xx) : 1.0F;
                dist = 1.0F - s * inv_norm * xn;
            }
            lds[j] = make_key(dist, id);
        }
    }
    __syncthreads();
    if (tid >= kWave) {
        return;
    }
    wave_bitonic_sort(lds, S, tid);
    for (uint32_t i = tid; i < k; i += kWave) {
        uint64_t key = lds[i];
        if (key == kInfKey) {
            ids[q * k + i] = VSAG_AMD_INVALID_ID;
            dists[q * k + i] = __builtin_inff();
        } else {
            ids[q * k + i] = static_cast<uint32_t>(key);
            dists[q * k + i] = ordered_to_float(static_cast<uint32_t>(key >> 32));
        }
    }
}

// Exact fp32 distance of every (query, inner id) pair, in the order given: what the rerank computes for a candidate,
// without the selection.  Sixteen lanes share a pair; ids beyond the rows (or VSAG_AMD_INVALID_ID) give -1.
__global__ void __launch_bounds__(kRerankThreads)
rows_distances_kernel(const float* raw, uint64_t n, uint32_t dim, int metric, const float* queries, const uint32_t* ids,
                      uint32_t count, float* dists) {
    const uint32_t tid = threadIdx.x;
    const uint32_t sub = tid >> 4, l = tid & 15;
    const uint64_t q = blockIdx.y;
    const float* qv = queries + q * dim;
    float inv_norm = 1.0F;
    if (metric == VSAG_AMD_METRIC_COSINE) {
        float s = 0.0F;
        for (uint32_t d = l; d < dim; d += 16) {
            s = fmaf(qv[d], qv[d], s);
        }
        for (int off = 8; off > 0; off >>= 1) {
            s += __shfl_xor(s, off);
        }
        inv_norm = s > 0.0F ? 1.0F / sqrtf(s) : 1.0F;
    }
    const uint32_t j = blockIdx.x * (kRerankThreads / 16) + sub;
    const uint32_t id = j < count ? ids[q * count + j] : VSAG_AMD_INVALID_ID;
    const bool live = id != VSAG_AMD_INVALID_ID && id < n;
    const float* x = raw + static_cast<uint64_t>(live ? id : 0) * dim;
    float s = 0.0F, xx = 0.0F;
    if (live) {
        if ((dim & 3) == 0) {
            for (uint32_t d = l * 4; d < dim; d += 64) {
                const float4 xv = *reinterpret_cast<const float4*>(x + d);
                const float4 qq = *reinterpret_cast<const float4*>(qv + d);
                if (metric == VSAG_AMD_METRIC_L2) {
                    const float t0 = qq.x - xv.x, t1 = qq.y - xv.y, t2 = qq.z - xv.z, t3 = qq.w - xv.w;
                    s = fmaf(t0, t0, s);
                    s = fmaf(t1, t1, s);
                    s = fmaf(t2, t2, s);
                    s = fmaf(t3, t3, s);
                } else {
                    s = fmaf(qq.x, xv.x, s);
                    s = fmaf(qq.y, xv.y, s);
                    s = fmaf(qq.z, xv.z, s);
                    s = fmaf(qq.w, xv.w, s);
                    xx = fmaf(xv.x, xv.x, xx);
                    xx = fmaf(xv.y, xv.y, xx);
                    xx = fmaf(xv.z, xv.z, xx);
                    xx = fmaf(xv.w, xv.w, xx);
                }
            }
        } else {
            for (uint32_t d = l; d < dim; d += 16) {
                const float xv = x[d];
                if (metric == VSAG_AMD_METRIC_L2) {
                    const float t = qv[d] - xv;
                    s = fmaf(t, t, s);
                } else {
                    s = fmaf(qv[d], xv, s);
                    xx = fmaf(xv, xv, xx);
                }
            }
        }
    }
    for (int off = 8; off > 0; off >>= 1) {
        s += __shfl_xor(s, off);
        xx += __shfl_xor(xx, off);
    }
    if (j < count && l == 0) {
        float dist = -1.0F;
        if (live) {
            if (metric == VSAG_AMD_METRIC_L2) {
                dist = s;
            } else if (metric == VSAG_AMD_METRIC_IP) {
                dist = 1.0F - s;
            } else {
                const float xn = xx > 0.0F ? 1.0F / sqrtf(xx) : 1.0F;
                dist = 1.0F - s * inv_norm * xn;
            }
        }
        dists[q * count + j] = dist;
    }
}

struct IvfBuffers {
    uint32_t* qtab;
    float* qmeta;
    uint8_t* qcodes;
    uint32_t* counts;     // nlist + 1
    uint32_t* cursor;     // nlist + 1
    uint32_t* pair_off;   // nlist + 1
    uint32_t* item_off;   // nlist + 1
    uint32_t* sorted_pair;
    uint32_t* hist;       // counting sort of many pairs: kRegroupGroups x nlist
    uint32_t* bound;
    uint32_t* seed;
    uint32_t* partial_cnt;
    uint64_t* partial;
    uint32_t* gate;       // mfma: nq + 3 (flags, raised gates, the pairs to scan again, the pairs queued)
    int32_t* tq;          // mfma: 2 (nq + 1)
    uint32_t* gpairs;     // mfma: pairs of gated queries, kGatedPairsCap
    uint8_t* q8;          // sq8 lists on the matrix cores: the planes of the queries, their scalars and thresholds
                          // (rabitq lists: the queries as bytes and their four factors)
    float* q8_u;
    uint32_t* q8_tau;
    float* res_term;      // residual lists: per pair
};

// Pairs of gated queries the direct fallback launch takes; more go through the per-list grouping.
constexpr uint32_t kGatedPairsCap = 32768;

static void
plan_ivf(const vsag_amd_store* s, uint64_t nq, uint32_t nprobe, uint32_t kcand, ScanPlanIvf* p, bool fine = true) {
    p->S = selector_slots(kcand);
    uint64_t npairs = nq * nprobe;
    uint64_t avg = s->nlist ? npairs / s->nlist : 1;
    int t = 4;
    if (s->kind == VSAG_AMD_KIND_RABITQ || ((s->kind == VSAG_AMD_KIND_SQ8 || s->kind == VSAG_AMD_KIND_SQ4) &&
                                            s->metric == VSAG_AMD_METRIC_L2)) {
        t = 2;
    }
    while (t > 1 && static_cast<uint64_t>(t) > avg) {
        t >>= 1;
    }
    while (t > 1 && static_cast<size_t>(t) * p->S * 8 > 65536) {
        t >>= 1;
    }
    p->T = t;
    p->ql = query_layout(s);
    p->qcode_bytes = query_staging_bytes(s, nq);
    p->npairs = npairs;
    // Enough (list, query group) items to fill the machine: every item walks its whole list, the nearest list
    // of every query goes first.  Otherwise lists are cut into chunks of at least four tiles for about 4096 items in all (a probed
    // list is taken as twice the average length), at most 64 chunks per list and 256 MiB of partial lists.
    // fp32 and sq8 codes against four queries an item make long items of many registers: from some 15 600 pairs on four times
    // as many keep the machine evenly busy to the end (fp32 l2 200k x 200, 512 lists, k 20, 1000 queries x 24: 480 -> 414 us,
    // k 100 568 -> 497; 200k x 768 1471 -> 1245; ip 1M x 96 459 -> 372; sq8 ip 200k x 200, 80 candidates, 457 -> 415; 60
    // points of these kinds, 1.02 times slower at most).  Fewer pairs lose (200k x 768, 1000 x 8: 646 -> 731), and so do two queries an
    // item (sq8 l2 1M x 96, 200 candidates, 2000 x 8: 1046 -> 1139; rabitq 590 -> 668) and sq4_uniform codes (533 -> 595).
    const uint64_t groups = div_up(npairs, static_cast<uint64_t>(t));
    p->chunked = groups < 8192 && s->max_list_tiles > 2;
    p->tiles_per_item = 0xFFFFFFFFU;
    p->chunks_max = 1;
    bool four_pays = false;
    uint64_t items = nprobe;  // of a query, in lists of average length
    if (p->chunked) {
        const uint64_t avg_tiles = std::max<uint64_t>(1, s->nlist ? s->ntiles / s->nlist : 1);
        const bool four = fine && t == 4 && groups >= 3900 && kcand <= 256 &&
                          (s->kind == VSAG_AMD_KIND_FP32 || s->kind == VSAG_AMD_KIND_SQ8);
        const uint64_t tpi = std::max<uint64_t>(4, div_up(groups * avg_tiles * 2, four ? 16384 : 4096));
        uint64_t cap = std::min<uint64_t>(64, div_up(s->max_list_tiles, tpi));
        while (cap > 1 && npairs * cap * kcand * 8 > (256ull << 20)) {
            cap /= 2;
        }
        p->tiles_per_item = static_cast<uint32_t>(std::min<uint64_t>(tpi, 0x7FFFFFFFU));
        p->chunks_max = static_cast<uint32_t>(cap);
        four_pays = four;
        items = nprobe * std::min<uint64_t>(cap, div_up(avg_tiles, tpi));
    }
    // Seeds give a bound once every one of kcand slots holds a minimum; with fewer items than that a query looks at its row of
    // them in vain, a wait for memory per tile (fp32 l2 200k x 200, 512 lists, k 100, 1000 queries x 24: 706 -> 667 us).
    const bool fills = kcand <= items;
    p->seeded = p->chunked && kcand <= 256 && fills;
    // Then the nearest list of every query goes ahead where its bound spares the others more selecting than its own scan costs: sq8
    // codes of up to 256 dimensions (cheap to scan), lists of four tiles or more but at most six times as many codes as are kept,
    // and 6000 (query, tile) pairs in that pass, which fewer leave as a chain of latencies on a chip that is not full.  173 points
    // of both sides, time without it over time with it: above the lines 0.95 to 1.37, 1.12 at the mean (sq8 ip 200k x 200, 512
    // lists, 80 kept, 1000 queries x 24: 560 -> 475 us; 55k x 100, 128 lists, 200 kept, 3136 x 8: 1088 -> 794; the worst, 658k x
    // 256, 2174 lists, 80 kept, 1165 x 17: 445 -> 469), below them 0.82 to 1.33, 1.01 at the mean and every third below 0.985.
    // Nor with ten times as many codes as are kept, 1M x 96, 1000 lists, 100 kept, 900 x 20: 407 -> 428; nor of 960 dimensions,
    // 300k, 1000 lists, 200 kept, 1500 x 12: 1516 -> 1701; nor fp32 codes, 200k x 200, k 100: 667 -> 736.
    p->nearest_first = p->chunked && four_pays && !fills && s->kind == VSAG_AMD_KIND_SQ8 && s->dpad <= 256 &&
                       s->ntiles >= 4ull * s->nlist && nq * s->ntiles >= 6000ull * s->nlist &&
                       s->ntiles * kWave <= 6ull * kcand * s->nlist;
    // Large batches on sq4_uniform (and sq8_uniform / l2) lists: the streaming kernel scans the nearest list of every query, the int8
    // matrix cores the other columns, into two private lists per (query, list) pair.
    p->mfma = !p->chunked && nprobe > 1 && scan_contraction_mode(s) >= 0 && ivf_i8_supports(s) &&
              s->residual_centroids_dev == nullptr &&
              npairs * ivf_i8_lists_per_pair() * kcand * 8 <= (8ull << 30);
    // sq8 lists of at most 128 dimensions: the same split with the two-plane test and an exact rescoring.
    p->planes = !p->mfma && !p->chunked && nprobe > 1 && scan_contraction_mode(s) >= 0 && ivf_sq8_i8_supports(s) &&
                kcand <= ivf_rescore_capacity() && npairs * ivf_i8_lists_per_pair() * kcand * 8 <= (8ull << 30);
    p->bits1 = !p->mfma && !p->planes && !p->chunked && nprobe > 1 && scan_contraction_mode(s) >= 0 && ivf_rb_supports(s) &&
               kcand <= ivf_rescore_capacity() && npairs * ivf_i8_lists_per_pair() * kcand * 8 <= (8ull << 30);
    p->pq = !p->mfma && !p->planes && !p->bits1 && !p->chunked && nprobe > 1 && scan_contraction_mode(s) >= 0 &&
            ivf_pq_supports(s) && s->residual_centroids_dev == nullptr &&
            npairs * ivf_i8_lists_per_pair() * kcand * 8 <= (8ull << 30);
    // sq8 lists of more than 128 dimensions: the fp16 matrix cores (mode 2 keeps the fp32 ones; residual lists too).
    p->h16 = !p->mfma && !p->planes && !p->bits1 && !p->pq && !p->chunked && nprobe > 1 && scan_contraction_mode(s) >= 0 &&
             (scan_contraction_mode(s) != 2 || s->kind == VSAG_AMD_KIND_SQ4) && ivf_h16_supports(s) &&
             kcand <= ivf_rescore_capacity() &&
             npairs * ivf_i8_lists_per_pair() * kcand * 8 <= (8ull << 30);
    // fp32 lists, sq8 lists the fp16 pass does not take: the fp32 matrix cores pre-select, the same exact rescoring.
    p->f32 = !p->h16 && !p->mfma && !p->planes && !p->bits1 && !p->pq && !p->chunked && nprobe > 1 && scan_contraction_mode(s) >= 0 &&
             ivf_f32_supports(s) && kcand <= ivf_rescore_capacity() &&
             npairs * ivf_i8_lists_per_pair() * kcand * 8 <= (8ull << 30);
    // (fp32 lists: the bf16 ones on two bf16 values per operand, unless mode 2 asks for the fp32 ones)
    p->b16 = p->f32 && scan_contraction_mode(s) != 2 && ivf_b16_supports(s);
    p->mfma = p->mfma || p->planes || p->bits1 || p->pq || p->h16 || p->f32;
    if (p->mfma) {
        p->chunks_max = ivf_i8_lists_per_pair();
    }
}

// Whether the pairs of a call are grouped by the counting sort (regroup_hist_kernel ...) rather than with an atomic
// per pair.
static bool
regroup_by_sort(const vsag_amd_store* s, uint64_t npairs) {
    return npairs >= 65536 && s->nlist <= kRegroupLists;
}

static size_t
carve_ivf(Carver& c, const vsag_amd_store* s, const ScanPlanIvf& p, uint64_t nq, uint32_t kcand, IvfBuffers* b) {
    b->qtab = c.take<uint32_t>((nq + 1) * p.ql.qstride);
    b->qmeta = c.take<float>((nq + 1) * p.ql.qmeta);
    b->qcodes = c.take<uint8_t>(p.qcode_bytes);
    b->counts = c.take<uint32_t>(s->nlist + 1);
    b->cursor = c.take<uint32_t>(s->nlist + 1);
    b->pair_off = c.take<uint32_t>(s->nlist + 1);
    b->item_off = c.take<uint32_t>(s->nlist + 1);
    b->sorted_pair = c.take<uint32_t>(p.npairs);
    b->hist = c.take<uint32_t>(regroup_by_sort(s, p.npairs) ? static_cast<size_t>(kRegroupGroups) * s->nlist : 0);
    b->bound = c.take<uint32_t>(nq);
    b->seed = c.take<uint32_t>(p.seeded ? nq * kcand : 0);
    b->partial_cnt = c.take<uint32_t>(p.npairs * p.chunks_max);
    b->partial = c.take<uint64_t>(p.npairs * p.chunks_max * kcand);
    b->gate = c.take<uint32_t>(p.mfma ? nq + 3 : 0);
    b->gpairs = c.take<uint32_t>(p.mfma ? kGatedPairsCap : 0);
    b->tq = c.take<int32_t>(p.mfma ? 2 * (nq + 1) : 0);  // thresholds, then (sq8_uniform) the sums of the query values
    b->q8 = c.take<uint8_t>(p.planes ? ivf_sq8_i8_query_bytes(nq) : p.bits1 ? ivf_rb_scratch_bytes(s, nq)
                            : p.h16  ? ivf_h16_scratch_bytes(s, nq) : p.b16 ? ivf_b16_scratch_bytes(s, nq) : 0);
    b->q8_u = c.take<float>(p.planes ? ivf_sq8_i8_scalar_floats(nq) : 0);
    b->q8_tau = c.take<uint32_t>(p.planes ? ivf_sq8_i8_tau_words(nq) : 0);
    b->res_term = c.take<float>(s->residual_centroids_dev != nullptr ? p.npairs : 0);
    return c.used;
}

static int
check_ivf(const vsag_amd_store* s, uint64_t nq, uint32_t nprobe, uint32_t kcand) {
    VA_CHECK_ARG(s != nullptr, "store is null");
    VA_CHECK_ARG(s->nlist > 0, "ivf scan on a flat store");
    VA_CHECK_ARG(kcand >= 1 && kcand <= kMaxTopK, "kcand must be in [1, %u], got %u", kMaxTopK, kcand);
    VA_CHECK_ARG(nprobe >= 1 && nprobe <= 65536, "nprobe must be in [1, 65536], got %u", nprobe);
    VA_CHECK_ARG(nq >= 1 && nq * nprobe < 0xFFFFFFFFull, "nq * nprobe must be below 2^32 - 1");
    return 0;
}

static inline uint32_t
blocks_for(uint64_t n) {
    return static_cast<uint32_t>(div_up(n ? n : 1, 256));
}

}  // namespace vsag_amd

using namespace vsag_amd;

extern "C" size_t
vsag_amd_ivf_route_workspace_bytes(const vsag_amd_store_t* centroids, uint64_t nq, uint32_t nprobe) {
    return vsag_amd_flat_scan_workspace_bytes(centroids, nq, nprobe);
}

extern "C" int
vsag_amd_ivf_route(const vsag_amd_store_t* centroids, const float* queries_dev, uint64_t nq, uint32_t nprobe,
                   int32_t* buckets_dev, float* dists_dev, void* workspace_dev, size_t workspace_bytes, void* stream) {
    VA_CHECK_ARG(centroids != nullptr && centroids->kind == VSAG_AMD_KIND_FP32,
                 "routing needs an fp32 store of centroids");
    // VSAG_AMD_INVALID_ID and -1 are the same 32 bits, so the id buffer is the bucket buffer.
    return vsag_amd_flat_scan_topk(centroids, queries_dev, nq, nprobe, reinterpret_cast<uint32_t*>(buckets_dev),
                                   dists_dev, workspace_dev, workspace_bytes, stream);
}

extern "C" size_t
vsag_amd_ivf_scan_workspace_bytes(const vsag_amd_store_t* s, uint64_t nq, uint32_t nprobe, uint32_t kcand) {
    if (check_ivf(s, nq, nprobe, kcand) != 0) {
        return 0;
    }
    ScanPlanIvf p;
    plan_ivf(s, nq, nprobe, kcand, &p);
    Carver c(nullptr, 0);
    IvfBuffers b;
    return carve_ivf(c, s, p, nq, kcand, &b) + 256;
}

extern "C" int
vsag_amd_ivf_scan_topk(const vsag_amd_store_t* s, const float* queries_dev, uint64_t nq, const int32_t* buckets_dev,
                       uint32_t nprobe, uint32_t kcand, uint32_t* ids_dev, float* dists_dev, void* workspace_dev,
                       size_t workspace_bytes, void* stream) {
    return vsag_amd_ivf_scan_topk_ex(s, queries_dev, nq, buckets_dev, nprobe, kcand, nullptr, ids_dev, dists_dev,
                                     workspace_dev, workspace_bytes, stream);
}

extern "C" int
vsag_amd_ivf_scan_topk_ex(const vsag_amd_store_t* s, const float* queries_dev, uint64_t nq, const int32_t* buckets_dev,
                          uint32_t nprobe, uint32_t kcand, const vsag_amd_search_options_t* options, uint32_t* ids_dev,
                          float* dists_dev, void* workspace_dev, size_t workspace_bytes, void* stream) {
    VA_TRY(ensure_init());
    VA_TRY(check_ivf(s, nq, nprobe, kcand));
    VA_CHECK_ARG(queries_dev && buckets_dev && ids_dev && dists_dev, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    ScanPlanIvf p;
    plan_ivf(s, nq, nprobe, kcand, &p);
    Carver c(workspace_dev, workspace_bytes);
    IvfBuffers b;
    carve_ivf(c, s, p, nq, kcand, &b);
    if (!c.ok()) {  // (sized for another batch: without room for four times the chunks)
        plan_ivf(s, nq, nprobe, kcand, &p, false);
        c = Carver(workspace_dev, workspace_bytes);
        carve_ivf(c, s, p, nq, kcand, &b);
    }
    VA_CHECK_ARG(c.ok(), "workspace too small: need %zu bytes, got %zu", c.used, workspace_bytes);

    const uint64_t nlists1 = static_cast<uint64_t>(s->nlist) + 1;
    const uint64_t nslots_all = p.npairs * p.chunks_max;
    const uint64_t nseed = p.seeded ? nq * kcand : 0;
    const FillJob start{{b.bound, b.partial_cnt, b.counts, b.cursor, b.seed},
                        {initial_bound(options), 0U, 0U, 0U, 0xFFFFFFFFU},
                        {nq, nslots_all, p.chunked ? 0 : nlists1, p.chunked ? 0 : nlists1, nseed}};
    // Row nq of the query tables is the all-zero row that idle slots of a query tile point at.
    VA_TRY(prepare_queries(s, queries_dev, nq, nq + 1, p.ql, b.qtab, b.qmeta, b.qcodes, &start, st));
    ScanArgs a = make_scan_args(s, p.ql, b.qtab, b.qmeta);
    IvfArgs v{};
    v.ids = s->ids_dev;
    v.list_tile = s->list_tile_dev;
    v.pair_off = b.pair_off;
    v.item_off = b.item_off;
    v.sorted_pair = b.sorted_pair;
    v.nlist = s->nlist;
    v.nprobe = nprobe;
    v.dummy_query = static_cast<uint32_t>(nq);
    v.k = kcand;
    v.S = p.S;
    v.deny = options != nullptr ? options->deny_bits_dev : nullptr;
    v.tiles_per_item = p.tiles_per_item;
    v.chunks_max = p.chunks_max;
    v.bound = b.bound;
    v.seed = p.seeded ? b.seed : nullptr;
    v.partial = b.partial;
    v.partial_cnt = b.partial_cnt;
    if (s->residual_centroids_dev != nullptr) {
        VA_TRY(launch_residual_terms(s, queries_dev, nq, buckets_dev, nprobe, b.res_term, st));
        v.res_term = b.res_term;
        v.res_bias = s->residual_bias_dev;
    }

    uint32_t waves = 4;
    while (waves > 1 && static_cast<size_t>(waves) * p.T * p.S * 8 > 65536) {
        waves >>= 1;
    }
    size_t lds = static_cast<size_t>(waves) * p.T * p.S * 8;
    // Whole lists: two passes, the nearest list of every query first (it seeds the per-query bound), then the
    // rest.  Chunked lists: all probe columns at once, or the nearest lists first (nearest_first).
    uint32_t cols[3] = {0, p.chunked && !p.nearest_first ? nprobe : 1, nprobe};
    // A pre-filter or a radius goes the streaming way (the matrix-core pass knows neither).
    const bool mfma = p.mfma && (options == nullptr || (options->deny_bits_dev == nullptr && options->use_radius == 0));
    // The pairs of columns [c0, c1) grouped by list (pair_off, sorted_pair) and the work items of every list (item_off).
    auto regroup = [&](uint32_t c0, uint32_t c1, uint64_t pairs, uint32_t per_item, uint32_t tiles_per_item,
                       uint32_t chunks_max) {
        if (b.hist != nullptr && pairs >= 65536) {
            hipLaunchKernelGGL(regroup_hist_kernel, dim3(kRegroupGroups), dim3(1024), 0, st, buckets_dev, nq, nprobe, c0,
                               c1, s->nlist, b.hist);
            hipLaunchKernelGGL(regroup_prefix_kernel, dim3(static_cast<uint32_t>(div_up(s->nlist, 256))), dim3(256), 0, st,
                               b.hist, kRegroupGroups, s->nlist, b.counts);
            hipLaunchKernelGGL(offsets_kernel, dim3(1), dim3(1024), 0, st, b.counts, s->list_tile_dev, s->nlist, per_item,
                               tiles_per_item, chunks_max, b.pair_off, b.item_off);
            hipLaunchKernelGGL(regroup_scatter_kernel, dim3(kRegroupGroups), dim3(1024), 0, st, buckets_dev, nq, nprobe,
                               c0, c1, s->nlist, b.pair_off, b.hist, b.sorted_pair);
            return;
        }
        hipLaunchKernelGGL(count_pairs_kernel, dim3(blocks_for(pairs)), dim3(256), 0, st, buckets_dev, nq, nprobe, c0, c1,
                           s->nlist, b.counts);
        hipLaunchKernelGGL(offsets_kernel, dim3(1), dim3(1024), 0, st, b.counts, s->list_tile_dev, s->nlist, per_item,
                           tiles_per_item, chunks_max, b.pair_off, b.item_off);
        hipLaunchKernelGGL(scatter_pairs_kernel, dim3(blocks_for(pairs)), dim3(256), 0, st, buckets_dev, nq, nprobe, c0,
                           c1, s->nlist, b.pair_off, b.cursor, b.sorted_pair);
    };
    timing_begin(st);
    for (int pass = 0; pass < 2; ++pass) {
        uint32_t p0 = cols[pass], p1 = cols[pass + 1];
        if (p1 <= p0) {
            continue;
        }
        uint64_t pairs = nq * (p1 - p0);
        if (pass == 1 && !p.chunked) {
            VA_TRY(launch_fill(FillJob{{b.counts, b.cursor, mfma ? b.gate : nullptr, nullptr, nullptr}, {0U, 0U, 0U, 0U, 0U},
                                       {nlists1, nlists1, mfma ? nq + 3 : 0, 0, 0}}, st));
        }
        if (pass == 1 && mfma) {
            // Pairs grouped by list once; workgroups of 256 pairs for the matrix cores, then -- for the queries whose
            // lists overflowed -- the streaming kernel's items over the same grouping.
            // ivf_i8.hip: items of 256 pairs, kIvfI8ChunkTiles, kIvfI8Chunks
            regroup(p0, p1, pairs,
                    p.bits1 ? ivf_rb_pairs_per_item() : p.pq ? ivf_pq_pairs_per_item() : p.h16 ? ivf_h16_pairs_per_item()
                    : p.b16 ? ivf_b16_pairs_per_item() : p.f32 ? ivf_f32_pairs_per_item() : 256U,
                    p.bits1 ? ivf_rb_chunk_tiles() : 32U, 4U);
            if (p.h16) {
                VA_TRY(launch_ivf_h16(s, a, nq, nprobe, p0, b.pair_off, b.item_off, b.sorted_pair, b.bound, kcand,
                                      reinterpret_cast<float*>(b.tq), b.q8, b.partial, b.partial_cnt, b.gate, st));
                VA_TRY(launch_ivf_clear_gated(b.gate, nq, nprobe, p0, b.partial_cnt, buckets_dev, b.gpairs,
                                              kGatedPairsCap, kcand, st));
                VA_TRY(launch_ivf_rescore(s, a, nq, nprobe, p0, kcand, p.chunks_max, b.partial, b.partial_cnt, b.bound,
                                          nullptr, st));
            } else if (p.f32) {
                if (p.b16) {
                    VA_TRY(launch_ivf_b16(s, a, nq, nprobe, p0, b.pair_off, b.item_off, b.sorted_pair, b.bound, kcand,
                                          reinterpret_cast<float*>(b.tq), b.q8, b.partial, b.partial_cnt, b.gate,
                                          v.res_term, st));
                } else {
                    VA_TRY(launch_ivf_f32(s, a, nq, nprobe, p0, b.pair_off, b.item_off, b.sorted_pair, b.bound, kcand,
                                          reinterpret_cast<float*>(b.tq), b.partial, b.partial_cnt, b.gate, v.res_term, st));
                }
                VA_TRY(launch_ivf_clear_gated(b.gate, nq, nprobe, p0, b.partial_cnt, buckets_dev, b.gpairs,
                                              kGatedPairsCap, kcand, st));
                VA_TRY(launch_ivf_rescore(s, a, nq, nprobe, p0, kcand, p.chunks_max, b.partial, b.partial_cnt, b.bound,
                                          v.res_term, st));
            } else if (p.pq) {
                VA_TRY(launch_ivf_pq(s, a, nq, nprobe, p0, kcand, b.pair_off, b.item_off, b.sorted_pair, b.bound, b.tq,
                                     b.partial, b.partial_cnt, b.gate, buckets_dev, b.gpairs, kGatedPairsCap, st));
            } else if (p.bits1) {
                VA_TRY(launch_ivf_rb(s, a, nq, nprobe, p0, b.pair_off, b.item_off, b.sorted_pair, b.bound, kcand, b.q8,
                                     b.partial, b.partial_cnt, b.gate, st));
                VA_TRY(launch_ivf_clear_gated(b.gate, nq, nprobe, p0, b.partial_cnt, buckets_dev, b.gpairs,
                                              kGatedPairsCap, kcand, st));
                VA_TRY(launch_ivf_rescore(s, a, nq, nprobe, p0, kcand, p.chunks_max, b.partial, b.partial_cnt, b.bound,
                                          nullptr, st));
            } else if (p.planes) {
                VA_TRY(launch_ivf_sq8_i8(s, reinterpret_cast<const float*>(a.qtab), a.qstride, a.qmeta, a.qmeta_stride, nq,
                                         nprobe, p0, b.pair_off, b.item_off, b.sorted_pair, b.bound, kcand, b.q8, b.q8_u,
                                         b.q8_tau, b.partial, b.partial_cnt, b.gate, st));
                VA_TRY(launch_ivf_clear_gated(b.gate, nq, nprobe, p0, b.partial_cnt, buckets_dev, b.gpairs,
                                              kGatedPairsCap, kcand, st));
                VA_TRY(launch_ivf_rescore(s, a, nq, nprobe, p0, kcand, p.chunks_max, b.partial, b.partial_cnt, b.bound,
                                          nullptr, st));
            } else {
                VA_TRY(launch_ivf_i8(s, a, nq, nprobe, p0, kcand, b.pair_off, b.item_off, b.sorted_pair, b.bound, b.tq,
                                     b.partial, b.partial_cnt, b.gate, buckets_dev, b.gpairs, kGatedPairsCap, st));
            }
            // Few gated pairs (the usual case): one wave per pair and chunk of its list.
            IvfArgs d = v;
            d.direct = b.gpairs;
            d.direct_count = b.gate + nq + 1;
            d.direct_cap = kGatedPairsCap;
            d.buckets = buckets_dev;
            d.tiles_per_item = 16;
            uint32_t dwaves = 4;
            while (dwaves > 1 && static_cast<size_t>(dwaves) * p.S * 8 > 65536) {
                dwaves >>= 1;
            }
            // (the waves of this grid take the queued items in turn: see ivf_scan_kernel)
            dim3 dgrid(static_cast<uint32_t>(std::min<uint64_t>(div_up(static_cast<uint64_t>(kGatedPairsCap) * d.chunks_max, dwaves),
                                                                8ull * static_cast<uint64_t>(device_cu_count()))));
            VA_TRY(launch_ivf(s, 1, dgrid, dim3(dwaves * kWave), static_cast<size_t>(dwaves) * p.S * 8, st, a, d));
            // Many: the streaming kernel's items over the same grouping (stands back otherwise).
            hipLaunchKernelGGL(offsets_kernel, dim3(1), dim3(1024), 0, st, b.counts, s->list_tile_dev, s->nlist,
                               static_cast<uint32_t>(p.T), 0xFFFFFFFFU, 1U, b.pair_off, b.item_off);
            v.gate = b.gate;
            v.direct_cap = kGatedPairsCap;
            uint64_t max_items = div_up(pairs, p.T) + std::min<uint64_t>(s->nlist, pairs);
            dim3 grid(static_cast<uint32_t>(div_up(max_items, waves)));
            VA_TRY(launch_ivf(s, p.T, grid, dim3(waves * kWave), lds, st, a, v));
            continue;
        }
        // The nearest-list pass ahead of the matrix cores: a list several times the average length (k-means leaves
        // such lists) would keep one wave busy long after the others are done, so lists are cut into chunks of about
        // the average list's length; a pair's chunks use the private lists the matrix-core pass has per pair anyway.
        IvfArgs first = v;
        const bool cut_first = mfma && pass == 0;
        // That pass lives on its selectors (no bound to start from), not on the list bytes: two queries per wave
        // instead of four mean twice the waves to overlap the flushes of each other (10M x 128, 64 lists: 0.59 ->
        // 0.45 ms).
        const bool nearest = p.nearest_first && pass == 0;
        const int t_pass = nearest ? 1 : cut_first ? std::min(p.T, 2) : p.T;
        if (nearest) {
            // An average list is one item, which gives the best bound; a list walked whole whatever its length was the chain that
            // the launch ended with (98k x 32, 413 lists of 237 codes and one of 20 000: 597 -> 775 us with the pass, cut 563).
            const uint32_t avg_tiles = static_cast<uint32_t>(s->ntiles / s->nlist);
            first.tiles_per_item = std::max<uint32_t>(8, avg_tiles + avg_tiles / 4);
            first.seed = nullptr;
        }
        if (cut_first) {
            const uint32_t avg_tiles = std::max<uint32_t>(1, static_cast<uint32_t>(s->ntiles / s->nlist));
            first.tiles_per_item = std::max<uint32_t>(std::max<uint32_t>(16, avg_tiles + avg_tiles / 4),
                                                      static_cast<uint32_t>(div_up(s->max_list_tiles, p.chunks_max)));
        }
        if (p.chunked) {
            const bool in_lds = s->nlist <= kRegroupLists, all = p0 == 0 && p1 == nprobe;
            auto kernel = in_lds ? (all ? regroup_small_kernel<true, true> : regroup_small_kernel<true, false>)
                                 : (all ? regroup_small_kernel<false, true> : regroup_small_kernel<false, false>);
            hipLaunchKernelGGL(kernel, dim3(1), dim3(1024), 0, st, buckets_dev, nq, nprobe, p0, p1, s->list_tile_dev, s->nlist,
                               static_cast<uint32_t>(t_pass), first.tiles_per_item, p.chunks_max, b.counts, b.cursor, b.pair_off,
                               b.item_off, b.sorted_pair);
        } else {
            regroup(p0, p1, pairs, static_cast<uint32_t>(t_pass), first.tiles_per_item, p.chunks_max);
        }
        // At most one partly filled query group per probed list, each cut into at most chunks_max items.
        const uint64_t most = nearest ? std::min<uint64_t>(p.chunks_max, div_up(s->max_list_tiles, first.tiles_per_item))
                                      : p.chunked || cut_first ? p.chunks_max : 1;
        uint64_t max_items =
            (div_up(pairs, t_pass) + std::min<uint64_t>(s->nlist, pairs)) * most;
        dim3 grid(static_cast<uint32_t>(div_up(max_items, waves)));
        VA_TRY(launch_ivf(s, t_pass, grid, dim3(waves * kWave), static_cast<size_t>(waves) * t_pass * p.S * 8, st, a, first));
    }
    if (!mfma) {
        timing_end(st);  // the matrix-core pass is timed on its own (ivf_i8.hip)
    }
    note_last_scan(mfma ? 256 : p.T, 0, 0);
    return launch_merge_partials(b.partial, b.partial_cnt, b.bound, nprobe * p.chunks_max, nprobe * p.chunks_max, kcand,
                                 p.S, nq, ids_dev, dists_dev, st);
}

namespace vsag_amd {
// Codes in the lists the queries probe, summed over all (query, probe) pairs.  Few pairs: one workgroup that stores the sum.
__global__ void __launch_bounds__(1024)
probed_codes_few_kernel(const int32_t* buckets, uint32_t npairs, uint32_t nlist, const uint32_t* list_sizes,
                        unsigned long long* total) {
    __shared__ unsigned long long part[16];
    unsigned long long mine = 0;
#pragma unroll 4
    for (uint32_t i = threadIdx.x; i < npairs; i += 1024) {
        const int32_t b = buckets[i];
        mine += b >= 0 && static_cast<uint32_t>(b) < nlist ? list_sizes[b] : 0;
    }
    for (int off = 32; off > 0; off >>= 1) {
        mine += __shfl_xor(mine, off);
    }
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x >> 6] = mine;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long sum = 0;
        for (uint32_t w = 0; w < 16; ++w) {
            sum += part[w];
        }
        *total = sum;
    }
}

__global__ void __launch_bounds__(256)
probed_codes_kernel(const int32_t* buckets, uint64_t npairs, uint32_t nlist, const uint32_t* list_sizes,
                    unsigned long long* total) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    unsigned long long mine = 0;
    if (i < npairs) {
        const int32_t b = buckets[i];
        if (b >= 0 && static_cast<uint32_t>(b) < nlist) {
            mine = list_sizes[b];
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        mine += __shfl_xor(mine, off);
    }
    if ((threadIdx.x & 63) == 0 && mine != 0) {
        atomicAdd(total, mine);
    }
}
}  // namespace vsag_amd

extern "C" int
vsag_amd_ivf_probed_codes(const vsag_amd_store_t* s, const int32_t* buckets_dev, uint64_t nq, uint32_t nprobe,
                          uint64_t* total_dev, void* stream) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG(s != nullptr && s->nlist > 0, "not a posting-list store");
    VA_CHECK_ARG(buckets_dev && total_dev, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    if (nq <= VSAG_AMD_PROBED_CODES_STORED && nq * nprobe <= VSAG_AMD_PROBED_CODES_STORED) {
        hipLaunchKernelGGL(probed_codes_few_kernel, dim3(1), dim3(1024), 0, st, buckets_dev,
                           static_cast<uint32_t>(nq * nprobe), s->nlist, s->list_sizes_dev,
                           reinterpret_cast<unsigned long long*>(total_dev));
        VA_HIP(hipGetLastError());
        return 0;
    }
    VA_TRY(launch_fill(FillJob{{reinterpret_cast<uint32_t*>(total_dev)}, {0}, {2}}, st));
    hipLaunchKernelGGL(probed_codes_kernel, dim3(blocks_for(nq * nprobe)), dim3(256), 0, st, buckets_dev, nq * nprobe,
                       s->nlist, s->list_sizes_dev, reinterpret_cast<unsigned long long*>(total_dev));
    VA_HIP(hipGetLastError());
    return 0;
}

extern "C" int
vsag_amd_rerank_fp32(const float* raw_dev, uint64_t n, uint32_t dim, int metric, const float* queries_dev, uint64_t nq,
                     const uint32_t* cand_ids_dev, uint32_t kcand, uint32_t k, uint32_t* ids_dev, float* dists_dev,
                     void* stream) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG(raw_dev && queries_dev && cand_ids_dev && ids_dev && dists_dev, "null pointer");
    VA_CHECK_ARG(kcand >= 1 && kcand <= 4096, "kcand must be in [1, 4096], got %u", kcand);
    VA_CHECK_ARG(k >= 1 && k <= kcand, "k must be in [1, kcand], got %u", k);
    VA_CHECK_ARG(metric >= VSAG_AMD_METRIC_L2 && metric <= VSAG_AMD_METRIC_COSINE, "unknown metric %d", metric);
    VA_CHECK_ARG(nq >= 1 && nq < (1ull << 31), "nq must be in [1, 2^31)");
    uint32_t S = 64;
    while (S < kcand) {
        S <<= 1;
    }
    hipLaunchKernelGGL(rerank_kernel, dim3(static_cast<uint32_t>(nq)), dim3(kRerankThreads), S * 8,
                       static_cast<hipStream_t>(stream), raw_dev, n, dim, metric, queries_dev, cand_ids_dev, kcand, k,
                       S, ids_dev, dists_dev);
    VA_HIP(hipGetLastError());
    return 0;
}

extern "C" int
vsag_amd_rows_distances_fp32(const float* raw_dev, uint64_t n, uint32_t dim, int metric, const float* queries_dev,
                             uint64_t nq, const uint32_t* ids_dev, uint32_t count, float* dists_dev, void* stream) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG(raw_dev && queries_dev && ids_dev && dists_dev, "null pointer");
    VA_CHECK_ARG(metric >= VSAG_AMD_METRIC_L2 && metric <= VSAG_AMD_METRIC_COSINE, "unknown metric %d", metric);
    VA_CHECK_ARG(nq >= 1 && nq <= 65535, "nq must be in [1, 65535]");
    VA_CHECK_ARG(count >= 1, "count must be positive");
    hipLaunchKernelGGL(rows_distances_kernel, dim3(static_cast<uint32_t>(div_up(count, kRerankThreads / 16)), static_cast<uint32_t>(nq)),
                       dim3(kRerankThreads), 0, static_cast<hipStream_t>(stream), raw_dev, n, dim, metric, queries_dev,
                       ids_dev, count, dists_dev);
    VA_HIP(hipGetLastError());
    return 0;
}
