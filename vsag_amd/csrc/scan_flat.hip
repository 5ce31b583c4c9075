// Flat scan with fused per-query top-k (BruteForce::SearchWithRequest hot loop,
// src/algorithm/bruteforce/bruteforce.cpp:481-597; FlattenDataCell::query,
// src/datacell/flatten_datacell.h:334-440), batched over queries: the streaming kernel.
//
// Work decomposition.  Grid x = query tile (T queries), y = chunk of code tiles.  A workgroup has up to
// four waves; wave w walks tiles chunk_begin + w, + W, ... with the next granule group already in flight,
// and keeps one LDS selector per query of the tile.  Workgroups that are resident together have
// consecutive x and the same y, so they stream the same chunk of codes at about the same time.
//
// Selection.  Every (wave, query) has a selector in LDS (topk.h).  Chunks and waves of one query share a
// per-query bound in global memory (the k-th best distance any of them has proven so far), so later
// work drops almost everything with one compare.  Each (chunk, wave) leaves a short counted list of the
// survivors that the bound still admits; a merge kernel picks the k best per query.  All waves of a query
// share a handful of addresses (its bound, its seed row), and atomics on one address serialise in L2, so
// every atomicMin is preceded by a plain load and issued only when it would lower the value.
#include "scan_flat.h"
#include "topk.h"

namespace vsag_amd {

// Cold start.  A wave that begins without a bound would have to sort its first tiles just to learn a
// threshold.  Instead every such wave publishes the smallest distance of its first tile into slot
// (global wave index mod k) of its query's seed row; waves own disjoint codes, so once all k slots are
// filled their maximum is a distance that k different codes reach -- a valid bound, usually far tighter
// than anything one wave could find alone.  A cold wave re-reads the row after each of its first
// kSeedTiles tiles; the host enables seeding only when there are at least 2k waves per query.
constexpr uint32_t kSeedTiles = 6;

template <int KIND, int METRIC, int T, bool SEED>
__global__ void __launch_bounds__(256)
flat_scan_kernel(ScanArgs a, FlatArgs f) {
    extern __shared__ uint64_t lds[];
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t nwaves = blockDim.x >> 6;
    const uint32_t S = f.S, k = f.k;
    uint64_t* sel = lds + static_cast<size_t>(wave) * T * S;

    uint32_t qidx[T];
    uint32_t thr[T];   // a candidate passes when its ordered distance is below thr
    uint32_t cnt[T];
    uint32_t cold[T];  // tiles after which this wave still looks at the seed row
    bool live[T];      // a real query that this launch serves
    bool any_live = false;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        qidx[t] = blockIdx.x * T + t;
        cnt[t] = 0;
        live[t] = qidx[t] < f.nq && (f.gate == nullptr || as_const(f.gate)[qidx[t]] != 0);
        any_live = any_live || live[t];
        uint32_t bs = live[t] ? __builtin_amdgcn_readfirstlane(__atomic_load_n(&f.bound[qidx[t]], __ATOMIC_RELAXED))
                              : 0xFFFFFFFFU;
        thr[t] = !live[t] ? 0U : bs == 0xFFFFFFFFU ? bs : bs + 1;
        cold[t] = SEED && live[t] && bs == 0xFFFFFFFFU ? kSeedTiles : 0;
    }
    if (!any_live) {
        return;
    }
    for (uint32_t i = lane; i < T * S; i += kWave) {
        sel[i] = kInfKey;
    }
    wave_lds_fence();
    const uint32_t seed_slot = (blockIdx.y * nwaves + wave) % k;

    const uint64_t tile_begin = f.tile0 + static_cast<uint64_t>(blockIdx.y) * f.tiles_per_chunk;
    uint64_t tile_end = tile_begin + f.tiles_per_chunk;
    if (tile_end > f.tile_end) {
        tile_end = f.tile_end;
    }
    // Software pipeline over granule groups: the loads of group g+1 (possibly of the next tile) are
    // issued before group g is consumed, so every wave keeps GROUP KiB in flight.  Two register buffers
    // alternate; the loop body is written out twice so that both are addressed statically.
    const QueryRows<T> qrows = query_rows<T>(a, qidx);
    constexpr int GROUP = GroupOf<T>::value;
    // RaBitQ codes have G = dim / 128 granules, often no multiple of the group (768 dimensions: 6).
    constexpr bool OVERLAP = KIND == VSAG_AMD_KIND_RABITQ || KIND == kKindRabitqF32;
    TileStream<GROUP, OVERLAP> cur{a.tiles, lane, tile_begin + wave, tile_end, nwaves, 0, a.G};
    TileStream<GROUP, OVERLAP> nxt = cur;
    uint4 buf_a[GROUP], buf_b[GROUP];
    if (cur.valid()) {
        cur.load(buf_a, cur.tile);
    }
    Acc<KIND, T> acc;
    acc_reset(acc);

    const uint32_t pend = selector_base(S, k);  // where a selector's pending keys start
    // Sorts selector t and folds its k-th key and the shared bound into thr[t].
    auto flush = [&](int t) __attribute__((always_inline)) {
        uint64_t* keys = sel + t * S;
        uint64_t th = selector_flush(keys, S, k, cnt[t], lane);
        cnt[t] = 0;
        cold[t] = 0;
        uint32_t tl = static_cast<uint32_t>(th >> 32);  // 0xFFFFFFFF while fewer than k seen
        uint32_t bs = 0xFFFFFFFFU;
        if (live[t]) {
            bs = lower_shared(&f.bound[qidx[t]], tl, lane);  // tl = 0xFFFFFFFF lowers nothing
        }
        uint32_t tb = bs == 0xFFFFFFFFU ? bs : bs + 1;
        thr[t] = tl < tb ? tl : tb;
    };

    // What a cold wave reads of its queries' seed rows (largest entry over this lane's share): fetched when a tile
    // begins, looked at when its distances are done, so that the read waits under the tile's arithmetic.
    uint32_t seed_seen[T];
    auto consume = [&](const uint4(&regs)[GROUP]) __attribute__((always_inline)) {
        const uint32_t first = cur.first();
        if (SEED && cur.j0 == 0) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                seed_seen[t] = 0;
                if (cold[t] != 0) {
                    const uint32_t* row = f.seed + static_cast<uint64_t>(qidx[t]) * k;
                    for (uint32_t i = lane; i < k; i += kWave) {
                        const uint32_t v = __atomic_load_n(&row[i], __ATOMIC_RELAXED);
                        seed_seen[t] = v > seed_seen[t] ? v : seed_seen[t];
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < GROUP; ++u) {
            const uint32_t g = first + u;
            if (g >= cur.j0 && g < a.G) {
                accumulate_granule<KIND, METRIC, T>(a, qrows, g, regs[u], acc);
            }
        }
        if (cur.j0 + GROUP < a.G) {
            return;
        }
        const uint64_t id = cur.tile * kWave + lane;
        float d[T];
        finish_distances<KIND, METRIC, T>(a, qidx, id, acc, d);
        acc_reset(acc);
        const bool valid = id < f.n && !denied(f.deny, id);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            // Inner ids grow along the scan, so "ordered distance < thr" is exactly the (distance, id)
            // order against the wave's own k-th key, and "<= bound" against the shared bound.
            uint32_t od = float_to_ordered(d[t]);
            if (SEED && cold[t] != 0) {
                uint32_t* row = f.seed + static_cast<uint64_t>(qidx[t]) * k;
                if (cold[t] == kSeedTiles) {
                    // This wave's entry (its own first look at the row came before it, the next one will see it).
                    uint32_t m = wave_min_u32(valid ? od : 0xFFFFFFFFU);
                    lower_shared(&row[seed_slot], m, lane);
                }
                --cold[t];
                const uint32_t mx = wave_max_u32(seed_seen[t]);
                if (mx != 0xFFFFFFFFU) {
                    // Every slot filled: k different codes reach mx.
                    cold[t] = 0;
                    const uint32_t b = lower_shared(&f.bound[qidx[t]], mx, lane);
                    thr[t] = b + 1 < thr[t] ? b + 1 : thr[t];
                }
            }
            bool pass = valid && od < thr[t];
            uint64_t mask = __ballot(pass);
            if (mask != 0) {
                uint32_t np = __popcll(mask);
                if (pend + cnt[t] + np > S) {
                    flush(t);
                }
                if (pass) {
                    sel[t * S + pend + cnt[t] + mask_rank(mask)] = (static_cast<uint64_t>(od) << 32) | static_cast<uint32_t>(id);
                }
                cnt[t] += np;
            }
        }
    };

    while (cur.valid()) {
        nxt.advance();
        nxt.load(buf_b, cur.tile);
        consume(buf_a);
        cur = nxt;
        if (!cur.valid()) {
            break;
        }
        nxt.advance();
        nxt.load(buf_a, cur.tile);
        consume(buf_b);
        cur = nxt;
    }

    const uint32_t slot = f.slot0 + blockIdx.y * nwaves + wave;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        if (!live[t]) {
            continue;
        }
        // Whatever lies above the shared bound is beaten by k candidates of other waves.  What remains is
        // usually less than k keys, which go out as they are; only a wave left with more sorts once more.
        uint64_t* keys = sel + t * S;
        wave_lds_fence();
        uint32_t bs = __builtin_amdgcn_readfirstlane(__atomic_load_n(&f.bound[qidx[t]], __ATOMIC_RELAXED));
        uint32_t total = pend + cnt[t];
        uint32_t admitted = selector_count_admitted(keys, total, bs, lane);
        if (admitted > k) {
            uint64_t th = selector_flush(keys, S, k, cnt[t], lane);
            bs = lower_shared(&f.bound[qidx[t]], static_cast<uint32_t>(th >> 32), lane);
            total = k;
            admitted = selector_count_admitted(keys, total, bs, lane);
        }
        const uint64_t list = static_cast<uint64_t>(qidx[t]) * f.nslots + slot;
        if (lane == 0) {
            f.partial_cnt[list] = admitted;
        }
        if (admitted != 0) {
            selector_copy_admitted(keys, total, bs, f.partial + list * k, lane);
        }
    }
}

template <int KIND, int METRIC, int T>
static void
launch_flat_s(dim3 grid, dim3 block, size_t lds, hipStream_t st, const ScanArgs& a, const FlatArgs& f) {
    if (f.seed != nullptr) {
        hipLaunchKernelGGL((flat_scan_kernel<KIND, METRIC, T, true>), grid, block, lds, st, a, f);
    } else {
        hipLaunchKernelGGL((flat_scan_kernel<KIND, METRIC, T, false>), grid, block, lds, st, a, f);
    }
}

template <int KIND, int METRIC>
static void
launch_flat_t(int T, dim3 grid, dim3 block, size_t lds, hipStream_t st, const ScanArgs& a, const FlatArgs& f) {
    switch (T) {
        case 1:
            launch_flat_s<KIND, METRIC, 1>(grid, block, lds, st, a, f);
            break;
        case 2:
            launch_flat_s<KIND, METRIC, 2>(grid, block, lds, st, a, f);
            break;
        case 4:
            launch_flat_s<KIND, METRIC, 4>(grid, block, lds, st, a, f);
            break;
        default:
            launch_flat_s<KIND, METRIC, 8>(grid, block, lds, st, a, f);
            break;
    }
}

template <int KIND>
static void
launch_flat_m(int metric, int T, dim3 grid, dim3 block, size_t lds, hipStream_t st, const ScanArgs& a,
              const FlatArgs& f) {
    // Cosine stores hold normalised vectors and scan as inner product (RaBitQ has its own formula).
    if (metric == VSAG_AMD_METRIC_L2) {
        launch_flat_t<KIND, VSAG_AMD_METRIC_L2>(T, grid, block, lds, st, a, f);
    } else if (metric == VSAG_AMD_METRIC_COSINE && (KIND == VSAG_AMD_KIND_RABITQ || KIND == kKindRabitqF32)) {
        launch_flat_t<KIND, VSAG_AMD_METRIC_COSINE>(T, grid, block, lds, st, a, f);
    } else {
        launch_flat_t<KIND, VSAG_AMD_METRIC_IP>(T, grid, block, lds, st, a, f);
    }
}

int
launch_flat(const vsag_amd_store* s, int T, dim3 grid, dim3 block, size_t lds, const ScanArgs& a, const FlatArgs& f,
            hipStream_t st) {
    switch (s->kind) {
        case VSAG_AMD_KIND_FP32:
            launch_flat_m<VSAG_AMD_KIND_FP32>(s->metric, T, grid, block, lds, st, a, f);
            break;
        case VSAG_AMD_KIND_SQ8:
            launch_flat_m<VSAG_AMD_KIND_SQ8>(s->metric, T, grid, block, lds, st, a, f);
            break;
        case VSAG_AMD_KIND_SQ4:
            launch_flat_m<VSAG_AMD_KIND_SQ4>(s->metric, T, grid, block, lds, st, a, f);
            break;
        case VSAG_AMD_KIND_SQ4_UNIFORM:
            launch_flat_m<VSAG_AMD_KIND_SQ4_UNIFORM>(s->metric, T, grid, block, lds, st, a, f);
            break;
        case VSAG_AMD_KIND_SQ8_UNIFORM:
            launch_flat_m<VSAG_AMD_KIND_SQ8_UNIFORM>(s->metric, T, grid, block, lds, st, a, f);
            break;
        case VSAG_AMD_KIND_PQFS:
            launch_flat_m<VSAG_AMD_KIND_PQFS>(s->metric, T, grid, block, lds, st, a, f);
            break;
        case VSAG_AMD_KIND_RABITQ:
            if (s->query_bits == 32) {
                launch_flat_m<kKindRabitqF32>(s->metric, T, grid, block, lds, st, a, f);
            } else {
                launch_flat_m<VSAG_AMD_KIND_RABITQ>(s->metric, T, grid, block, lds, st, a, f);
            }
            break;
        default:
            return fail(VSAG_AMD_INVALID_ARGUMENT, "unknown store kind %d", s->kind);
    }
    VA_HIP(hipGetLastError());
    return 0;
}

}  // namespace vsag_amd
