// The streaming kernel over posting lists: a wave takes a work item, up to T of the queries that probe a list against the
// list or a chunk of it (ivf.hip plans the items).
#include "ivf_scan.h"
#include "topk.h"

namespace vsag_amd {

constexpr uint32_t kIvfSeedTiles = 4;

// CHUNKED: work items are chunks of lists and start cold together (few queries); otherwise whole lists.
template <int KIND, int METRIC, int T, bool CHUNKED>
__device__ __forceinline__ void
ivf_scan_item(const ScanArgs& a, const IvfArgs& v, uint64_t* lds, uint32_t item) {
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    uint32_t list_begin, list_end, local, pfirst, plast;
    cu32_p pairs_src = as_const(v.sorted_pair);
    if (v.direct != nullptr) {
        const uint32_t count = as_const(v.direct_count)[0];
        const uint32_t vi = item / v.chunks_max;
        if (count > v.direct_cap || vi >= count) {
            return;
        }
        pairs_src = as_const(v.direct);
        const int32_t bk = v.buckets[pairs_src[vi]];  // a real list: pairs without one are never queued
        list_begin = as_const(v.list_tile)[2 * bk];
        list_end = as_const(v.list_tile)[2 * bk + 1];
        local = item % v.chunks_max;
        pfirst = vi;
        plast = vi + 1;
    } else {
        const uint32_t total = as_const(v.item_off)[v.nlist];
        if (item >= total) {
            return;
        }
        if (v.gate != nullptr) {
            // Words nq and nq + 1 of the gate array count the raised gates and their pairs: nothing to serve, or
            // few enough for the direct launch.
            const uint32_t raised = as_const(v.gate)[v.dummy_query];
            if (raised == 0 || (v.direct_cap != 0 && as_const(v.gate)[v.dummy_query + 1] <= v.direct_cap)) {
                return;
            }
        }
        // Which list: last b with item_off[b] <= item.
        cu32_p ioff = as_const(v.item_off);
        uint32_t lo = 0, hi = v.nlist;
        while (hi - lo > 1) {
            uint32_t mid = (lo + hi) >> 1;
            if (ioff[mid] <= item) {
                lo = mid;
            } else {
                hi = mid;
            }
        }
        list_begin = as_const(v.list_tile)[2 * lo];
        list_end = as_const(v.list_tile)[2 * lo + 1];
        local = item - ioff[lo];
        pfirst = as_const(v.pair_off)[lo];
        plast = as_const(v.pair_off)[lo + 1];
    }
    uint32_t group = local, chunk = 0;
    uint32_t tbeg = list_begin, tend = list_end;
    if (CHUNKED) {
        const uint32_t tiles = list_end - list_begin;
        const uint32_t chunks = list_chunks(tiles, v.tiles_per_item, v.chunks_max);
        if (chunks == 0) {
            return;
        }
        const uint32_t per = (tiles + chunks - 1) / chunks;
        chunk = group % chunks;
        group = group / chunks;
        tbeg = list_begin + chunk * per;
        tbeg = tbeg < list_end ? tbeg : list_end;
        tend = tbeg + per < list_end ? tbeg + per : list_end;
    }
    const uint32_t pbeg = pfirst + group * T;
    const uint32_t pend = plast;

    const uint32_t S = v.S, k = v.k;
    const uint32_t spend = selector_base(S, k);  // where a selector's pending keys start
    uint64_t* sel = lds + static_cast<size_t>(wave) * T * S;
    uint32_t qidx[T], pair[T];
    uint64_t tau[T];
    uint32_t cnt[T];
    uint32_t cold[T];  // tiles after which this item still looks at the seed row (see the flat scan)
    bool any_live = false;
#pragma unroll
    for (int t = 0; t < T; ++t) {
        bool live = pbeg + t < pend;
        pair[t] = live ? pairs_src[pbeg + t] : 0xFFFFFFFFU;
        if (live && v.gate != nullptr && as_const(v.gate)[pair[t] / v.nprobe] == 0) {
            live = false;
            pair[t] = 0xFFFFFFFFU;
        }
        any_live = any_live || live;
        qidx[t] = live ? pair[t] / v.nprobe : v.dummy_query;
        cnt[t] = 0;
        uint32_t bound = live ? __builtin_amdgcn_readfirstlane(__atomic_load_n(&v.bound[qidx[t]], __ATOMIC_RELAXED))
                              : 0U;
        // Everything at or below the bound passes, whatever its id.
        tau[t] = (static_cast<uint64_t>(bound) << 32) | 0xFFFFFFFFULL;
        cold[t] = CHUNKED && v.seed != nullptr && live && bound == 0xFFFFFFFFU ? kIvfSeedTiles : 0;
    }
    if (!any_live) {
        return;  // nothing but gated-off queries
    }
    const uint32_t seed_slot = item % k;
    for (uint32_t i = lane; i < T * S; i += kWave) {
        sel[i] = kInfKey;
    }
    wave_lds_fence();

    const QueryRows<T> qrows = query_rows<T>(a, qidx);
    float rterm[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        rterm[t] = v.res_term != nullptr && pair[t] != 0xFFFFFFFFU ? v.res_term[pair[t]] : 0.0F;
    }
    constexpr int GROUP = GroupOf<T>::value;
    TileStream<GROUP> cur{a.tiles, lane, tbeg, tend, 1, 0, a.G};
    TileStream<GROUP> nxt = cur;
    uint4 buf_a[GROUP], buf_b[GROUP];
    if (cur.valid()) {
        cur.load(buf_a, cur.tile);
    }
    Acc<KIND, T> acc;
    acc_reset(acc);

    auto consume = [&](const uint4(&regs)[GROUP]) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < GROUP; ++u) {
            if (cur.j0 + u < a.G) {
                accumulate_granule<KIND, METRIC, T>(a, qrows, cur.j0 + u, regs[u], acc);
            }
        }
        if (cur.j0 + GROUP < a.G) {
            return;
        }
        const uint64_t slot = cur.tile * kWave + lane;
        float d[T];
        finish_distances<KIND, METRIC, T>(a, qidx, slot, acc, d);
        acc_reset(acc);
        if (v.res_term != nullptr) {
            const float bias = v.res_bias != nullptr ? v.res_bias[slot] : 0.0F;
#pragma unroll
            for (int t = 0; t < T; ++t) {
                d[t] = (d[t] - bias) - rterm[t];
            }
        }
        const uint32_t id = v.ids[slot];
        const bool valid = id != VSAG_AMD_INVALID_ID && !denied(v.deny, id);
#pragma unroll
        for (int t = 0; t < T; ++t) {
            uint64_t key = make_key(d[t], id);
            if (CHUNKED && cold[t] != 0) {
                uint32_t* row = v.seed + static_cast<uint64_t>(qidx[t]) * k;
                if (cold[t] == kIvfSeedTiles) {
                    uint32_t m = wave_min_u32(valid ? static_cast<uint32_t>(key >> 32) : 0xFFFFFFFFU);
                    lower_shared(&row[seed_slot], m, lane);
                }
                --cold[t];
                uint32_t mx = 0;
                for (uint32_t i = lane; i < k; i += kWave) {
                    uint32_t sv = __atomic_load_n(&row[i], __ATOMIC_RELAXED);
                    mx = sv > mx ? sv : mx;
                }
                mx = wave_max_u32(mx);
                if (mx != 0xFFFFFFFFU) {
                    cold[t] = 0;
                    mx = lower_shared(&v.bound[qidx[t]], mx, lane);
                    uint64_t shared_tau = (static_cast<uint64_t>(mx) << 32) | 0xFFFFFFFFULL;
                    tau[t] = tau[t] < shared_tau ? tau[t] : shared_tau;
                }
            }
            bool pass = valid && key < tau[t];
            uint64_t mask = __ballot(pass);
            if (mask == 0) {
                continue;
            }
            uint64_t* keys = sel + t * S;
            uint32_t np = __popcll(mask);
            if (spend + cnt[t] + np > S) {
                uint64_t th = selector_flush(keys, S, k, cnt[t], lane);
                cnt[t] = 0;
                cold[t] = 0;
                if (pair[t] != 0xFFFFFFFFU) {
                    // th finite: this pair alone already holds k candidates at or below th.
                    uint32_t bound = lower_shared(&v.bound[qidx[t]], static_cast<uint32_t>(th >> 32), lane);
                    uint64_t shared_tau = (static_cast<uint64_t>(bound) << 32) | 0xFFFFFFFFULL;
                    tau[t] = th < shared_tau ? th : shared_tau;
                }
            }
            if (pass) {
                keys[spend + cnt[t] + mask_rank(mask)] = key;
            }
            cnt[t] += np;
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
#pragma unroll
    for (int t = 0; t < T; ++t) {
        if (pair[t] == 0xFFFFFFFFU) {
            continue;
        }
        // What the shared bound still admits is usually less than k keys, which go out unsorted; only a
        // pair left with more sorts once more (and then has a k-th key to lower the bound with).
        uint64_t* keys = sel + t * S;
        wave_lds_fence();
        uint32_t bs = __builtin_amdgcn_readfirstlane(__atomic_load_n(&v.bound[qidx[t]], __ATOMIC_RELAXED));
        uint32_t total = spend + cnt[t];
        uint32_t admitted = selector_count_admitted(keys, total, bs, lane);
        if (admitted > k) {
            uint64_t th = selector_flush(keys, S, k, cnt[t], lane);
            bs = lower_shared(&v.bound[qidx[t]], static_cast<uint32_t>(th >> 32), lane);
            total = k;
            admitted = selector_count_admitted(keys, total, bs, lane);
        } else if (admitted == k) {
            // Exactly k admitted keys: their largest distance is a bound other pairs can use.
            uint32_t mx = 0;
            for (uint32_t i = lane; i < total; i += kWave) {
                uint64_t key = keys[i];
                uint32_t od = static_cast<uint32_t>(key >> 32);
                mx = key != kInfKey && od <= bs && od > mx ? od : mx;
            }
            lower_shared(&v.bound[qidx[t]], wave_max_u32(mx), lane);  // bs itself must stay what was counted with
        }
        const uint64_t list = static_cast<uint64_t>(pair[t]) * v.chunks_max + chunk;
        if (lane == 0) {
            v.partial_cnt[list] = admitted;
        }
        if (admitted != 0) {
            selector_copy_admitted(keys, total, bs, v.partial + list * k, lane);
        }
    }
}

// A wave is a work item.  The direct launch (v.direct) serves a queue whose length only the device knows: a grid sized
// for its capacity would be tens of thousands of workgroups that find nothing to do, so there the waves of a smaller
// grid take the items in turn.
template <int KIND, int METRIC, int T, bool CHUNKED>
__global__ void __launch_bounds__(256)
ivf_scan_kernel(ScanArgs a, IvfArgs v) {
    extern __shared__ uint64_t lds[];
    const uint32_t waves = blockDim.x >> 6;
    uint32_t item = blockIdx.x * waves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (v.direct == nullptr) {
        ivf_scan_item<KIND, METRIC, T, CHUNKED>(a, v, lds, item);
        return;
    }
    const uint32_t count = as_const(v.direct_count)[0];
    const uint32_t stride = gridDim.x * waves;
    const uint32_t limit = count <= v.direct_cap ? count * v.chunks_max : 0;
    for (; item < limit; item += stride) {
        ivf_scan_item<KIND, METRIC, T, CHUNKED>(a, v, lds, item);
        // the selectors of the item in LDS have been read before the next item resets them
        wave_lds_fence();
    }
}

template <int KIND, int METRIC, int T>
static void
launch_ivf_c(dim3 grid, dim3 block, size_t lds, hipStream_t st, const ScanArgs& a, const IvfArgs& v) {
    if (v.tiles_per_item != 0xFFFFFFFFU) {
        hipLaunchKernelGGL((ivf_scan_kernel<KIND, METRIC, T, true>), grid, block, lds, st, a, v);
    } else {
        hipLaunchKernelGGL((ivf_scan_kernel<KIND, METRIC, T, false>), grid, block, lds, st, a, v);
    }
}

template <int KIND, int METRIC>
static void
launch_ivf_t(int T, dim3 grid, dim3 block, size_t lds, hipStream_t st, const ScanArgs& a, const IvfArgs& v) {
    switch (T) {
        case 1:
            launch_ivf_c<KIND, METRIC, 1>(grid, block, lds, st, a, v);
            break;
        case 2:
            launch_ivf_c<KIND, METRIC, 2>(grid, block, lds, st, a, v);
            break;
        default:
            launch_ivf_c<KIND, METRIC, 4>(grid, block, lds, st, a, v);
            break;
    }
}

template <int KIND>
static void
launch_ivf_m(int metric, int T, dim3 grid, dim3 block, size_t lds, hipStream_t st, const ScanArgs& a,
             const IvfArgs& v) {
    if (metric == VSAG_AMD_METRIC_L2) {
        launch_ivf_t<KIND, VSAG_AMD_METRIC_L2>(T, grid, block, lds, st, a, v);
    } else if (metric == VSAG_AMD_METRIC_COSINE && (KIND == VSAG_AMD_KIND_RABITQ || KIND == kKindRabitqF32)) {
        launch_ivf_t<KIND, VSAG_AMD_METRIC_COSINE>(T, grid, block, lds, st, a, v);
    } else {
        launch_ivf_t<KIND, VSAG_AMD_METRIC_IP>(T, grid, block, lds, st, a, v);
    }
}

int
launch_ivf(const vsag_amd_store* s, int T, dim3 grid, dim3 block, size_t lds, hipStream_t st, const ScanArgs& a,
           const IvfArgs& v) {
    switch (s->kind) {
        case VSAG_AMD_KIND_FP32:
            launch_ivf_m<VSAG_AMD_KIND_FP32>(s->metric, T, grid, block, lds, st, a, v);
            break;
        case VSAG_AMD_KIND_SQ8:
            launch_ivf_m<VSAG_AMD_KIND_SQ8>(s->metric, T, grid, block, lds, st, a, v);
            break;
        case VSAG_AMD_KIND_SQ4:
            launch_ivf_m<VSAG_AMD_KIND_SQ4>(s->metric, T, grid, block, lds, st, a, v);
            break;
        case VSAG_AMD_KIND_SQ4_UNIFORM:
            launch_ivf_m<VSAG_AMD_KIND_SQ4_UNIFORM>(s->metric, T, grid, block, lds, st, a, v);
            break;
        case VSAG_AMD_KIND_SQ8_UNIFORM:
            launch_ivf_m<VSAG_AMD_KIND_SQ8_UNIFORM>(s->metric, T, grid, block, lds, st, a, v);
            break;
        case VSAG_AMD_KIND_PQFS:
            launch_ivf_m<VSAG_AMD_KIND_PQFS>(s->metric, T, grid, block, lds, st, a, v);
            break;
        case VSAG_AMD_KIND_RABITQ:
            if (s->query_bits == 32) {
                launch_ivf_m<kKindRabitqF32>(s->metric, T, grid, block, lds, st, a, v);
            } else {
                launch_ivf_m<VSAG_AMD_KIND_RABITQ>(s->metric, T, grid, block, lds, st, a, v);
            }
            break;
        default:
            return fail(VSAG_AMD_INVALID_ARGUMENT, "unknown store kind %d", s->kind);
    }
    VA_HIP(hipGetLastError());
    return 0;
}

}  // namespace vsag_amd
