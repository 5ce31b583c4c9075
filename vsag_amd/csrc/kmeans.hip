// k-means assignment as an fp32 MFMA contraction with a fused argmin, centroid update and Lloyd driver
// (KMeansCluster::find_nearest_one_with_blas / Run, src/impl/cluster/kmeans_cluster.cpp:46-305).
//
// The reference forms distances = -2 C X^T with SGEMM into a k x 65536 buffer, then makes a second pass
// adding ||c||^2 and taking std::min_element per row.  Here one kernel does both: a workgroup owns a
// 128-row tile of X and walks the centroid tiles of its group; v_mfma_f32_32x32x2_f32 accumulates
// <c_m, x_n> with centroids as the M side and data rows as the N side, so that after the K loop every
// lane holds 16 centroid values of ONE data row and the argmin needs no cross-lane traffic until the
// very end.  Candidates are (ordered distance, centroid index) keys, so the smallest index wins ties
// exactly like std::min_element.
//
// Grid: x = centroid group (tile t belongs to group t % groups, groups <= 8), y = row tile.  Workgroups
// are dealt round-robin to the eight XCDs in x-major order, so one XCD always works on the same
// quarter-to-eighth of the centroids and keeps them in its own L2, while the X tile is what streams.
#include <hipcub/hipcub.hpp>

#include <mutex>
#include <random>
#include <vector>

#include "common.h"
#include "kmeans_h16.h"

namespace vsag_amd {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int BM = 128;  // centroids per tile
constexpr int BN = 128;  // data rows per tile
constexpr int BK = 32;   // contraction depth per stage
constexpr int kPlane = BM;  // float4 slots per (parity, chunk) plane

// LDS operand layout for one stage: [parity h = k & 1][chunk c = (k >> 1) / 4][row] of float4, element e
// of the float4 is k = 2 (4 c + e) + h.  A lane of the MFMA (row = lane % 32, h = lane / 32) then reads
// its operand for four consecutive k-steps with one conflict-free ds_read_b128.
struct Stage {
    float4 a[2 * 4 * kPlane];
    float4 b[2 * 4 * kPlane];
};

__device__ inline float4
load_row_chunk(const float* base, uint64_t row, uint64_t rows, uint32_t k0, uint32_t dim, bool aligned) {
    float4 v = make_float4(0.0F, 0.0F, 0.0F, 0.0F);
    if (row < rows) {
        const float* p = base + row * dim + k0;
        if (aligned && k0 + 4 <= dim) {
            v = *reinterpret_cast<const float4*>(p);
        } else {
            if (k0 < dim) {
                v.x = p[0];
            }
            if (k0 + 1 < dim) {
                v.y = p[1];
            }
            if (k0 + 2 < dim) {
                v.z = p[2];
            }
            if (k0 + 3 < dim) {
                v.w = p[3];
            }
        }
    }
    return v;
}

// Scatter one global float4 (k = 4g .. 4g+3 of `row`) into the parity planes.
__device__ inline void
stage_store(float4* plane, uint32_t row, uint32_t g, float4 v) {
    uint32_t c = g >> 1, e = (g & 1) * 2;
    float* even = reinterpret_cast<float*>(&plane[(0 * 4 + c) * kPlane + row]) + e;
    float* odd = reinterpret_cast<float*>(&plane[(1 * 4 + c) * kPlane + row]) + e;
    *reinterpret_cast<float2*>(even) = make_float2(v.x, v.z);
    *reinterpret_cast<float2*>(odd) = make_float2(v.y, v.w);
}

// Which rows an assignment kernel works on: all (null pointers) or those that the fp16 pre-selection left open
// (kmeans_h16.hip): a flag per row, a word per 64 rows that says whether one of them is set, and one for all rows.  Such a
// launch has a workgroup per compute unit that walks the tiles, so that it costs little when nothing is open (a workgroup
// per tile, each of which found its rows done, took 178 us at 1M rows x 4096 centroids).
struct OpenRows {
    const uint8_t* row;
    const uint32_t* per64;
    const uint32_t* all;
    __device__ bool
    none() const {
        return all != nullptr && *all == 0;
    }
    OpenRows
    from(uint64_t r0) const {  // r0: a multiple of 64
        return row == nullptr ? *this : OpenRows{row + r0, per64 + r0 / 64, all};
    }
    __device__ bool
    any(uint64_t row0, uint32_t count, uint64_t n) const {
        if (per64 == nullptr) {
            return true;
        }
        uint32_t found = 0;
        for (uint64_t r = row0; r < row0 + count && r < n; r += 64) {
            found |= per64[r / 64];
        }
        return found != 0;
    }
    __device__ bool
    has(uint64_t r) const {
        return row == nullptr || row[r] != 0;
    }
};

__global__ void __launch_bounds__(256, 2)
kmeans_assign_kernel(const float* __restrict__ X, uint64_t n, const float* __restrict__ C, uint32_t k, uint32_t dim,
                     const float* __restrict__ ynorm, unsigned long long* __restrict__ best, uint32_t groups,
                     OpenRows open) {
    __shared__ Stage stage[2];  // 64 KiB: two workgroups fit the 160 KiB of a gfx950 CU
    if (open.none()) {
        return;
    }

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = tid >> 6;
    const uint32_t wm = wave & 1;   // which 64 centroids of the tile
    const uint32_t wn = wave >> 1;  // which 64 data rows of the tile
    const uint32_t half = lane >> 5;
    const uint32_t l32 = lane & 31;
    const bool aligned = (dim & 3) == 0;
    const uint32_t ktiles = (dim + BK - 1) / BK;
    const uint32_t ctiles = (k + BM - 1) / BM;

    // Loader roles: 1024 float4 per operand per stage, four per thread.
    uint32_t ld_row[4], ld_g[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        uint32_t idx = tid + 256 * r;
        ld_row[r] = idx >> 3;
        ld_g[r] = idx & 7;
    }

    for (uint64_t row0 = static_cast<uint64_t>(blockIdx.y) * BN; row0 < n; row0 += static_cast<uint64_t>(gridDim.y) * BN) {
    if (!open.any(row0, BN, n)) {
        continue;
    }
    unsigned long long my_best[2] = {~0ull, ~0ull};  // per n-block of this wave, for row l32

    for (uint32_t ct = blockIdx.x; ct < ctiles; ct += groups) {
        const uint64_t c0 = static_cast<uint64_t>(ct) * BM;
        floatx16 acc[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    acc[i][j][e] = 0.0F;
                }
            }
        }
        __syncthreads();  // the previous tile's readers of the stages are done
        float4 ra[4], rb[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            ra[r] = load_row_chunk(C, c0 + ld_row[r], k, 4 * ld_g[r], dim, aligned);
            rb[r] = load_row_chunk(X, row0 + ld_row[r], n, 4 * ld_g[r], dim, aligned);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            stage_store(stage[0].a, ld_row[r], ld_g[r], ra[r]);
            stage_store(stage[0].b, ld_row[r], ld_g[r], rb[r]);
        }
        __syncthreads();
        for (uint32_t kt = 0; kt < ktiles; ++kt) {
            const uint32_t cur = kt & 1;
            if (kt + 1 < ktiles) {
                uint32_t k0 = (kt + 1) * BK;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    ra[r] = load_row_chunk(C, c0 + ld_row[r], k, k0 + 4 * ld_g[r], dim, aligned);
                    rb[r] = load_row_chunk(X, row0 + ld_row[r], n, k0 + 4 * ld_g[r], dim, aligned);
                }
            }
            const float4* pa = stage[cur].a + half * 4 * kPlane + wm * 64 + l32;
            const float4* pb = stage[cur].b + half * 4 * kPlane + wn * 64 + l32;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                float4 a0 = pa[c * kPlane];
                float4 a1 = pa[c * kPlane + 32];
                float4 b0 = pb[c * kPlane];
                float4 b1 = pb[c * kPlane + 32];
                const float av0[4] = {a0.x, a0.y, a0.z, a0.w};
                const float av1[4] = {a1.x, a1.y, a1.z, a1.w};
                const float bv0[4] = {b0.x, b0.y, b0.z, b0.w};
                const float bv1[4] = {b1.x, b1.y, b1.z, b1.w};
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    acc[0][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(av0[e], bv0[e], acc[0][0], 0, 0, 0);
                    acc[0][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av0[e], bv1[e], acc[0][1], 0, 0, 0);
                    acc[1][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(av1[e], bv0[e], acc[1][0], 0, 0, 0);
                    acc[1][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av1[e], bv1[e], acc[1][1], 0, 0, 0);
                }
            }
            if (kt + 1 < ktiles) {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    stage_store(stage[cur ^ 1].a, ld_row[r], ld_g[r], ra[r]);
                    stage_store(stage[cur ^ 1].b, ld_row[r], ld_g[r], rb[r]);
                }
            }
            __syncthreads();
        }
        // Fused argmin: acc[i][j][e] = <c_m, x_n> with m = c0 + wm*64 + i*32 + 8*(e/4) + 4*half + e%4 and
        // n = row0 + wn*64 + j*32 + l32.  m grows with (i, e), so a strict `<` keeps the first minimum.
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            float bd = __builtin_inff();
            uint32_t bi = 0xFFFFFFFFU;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    uint32_t ml = wm * 64 + i * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
                    bool ok = c0 + ml < k;
                    float dist = (ok ? ynorm[c0 + ml] : 0.0F) + (-2.0F * acc[i][j][e]);
                    if (ok && dist < bd) {
                        bd = dist;
                        bi = static_cast<uint32_t>(c0) + ml;
                    }
                }
            }
            if (bi != 0xFFFFFFFFU) {
                unsigned long long key = make_key(bd, bi);
                if (key < my_best[j]) {
                    my_best[j] = key;
                }
            }
        }
    }
    // Combine the two halves of the wave (they hold different centroids of the same data row), then
    // publish with one 64-bit atomic per row and wave.
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        unsigned long long other = __shfl_xor(my_best[j], 32);
        unsigned long long key = other < my_best[j] ? other : my_best[j];
        uint64_t row = row0 + wn * 64 + j * 32 + l32;
        if (half == 0 && row < n && key != ~0ull && open.has(row)) {
            atomicMin(&best[row], key);
        }
    }
    }
}

// v or zeros, component by component (a conditional on the whole float4 would go through memory).
__device__ inline float4
keep_if(bool in, float4 v) {
    v.x = in ? v.x : 0.0F;
    v.y = in ? v.y : 0.0F;
    v.z = in ? v.z : 0.0F;
    v.w = in ? v.w : 0.0F;
    return v;
}

// The same contraction for dim % 4 == 0 (every row is a whole number of float4), one (row tile, centroid tile) per
// workgroup of eight waves: 256 data rows x (64 MI) centroids, MI = 2 or 4.  What bounds this kernel next to the matrix
// pipe is the stream of operand tiles from L2 into the CUs, so the tile is as large as LDS and registers allow: one
// workgroup per CU, 16 MI accumulator registers per 32 data rows.
//
// Stages of 16 k travel through a ring of three LDS slots.  In iteration s a wave stores the rows it loaded for
// stage s + 2 (the loads went out an iteration ago), sends the loads for stage s + 3, and contracts stage s; the
// operands of the first MFMAs of stage s + 1 are read from LDS while the last ones of stage s run, so the matrix pipe
// never waits for LDS across the one barrier per stage.  Slot (s + 2) % 3 last held stage s - 1, which every wave
// finished before the barrier that ended iteration s - 1.
//
// LDS layout per slot and operand: four planes of float4, plane g = 2c + h holds for every row the float4 of
// k = 8c + 4h .. 8c + 4h + 3 of the stage.  The contraction runs over all k, so the k a lane feeds to an MFMA step may
// be any bijection as long as both operands use the same one: lane (row, h) takes k = 8c + 4h + e in step 4c + e,
// which makes a global float4 one ds_write_b128 and a lane's operands for four steps one ds_read_b128.  Row r of
// plane g sits in slot r ^ (10 (g & 1) + 4 (g >> 1)): the float4 written by 8 (16) neighbouring lanes, 2 (4) rows of
// all planes, fall into different 16-byte columns of a 128 (256) byte bank period, and a read of 32 consecutive rows
// stays a permutation of 32 consecutive slots.
//
// Grid: one dimension.  Workgroups are dealt round-robin to the eight XCDs, so id % 8 is the XCD; the ids of one XCD
// walk macro tiles of (32 / mc) row tiles x mc centroid tiles, the 32 workgroups that run at the same time on that
// XCD and advance through k together: a k-slice of a row tile or centroid tile is fetched into the XCD's L2 once and
// hit by the other workgroups of its macro row / column.
struct TilePlan {
    uint32_t rtiles, ctiles;
    uint32_t mc_log2;  // macro tile: (32 >> mc_log2) row tiles x (1 << mc_log2) centroid tiles
    uint32_t mcols;    // macro tiles per macro row
    uint64_t ld;       // STORE: floats per row of the output
    float alpha;       // STORE: factor of the product
    uint32_t macros;
    OpenRows open;
};

constexpr int kTileRows = 256;  // data rows per workgroup tile
constexpr int kTileThreads = 512;
constexpr int kStageK = 16;     // contraction depth per stage
constexpr int kRing = 3;

constexpr size_t
tile_lds_bytes(int mi) {
    return kRing * static_cast<size_t>(4 * (64 * mi + kTileRows)) * sizeof(float4);
}

// STORE: instead of the argmin, every product goes out as out[m * plan.ld + n] = (ynorm ? ynorm[n] : 0) + plan.alpha *
// <c_m, x_n> (m a row of C, n a row of X; `best` is that float matrix, ynorm is indexed by rows of X): the table of
// approximate distances a routing call selects from (scan.hip, route_select_kernel).
template <int MI, bool STORE, bool OPEN>
__device__ __forceinline__ void
assign_tile(const float* __restrict__ X, uint64_t n, const float* __restrict__ C, uint32_t k, uint32_t dim,
            const float* __restrict__ ynorm, unsigned long long* __restrict__ best, const TilePlan& plan, uint32_t id) {
    constexpr uint32_t TM = 64 * MI;                   // centroids per tile
    constexpr uint32_t kSlot = 4 * (TM + kTileRows);   // float4 per ring slot: A planes, then B planes
    constexpr int RA = MI / 2;                         // float4 of A a thread loads per stage
    extern __shared__ float4 lds[];

    const uint32_t xcd = id & 7;
    const uint32_t local = id >> 3;
    const uint32_t macro = (local >> 5) * 8 + xcd;
    if (macro >= plan.macros) {
        return;
    }
    const uint32_t within = local & 31;
    const uint32_t rt = (macro / plan.mcols) * (32U >> plan.mc_log2) + (within >> plan.mc_log2);
    const uint32_t ct = ((macro % plan.mcols) << plan.mc_log2) + (within & ((1U << plan.mc_log2) - 1));
    if (rt >= plan.rtiles || ct >= plan.ctiles) {
        return;
    }
    if (OPEN && !plan.open.any(static_cast<uint64_t>(rt) * kTileRows, kTileRows, n)) {
        return;
    }

    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = tid >> 6;
    const uint32_t wm = wave & 1;   // which half of the tile's centroids
    const uint32_t wn = wave >> 1;  // which 64 data rows of the tile
    const uint32_t half = lane >> 5;
    const uint32_t l32 = lane & 31;
    const uint64_t row0 = static_cast<uint64_t>(rt) * kTileRows;
    const uint64_t c0 = static_cast<uint64_t>(ct) * TM;
    const uint32_t stages = (dim + kStageK - 1) / kStageK;

    // Loader: thread (r, g) of 128 x 4 moves float4 g of rows r, r + 128 of both operands (A: one row when the tile
    // has 128 centroids).  Rows past the end repeat the last one: their results are dropped at the end.
    const uint32_t lr = tid >> 2, lg = tid & 3;
    const float* pa[RA];
    const float* pb[2];
#pragma unroll
    for (int r = 0; r < RA; ++r) {
        const uint64_t ca = c0 + lr + 128 * r;
        pa[r] = C + (ca < k ? ca : k - 1) * dim;
    }
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const uint64_t xb = row0 + lr + 128 * r;
        pb[r] = X + (xb < n ? xb : n - 1) * dim;
    }
    const uint32_t wslot = lr ^ (10 * (lg & 1) + 4 * (lg >> 1));  // + 128 r
    const uint32_t wa = lg * TM + wslot;
    const uint32_t wb = 4 * TM + lg * kTileRows + wslot;
    // Reader: lane (l32, half) takes plane 2c + half, rows wm * 32 MI + 32 i + l32 of A and wn * 64 + 32 j + l32 of B.
    uint32_t ra_off[2], rb_off[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const uint32_t sw = 10 * half + 4 * c;
        ra_off[c] = (2 * c + half) * TM + wm * 32 * MI + (l32 ^ sw);
        rb_off[c] = 4 * TM + (2 * c + half) * kTileRows + wn * 64 + (l32 ^ sw);
    }

    floatx16 acc[MI][2];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] = 0.0F;
            }
        }
    }
    float4 ga[RA], gb[2];
    // Loads of stage t; past the last stage they repeat it and what they bring is never read.
    auto load_column = [&](uint32_t t) {
        const uint32_t k0 = (t < stages ? t : stages - 1) * kStageK + 4 * lg;
        return k0 < dim ? k0 : 0;
    };
    auto issue_loads = [&](uint32_t t) {
        const uint32_t col = load_column(t);
#pragma unroll
        for (int r = 0; r < RA; ++r) {
            ga[r] = *reinterpret_cast<const float4*>(pa[r] + col);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            gb[r] = *reinterpret_cast<const float4*>(pb[r] + col);
        }
    };
    auto store_stage = [&](uint32_t t, float4* slot) {
        const bool in = t * kStageK + 4 * lg < dim;
#pragma unroll
        for (int r = 0; r < RA; ++r) {
            slot[wa + 128 * r] = keep_if(in, ga[r]);
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            slot[wb + 128 * r] = keep_if(in, gb[r]);
        }
    };
    float4 fa[2][MI], fb[2][2];
    // Operand m of 6 (MI = 4) or 4 (MI = 2) of chunk c of a slot into buffer u.
    auto read_operand = [&](const float4* slot, int c, int u, int m) {
        if (m < MI) {
            fa[u][m] = slot[ra_off[c] + 32 * m];
        } else {
            fb[u][m - MI] = slot[rb_off[c] + 32 * (m - MI)];
        }
    };
    // The 2 MI MFMAs of step e of the chunk in buffer u; side(m) runs behind the m-th of them, so that the loads,
    // stores and LDS reads of the pipeline are issued while the matrix pipe works on an MFMA of this wave.
    auto mfma_step = [&](int u, int e, auto side) {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
            const float av = e == 0 ? fa[u][i].x : e == 1 ? fa[u][i].y : e == 2 ? fa[u][i].z : fa[u][i].w;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float bv = e == 0 ? fb[u][j].x : e == 1 ? fb[u][j].y : e == 2 ? fb[u][j].z : fb[u][j].w;
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc[i][j], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                side(2 * i + j);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    auto nothing = [](int) {};
    float4* s0 = lds;              // slot of the stage being contracted
    float4* s1 = lds + kSlot;      // of the next one
    float4* s2 = lds + 2 * kSlot;  // of the one after
    issue_loads(0);
    store_stage(0, s0);
    issue_loads(1);
    store_stage(1, s1);
    issue_loads(2);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MI + 2; ++m) {
        read_operand(s0, 0, 0, m);
    }
    for (uint32_t st = 0; st < stages; ++st) {
        const bool in = (st + 2) * kStageK + 4 * lg < dim;
        const uint32_t col = load_column(st + 3);
        // chunk 0; the operands of chunk 1 are read behind its first MFMAs
        mfma_step(0, 0, [&](int m) {
            if (m < MI + 2) {
                read_operand(s0, 1, 1, m);
            }
        });
        mfma_step(0, 1, nothing);
        mfma_step(0, 2, nothing);
        mfma_step(0, 3, nothing);
        // chunk 1; behind it the first operands of stage st + 1 (stored an iteration ago, behind the last barrier),
        // then the rows loaded for stage st + 2 go to LDS and the loads of stage st + 3 go out
        mfma_step(1, 0, [&](int m) {
            if (m < MI + 2) {
                read_operand(s1, 0, 0, m);
            }
        });
        mfma_step(1, 1, [&](int m) {
            if (m < RA) {
                s2[wa + 128 * m] = keep_if(in, ga[m]);
            } else if (m < RA + 2) {
                s2[wb + 128 * (m - RA)] = keep_if(in, gb[m - RA]);
            }
        });
        mfma_step(1, 2, [&](int m) {
            if (m < RA) {
                ga[m] = *reinterpret_cast<const float4*>(pa[m] + col);
            } else if (m < RA + 2) {
                gb[m - RA] = *reinterpret_cast<const float4*>(pb[m - RA] + col);
            }
        });
        mfma_step(1, 3, nothing);
        __syncthreads();
        float4* t = s0;
        s0 = s1;
        s1 = s2;
        s2 = t;
    }
    if constexpr (STORE) {
        float* out = reinterpret_cast<float*>(best);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint64_t row = row0 + wn * 64 + j * 32 + l32;
            const float base = row < n && ynorm != nullptr ? ynorm[row] : 0.0F;
#pragma unroll
            for (int i = 0; i < MI; ++i) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const uint32_t ml = wm * 32 * MI + i * 32 + 8 * (e >> 2) + 4 * half + (e & 3);
                    if (row < n && c0 + ml < k) {
                        out[(c0 + ml) * plan.ld + row] = base + plan.alpha * acc[i][j][e];
                    }
                }
            }
        }
        return;
    }
    // Fused argmin: acc[i][j][e] = <c_m, x_n> with m = c0 + wm*32*MI + i*32 + 8*(e/4) + 4*half + e%4 and
    // n = row0 + wn*64 + j*32 + l32.  m grows with (i, e), so a strict `<` keeps the first minimum.  |c|^2 comes four
    // centroids a load, once for both j, and is infinite past the last centroid, where nothing is ever less (with a load and
    // a test of the index for every product 747 490 x 96 rows and 436 centroids took 910 us, now 786).
    const bool whole = c0 + TM <= k;
    float bd[2] = {__builtin_inff(), __builtin_inff()};
    uint32_t bi[2] = {0xFFFFFFFFU, 0xFFFFFFFFU};
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        float yn[16];
        const uint64_t m0 = c0 + wm * 32 * MI + i * 32 + 4 * half;
        if (whole) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float4 v = *reinterpret_cast<const float4*>(ynorm + m0 + 8 * g);
                yn[4 * g] = v.x;
                yn[4 * g + 1] = v.y;
                yn[4 * g + 2] = v.z;
                yn[4 * g + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const uint64_t m = m0 + 8 * (e >> 2) + (e & 3);
                const float v = ynorm[m < k ? m : k - 1];
                yn[e] = m < k ? v : __builtin_inff();
            }
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                const float dist = yn[e] + (-2.0F * acc[i][j][e]);
                if (dist < bd[j]) {
                    bd[j] = dist;
                    bi[j] = static_cast<uint32_t>(m0) + 8 * (e >> 2) + (e & 3);
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        // the two halves of the wave hold different centroids of the same data row
        unsigned long long key = bi[j] != 0xFFFFFFFFU ? make_key(bd[j], bi[j]) : ~0ull;
        const unsigned long long other = __shfl_xor(key, 32);
        key = other < key ? other : key;
        const uint64_t row = row0 + wn * 64 + j * 32 + l32;
        if (half == 0 && row < n && key != ~0ull && (!OPEN || plan.open.has(row))) {
            atomicMin(&best[row], key);
        }
    }
}

// PAIR: two workgroups to a compute unit, so that one's start and end lie beside the other's contraction.  That leaves a lane 128
// registers, of which tiles of 128 centroids spill 21, so it is for calls with more workgroups than the chip holds at once:
// 1M x 128 rows, 100 centroids 940 -> 918 us an iteration, 1M x 960 3582 -> 3536, 150k x 24, 380 centroids 142 -> 136; with 79 to
// 391 workgroups it was slower, 20k x 128, 64 centroids 70.2 -> 72.8, 100k x 128, 128 centroids 120.4 -> 121.8.
template <int MI, bool STORE = false, bool PAIR = false>
__global__ void __launch_bounds__(kTileThreads, PAIR ? 4 : 1)
kmeans_assign_tile_kernel(const float* __restrict__ X, uint64_t n, const float* __restrict__ C, uint32_t k, uint32_t dim,
                          const float* __restrict__ ynorm, unsigned long long* __restrict__ best, TilePlan plan) {
    assign_tile<MI, STORE, false>(X, n, C, k, dim, ynorm, best, plan, blockIdx.x);
}

// The tiles that hold an open row; gridDim.x is a multiple of 8, so a workgroup's tiles stay on its XCD.
template <int MI>
__global__ void __launch_bounds__(kTileThreads, 1)
kmeans_assign_open_kernel(const float* __restrict__ X, uint64_t n, const float* __restrict__ C, uint32_t k, uint32_t dim,
                          const float* __restrict__ ynorm, unsigned long long* __restrict__ best, TilePlan plan,
                          uint32_t tiles) {
    if (plan.open.none()) {
        return;
    }
    for (uint32_t id = blockIdx.x; id < tiles; id += gridDim.x) {
        assign_tile<MI, false, true>(X, n, C, k, dim, ynorm, best, plan, id);
        __syncthreads();  // the next tile's first stages overwrite LDS
    }
}

__global__ void
fill_u64_kernel(unsigned long long* p, unsigned long long v, uint64_t n) {
    uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) {
        p[i] = v;
    }
}

// ||row||^2 for every row.  It is a read of the rows and nothing else, so what counts is bytes in flight: 16 lanes take a
// row in runs of 16 bytes each, four rows at once, and every component has a sum of its own.  The sums are those of a wave
// that takes dimension d in lane d % 64 and folds its lanes 32, 16, ... 1, bit for bit: with another order some rows between
// two centroids change their label.  904 914 x 416 rows: a wave per row and 4 bytes per lane 488 us (3.1 TB/s), this
// 242 us (6.2 TB/s); 747 490 x 96: 150 -> 46 us.
constexpr uint32_t kNormRows = 4;                       // rows of a group of 16 lanes
constexpr uint32_t kNormBlock = 16 * kNormRows;         // rows of a workgroup
typedef float float4_any __attribute__((ext_vector_type(4), aligned(4)));  // rows need not be 16-byte aligned

__global__ void __launch_bounds__(256)
row_sqnorm_kernel(const float* x, uint64_t n, uint32_t dim, float* out) {
    const uint32_t l16 = threadIdx.x & 15;
    const uint64_t row0 = static_cast<uint64_t>(blockIdx.x) * kNormBlock + (threadIdx.x >> 4) * kNormRows;
    const float* rows[kNormRows];
    float4_any sums[kNormRows];
#pragma unroll
    for (uint32_t r = 0; r < kNormRows; ++r) {  // (rows past the end repeat the last one)
        rows[r] = x + (row0 + r < n ? row0 + r : n - 1) * dim;
        sums[r] = float4_any{0.0F, 0.0F, 0.0F, 0.0F};
    }
    const uint32_t whole = dim & ~3U;
    for (uint32_t d = 4 * l16; d < whole; d += 64) {
        float4_any v[kNormRows];
#pragma unroll
        for (uint32_t r = 0; r < kNormRows; ++r) {
            v[r] = *reinterpret_cast<const float4_any*>(rows[r] + d);
        }
#pragma unroll
        for (uint32_t r = 0; r < kNormRows; ++r) {
#pragma unroll
            for (uint32_t e = 0; e < 4; ++e) {
                sums[r][e] = fmaf(v[r][e], v[r][e], sums[r][e]);
            }
        }
    }
    // Dimension d belongs to component d % 4 of lane (d % 64) / 4, behind those that the lane has summed above.
    if (whole < dim && l16 == (whole & 63) >> 2) {
#pragma unroll
        for (uint32_t r = 0; r < kNormRows; ++r) {
#pragma unroll
            for (uint32_t e = 0; e < 3; ++e) {
                if (whole + e < dim) {
                    const float v = rows[r][whole + e];
                    sums[r][e] = fmaf(v, v, sums[r][e]);
                }
            }
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < kNormRows; ++r) {
#pragma unroll
        for (uint32_t e = 0; e < 4; ++e) {
            for (int off = 8; off > 0; off >>= 1) {
                sums[r][e] += __shfl_down(sums[r][e], off, 16);
            }
        }
        if (l16 == 0 && row0 + r < n) {
            out[row0 + r] = (sums[r][0] + sums[r][2]) + (sums[r][1] + sums[r][3]);
        }
    }
}

// labels / min distances out of the keys, and the loss: sum over rows of double(float(min + ||x||^2))
// (kmeans_cluster.cpp:279-304).  Block partial sums go to `partial` and are added in block order by the
// last kernel, so the result does not depend on scheduling.
__global__ void __launch_bounds__(256)
kmeans_finalize_kernel(const unsigned long long* best, const float* xnorm, uint64_t n, int32_t* labels,
                       float* min_dist, double* partial) {
    __shared__ double red[4];
    uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    double v = 0.0;
    if (i < n) {
        unsigned long long key = best[i];
        float md = ordered_to_float(static_cast<uint32_t>(key >> 32));
        labels[i] = static_cast<int32_t>(static_cast<uint32_t>(key));
        if (min_dist != nullptr) {
            min_dist[i] = md;
        }
        v = static_cast<double>(md + xnorm[i]);
    }
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_down(v, off);
    }
    if ((threadIdx.x & 63) == 0) {
        red[threadIdx.x >> 6] = v;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        partial[blockIdx.x] = red[0] + red[1] + red[2] + red[3];
    }
}

// The block sums in a fixed order: a thread every 1024th of them, then a tree over the threads (one thread took 197 us for the
// 3907 sums of 1M rows).
__global__ void __launch_bounds__(1024)
loss_reduce_kernel(const double* partial, uint64_t count, uint64_t n, double* loss) {
    __shared__ double sums[1024];
    double s = 0.0;
    for (uint64_t i = threadIdx.x; i < count; i += blockDim.x) {
        s += partial[i];
    }
    sums[threadIdx.x] = s;
    __syncthreads();
    for (uint32_t w = 512; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            sums[threadIdx.x] += sums[threadIdx.x + w];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        *loss = sums[0] / static_cast<float>(n);
    }
}

// ------------------------------------------------------------------ centroid update
__global__ void
iota_u32_kernel(uint32_t* p, uint64_t n) {
    uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) {
        p[i] = static_cast<uint32_t>(i);
    }
}

__global__ void
count_labels_kernel(const int32_t* labels, uint64_t n, uint32_t k, uint32_t* counts) {
    uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < n) {
        int32_t l = labels[i];
        if (l >= 0 && static_cast<uint32_t>(l) < k) {
            atomicAdd(&counts[l], 1U);
        }
    }
}

// Exclusive prefix sum of k counts by one workgroup (k is a few thousand).
__global__ void __launch_bounds__(1024)
exclusive_scan_kernel(const uint32_t* counts, uint32_t k, uint32_t* offsets) {
    __shared__ uint32_t sums[16];
    uint32_t per = (k + blockDim.x - 1) / blockDim.x;
    uint32_t begin = threadIdx.x * per;
    uint32_t end = begin + per < k ? begin + per : k;
    uint32_t s = 0;
    for (uint32_t i = begin; i < end; ++i) {
        s += counts[i];
    }
    uint32_t upto = s;  // inclusive sums: over the lanes of a wave, then over the waves
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(upto, off);
        upto += static_cast<int>(threadIdx.x & 63) >= off ? v : 0;
    }
    if ((threadIdx.x & 63) == 63) {
        sums[threadIdx.x >> 6] = upto;
    }
    __syncthreads();
    uint32_t run = upto - s;
    for (uint32_t w = 0; w < (threadIdx.x >> 6); ++w) {
        run += sums[w];
    }
    if (threadIdx.x == blockDim.x - 1) {
        offsets[k] = run + s;
    }
    for (uint32_t i = begin; i < end; ++i) {
        offsets[i] = run;
        run += counts[i];
    }
}

// The rows of every label, in row order: a stable counting sort.  A unit is a run of rows; the units' counts per label
// stand in a table, a column of which is summed over the units, and one wave per unit then gives its rows their places.
// (Every row counted by an atomic on its label's counter in memory, and the rows sorted by hipCUB in up to 20 launches,
// took 1.41 ms for 904 914 rows of 98 labels, most of it the atomics that meet at a counter, and 0.15 ms for 1M rows of
// 4096; this takes 32 us for the first, 24-35 us for anything between.)
constexpr uint32_t kGroupMaxLabels = 16384;  // a unit's counters stand in 64 KB of LDS
constexpr uint32_t kGroupMinRows = 1024;     // rows of a unit, at least
constexpr uint32_t kGroupChunks = 16;        // parts of a column that are summed side by side

struct GroupPlan {
    uint32_t unit_rows, units;
};

// The table has units x k words and lies in the 2 n words of the buffers that the general sort keeps its pairs in.
static GroupPlan
group_plan(uint64_t n, uint32_t k) {
    GroupPlan p;
    p.unit_rows = static_cast<uint32_t>(round_up(k / 2 + 1 > kGroupMinRows ? k / 2 + 1 : kGroupMinRows, 64));
    p.units = static_cast<uint32_t>(div_up(n, p.unit_rows));
    return p;
}

static bool
group_takes(uint64_t n, uint32_t k) {
    return k <= kGroupMaxLabels && static_cast<uint64_t>(group_plan(n, k).units) * k <= 2 * n;
}

__global__ void __launch_bounds__(256)
group_count_kernel(const int32_t* labels, uint64_t n, uint32_t k, uint32_t unit_rows, uint32_t* table) {
    extern __shared__ uint32_t counters[];
    for (uint32_t l = threadIdx.x; l < k; l += blockDim.x) {
        counters[l] = 0;
    }
    __syncthreads();
    const uint64_t first = static_cast<uint64_t>(blockIdx.x) * unit_rows;
    const uint64_t last = first + unit_rows < n ? first + unit_rows : n;
    for (uint64_t i = first + threadIdx.x; i < last; i += blockDim.x) {
        const uint32_t l = static_cast<uint32_t>(labels[i]);
        if (l < k) {  // (a negative label is a large one here: no row of any centroid)
            atomicAdd(&counters[l], 1U);
        }
    }
    __syncthreads();
    for (uint32_t l = threadIdx.x; l < k; l += blockDim.x) {
        table[static_cast<uint64_t>(blockIdx.x) * k + l] = counters[l];
    }
}

// table[u][l] becomes the rows of label l in the units before u, counts[l] those of all units.  64 labels a workgroup (a
// lane each: whole lines), a wave for each part of the column.
__global__ void __launch_bounds__(64 * kGroupChunks)
group_columns_kernel(uint32_t* table, uint32_t units, uint32_t k, uint32_t* counts) {
    __shared__ uint32_t part[kGroupChunks][64];
    const uint32_t lane = threadIdx.x & 63, chunk = threadIdx.x >> 6;
    const uint32_t l = blockIdx.x * 64 + lane;
    const uint32_t per = (units + kGroupChunks - 1) / kGroupChunks;
    const uint32_t begin = chunk * per < units ? chunk * per : units;
    const uint32_t end = begin + per < units ? begin + per : units;
    uint32_t* column = table + (l < k ? l : k - 1);
    uint32_t sum = 0;
#pragma unroll 8
    for (uint32_t u = begin; u < end; ++u) {
        sum += column[static_cast<uint64_t>(u) * k];
    }
    part[chunk][lane] = sum;
    __syncthreads();
    uint32_t run = 0;
    for (uint32_t c = 0; c < chunk; ++c) {
        run += part[c][lane];
    }
    if (l >= k) {
        return;
    }
    if (chunk == kGroupChunks - 1) {
        counts[l] = run + sum;
    }
    for (uint32_t u0 = begin; u0 < end; u0 += 8) {  // eight loads on their way before the first store behind them
        uint32_t c[8];
#pragma unroll
        for (uint32_t v = 0; v < 8; ++v) {
            c[v] = column[static_cast<uint64_t>(u0 + v < end ? u0 + v : end - 1) * k];
        }
#pragma unroll
        for (uint32_t v = 0; v < 8; ++v) {
            if (u0 + v < end) {
                column[static_cast<uint64_t>(u0 + v) * k] = run;
                run += c[v];
            }
        }
    }
}

// One wave per unit: 64 rows at a time find, ballot by ballot over the bits of their labels, the lanes that share theirs;
// a row's place is its label's next one plus the lanes before it, and the last of them moves the label on.
__global__ void __launch_bounds__(64)
group_scatter_kernel(const int32_t* labels, uint64_t n, uint32_t k, uint32_t bits, uint32_t unit_rows,
                     const uint32_t* table, const uint32_t* offsets, uint32_t* rows_out) {
    extern __shared__ uint32_t next[];
    const uint32_t lane = threadIdx.x;
    for (uint32_t l = lane; l < k; l += 64) {
        next[l] = offsets[l] + table[static_cast<uint64_t>(blockIdx.x) * k + l];
    }
    __syncthreads();
    const uint64_t first = static_cast<uint64_t>(blockIdx.x) * unit_rows;
    const uint64_t last = first + unit_rows < n ? first + unit_rows : n;
    const uint64_t before = (1ull << lane) - 1;
    uint32_t l = first + lane < last ? static_cast<uint32_t>(labels[first + lane]) : 0xFFFFFFFFU;
    for (uint64_t i0 = first; i0 < last; i0 += 64) {
        const uint64_t ahead = i0 + 64 + lane;
        const uint32_t l_next = ahead < last ? static_cast<uint32_t>(labels[ahead]) : 0xFFFFFFFFU;
        const bool valid = l < k;
        uint64_t same = __ballot(valid);
        for (uint32_t b = 0; b < bits; ++b) {
            const bool bit = ((l >> b) & 1) != 0;
            const uint64_t set = __ballot(bit);
            same &= bit ? set : ~set;
        }
        if (valid) {
            const uint32_t place = next[l] + static_cast<uint32_t>(__popcll(same & before));
            rows_out[place] = static_cast<uint32_t>(i0 + lane);
            if ((same >> lane) == 1) {  // the last lane of its label
                next[l] = place + 1;
            }
        }
        __syncthreads();  // (one wave: the next rows read what was written above)
        l = l_next;
    }
}

// Mean of a centroid's member rows (rows sorted by label, in row order), fp32 running sums per dimension in row order.
// Empty clusters keep their centroid.
//
// A workgroup takes 64 dimensions of a centroid.  What bounds it is memory: the rows of a cluster lie anywhere, and the
// sums of a dimension are one chain, so the rows have to be on their way long before their turn.  256 threads bring 64
// rows at a time (16 lanes a 256-byte run) through registers into LDS, two such stages are in flight and the row numbers
// a stage further ahead; a fifth wave does nothing but add from LDS, so that the chain of a large cluster, which the launch
// ends with, does not wait for loads, addresses and LDS writes of its own wave (904 914 x 416 rows in 98 uneven clusters:
// 720 -> 660 us).
//
// An iteration on 1M x 960 rows and 4096 centroids 14.45 -> 13.81 ms with clusters of about 244 rows; where clusters are
// uneven (uniform rows: a workgroup per centroid with eight rows in flight took 7.9 ms for the largest), ten Lloyd
// iterations take 0.133 s.  The build of an ivf index from 120 000 x 96 rows, 256 lists: 33.2 -> 31.3 ms.
constexpr uint32_t kMeanDims = 64;
constexpr uint32_t kMeanRows = 64;   // per stage
constexpr uint32_t kMeanLoads = kMeanRows / 16;
constexpr uint32_t kMeanThreads = 256 + 64;  // four waves that load, one that adds
constexpr uint64_t kMeanGrid = 1ull << 22;

// QUADS: the dimension is a multiple of 4, a run of four dimensions lies in one row.
template <bool QUADS>
__global__ void __launch_bounds__(kMeanThreads)
centroid_mean_kernel(const float* x, uint32_t dim, uint32_t k, const uint32_t* sorted_rows, const uint32_t* offsets,
                     float* centroids, int32_t* counts_out) {
    __shared__ __align__(16) float stage[2][kMeanRows][kMeanDims];
    const uint32_t tid = threadIdx.x;
    const uint32_t quad = 4 * (tid & 15), slot = tid >> 4;
    const uint32_t chunks = (dim + kMeanDims - 1) / kMeanDims;
    const uint64_t tasks = static_cast<uint64_t>(k) * chunks;
    for (uint64_t task = blockIdx.x; task < tasks; task += gridDim.x) {
        const uint32_t j = static_cast<uint32_t>(task / chunks);
        const uint32_t d0 = static_cast<uint32_t>(task - static_cast<uint64_t>(j) * chunks) * kMeanDims;
        const uint32_t begin = offsets[j], end = offsets[j + 1];
        if (d0 == 0 && tid == 0) {
            counts_out[j] = static_cast<int32_t>(end - begin);
        }
        if (end == begin) {
            continue;
        }
        // (no branch around a load, or the wait for one stage would become a wait for all that are in flight: what lies
        // past the rows or the dimensions repeats the last of them and is not added)
        uint32_t rows[kMeanLoads];
        float4_any regs[2][kMeanLoads];
        auto number = [&](uint32_t first) {
#pragma unroll
            for (uint32_t u = 0; u < kMeanLoads; ++u) {
                const uint32_t p = first + 16 * u + slot;
                rows[u] = sorted_rows[p < end ? p : end - 1];
            }
        };
        auto fetch = [&](float4_any(&to)[kMeanLoads]) {
#pragma unroll
            for (uint32_t u = 0; u < kMeanLoads; ++u) {
                const float* row = x + static_cast<uint64_t>(rows[u]) * dim;
                if constexpr (QUADS) {
                    const uint32_t d = d0 + quad;
                    to[u] = *reinterpret_cast<const float4_any*>(row + (d < dim ? d : dim - 4));
                } else {
#pragma unroll
                    for (uint32_t e = 0; e < 4; ++e) {
                        const uint32_t d = d0 + quad + e;
                        to[u][e] = row[d < dim ? d : dim - 1];
                    }
                }
            }
        };
        if (tid < 256) {
            number(begin);
            fetch(regs[0]);
            number(begin + kMeanRows);
            fetch(regs[1]);
            number(begin + 2 * kMeanRows);
            for (uint32_t base = begin; base < end; base += 2 * kMeanRows) {
#pragma unroll
                for (uint32_t a = 0; a < 2; ++a) {
                    const uint32_t first = base + a * kMeanRows;
                    if (first >= end) {
                        break;
                    }
                    // Buffer a was last read two stages ago, a barrier ago.
#pragma unroll
                    for (uint32_t u = 0; u < kMeanLoads; ++u) {
                        const float4_any v = regs[a][u];
                        *reinterpret_cast<float4*>(&stage[a][16 * u + slot][quad]) = make_float4(v.x, v.y, v.z, v.w);
                    }
                    fetch(regs[a]);
                    number(first + 3 * kMeanRows);
                    __syncthreads();
                }
            }
        } else {
            __builtin_amdgcn_s_setprio(3);
            const uint32_t d = tid - 256;
            float s = 0.0F;
            uint32_t a = 0;
            for (uint32_t first = begin; first < end; first += kMeanRows, a ^= 1) {  // a barrier per stage, as above
                __syncthreads();
                if (end - first >= kMeanRows) {
#pragma unroll
                    for (uint32_t r = 0; r < kMeanRows; ++r) {
                        s += stage[a][r][d];
                    }
                } else {
                    for (uint32_t r = 0; r < end - first; ++r) {
                        s += stage[a][r][d];
                    }
                }
            }
            if (d0 + d < dim) {
                centroids[static_cast<uint64_t>(j) * dim + d0 + d] = s * (1.0F / static_cast<float>(end - begin));
            }
        }
        __syncthreads();  // the next task's first stages overwrite LDS
    }
}

void timing_begin(hipStream_t st);
void timing_end(hipStream_t st);

// out[m * ld + n] = (base ? base[n] : 0) + alpha <c_m, x_n> for the rows x_n of x (nx x dim) and c_m of c (nc x dim), on
// the fp32 matrix cores; dim a multiple of 4, rows 16-byte aligned.
int
launch_row_products(const float* x, uint64_t nx, const float* c, uint32_t nc, uint32_t dim, const float* base, float alpha,
                    float* out, uint64_t ld, hipStream_t st) {
    if ((dim & 3) != 0 || nx == 0 || nc == 0 || nx > (1ull << 20) * kTileRows) {
        return fail(VSAG_AMD_INVALID_ARGUMENT, "row products: the dimension must be a multiple of 4");
    }
    static std::once_flag lds_once;
    static hipError_t lds_rc = hipSuccess;
    std::call_once(lds_once, []() {
        lds_rc = hipFuncSetAttribute(reinterpret_cast<const void*>(kmeans_assign_tile_kernel<4, true>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(tile_lds_bytes(4)));
    });
    VA_HIP(lds_rc);
    TilePlan plan;
    plan.rtiles = static_cast<uint32_t>(div_up(nx, kTileRows));
    plan.ctiles = (nc + 255) / 256;
    plan.mc_log2 = plan.ctiles >= 8 ? 3 : plan.ctiles >= 4 ? 2 : plan.ctiles >= 2 ? 1 : 0;
    plan.mcols = (plan.ctiles + (1U << plan.mc_log2) - 1) >> plan.mc_log2;
    const uint32_t mrows = (plan.rtiles + (32U >> plan.mc_log2) - 1) / (32U >> plan.mc_log2);
    plan.macros = mrows * plan.mcols;
    plan.ld = ld;
    plan.alpha = alpha;
    plan.open = {nullptr, nullptr, nullptr};
    const uint32_t per_xcd = (plan.macros + 7) / 8;
    const dim3 grid(per_xcd * 32 * 8);
    hipLaunchKernelGGL((kmeans_assign_tile_kernel<4, true>), grid, dim3(kTileThreads), tile_lds_bytes(4), st, x, nx, c, nc,
                       dim, base, reinterpret_cast<unsigned long long*>(out), plan);
    VA_HIP(hipGetLastError());
    return 0;
}

// The largest finite value of out[0, n) as float bits (norms: not negative, so the bits order like the values); one
// workgroup.
__global__ void __launch_bounds__(1024)
max_norm_kernel(const float* out, uint64_t n, uint32_t* max_bits) {
    __shared__ float part[16];
    float m = 0.0F;
    for (uint64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const float v = out[i];
        m = v < __builtin_inff() ? fmaxf(m, v) : m;
    }
    for (int off = 32; off > 0; off >>= 1) {
        m = fmaxf(m, __shfl_xor(m, off));
    }
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x >> 6] = m;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (uint32_t w = 1; w < blockDim.x / 64; ++w) {
            m = fmaxf(m, part[w]);
        }
        *max_bits = __float_as_uint(m);
    }
}

// ||row||^2 of nx rows and the largest of them (as float bits).
int
launch_row_sqnorms(const float* x, uint64_t nx, uint32_t dim, float* out, uint32_t* max_bits, hipStream_t st) {
    hipLaunchKernelGGL(row_sqnorm_kernel, dim3(static_cast<uint32_t>(div_up(nx, kNormBlock))), dim3(256), 0, st, x, nx, dim, out);
    hipLaunchKernelGGL(max_norm_kernel, dim3(1), dim3(1024), 0, st, out, nx, max_bits);
    VA_HIP(hipGetLastError());
    return 0;
}

struct AssignBuffers {
    float* ynorm;
    float* xnorm;
    unsigned long long* best;
    double* partial;
    double* loss_tmp;
    bool h16;  // the fp16 pre-selection comes first (kmeans_h16.hip)
    KmeansH16Buffers pre;
};

// The pre-selection's buffers are up to 400 MB beside what the fp32 kernels need (12 bytes a row); a workspace without room
// for them is served by those (`preselect` false).
static size_t
carve_assign(Carver& c, uint64_t n, uint32_t dim, uint32_t k, bool preselect, AssignBuffers* b) {
    b->ynorm = c.take<float>(k);
    b->xnorm = c.take<float>(n);
    b->best = c.take<unsigned long long>(n);
    b->partial = c.take<double>(div_up(n, 256));
    b->loss_tmp = c.take<double>(1);
    b->h16 = preselect && kmeans_h16_takes(n, dim, k);
    if (b->h16) {
        carve_kmeans_h16(c, n, dim, k, &b->pre);
    }
    return c.used;
}

static int
assign_launch(const float* x, uint64_t n, uint32_t dim, const float* cent, uint32_t k, int32_t* labels,
              float* min_dist, double* loss_dev, const AssignBuffers& b, int iteration, hipStream_t st) {
    hipLaunchKernelGGL(row_sqnorm_kernel, dim3(static_cast<uint32_t>(div_up(k, kNormBlock))), dim3(256), 0, st, cent,
                       static_cast<uint64_t>(k), dim, b.ynorm);
    if (iteration == 0 && !b.h16) {  // (from the second Lloyd iteration on |x|^2 is there)
        hipLaunchKernelGGL(row_sqnorm_kernel, dim3(static_cast<uint32_t>(div_up(n, kNormBlock))), dim3(256), 0, st, x, n, dim,
                           b.xnorm);
    }
    if (!b.h16) {
        hipLaunchKernelGGL(fill_u64_kernel, dim3(static_cast<uint32_t>(div_up(n, 256))), dim3(256), 0, st, b.best, ~0ull,
                           n);
    }
    uint32_t ctiles = (k + BM - 1) / BM;
    timing_begin(st);
    OpenRows open = {nullptr, nullptr, nullptr};
    if (b.h16) {
        VA_TRY(launch_kmeans_h16(x, n, dim, cent, k, b.ynorm, b.xnorm, iteration, b.best, b.pre, st));
        // what follows does the rows that were left open: usually none, and its workgroups return at once
        open = {b.pre.row_open, b.pre.open64, &b.pre.state->any_open};
    }
    if ((dim & 3) == 0) {
        // 256 centroids per tile when there are enough of them to fill it, else 128
        const int mi = k > 384 ? 4 : 2;
        const uint32_t tile_m = 64 * mi;
        static std::once_flag lds_once;
        static hipError_t lds_rc = hipSuccess;
        std::call_once(lds_once, []() {
            auto allow = [](const void* kernel, int mi_of) {
                if (lds_rc == hipSuccess) {
                    lds_rc = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                 static_cast<int>(tile_lds_bytes(mi_of)));
                }
            };
            allow(reinterpret_cast<const void*>(kmeans_assign_tile_kernel<2>), 2);
            allow(reinterpret_cast<const void*>(kmeans_assign_tile_kernel<2, false, true>), 2);
            allow(reinterpret_cast<const void*>(kmeans_assign_tile_kernel<4>), 4);
            allow(reinterpret_cast<const void*>(kmeans_assign_open_kernel<2>), 2);
            allow(reinterpret_cast<const void*>(kmeans_assign_open_kernel<4>), 4);
        });
        VA_HIP(lds_rc);
        // rows go slab by slab so that the tile count stays far inside the grid limit
        const uint64_t slab_rows = (1ull << 20) * kTileRows;
        for (uint64_t r0 = 0; r0 < n; r0 += slab_rows) {
            const uint64_t rows = n - r0 < slab_rows ? n - r0 : slab_rows;
            TilePlan plan;
            plan.rtiles = static_cast<uint32_t>(div_up(rows, kTileRows));
            plan.ctiles = (k + tile_m - 1) / tile_m;
            plan.mc_log2 = plan.ctiles >= 8 ? 3 : plan.ctiles >= 4 ? 2 : plan.ctiles >= 2 ? 1 : 0;
            plan.mcols = (plan.ctiles + (1U << plan.mc_log2) - 1) >> plan.mc_log2;
            const uint32_t mrows = (plan.rtiles + (32U >> plan.mc_log2) - 1) / (32U >> plan.mc_log2);
            plan.macros = mrows * plan.mcols;
            plan.ld = 0;
            plan.alpha = 0.0F;
            plan.open = open.from(r0);
            const uint32_t per_xcd = (plan.macros + 7) / 8;
            const uint32_t tiles = per_xcd * 32 * 8;
            const dim3 grid(tiles);
            if (b.h16) {
                const uint32_t cus = static_cast<uint32_t>(device_cu_count()) / 8 * 8;
                const dim3 few(tiles < cus || cus == 0 ? tiles : cus);
                if (mi == 4) {
                    hipLaunchKernelGGL(kmeans_assign_open_kernel<4>, few, dim3(kTileThreads), tile_lds_bytes(4), st,
                                       x + r0 * dim, rows, cent, k, dim, b.ynorm, b.best + r0, plan, tiles);
                } else {
                    hipLaunchKernelGGL(kmeans_assign_open_kernel<2>, few, dim3(kTileThreads), tile_lds_bytes(2), st,
                                       x + r0 * dim, rows, cent, k, dim, b.ynorm, b.best + r0, plan, tiles);
                }
            } else if (mi == 4) {
                hipLaunchKernelGGL(kmeans_assign_tile_kernel<4>, grid, dim3(kTileThreads), tile_lds_bytes(4), st,
                                   x + r0 * dim, rows, cent, k, dim, b.ynorm, b.best + r0, plan);
            } else {
                const bool pair = static_cast<uint64_t>(plan.rtiles) * plan.ctiles > 2ull * device_cu_count();
                hipLaunchKernelGGL((pair ? kmeans_assign_tile_kernel<2, false, true> : kmeans_assign_tile_kernel<2>), grid,
                                   dim3(kTileThreads), tile_lds_bytes(2), st, x + r0 * dim, rows, cent, k, dim, b.ynorm,
                                   b.best + r0, plan);
            }
        }
    } else {
        uint32_t groups = ctiles < 8 ? ctiles : 8;
        // grid.y is limited to 65535 row tiles: larger inputs go slab by slab.
        const uint64_t slab_rows = 65535ull * BN;
        for (uint64_t r0 = 0; r0 < n; r0 += slab_rows) {
            uint64_t rows = n - r0 < slab_rows ? n - r0 : slab_rows;
            const uint32_t rtiles = static_cast<uint32_t>(div_up(rows, BN));
            dim3 grid(groups, b.h16 && rtiles > 128 ? 128 : rtiles);
            hipLaunchKernelGGL(kmeans_assign_kernel, grid, dim3(256), 0, st, x + r0 * dim, rows, cent, k, dim, b.ynorm,
                               b.best + r0, groups, open.from(r0));
        }
    }
    timing_end(st);
    hipLaunchKernelGGL(kmeans_finalize_kernel, dim3(static_cast<uint32_t>(div_up(n, 256))), dim3(256), 0, st, b.best,
                       b.xnorm, n, labels, min_dist, b.partial);
    hipLaunchKernelGGL(loss_reduce_kernel, dim3(1), dim3(1024), 0, st, b.partial, div_up(n, 256), n,
                       loss_dev ? loss_dev : b.loss_tmp);
    VA_HIP(hipGetLastError());
    return 0;
}

struct UpdateBuffers {
    uint32_t* counts;
    uint32_t* offsets;
    uint32_t* rows_in;
    uint32_t* rows_out;
    int32_t* keys_out;
    void* sort_tmp;
    size_t sort_tmp_bytes;
};

static size_t
sort_temp_bytes(uint64_t n) {
    size_t bytes = 0;
    // A size query only; a failure leaves 0 and the sort that follows reports it.
    if (hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, static_cast<const int32_t*>(nullptr),
                                           static_cast<int32_t*>(nullptr), static_cast<const uint32_t*>(nullptr),
                                           static_cast<uint32_t*>(nullptr), static_cast<int>(n), 0, 32,
                                           nullptr) != hipSuccess) {
        bytes = 0;
    }
    return bytes;
}

static size_t
carve_update(Carver& c, uint64_t n, uint32_t k, UpdateBuffers* b) {
    b->counts = c.take<uint32_t>(k + 1);
    b->offsets = c.take<uint32_t>(k + 1);
    b->rows_out = c.take<uint32_t>(n);
    b->rows_in = c.take<uint32_t>(n);  // (with keys_out behind it: the counting sort's table)
    b->keys_out = c.take<int32_t>(n);
    b->sort_tmp_bytes = sort_temp_bytes(n);
    b->sort_tmp = c.take<uint8_t>(b->sort_tmp_bytes);
    return c.used;
}

// Few, short centroids (the 16 centroids of a product-quantizer subspace): sorting the rows by label and giving a
// workgroup to each centroid leaves the machine idle.  Instead a workgroup sums a block of 1024 rows per (centroid,
// dimension) in row order, and a second launch adds the block sums in block order -- the order of the reference's own
// update, which sums per task of 1024 rows and merges the tasks (kmeans_cluster.cpp:108-154).
constexpr uint32_t kSmallUpdateRows = 1024;

__global__ void __launch_bounds__(256)
small_update_partial_kernel(const float* x, const int32_t* labels, uint64_t n, uint32_t dim, uint32_t k, float* psum,
                            uint32_t* pcount) {
    __shared__ int32_t lab[kSmallUpdateRows];
    const uint64_t row0 = static_cast<uint64_t>(blockIdx.x) * kSmallUpdateRows;
    const uint32_t rows = static_cast<uint32_t>(n - row0 < kSmallUpdateRows ? n - row0 : kSmallUpdateRows);
    for (uint32_t r = threadIdx.x; r < rows; r += blockDim.x) {
        lab[r] = labels[row0 + r];
    }
    __syncthreads();
    const uint32_t entries = k * dim;
    for (uint32_t e = threadIdx.x; e < entries; e += blockDim.x) {
        const int32_t c = static_cast<int32_t>(e / dim);
        const uint32_t d = e % dim;
        const float* col = x + row0 * dim + d;
        float s = 0.0F;
        uint32_t cnt = 0;
        for (uint32_t r = 0; r < rows; ++r) {
            if (lab[r] == c) {
                s += col[static_cast<uint64_t>(r) * dim];
                ++cnt;
            }
        }
        psum[static_cast<uint64_t>(blockIdx.x) * entries + e] = s;
        if (d == 0) {
            pcount[static_cast<uint64_t>(blockIdx.x) * k + c] = cnt;
        }
    }
}

__global__ void __launch_bounds__(256)
small_update_final_kernel(const float* psum, const uint32_t* pcount, uint32_t blocks, uint32_t dim, uint32_t k,
                          float* centroids, int32_t* counts_out) {
    const uint32_t e = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t entries = k * dim;
    if (e >= entries) {
        return;
    }
    const uint32_t c = e / dim;
    float s = 0.0F;
    uint32_t cnt = 0;
    for (uint32_t b = 0; b < blocks; ++b) {
        const uint32_t bc = pcount[static_cast<uint64_t>(b) * k + c];
        if (bc != 0) {
            s += psum[static_cast<uint64_t>(b) * entries + e];
            cnt += bc;
        }
    }
    if (e % dim == 0) {
        counts_out[c] = static_cast<int32_t>(cnt);
    }
    if (cnt != 0) {
        centroids[e] = s * (1.0F / static_cast<float>(cnt));  // empty clusters keep their centroid
    }
}

static int
update_launch(const float* x, const int32_t* labels, uint64_t n, uint32_t dim, uint32_t k, float* cent,
              int32_t* counts_dev, const UpdateBuffers& b, hipStream_t st) {
    const uint64_t small_blocks = div_up(n, static_cast<uint64_t>(kSmallUpdateRows));
    if (k <= 64 && static_cast<uint64_t>(k) * dim <= 512 && small_blocks * k * dim <= n && small_blocks * k <= n) {
        // the block sums and counts live where the sort of the general path keeps its row lists
        float* psum = reinterpret_cast<float*>(b.rows_in);
        uint32_t* pcount = b.rows_out;
        hipLaunchKernelGGL(small_update_partial_kernel, dim3(static_cast<uint32_t>(small_blocks)), dim3(256), 0, st, x,
                           labels, n, dim, k, psum, pcount);
        hipLaunchKernelGGL(small_update_final_kernel, dim3((k * dim + 255) / 256), dim3(256), 0, st, psum, pcount,
                           static_cast<uint32_t>(small_blocks), dim, k, cent, counts_dev);
        VA_HIP(hipGetLastError());
        return 0;
    }
    int end_bit = 1;
    while ((1ull << end_bit) < k) {
        ++end_bit;
    }
    if (group_takes(n, k)) {
        const GroupPlan p = group_plan(n, k);
        hipLaunchKernelGGL(group_count_kernel, dim3(p.units), dim3(256), k * sizeof(uint32_t), st, labels, n, k, p.unit_rows,
                           b.rows_in);
        hipLaunchKernelGGL(group_columns_kernel, dim3((k + 63) / 64), dim3(64 * kGroupChunks), 0, st, b.rows_in, p.units, k,
                           b.counts);
        hipLaunchKernelGGL(exclusive_scan_kernel, dim3(1), dim3(1024), 0, st, b.counts, k, b.offsets);
        hipLaunchKernelGGL(group_scatter_kernel, dim3(p.units), dim3(64), k * sizeof(uint32_t), st, labels, n, k,
                           static_cast<uint32_t>(end_bit), p.unit_rows, b.rows_in, b.offsets, b.rows_out);
    } else {
        // more labels than a unit has counters for
        uint32_t blocks = static_cast<uint32_t>(div_up(n, 256));
        hipLaunchKernelGGL(fill_u64_kernel, dim3((k / 2 + 1 + 255) / 256), dim3(256), 0, st,
                           reinterpret_cast<unsigned long long*>(b.counts), 0ull, static_cast<uint64_t>(k / 2 + 1));
        hipLaunchKernelGGL(count_labels_kernel, dim3(blocks), dim3(256), 0, st, labels, n, k, b.counts);
        hipLaunchKernelGGL(exclusive_scan_kernel, dim3(1), dim3(1024), 0, st, b.counts, k, b.offsets);
        hipLaunchKernelGGL(iota_u32_kernel, dim3(blocks), dim3(256), 0, st, b.rows_in, n);
        size_t tmp_bytes = b.sort_tmp_bytes;
        VA_HIP(hipcub::DeviceRadixSort::SortPairs(b.sort_tmp, tmp_bytes, labels, b.keys_out, b.rows_in, b.rows_out,
                                                  static_cast<int>(n), 0, end_bit, st));
    }
    const uint64_t tasks = static_cast<uint64_t>(k) * div_up(dim, kMeanDims);
    const dim3 grid(static_cast<uint32_t>(tasks < kMeanGrid ? tasks : kMeanGrid));
    if ((dim & 3) == 0) {
        hipLaunchKernelGGL(centroid_mean_kernel<true>, grid, dim3(kMeanThreads), 0, st, x, dim, k, b.rows_out, b.offsets, cent,
                           counts_dev);
    } else {
        hipLaunchKernelGGL(centroid_mean_kernel<false>, grid, dim3(kMeanThreads), 0, st, x, dim, k, b.rows_out, b.offsets, cent,
                           counts_dev);
    }
    VA_HIP(hipGetLastError());
    return 0;
}

static int
check_kmeans(const void* x, uint64_t n, uint32_t dim, const void* cent, uint32_t k) {
    VA_CHECK_ARG(k >= 1, "k must be positive");
    VA_CHECK_ARG(n >= 1, "count must be positive");
    VA_CHECK_ARG(x != nullptr && cent != nullptr, "datas cannot be null");
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    VA_CHECK_ARG(n < (1ull << 31), "n must be below 2^31");
    return 0;
}

// ---- k-means++ seeding (KMeansCluster::select_initial_centroids_kmeans_plus_plus, kmeans_cluster.cpp:383-435) -------
// One step = two launches: the distance of every row to the centroid chosen last lowers the row's smallest distance
// so far, and a row is drawn with a probability proportional to that distance -- the first row at which the running
// sum of the distances (a double, in row order) reaches the step's threshold draw * total.  The reference sums
// sequentially; here a block of 64 rows is summed in row order, blocks in chunks in block order, chunks in chunk
// order, chunks in runs: the same sums apart from the association of the double additions.
constexpr uint32_t kPpRows = 64;      // rows per workgroup of the distance launch (one wave, a lane per row)
constexpr uint32_t kPpChunks = 1024;  // threads of the picking workgroup: each sums a run of block sums

__global__ void __launch_bounds__(64)
kpp_distance_kernel(const float* x, uint64_t n, uint32_t dim, const float* centroid, float* min_dist, double* block_sum,
                    int first_step) {
    __shared__ float rows[kPpRows][kPpRows + 1];
    __shared__ float cent[kPpRows];
    __shared__ float md[kPpRows];
    const uint32_t lane = threadIdx.x;
    const uint64_t row0 = static_cast<uint64_t>(blockIdx.x) * kPpRows;
    // FP32ComputeL2Sqr in element order (simd/generic.cpp): result += (a - b) * (a - b), one row per lane.
    float result = 0.0F;
    for (uint32_t c0 = 0; c0 < dim; c0 += kPpRows) {
        const uint32_t d = c0 + lane;
        cent[lane] = d < dim ? centroid[d] : 0.0F;
        // All 64 loads of the chunk are issued before the first is used (no branch around a load: addresses are
        // clamped, what lies beyond the data is never used).
        const uint32_t dc = d < dim ? d : dim - 1;
        float v[kPpRows];
#pragma unroll
        for (uint32_t r = 0; r < kPpRows; ++r) {
            const uint64_t row = row0 + r < n ? row0 + r : n - 1;
            v[r] = x[row * dim + dc];
        }
#pragma unroll
        for (uint32_t r = 0; r < kPpRows; ++r) {
            rows[r][lane] = v[r];
        }
        __syncthreads();
        const uint32_t width = dim - c0 < kPpRows ? dim - c0 : kPpRows;
        for (uint32_t j = 0; j < width; ++j) {
            const float diff = rows[lane][j] - cent[j];
            result += diff * diff;
        }
        __syncthreads();
    }
    const uint64_t row = row0 + lane;
    float m = 0.0F;
    if (row < n) {
        const float old = first_step ? 3.402823466e38F : min_dist[row];
        m = result < old ? result : old;  // std::min(min_distances[i], dist)
        min_dist[row] = m;
    }
    md[lane] = m;
    __syncthreads();
    if (lane == 0) {
        double sum = 0.0;
        for (uint32_t r = 0; r < kPpRows; ++r) {
            sum += static_cast<double>(md[r]);
        }
        block_sum[blockIdx.x] = sum;
    }
}

// One workgroup.  The walk along the running sum goes down four levels -- 32 runs of 32 chunks, the chunks of a run,
// the block sums of a chunk, the 64 rows of a block -- and one thread does each walk over values the others have
// brought into LDS, so that no step of a walk waits for global memory.
__global__ void __launch_bounds__(kPpChunks)
kpp_pick_kernel(const float* x, uint64_t n, uint32_t dim, const float* min_dist, const double* block_sum,
                uint64_t nblocks, double draw, float* centroid_out, uint64_t* pick_out) {
    constexpr uint32_t kRuns = 32, kPerRun = kPpChunks / kRuns;
    __shared__ double chunk_sum[kPpChunks];
    __shared__ double run_sum[kRuns];
    __shared__ double staged[kPpChunks];
    __shared__ double cumulative_s, threshold_s;
    __shared__ uint64_t at_s;  // the chunk, then the block, then the row the walk has reached
    __shared__ int done_s;
    const uint32_t t = threadIdx.x;
    const uint64_t per = (nblocks + kPpChunks - 1) / kPpChunks;
    const uint64_t b0 = t * per, b1 = b0 + per < nblocks ? b0 + per : nblocks;
    double mine = 0.0;
    for (uint64_t b = b0; b < b1; ++b) {
        mine += block_sum[b];
    }
    chunk_sum[t] = mine;
    __syncthreads();
    if (t < kRuns) {
        double r = 0.0;
        for (uint32_t c = 0; c < kPerRun; ++c) {
            r += chunk_sum[t * kPerRun + c];
        }
        run_sum[t] = r;
    }
    __syncthreads();
    if (t == 0) {
        double total = 0.0;
        for (uint32_t r = 0; r < kRuns; ++r) {
            total += run_sum[r];
        }
        done_s = 0;
        if (!(total > 0.0)) {
            // Every row coincides with a centroid: any row (uniform_int_distribution in the reference).
            const double f = draw * static_cast<double>(n);
            at_s = f >= static_cast<double>(n - 1) ? n - 1 : static_cast<uint64_t>(f);
            done_s = 1;
        } else {
            const double threshold = draw * total;
            double cumulative = 0.0;
            uint32_t r = 0;
            while (r + 1 < kRuns && !(cumulative + run_sum[r] >= threshold)) {
                cumulative += run_sum[r];
                ++r;
            }
            uint32_t c = r * kPerRun;
            while (c + 1 < (r + 1) * kPerRun && !(cumulative + chunk_sum[c] >= threshold)) {
                cumulative += chunk_sum[c];
                ++c;
            }
            cumulative_s = cumulative;
            threshold_s = threshold;
            at_s = c;
        }
    }
    __syncthreads();
    if (done_s == 0) {
        // The block sums of the chunk, kPpChunks at a time.
        const uint64_t first = at_s * per;
        const uint64_t last = first + per < nblocks ? first + per : nblocks;  // may be <= first: a chunk without blocks
        __syncthreads();
        if (t == 0) {
            at_s = last > first ? last - 1 : (nblocks - 1);
        }
        for (uint64_t base = first; base < last; base += kPpChunks) {
            if (base + t < last) {
                staged[t] = block_sum[base + t];
            }
            __syncthreads();
            if (t == 0 && done_s == 0) {
                const uint64_t m = last - base < kPpChunks ? last - base : kPpChunks;
                double cumulative = cumulative_s;
                for (uint64_t i = 0; i < m; ++i) {
                    if (base + i + 1 == last || cumulative + staged[i] >= threshold_s) {
                        at_s = base + i;
                        done_s = 2;
                        break;
                    }
                    cumulative += staged[i];
                }
                cumulative_s = cumulative;
            }
            __syncthreads();
            if (done_s != 0) {
                break;
            }
        }
        __syncthreads();
        const uint64_t blk = at_s;
        const uint64_t r0 = blk * kPpRows, r1 = r0 + kPpRows < n ? r0 + kPpRows : n;
        if (t < kPpRows) {
            staged[t] = r0 + t < r1 ? static_cast<double>(min_dist[r0 + t]) : 0.0;
        }
        __syncthreads();
        if (t == 0) {
            uint64_t idx = r1 - 1;
            double cumulative = cumulative_s;
            for (uint64_t r = r0; r < r1; ++r) {
                cumulative += staged[r - r0];
                if (cumulative >= threshold_s) {
                    idx = r;
                    break;
                }
            }
            at_s = idx;
        }
        __syncthreads();
    }
    const uint64_t idx = at_s;
    if (t == 0 && pick_out != nullptr) {
        *pick_out = idx;
    }
    for (uint32_t d = t; d < dim; d += kPpChunks) {
        centroid_out[d] = x[idx * dim + d];
    }
}

}  // namespace vsag_amd

using namespace vsag_amd;

extern "C" size_t
vsag_amd_kmeans_init_plus_plus_workspace_bytes(uint64_t n) {
    Carver c(nullptr, 0);
    c.take<float>(n);
    c.take<double>(div_up(n, static_cast<uint64_t>(kPpRows)));
    return c.used + 256;
}

extern "C" int
vsag_amd_kmeans_init_plus_plus(const float* x_dev, uint64_t n, uint32_t dim, uint32_t k, uint64_t first,
                               const double* draws, float* centroids_dev, uint64_t* picks_dev, void* workspace_dev,
                               size_t workspace_bytes, void* stream) {
    VA_TRY(ensure_init());
    VA_TRY(check_kmeans(x_dev, n, dim, centroids_dev, k));
    VA_CHECK_ARG(k <= n, "k cannot be larger than count");
    VA_CHECK_ARG(first < n, "the first centroid must be a row of the data");
    VA_CHECK_ARG(k == 1 || draws != nullptr, "draws is null");
    for (uint32_t c = 1; c < k; ++c) {
        VA_CHECK_ARG(draws[c - 1] >= 0.0 && draws[c - 1] < 1.0, "draws must lie in [0, 1)");
    }
    hipStream_t st = static_cast<hipStream_t>(stream);
    Carver c(workspace_dev, workspace_bytes);
    float* min_dist = c.take<float>(n);
    const uint64_t nblocks = div_up(n, static_cast<uint64_t>(kPpRows));
    double* block_sum = c.take<double>(nblocks);
    VA_CHECK_ARG(c.ok(), "workspace too small: need %zu bytes, got %zu", c.used, workspace_bytes);
    VA_HIP(hipMemcpyAsync(centroids_dev, x_dev + first * dim, dim * sizeof(float), hipMemcpyDeviceToDevice, st));
    if (picks_dev != nullptr) {
        VA_HIP(hipMemcpyAsync(picks_dev, &first, sizeof(uint64_t), hipMemcpyHostToDevice, st));
        VA_HIP(hipStreamSynchronize(st));  // `first` lives on this frame
    }
    for (uint32_t j = 1; j < k; ++j) {
        hipLaunchKernelGGL(kpp_distance_kernel, dim3(static_cast<uint32_t>(nblocks)), dim3(kPpRows), 0, st, x_dev, n, dim,
                           centroids_dev + static_cast<uint64_t>(j - 1) * dim, min_dist, block_sum, j == 1 ? 1 : 0);
        hipLaunchKernelGGL(kpp_pick_kernel, dim3(1), dim3(kPpChunks), 0, st, x_dev, n, dim, min_dist, block_sum, nblocks,
                           draws[j - 1], centroids_dev + static_cast<uint64_t>(j) * dim,
                           picks_dev != nullptr ? picks_dev + j : nullptr);
    }
    VA_HIP(hipGetLastError());
    return 0;
}

extern "C" size_t
vsag_amd_kmeans_assign_workspace_bytes(uint64_t n, uint32_t dim, uint32_t k) {
    Carver c(nullptr, 0);
    AssignBuffers b;
    return carve_assign(c, n, dim, k, true, &b) + 256;
}

extern "C" int
vsag_amd_kmeans_assign(const float* x_dev, uint64_t n, uint32_t dim, const float* centroids_dev, uint32_t k,
                       int32_t* labels_dev, float* min_dist_dev, double* loss_dev, void* workspace_dev,
                       size_t workspace_bytes, void* stream) {
    VA_TRY(ensure_init());
    VA_TRY(check_kmeans(x_dev, n, dim, centroids_dev, k));
    VA_CHECK_ARG(labels_dev != nullptr, "labels_dev is null");
    Carver c(workspace_dev, workspace_bytes);
    AssignBuffers b;
    carve_assign(c, n, dim, k, true, &b);
    if (!c.ok() && b.h16) {
        c = Carver(workspace_dev, workspace_bytes);
        carve_assign(c, n, dim, k, false, &b);
    }
    VA_CHECK_ARG(c.ok(), "workspace too small: need %zu bytes, got %zu", c.used, workspace_bytes);
    return assign_launch(x_dev, n, dim, centroids_dev, k, labels_dev, min_dist_dev, loss_dev, b, 0,
                         static_cast<hipStream_t>(stream));
}

extern "C" size_t
vsag_amd_kmeans_update_workspace_bytes(uint64_t n, uint32_t dim, uint32_t k) {
    (void)dim;
    if (ensure_init() != 0) {
        return 0;
    }
    Carver c(nullptr, 0);
    UpdateBuffers b;
    return carve_update(c, n, k, &b) + 256;
}

extern "C" int
vsag_amd_kmeans_update(const float* x_dev, const int32_t* labels_dev, uint64_t n, uint32_t dim, uint32_t k,
                       float* centroids_dev, int32_t* counts_dev, void* workspace_dev, size_t workspace_bytes,
                       void* stream) {
    VA_TRY(ensure_init());
    VA_TRY(check_kmeans(x_dev, n, dim, centroids_dev, k));
    VA_CHECK_ARG(labels_dev != nullptr && counts_dev != nullptr, "null labels / counts");
    Carver c(workspace_dev, workspace_bytes);
    UpdateBuffers b;
    carve_update(c, n, k, &b);
    VA_CHECK_ARG(c.ok(), "workspace too small: need %zu bytes, got %zu", c.used, workspace_bytes);
    return update_launch(x_dev, labels_dev, n, dim, k, centroids_dev, counts_dev, b, static_cast<hipStream_t>(stream));
}

namespace vsag_amd {
struct RunBuffers {
    AssignBuffers assign;
    UpdateBuffers update;
    int32_t* counts;
};

static size_t
carve_run(Carver& c, uint64_t n, uint32_t dim, uint32_t k, bool preselect, RunBuffers* b) {
    carve_assign(c, n, dim, k, preselect, &b->assign);
    carve_update(c, n, k, &b->update);
    b->counts = c.take<int32_t>(k);
    return c.used;
}
}  // namespace vsag_amd

extern "C" size_t
vsag_amd_kmeans_run_workspace_bytes(uint64_t n, uint32_t dim, uint32_t k) {
    if (ensure_init() != 0) {
        return 0;
    }
    Carver c(nullptr, 0);
    RunBuffers b;
    return carve_run(c, n, dim, k, true, &b) + 256;
}

extern "C" int
vsag_amd_kmeans_run(const float* x_dev, uint64_t n, uint32_t dim, float* centroids_dev, uint32_t k, int iters,
                    uint64_t seed, int32_t* labels_dev, double* loss, void* workspace_dev, size_t workspace_bytes,
                    void* stream) {
    VA_TRY(ensure_init());
    VA_TRY(check_kmeans(x_dev, n, dim, centroids_dev, k));
    VA_CHECK_ARG(k <= n, "k cannot be larger than count");
    VA_CHECK_ARG(labels_dev != nullptr, "labels_dev is null");
    VA_CHECK_ARG(iters >= 0, "iters must not be negative");
    hipStream_t st = static_cast<hipStream_t>(stream);
    Carver c(workspace_dev, workspace_bytes);
    RunBuffers b;
    carve_run(c, n, dim, k, true, &b);
    if (!c.ok() && b.assign.h16) {
        c = Carver(workspace_dev, workspace_bytes);
        carve_run(c, n, dim, k, false, &b);
    }
    const AssignBuffers& a = b.assign;
    const UpdateBuffers& u = b.update;
    int32_t* const counts_dev = b.counts;
    VA_CHECK_ARG(c.ok(), "workspace too small: need %zu bytes, got %zu", c.used, workspace_bytes);

    std::mt19937 gen(static_cast<uint32_t>(seed));
    std::vector<int32_t> counts(k);
    double last = 0.0;
    for (int it = 0; it < iters; ++it) {
        VA_TRY(assign_launch(x_dev, n, dim, centroids_dev, k, labels_dev, nullptr, a.loss_tmp, a, it, st));
        VA_TRY(update_launch(x_dev, labels_dev, n, dim, k, centroids_dev, counts_dev, u, st));
        VA_HIP(hipMemcpyAsync(counts.data(), counts_dev, k * sizeof(int32_t), hipMemcpyDeviceToHost, st));
        VA_HIP(hipMemcpyAsync(&last, a.loss_tmp, sizeof(double), hipMemcpyDeviceToHost, st));
        VA_HIP(hipStreamSynchronize(st));
        // Empty clusters restart from a random data row (kmeans_cluster.cpp:156-171).
        std::uniform_int_distribution<uint64_t> dis(0, n - 1);
        for (uint32_t j = 0; j < k; ++j) {
            if (counts[j] == 0) {
                uint64_t idx = dis(gen);
                VA_HIP(hipMemcpyAsync(centroids_dev + static_cast<uint64_t>(j) * dim, x_dev + idx * dim,
                                      dim * sizeof(float), hipMemcpyDeviceToDevice, st));
            }
        }
    }
    VA_HIP(hipStreamSynchronize(st));
    if (loss != nullptr) {
        *loss = last;
    }
    return 0;
}
