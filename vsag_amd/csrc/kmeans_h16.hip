// Pre-selection of the k-means assignment on the fp16 matrix cores.
//
// The fp32 contraction of kmeans.hip is bound by the fp32 matrix rate (1M rows x 960 x 4096 centroids: 62 ms at 127
// TFLOP/s, 80 % of that peak).  The fp16 instruction is sixteen times as fast, and almost every centroid of a row can be
// ruled out with far less than fp32 accuracy, so the contraction runs on rows and centroids rounded to fp16 and only
// decides which centroids are still possible; those get their distance from the fp32 values by the chain of fma that the
// fp32 kernels run, and the smallest (distance, index) wins: the result is theirs bit for bit.
//
// What the test rests on.  With a centre m (any point; the mean of some centroids keeps the lengths small), x' = x - m,
// c' = c - m and their fp16 forms X, C:  |x - c|^2 - |x'|^2 = |c'|^2 - 2 <x', c'>, and
//     |<x', c'> - <X, C>| <= |x' - X| |c'| + |X| |c' - C|
// with the lengths of the actual remainders, summed per row and centroid when they are rounded.  Together with the
// roundings of the accumulation, of |c'|^2, of the stored value and of the final fp32 distances that is the row's error
// bound E (largest |c'| and |c' - C| taken): a centroid is possible only if its approximate distance is within 2 E of the
// row's least one.
//
// The contraction leaves, per row and group of 64 centroids, the three least approximate distances, the low six mantissa
// bits of each saying which centroid: 12 bytes where the products would be 256.  A group brings those of the first two
// that are possible, or all its 64 centroids where the third is possible too (with two values per group, and a group
// open once its second was possible, a first form of the rescoring took 4.2 ms and not 1.9: every group of 64 is 64
// distances).  Rows with more than kMaxWork distances to form, and rows that are not finite or too large, are
// marked and left to the fp32 kernels.  What those cost does not depend on how many rows of a
// tile of 256 are open, so a few in a hundred, scattered, cost what all do: where a common offset of rows and centroids is
// many times their spread (the fp32 distances themselves are rounded to that), or centroids are missing from whole clusters,
// a call can pay for both.  So every fourth slab (of one slab: every fourth Lloyd iteration) is a probe, and where it left
// rows open in more than half of its groups of 64, the three behind it go to the fp32 kernels at once.  Clusters of width 0.05
// ten times the centres' range from the origin, fp32 kernels / every slab tried / this, ms: 1M x 960, k 4096 63.3 / 77.4 /
// 67.9; 480k x 960, k 256 2.42 / 3.51 / 2.68; of a single slab (65536 x 128, k 512) 0.12 / 0.18 / 0.18.  Where nothing is
// open, asking costs 0.5 to 1 %.
//
// 1M x 960 rows, 4096 centroids (one assignment): 63.3 -> 11.2 ms.  Of that the contraction takes 7.4 to 7.8 (7.9e12 flop: 1010
// to 1070 TFLOP/s, from card to card, where matrix instructions on random operands in registers reach 1730 and with their reads
// of LDS 1610, bound by power: 2330 and 2240 on zeros), the rounding of the rows 1.25 (5.8 GB at 4.6 TB/s) and the rescoring 2.4
// (3.8 GB of rows, 0.8 GB of table, one to three centroids a row).
#include "kmeans_h16.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace vsag_amd {

typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef float float4_v __attribute__((ext_vector_type(4)));

constexpr uint32_t kTile = 256;        // centroids x rows of a workgroup's tile
constexpr uint32_t kThreads = 512;
constexpr uint32_t kStage = 64;        // dimensions per stage: a row's part is one 128-byte line
constexpr uint32_t kSlots = kStage / 8;
constexpr uint32_t kGroup = 64;        // centroids per entry of the table
constexpr uint32_t kRowsPerBlock = 64; // rescoring: rows of a workgroup
constexpr uint32_t kParts = 4;         // rescoring: waves of a workgroup
constexpr uint32_t kPairs = 128;       // rescoring: (row, centroid) pairs at a time
constexpr uint32_t kPiece = 32;        // rescoring: dimensions at a time
constexpr uint32_t kPitch = kPiece + 4;
constexpr uint32_t kMaxList = 24;      // rescoring: entries (a centroid, or a whole group) per row
constexpr uint32_t kMaxWork = 160;     // rescoring: distances per row
constexpr uint32_t kProbes = 4;        // every fourth slab or iteration is a probe
constexpr uint32_t kProbeStep = 16;    // of which every 16th workgroup counts (all of them: 60 us of atomics on one word)
constexpr uint64_t kSlabHalves = 64ull << 20;  // fp16 values per slab: 128 MB stay in the 256 MB memory-side cache
constexpr uint64_t kTableBytes = 256ull << 20;  // the table of a slab: the rows get fewer as the centroids get more ...
constexpr uint64_t kMinSlabRows = 4096;         // ... down to this
constexpr uint32_t kMaxDim = 8192;

static uint32_t
padded_dim(uint32_t dim) {
    return static_cast<uint32_t>(round_up(dim, kStage));
}
static uint64_t
tile_count(uint32_t k) {
    return div_up(k, kTile);
}
static uint64_t
table_row_bytes(uint32_t k) {
    return tile_count(k) * (kTile / kGroup) * 3 * sizeof(float);
}
static uint64_t
slab_rows(uint64_t n, uint32_t dim, uint32_t k) {
    const uint64_t rows = std::min({kSlabHalves / padded_dim(dim), kTableBytes / table_row_bytes(k), uint64_t{1} << 18}) /
                          kTile * kTile;
    return n < rows ? round_up(n, kTile) : rows;
}

// Where it pays: rounding and rescoring cost a row about 0.7 ns up to 128 dimensions (one read of it each), which the
// fp32 kernels need for 40 000 products at 110 TFLOP/s; the six launches before and after the contraction take 40 us, and
// a tile holds 256 centroids.  Measured, fp32 -> this, ms: 131072 x 128, k 256 0.148 -> 0.156 (not taken); 65536 x 128,
// k 512 0.128 -> 0.112; 300000 x 101, k 512 0.65 -> 0.43; 22000 x 960, k 200 0.165 -> 0.175 (not taken); 1M x 960, k 256
// 5.28 -> 3.65; 1M x 32, k 256 0.62 -> 0.85 (not taken); 1M x 37, k 4096 7.4 -> 2.5.
bool
kmeans_h16_takes(uint64_t n, uint32_t dim, uint32_t k) {
    const double products = static_cast<double>(k) * dim;
    return dim >= 32 && dim <= kMaxDim && k >= 256 && products >= 49152.0 && static_cast<double>(n) * products >= 4.0e9 &&
           slab_rows(n, dim, k) >= std::min(n, kMinSlabRows);
}

void
carve_kmeans_h16(Carver& c, uint64_t n, uint32_t dim, uint32_t k, KmeansH16Buffers* b) {
    const uint64_t rows = slab_rows(n, dim, k);
    const uint32_t dpad = padded_dim(dim);
    b->x16 = c.take<uint16_t>(rows * dpad);
    b->c16 = c.take<uint16_t>(static_cast<uint64_t>(k) * dpad);
    b->xinfo = c.take<float2>(rows);
    b->xscale = c.take<float>(rows);
    b->group_min = c.take<float>(table_row_bytes(k) / sizeof(float) * rows);
    b->centre = c.take<float>(dim);
    b->cnorm = c.take<float>(k);
    b->state = c.take<KmeansH16State>(1);
    b->row_open = c.take<uint8_t>(n);
    b->open64 = c.take<uint32_t>(div_up(n, kRowsPerBlock));
}

__device__ inline void
reset_state(KmeansH16State* state, uint32_t open_groups) {
    *state = {0, 0, 0, 0, 0, __float_as_uint(__builtin_inff()), open_groups};
}

// A centre: per dimension, sixteen means of sixteen centroids each, the middle half of them averaged -- a few centroids far
// out do not move it.  64 dimensions per workgroup; finite whatever the centroids hold.
__global__ void __launch_bounds__(1024)
kmeans_centre_kernel(const float* cent, uint32_t k, uint32_t dim, float* centre, KmeansH16State* state) {
    __shared__ float part[16][64];
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        reset_state(state, 0);
    }
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t d = blockIdx.x * 64 + lane;
    const uint32_t step = k / 256;  // k >= 256
    float s = 0.0F;
    if (d < dim) {
        for (uint32_t i = w; i < 256; i += 16) {
            s += cent[static_cast<uint64_t>(i) * step * dim + d];
        }
    }
    s *= 1.0F / 16.0F;
    part[w][lane] = s - s == 0.0F ? s : 3.0e38F;
    __syncthreads();
    if (w == 0 && d < dim) {
        float t = 0.0F;
        for (uint32_t i = 0; i < 16; ++i) {
            const float v = part[i][lane];
            uint32_t rank = 0;
            for (uint32_t j = 0; j < 16; ++j) {
                const float o = part[j][lane];
                rank += o < v || (o == v && j < i) ? 1U : 0U;
            }
            t += rank >= 4 && rank < 12 ? v : 0.0F;
        }
        t *= 1.0F / 8.0F;
        centre[d] = t - t == 0.0F ? t : 0.0F;
    }
}

__global__ void
kmeans_reset_kernel(KmeansH16State* state, int probe) {
    if (threadIdx.x == 0) {
        reset_state(state, probe != 0 ? 0 : state->open_groups);
    }
}

__device__ inline float4
load4(const float* row, uint32_t d, uint32_t dim, bool wide) {
    if (wide) {
        return *reinterpret_cast<const float4*>(row + d);
    }
    float4 v;
    v.x = row[d];
    v.y = d + 1 < dim ? row[d + 1] : 0.0F;
    v.z = d + 2 < dim ? row[d + 2] : 0.0F;
    v.w = d + 3 < dim ? row[d + 3] : 0.0F;
    return v;
}

// Not negative: orders like the value, NaN above infinity.
__device__ inline uint32_t
magnitude_bits(float v) {
    return __float_as_uint(v) & 0x7FFFFFFFU;
}

__device__ inline float
wave_sum(float v) {
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_xor(v, off);
    }
    return v;
}

// |c'|^2 per centroid, a wave each.
__global__ void __launch_bounds__(1024)
kmeans_cnorm_kernel(const float* cent, uint32_t k, uint32_t dim, const float* centre, float* cnorm) {
    const uint32_t lane = threadIdx.x & 63;
    for (uint32_t c = blockIdx.x * kGroup + (threadIdx.x >> 6); c < (blockIdx.x + 1) * kGroup && c < k; c += 16) {
        const float* row = cent + static_cast<uint64_t>(c) * dim;
        float s = 0.0F;
        for (uint32_t d = lane; d < dim; d += 64) {
            const float v = row[d] - centre[d];
            s = fmaf(v, v, s);
        }
        s = wave_sum(s);
        if (lane == 0) {
            cnorm[c] = s;
        }
    }
}

// 2^e with 2^e sqrt(sq) in [2^13, 2^14): no entry exceeds the length, so none leaves the fp16 range.  The exponent is
// kept within bounds that leave products of two scales normal; below them fp16 holds fewer bits, which the remainders say.
__device__ inline int
scale_exponent(float sq) {
    int e = 0;
    (void)frexpf(sqrtf(sq), &e);
    e = 14 - e;
    return e > 50 ? 50 : e < -49 ? -49 : e;
}

// Rounds a row (less the centre, times 2^e) to fp16, zeros up to dpad; what is left out (|x' - X|^2) and kept (|X|^2),
// in the scale of the row.  x - m is taken in fp32 and its own rounding (2^-24 of it) added to the remainder.
__device__ inline void
round_row(const float* row, uint32_t dim, uint32_t dpad, const float* centre, bool wide, float up, uint16_t* out,
          float* missed, float* kept) {
    const uint32_t lane = threadIdx.x & 63;
    float ms = 0.0F, ks = 0.0F;
    for (uint32_t d = 4 * lane; d < dpad; d += 256) {
        float v[4] = {0.0F, 0.0F, 0.0F, 0.0F};
        if (d < dim) {
            const float4 a = load4(row, d, dim, wide);
            const float4 m = load4(centre, d, dim, wide);
            v[0] = (a.x - m.x) * up;
            v[1] = (a.y - m.y) * up;
            v[2] = (a.z - m.z) * up;
            v[3] = (a.w - m.w) * up;
        }
        halfx4 h;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h[i] = static_cast<_Float16>(v[i]);
            const float back = static_cast<float>(h[i]);
            const float left = fabsf(v[i] - back) + 6.0e-8F * fabsf(v[i]);
            ms = fmaf(left, left, ms);
            ks = fmaf(back, back, ks);
        }
        *reinterpret_cast<halfx4*>(out + d) = h;
    }
    *missed = wave_sum(ms);
    *kept = wave_sum(ks);
}

// The error bound of every row holds the largest centroid, so one far out would make all centroids of all rows possible.
// Those are left out instead (zeros, and the contraction takes them for padding), and a row asks whether the nearest of them
// can be ruled out by the triangle inequality alone.  Far: 32 times as far from the centre as all but one in 64 of (up to
// 4096 of) the centroids, rounded up to the next power of two, or not finite.  (1M x 960, k 4096 with one centroid a thousand
// times as long as the rest, or one NaN: 75 -> 13.0 ms, as without it.)
__global__ void __launch_bounds__(1024)
kmeans_round_centroids_kernel(const float* cent, uint32_t k, uint32_t dim, uint32_t dpad, const float* centre, int wide,
                              const float* cnorm_raw, const float* cnorm, uint16_t* c16, KmeansH16State* state) {
    __shared__ uint32_t hist[256], most[3], nearest_far;
    __shared__ float far_from;
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    if (tid < 256) {
        hist[tid] = 0;
    }
    if (tid < 3) {
        most[tid] = 0;
    }
    if (tid == 0) {
        nearest_far = __float_as_uint(__builtin_inff());
    }
    __syncthreads();
    const uint32_t take = k < 4096 ? k : 4096, step = k / take;
    for (uint32_t i = tid; i < take; i += 1024) {
        atomicAdd(&hist[magnitude_bits(cnorm[static_cast<uint64_t>(i) * step]) >> 23], 1U);
    }
    __syncthreads();
    if (tid < 64) {
        uint32_t incl = 0;
        for (uint32_t i = 0; i < 4; ++i) {
            incl += hist[4 * lane + i];
        }
        const uint32_t sum = incl;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t up = __shfl_up(incl, off);
            incl += lane >= static_cast<uint32_t>(off) ? up : 0;
        }
        const uint32_t want = take - take / 64;
        uint32_t before = incl - sum;
        if (before < want && want <= incl) {
            uint32_t bin = 4 * lane;  // |c'|^2 in [2^(bin - 127), 2^(bin - 126))
            while (before + hist[bin] < want) {
                before += hist[bin];
                ++bin;
            }
            far_from = bin > 215 ? 1.0e30F : ldexpf(1.0F, static_cast<int>(bin) - 126 + 10);
        }
    }
    __syncthreads();
    const float limit = far_from;
    const int e = scale_exponent(limit);
    for (uint32_t c = blockIdx.x * kGroup + (tid >> 6); c < (blockIdx.x + 1) * kGroup && c < k; c += 16) {
        const float sq = cnorm[c], raw = cnorm_raw[c];
        const bool near = sq <= limit;  // false for NaN as well
        float missed, kept;
        round_row(cent + static_cast<uint64_t>(c) * dim, near ? dim : 0, dpad, centre, wide != 0, ldexpf(1.0F, e),
                  c16 + static_cast<uint64_t>(c) * dpad, &missed, &kept);
        if (lane == 0) {
            if (near) {
                atomicMax(&most[0], magnitude_bits(sq));
                atomicMax(&most[1], magnitude_bits(raw));
                atomicMax(&most[2], magnitude_bits(ldexpf(sqrtf(missed), -e)));
            } else if (raw - raw == 0.0F) {  // (the fp32 kernels choose none whose |c|^2 is not finite)
                atomicMin(&nearest_far, magnitude_bits(fminf(sq, 3.0e38F)));
            }
        }
    }
    __syncthreads();
    if (tid == 0) {
        atomicMax(&state->centred, most[0]);
        atomicMax(&state->raw, most[1]);
        atomicMax(&state->missed, most[2]);
        atomicMin(&state->nearest_far, nearest_far);
        state->far_from = __float_as_uint(limit);  // (all workgroups the same)
    }
}

// Whether a slab goes to the fp32 kernels without the pre-selection: the probe before it left rows open in open_groups of the
// `probed` groups that were looked at (0: this slab is a probe itself, whose count is being formed).  The kernels read the
// count first and ask late, so that its way from memory is hidden (1M x 128, k 1024: 1.185 ms without, 1.23 ms with waves
// that wait for it).
__device__ inline bool
given_up(uint32_t open_groups, uint32_t probed) {
    return probed != 0 && open_groups > probed / 2;
}

// A wave per row: |x|^2 (unless it is known), the row in fp16 and its lengths.  The row is read twice, the second time
// from the caches.
__global__ void __launch_bounds__(256)
kmeans_round_rows_kernel(const float* x, uint64_t rows, uint32_t dim, uint32_t dpad, const float* centre, int wide,
                         KmeansH16State* state, uint32_t probed, uint16_t* x16, float2* xinfo, float* xscale,
                         float* xnorm) {
    const uint64_t r = static_cast<uint64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (r >= rows) {
        return;
    }
    const uint32_t open_groups = state->open_groups;
    if (probed == 0 && r == 0 && threadIdx.x == 0) {
        state->open_groups = 0;  // the rescoring of this slab counts
    }
    const uint32_t lane = threadIdx.x & 63;
    const float* row = x + r * dim;
    float sq = 0.0F, raw = 0.0F;
    for (uint32_t d = 4 * lane; d < dim; d += 256) {
        const float4 a = load4(row, d, dim, wide != 0);
        const float4 m = load4(centre, d, dim, wide != 0);
        raw = fmaf(a.x, a.x, fmaf(a.y, a.y, fmaf(a.z, a.z, fmaf(a.w, a.w, raw))));
        // entries past the dimension are zero on both sides
        const float vx = a.x - m.x, vy = a.y - m.y, vz = a.z - m.z, vw = a.w - m.w;
        sq = fmaf(vx, vx, fmaf(vy, vy, fmaf(vz, vz, fmaf(vw, vw, sq))));
    }
    sq = wave_sum(sq);
    if (xnorm != nullptr) {
        raw = wave_sum(raw);
        if (lane == 0) {
            xnorm[r] = raw;
        }
    }
    if (given_up(open_groups, probed)) {
        return;
    }
    const bool usable = sq < 1.0e30F;  // false for NaN as well
    const int e = usable ? scale_exponent(sq) : 0;
    float missed, kept;
    round_row(row, usable ? dim : 0, dpad, centre, wide != 0, ldexpf(1.0F, e), x16 + r * dpad, &missed, &kept);
    if (lane == 0) {
        const float down = ldexpf(1.0F, -e);
        xinfo[r] = make_float2(usable ? sqrtf(missed) * down : __builtin_inff(), sqrtf(kept) * down);
        xscale[r] = down;
    }
}

__device__ inline uint32_t
lds_offset(const void* p) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>(
        (__attribute__((address_space(3))) const void*)p));  // NOLINT: an address-space cast
}

// Lane l's 16 bytes (touch_line: 4, for the sake of their line) at base + bytes go to LDS at to + 16 l (4 l); `to` is the same
// in all lanes.  In assembly because the compiler would wait for all such loads before any read of LDS; who reads what they
// bring waits for vmcnt and a barrier itself.  (m0 is reserved: the compiler keeps nothing in it from one instruction to the
// next, sets it itself where it needs it, and takes it in no list of clobbers.)
__device__ inline void
load_to_lds(const void* base, uint32_t bytes, uint32_t to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(to), "v"(bytes), "s"(base) : "memory");
}

__device__ inline void
touch_line(const void* base, uint32_t bytes, uint32_t to) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" : : "s"(to), "v"(bytes), "s"(base) : "memory");
}

struct KmeansH16Args {
    const uint4* x16;  // [rows][dpad / 8]
    const uint4* c16;  // [k][dpad / 8]
    uint64_t rows;
    uint32_t k;
    uint32_t slots;    // dpad / 8
    const float* xscale;
    const float* cnorm;
    const KmeansH16State* state;
    uint32_t probed;   // see given_up
    float* group_min;
    uint64_t ld;       // the table: [group][3][ld]
    uint32_t rtiles, ctiles, mc_log2, mcols, macros;
};

// 256 centroids (the M side, so that a lane's sixteen results belong to one row) x 256 rows, eight waves of 128 x 64.  A
// stage of 64 dimensions is 64 KB; two are in LDS, the next one's loads go straight there while a stage is multiplied, and
// there is one barrier per stage, with the products of a stage's last step behind it, beside the reads of the next stage's
// first operands.  The lines of the stage after that are touched, so that they are in the XCD's L2 when they are asked for.
// Launch of 69 888 x 960 rows, k 4096, us: loads through registers, each stage's first reads exposed 628; as above without
// the touch 536; with it 510.  (Two workgroups of four waves, 256 x 128 and stages of 32 dimensions three deep to a compute
// unit, so that one looks through its products beside the other's contraction: 557; it moves half as much again.)
//
// LDS: 16-byte slots [row][8], slot s of row r at position s ^ ((r >> 1) & 7): the 16 consecutive rows that a
// ds_read_b128 serves at a time fall on the sixteen 16-byte columns of the 64 banks, and a global line of a row stays one
// 128-byte run on the way in.
//
// Grid: as kmeans_assign_tile_kernel, id % 8 is the XCD, and the 32 workgroups that run on an XCD at the same time form a
// macro tile whose rows and centroids they share through that XCD's L2.
__global__ void __launch_bounds__(kThreads, 2)
kmeans_h16_kernel(KmeansH16Args p) {
    extern __shared__ uint4 lds[];  // [2][A: kTile x kSlots, B: kTile x kSlots], then |c'|^2 of the tile
    const uint32_t xcd = blockIdx.x & 7;
    const uint32_t local = blockIdx.x >> 3;
    const uint32_t macro = (local >> 5) * 8 + xcd;
    if (macro >= p.macros) {
        return;
    }
    const uint32_t within = local & 31;
    const uint32_t rt = (macro / p.mcols) * (32U >> p.mc_log2) + (within >> p.mc_log2);
    const uint32_t ct = ((macro % p.mcols) << p.mc_log2) + (within & ((1U << p.mc_log2) - 1));
    if (rt >= p.rtiles || ct >= p.ctiles) {
        return;
    }
    constexpr uint32_t kSide = kTile * kSlots;
    float* cn = reinterpret_cast<float*>(lds + 4 * kSide);
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = tid >> 6;
    const uint32_t wm = wave & 1;   // which 128 centroids
    const uint32_t wn = wave >> 1;  // which 64 rows
    const uint32_t half = lane >> 5;
    const uint32_t l32 = lane & 31;
    const uint64_t row0 = static_cast<uint64_t>(rt) * kTile;
    const uint32_t c0 = ct * kTile;
    const uint32_t stages = p.slots / kSlots;

    // Loader: from memory into LDS without a stop in registers, 16 bytes a lane, eight rows a wave at a time; wave w brings
    // rows 8 w + 64 i of both sides.  LDS takes the lanes' pieces in order, so the lane chooses the slot that belongs where
    // it lands; rows past the end repeat the last one.
    const uint32_t lr = tid >> 3, ls = (tid & 7) ^ ((lr >> 1) & 7);
    const uint4* side_a = p.c16 + static_cast<uint64_t>(c0) * p.slots;
    const uint4* side_b = p.x16 + row0 * p.slots;
    const uint32_t a_last = p.k - 1 - c0;
    const uint32_t b_last = static_cast<uint32_t>(p.rows - 1 - row0 < kTile ? p.rows - 1 - row0 : kTile);
    auto offset = [&](uint32_t r, uint32_t last) __attribute__((always_inline)) {
        return ((r < last ? r : last) * p.slots + ls) * 16;
    };
    const uint32_t oa0 = offset(lr, a_last), oa1 = offset(lr + 64, a_last), oa2 = offset(lr + 128, a_last),
                   oa3 = offset(lr + 192, a_last);
    const uint32_t ob0 = offset(lr, b_last), ob1 = offset(lr + 64, b_last), ob2 = offset(lr + 128, b_last),
                   ob3 = offset(lr + 192, b_last);
    const uint32_t lds_wave = __builtin_amdgcn_readfirstlane(lds_offset(lds) + wave * 8 * kSlots * 16);
    const uint32_t open_groups = p.state->open_groups;
    if (tid < kTile) {
        const float sq = c0 + tid < p.k ? p.cnorm[c0 + tid] : 3.0e38F;
        cn[tid] = sq <= __uint_as_float(p.state->far_from) ? sq : 3.0e38F;
    }

    auto fetch = [&](uint32_t st) __attribute__((always_inline)) {
        const uint4* a = side_a + st * kSlots;
        const uint4* b = side_b + st * kSlots;
        const uint32_t to = lds_wave + (st & 1) * 2 * kSide * 16;
        constexpr uint32_t kStep = 64 * kSlots * 16;
        load_to_lds(a, oa0, to);
        load_to_lds(a, oa1, to + kStep);
        load_to_lds(a, oa2, to + 2 * kStep);
        load_to_lds(a, oa3, to + 3 * kStep);
        load_to_lds(b, ob0, to + 4 * kStep);
        load_to_lds(b, ob1, to + 5 * kStep);
        load_to_lds(b, ob2, to + 6 * kStep);
        load_to_lds(b, ob3, to + 7 * kStep);
    };
    // One line of the stage after that per thread, into the XCD's L2: a word of it goes to a corner of LDS that nobody reads.
    const uint32_t side = wave >> 2;  // the first four waves: centroids
    const uint32_t tr = tid & (kTile - 1);
    const uint32_t touch_off = (tr < (side == 0 ? a_last : b_last) ? tr : (side == 0 ? a_last : b_last)) * p.slots * 16;
    const uint32_t touch_to = __builtin_amdgcn_readfirstlane(lds_offset(cn + kTile) + wave * 256);
    const uint32_t side_u = __builtin_amdgcn_readfirstlane(side);
    auto touch = [&](uint32_t st) __attribute__((always_inline)) {
        touch_line((side_u == 0 ? side_a : side_b) + st * kSlots, touch_off, touch_to);
    };
    // What this wave asked for but for its last load (the line) has landed, and its reads of LDS are done; then the others'.
    auto landed = [&](auto touched) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(touched ? 0x0071 : 0x0070);  // vmcnt 1 or 0, lgkmcnt 0
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const uint32_t swap = (l32 >> 1) & 7;
    const uint32_t a_row = (wm * 128 + l32) * kSlots;
    const uint32_t b_row = kSide + (wn * 64 + l32) * kSlots;

    floatx16 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                acc[i][j][e] = 0.0F;
            }
        }
    }
    // One step of sixteen dimensions; its six operands are in registers a step ahead.
    halfx8 fa[2][4], fb[2][2];
    auto operands = [&](const uint4* buf, uint32_t step, int u) __attribute__((always_inline)) {
        const uint32_t at = (2 * step + half) ^ swap;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            fa[u][i] = __builtin_bit_cast(halfx8, buf[a_row + 32 * i * kSlots + at]);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            fb[u][j] = __builtin_bit_cast(halfx8, buf[b_row + 32 * j * kSlots + at]);
        }
    };
    auto multiply = [&](int u) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[u][i], fb[u][j], acc[i][j], 0, 0, 0);
            }
        }
    };

    if (given_up(open_groups, p.probed)) {
        return;
    }
    using Yes = std::true_type;
    using No = std::false_type;
    fetch(0);
    if (stages > 1) {
        touch(1);
        landed(Yes{});
    } else {
        landed(No{});  // (a wave must not end with a write to LDS on its way)
    }
    operands(lds, 0, 0);
    // (The barriers to the scheduler keep every step's reads a step ahead of its products, where it would read them late to
    // save registers.)
    auto stage = [&](uint32_t st, auto fetches, auto touches) __attribute__((always_inline)) {
        const uint4* cur = lds + (st & 1) * 2 * kSide;
        if constexpr (fetches) {
            fetch(st + 1);  // the last readers of its buffer passed the barrier that ended stage st - 1
        }
        if constexpr (touches) {
            touch(st + 2);
        }
        operands(cur, 1, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0);
        __builtin_amdgcn_sched_barrier(0);
        operands(cur, 2, 0);
        __builtin_amdgcn_sched_barrier(0);
        multiply(1);
        __builtin_amdgcn_sched_barrier(0);
        operands(cur, 3, 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(0);
        __builtin_amdgcn_sched_barrier(0);
        // The last step is multiplied behind the barrier, beside the reads of the next stage's first operands.
        if constexpr (fetches) {
            landed(touches);
            operands(lds + ((st + 1) & 1) * 2 * kSide, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        multiply(1);
        __builtin_amdgcn_sched_barrier(0);
    };
    uint32_t st = 0;
    for (; st + 2 < stages; ++st) {
        stage(st, Yes{}, Yes{});
    }
    if (st + 1 < stages) {
        stage(st, Yes{}, No{});
        ++st;
    }
    stage(st, No{}, No{});

    // acc[i][j][e] = <C, X> (scaled) of centroid c0 + wm 128 + 32 i + 8 (e / 4) + 4 half + e % 4 and row wn 64 + 32 j + l32:
    // the 64 of a lane are one group of the table, 16 i + e the place in it.
    const float cdown = ldexpf(-2.0F, -scale_exponent(__uint_as_float(p.state->far_from)));
    const uint32_t group = (ct * 2 + wm) * 2 + half;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint64_t row = row0 + wn * 64 + 32 * j + l32;
        const float factor = (row < p.rows ? p.xscale[row] : 0.0F) * cdown;
        float least = __builtin_inff(), second = __builtin_inff(), third = __builtin_inff();
#pragma unroll
        for (int i = 0; i < 4; ++i) {
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const float4 n4 = *reinterpret_cast<const float4*>(cn + wm * 128 + 32 * i + 8 * e4 + 4 * half);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float base = e == 0 ? n4.x : e == 1 ? n4.y : e == 2 ? n4.z : n4.w;
                    const float d = fmaf(factor, acc[i][j][4 * e4 + e], base);
                    const float v = __uint_as_float((__float_as_uint(d) & ~63U) | (16U * i + 4U * e4 + e));
                    third = __builtin_amdgcn_fmed3f(second, third, v);
                    second = __builtin_amdgcn_fmed3f(least, second, v);
                    // (fminf would make v canonical first, one instruction in six here)
                    asm("v_min_f32 %0, %1, %2" : "=v"(least) : "v"(least), "v"(v));
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // keeps the reads of cn from piling up in registers
        }
        if (row < p.rows) {
            float* entry = p.group_min + static_cast<uint64_t>(group) * 3 * p.ld + row;
            entry[0] = least;
            entry[p.ld] = second;
            entry[2 * p.ld] = third;
        }
    }
}

struct KmeansRescoreArgs {
    const float* x;  // the slab's rows
    uint64_t rows;
    uint32_t dim;
    const float* cent;
    uint32_t k;
    uint32_t groups;
    const float* group_min;
    uint64_t ld;
    const float2* xinfo;
    const float* xnorm;
    const float* cnorm_raw;
    KmeansH16State* state;
    uint32_t probed;  // see given_up
    int wide;
    int natural;  // order of the products, see the kernel
    unsigned long long* best;
    uint8_t* row_open;
    uint32_t* open64;
};

// 64 rows per workgroup.  First four threads a row look through the table (coalesced along the rows); then a lane per
// (row, centroid) that is still possible forms the distance exactly as the fp32 kernels do, one fma after the other in the
// order of their matrix instructions (natural: k = 0, 1, 2, ...; else, for dimensions that are a multiple of 4, k = 0, 4,
// 1, 5, 2, 6, 3, 7 of every eight), so labels and distances are those of the fp32 kernels bit for bit.  128 pairs at a
// time; their rows come through LDS in pieces of 32 dimensions (whole 128-byte lines in, a pitch of 36 floats so that
// the lanes' reads fall on all banks), the next piece in flight while one is summed.
__global__ void __launch_bounds__(256)
kmeans_h16_rescore_kernel(KmeansRescoreArgs p) {
    __shared__ __align__(16) float seg_x[kPairs][kPitch], seg_c[kPairs][kPitch];
    __shared__ uint32_t least_bits[kRowsPerBlock], count[kRowsPerBlock], cost[kRowsPerBlock], offset[kRowsPerBlock + 1];
    __shared__ uint32_t list[kRowsPerBlock][kMaxList];
    __shared__ uint32_t pair_row[kPairs], pair_c[kPairs];
    __shared__ unsigned long long best[kRowsPerBlock];
    __shared__ uint32_t any;
    const uint32_t tid = threadIdx.x;
    const uint32_t rl = tid & 63, part = tid >> 6;
    const uint64_t block_row = static_cast<uint64_t>(blockIdx.x) * kRowsPerBlock;
    const uint64_t row = block_row + rl;
    const uint32_t open_groups = p.state->open_groups;
    if (tid < kRowsPerBlock) {
        count[tid] = 0;
        cost[tid] = 0;
        least_bits[tid] = 0xFFFFFFFFU;
        best[tid] = ~0ull;
    }
    if (tid == 0) {
        any = 0;
    }
    __syncthreads();
    float least = __builtin_inff();
    if (row < p.rows) {
#pragma unroll 8
        for (uint32_t g = part; g < p.groups; g += kParts) {
            least = fminf(least, p.group_min[static_cast<uint64_t>(g) * 3 * p.ld + row]);
        }
        atomicMin(&least_bits[rl], float_to_ordered(least));
    }
    if (given_up(open_groups, p.probed)) {  // (the table is not this slab's: nothing of it was used)
        if (tid < kRowsPerBlock && row < p.rows) {
            p.row_open[row] = 1;
            p.best[row] = ~0ull;
        }
        if (tid == 0) {
            p.open64[blockIdx.x] = 1;
            p.state->any_open = 1;
        }
        return;
    }
    __syncthreads();
    if (row < p.rows) {
        least = ordered_to_float(least_bits[rl]);
        constexpr float kU = 5.9604645e-8F;  // 2^-24
        const float2 info = p.xinfo[row];
        // Squares and products that underflow lose bits that no relative term covers: kTinyLength^2 is what 8192 squares can
        // lose, kTinyRest the same for the remainders (in scales of 2^14 and more), kTinySquare what the products can.  Rows and
        // centroids that small have every centroid possible and go to the fp32 kernels.
        constexpr float kTinyLength = 2.0e-17F, kTinyRest = 1.0e-20F, kTinySquare = 1.0e-33F;
        const float cmax = sqrtf(__uint_as_float(p.state->centred)) * 1.00001F + kTinyLength;
        const float craw = sqrtf(__uint_as_float(p.state->raw)) * 1.00001F + kTinyLength;
        const float cmiss = __uint_as_float(p.state->missed) * 1.00001F + kTinyRest;
        const float missed = info.x * 1.00001F + kTinyRest, kept = info.y * 1.00001F + kTinyRest;
        const float xraw = sqrtf(p.xnorm[row]) * 1.00001F + kTinyLength;
        const float steps = static_cast<float>(p.dim);
        // 2 |<x', c'> - <X, C>|
        float err = 2.0F * (missed * cmax + kept * cmiss);
        // four roundings of the absolute sum per matrix instruction of sixteen dimensions; |c'|^2 summed by a wave, the
        // fma that adds it, and six mantissa bits of the stored value
        const float big = cmax * cmax + 2.0F * (kept + missed) * (cmax + cmiss);
        err += 2.0F * 4.0F * (steps / 16.0F + 5.0F) * kU * kept * (cmax + cmiss);
        err += (steps / 64.0F + 12.0F) * 2.0F * kU * cmax * cmax + 66.0F * 2.0F * kU * big;
        // the distances formed below: |c|^2 by a wave, <x, c> by a chain of dim roundings, the sum of the two
        err += (steps / 64.0F + 12.0F) * 2.0F * kU * craw * craw;
        err += 2.0F * (steps + 4.0F) * kU * xraw * craw + kTinySquare;
        const float limit = least + 2.0F * err;
        // A far centroid at r from the centre: |c'|^2 - 2 <x', c'> >= r^2 - 2 r |x'|, which as well as its fp32 distance
        // (roundings: 1e-3 |x| |c| and 2e-5 |c|^2 at most, up to 8192 dimensions; |c| <= r + |x| + |x'|) grows with r from
        // four times |x| + |x'| on, so that the nearest one speaks for all.
        const float far = sqrtf(__uint_as_float(p.state->nearest_far)) * 0.9999F;
        const float len = kept + missed, both = len + xraw;
        const bool far_out = p.state->nearest_far == __float_as_uint(__builtin_inff()) ||
                             (far >= 4.0F * both &&
                              0.99F * far * far - 2.0F * far * len - 2.0e-3F * xraw * (far + both) > limit);
        if (!(err < 1.0e30F) || !(fabsf(limit) < 1.0e30F) || !far_out) {
            cost[rl] = kMaxWork + 1;  // (its threads write the same)
        } else {
#pragma unroll 4
            for (uint32_t g = part; g < p.groups; g += kParts) {
                const float* entry = p.group_min + static_cast<uint64_t>(g) * 3 * p.ld + row;
                const float v1 = entry[0];
                if (v1 <= limit) {
                    const float v2 = entry[p.ld], v3 = entry[2 * p.ld];
                    const uint32_t more = v3 <= limit ? 0 : v2 <= limit ? 2 : 1;  // 0: the whole group
                    const uint32_t at = atomicAdd(&count[rl], more == 2 ? 2U : 1U);
                    atomicAdd(&cost[rl], more == 0 ? kGroup : more);
                    if (at < kMaxList) {
                        list[rl][at] = (g << 7) | (more == 0 ? 64U : (__float_as_uint(v1) & 63U));
                    }
                    if (more == 2 && at + 1 < kMaxList) {
                        list[rl][at + 1] = (g << 7) | (__float_as_uint(v2) & 63U);
                    }
                }
            }
        }
    }
    __syncthreads();
    if (part == 0) {
        const bool real = row < p.rows;
        const bool open = real && (count[rl] == 0 || count[rl] > kMaxList || cost[rl] > kMaxWork);
        if (real) {
            p.row_open[row] = open ? 1 : 0;
        }
        if (open) {
            any = 1;
        }
        // where the pairs of each row begin
        const uint32_t mine = real && !open ? cost[rl] : 0;
        uint32_t sum = mine;
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t up = __shfl_up(sum, off);
            sum += rl >= static_cast<uint32_t>(off) ? up : 0;
        }
        offset[rl] = sum - mine;
        if (rl == 63) {
            offset[64] = sum;
        }
    }
    __syncthreads();
    if (tid == 0) {
        p.open64[blockIdx.x] = any;
        if (any != 0) {
            p.state->any_open = 1;
            if (p.probed == 0 && blockIdx.x % kProbeStep == 0) {
                atomicAdd(&p.state->open_groups, 1U);
            }
        }
    }

    const uint32_t total = offset[kRowsPerBlock];
    const uint32_t pieces = (p.dim + kPiece - 1) / kPiece;
    const uint32_t quad = 4 * (tid & 7);
    for (uint32_t base = 0; base < total; base += kPairs) {
        if (tid < kPairs) {
            uint32_t r = 0, c = 0xFFFFFFFFU;
            const uint32_t t = base + tid;
            if (t < total) {
                for (uint32_t step = 32; step > 0; step >>= 1) {
                    r += offset[r + step] <= t ? step : 0;  // the last row whose pairs begin at or before t
                }
                uint32_t at = t - offset[r], i = 0;
                while ((list[r][i] & 64U) != 0 ? at >= kGroup : at >= 1) {
                    at -= (list[r][i] & 64U) != 0 ? kGroup : 1;
                    ++i;
                }
                // group g = (tile, half of the tile, lane half); place 16 i + j of it is centroid
                // 32 i + 8 (j / 4) + 4 half + j % 4
                const uint32_t e = list[r][i], g = e >> 7, j = (e & 64U) != 0 ? at : e & 63U;
                c = (g >> 1) * 128 + 4 * (g & 1) + 32 * (j >> 4) + 8 * ((j >> 2) & 3) + (j & 3);
                c = c < p.k ? c : p.k - 1;  // past the end: once more the last centroid, a true distance all the same
            }
            pair_row[tid] = r;
            pair_c[tid] = c;
        }
        __syncthreads();
        // Two pieces are on their way while one is summed (with one, 69 888 x 960 rows took 200 us, a wait of 2 us per piece;
        // 168 now).
        const float *xrow[4], *crow[4];
        bool used[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t pr = (tid >> 3) + 32 * i;
            const uint32_t c = pair_c[pr];
            used[i] = c != 0xFFFFFFFFU;
            xrow[i] = p.x + (block_row + pair_row[pr]) * p.dim;
            crow[i] = p.cent + static_cast<uint64_t>(used[i] ? c : 0) * p.dim;
        }
        float4_v gx[2][4], gc[2][4];
        auto fetch = [&](uint32_t d, int b) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                gx[b][i] = gc[b][i] = float4_v{0.0F, 0.0F, 0.0F, 0.0F};
                if (used[i] && d < p.dim) {
                    const float4 vx = load4(xrow[i], d, p.dim, p.wide != 0), vc = load4(crow[i], d, p.dim, p.wide != 0);
                    gx[b][i] = float4_v{vx.x, vx.y, vx.z, vx.w};
                    gc[b][i] = float4_v{vc.x, vc.y, vc.z, vc.w};
                }
            }
        };
        float acc = 0.0F;
        auto sum = [&](uint32_t piece, int b) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t pr = (tid >> 3) + 32 * i;
                *reinterpret_cast<float4_v*>(&seg_x[pr][quad]) = gx[b][i];
                *reinterpret_cast<float4_v*>(&seg_c[pr][quad]) = gc[b][i];
            }
            __syncthreads();
            fetch((piece + 2) * kPiece + quad, b);  // (nothing past the dimension)
            if (tid < kPairs) {
#pragma unroll
                for (uint32_t d = 0; d < kPiece; d += 8) {
                    const float4 xa = *reinterpret_cast<const float4*>(&seg_x[tid][d]);
                    const float4 xb = *reinterpret_cast<const float4*>(&seg_x[tid][d + 4]);
                    const float4 ca = *reinterpret_cast<const float4*>(&seg_c[tid][d]);
                    const float4 cb = *reinterpret_cast<const float4*>(&seg_c[tid][d + 4]);
                    if (p.natural != 0) {
                        acc = fmaf(xa.w, ca.w, fmaf(xa.z, ca.z, fmaf(xa.y, ca.y, fmaf(xa.x, ca.x, acc))));
                        acc = fmaf(xb.w, cb.w, fmaf(xb.z, cb.z, fmaf(xb.y, cb.y, fmaf(xb.x, cb.x, acc))));
                    } else {
                        acc = fmaf(xb.y, cb.y, fmaf(xa.y, ca.y, fmaf(xb.x, cb.x, fmaf(xa.x, ca.x, acc))));
                        acc = fmaf(xb.w, cb.w, fmaf(xa.w, ca.w, fmaf(xb.z, cb.z, fmaf(xa.z, ca.z, acc))));
                    }
                }
            }
            __syncthreads();
        };
        fetch(quad, 0);
        fetch(kPiece + quad, 1);
        for (uint32_t piece = 0; piece < pieces; piece += 2) {
            sum(piece, 0);
            if (piece + 1 < pieces) {
                sum(piece + 1, 1);
            }
        }
        if (base + tid < total && tid < kPairs) {
            const uint32_t c = pair_c[tid];
            const float dist = p.cnorm_raw[c] + (-2.0F * acc);
            if (dist < __builtin_inff()) {  // (a whole group may hold a centroid that is not finite: nobody chooses it)
                atomicMin(&best[pair_row[tid]], static_cast<unsigned long long>(make_key(dist, c)));
            }
        }
        __syncthreads();  // pair_row / pair_c are written again
    }
    if (tid < kRowsPerBlock && row < p.rows) {
        p.best[row] = best[tid];
    }
}

int
launch_kmeans_h16(const float* x, uint64_t n, uint32_t dim, const float* cent, uint32_t k, const float* cnorm_raw,
                  float* xnorm, int iteration, unsigned long long* best, const KmeansH16Buffers& b, hipStream_t st) {
    constexpr size_t lds_bytes = 4 * static_cast<size_t>(kTile) * kSlots * sizeof(uint4) + kTile * sizeof(float) +
                                 kThreads * sizeof(uint32_t);
    static std::once_flag lds_once;
    static hipError_t lds_rc = hipSuccess;
    std::call_once(lds_once, []() {
        lds_rc = hipFuncSetAttribute(reinterpret_cast<const void*>(kmeans_h16_kernel),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds_bytes));
    });
    VA_HIP(lds_rc);
    const uint32_t dpad = padded_dim(dim);
    const uint64_t slab = slab_rows(n, dim, k);
    const int wide = (dim & 3) == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(cent)) & 15) == 0;
    const bool have_xnorm = iteration > 0;
    const bool kept = have_xnorm && n <= slab;  // the rows' fp16 form of the call before, and the centre it was formed with
    const uint32_t cblocks = (k + kGroup - 1) / kGroup;
    const uint32_t probe_groups = static_cast<uint32_t>(div_up(std::min(n, slab), kRowsPerBlock * kProbeStep));
    if (!kept) {
        hipLaunchKernelGGL(kmeans_centre_kernel, dim3((dim + 63) / 64), dim3(1024), 0, st, cent, k, dim, b.centre, b.state);
    } else {
        hipLaunchKernelGGL(kmeans_reset_kernel, dim3(1), dim3(64), 0, st, b.state, iteration % kProbes == 0 ? 1 : 0);
    }
    hipLaunchKernelGGL(kmeans_cnorm_kernel, dim3(cblocks), dim3(1024), 0, st, cent, k, dim, b.centre, b.cnorm);
    hipLaunchKernelGGL(kmeans_round_centroids_kernel, dim3(cblocks), dim3(1024), 0, st, cent, k, dim, dpad, b.centre, wide,
                       cnorm_raw, b.cnorm, b.c16, b.state);
    for (uint64_t r0 = 0; r0 < n; r0 += slab) {
        const uint64_t rows = n - r0 < slab ? n - r0 : slab;
        const bool probe = (kept ? static_cast<uint64_t>(iteration) : r0 / slab) % kProbes == 0;
        const uint32_t probed = probe ? 0 : probe_groups;
        if (!kept) {
            hipLaunchKernelGGL(kmeans_round_rows_kernel, dim3(static_cast<uint32_t>(div_up(rows, 4))), dim3(256), 0, st,
                               x + r0 * dim, rows, dim, dpad, b.centre, wide, b.state, probed, b.x16, b.xinfo, b.xscale,
                               have_xnorm ? nullptr : xnorm + r0);
        }
        KmeansH16Args a;
        a.x16 = reinterpret_cast<const uint4*>(b.x16);
        a.c16 = reinterpret_cast<const uint4*>(b.c16);
        a.rows = rows;
        a.k = k;
        a.slots = dpad / 8;
        a.xscale = b.xscale;
        a.cnorm = b.cnorm;
        a.state = b.state;
        a.probed = probed;
        a.group_min = b.group_min;
        a.ld = slab;
        a.rtiles = static_cast<uint32_t>(div_up(rows, kTile));
        a.ctiles = static_cast<uint32_t>(tile_count(k));
        a.mc_log2 = a.ctiles >= 8 ? 3 : a.ctiles >= 4 ? 2 : a.ctiles >= 2 ? 1 : 0;
        a.mcols = (a.ctiles + (1U << a.mc_log2) - 1) >> a.mc_log2;
        const uint32_t mrows = (a.rtiles + (32U >> a.mc_log2) - 1) / (32U >> a.mc_log2);
        a.macros = mrows * a.mcols;
        hipLaunchKernelGGL(kmeans_h16_kernel, dim3((a.macros + 7) / 8 * 32 * 8), dim3(kThreads), lds_bytes, st, a);

        KmeansRescoreArgs s;
        s.x = x + r0 * dim;
        s.rows = rows;
        s.dim = dim;
        s.cent = cent;
        s.k = k;
        s.groups = a.ctiles * (kTile / kGroup);
        s.group_min = b.group_min;
        s.ld = slab;
        s.xinfo = b.xinfo;
        s.xnorm = xnorm + r0;
        s.cnorm_raw = cnorm_raw;
        s.state = b.state;
        s.probed = probed;
        s.wide = wide;
        s.natural = (dim & 3) != 0;
        s.best = best + r0;
        s.row_open = b.row_open + r0;
        s.open64 = b.open64 + r0 / kRowsPerBlock;
        const dim3 grid(static_cast<uint32_t>(div_up(rows, kRowsPerBlock)));
        hipLaunchKernelGGL(kmeans_h16_rescore_kernel, grid, dim3(256), 0, st, s);
    }
    VA_HIP(hipGetLastError());
    return 0;
}

}  // namespace vsag_amd
