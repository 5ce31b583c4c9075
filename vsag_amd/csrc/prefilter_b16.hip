// Pre-selection for query batches on the bf16 matrix cores: flat fp32, sq8, sq4, sq8_uniform and sq4_uniform stores, fp32
// posting lists.
//
// The inner product <b, c> of a query with a code is formed from two bf16 values per operand, x = h + l + r with h =
// bf16(x), l = bf16(x - h), |l| <= 2^-8 |x| and |r| <= 2^-17 |x| (bf16 keeps eight bits, rounded to nearest: half a unit in
// the last place is 2^-8 of the power of two below x, and of l at most 2^-9 of 2^-8).  A code byte or nibble is one bf16
// value exactly, so
//   sq8, sq4   <b, c>  ~  <h_b, c> + <l_b, c>                        (b: the query with the scale folded in)
//   fp32       <a, y>  ~  <h_a, h_y> + <l_a, h_y> + <h_a, l_y>
//   uniform    <b, c>  =  the integer product of two rows of bytes: one part each
// one to three v_mfma_f32_32x32x16_bf16 for sixteen dimensions.  The products are exact in the fp32 accumulator; what is
// left out is known (the remainders of the query are summed, those of an fp32 code are at most 2^-17 of it), so the value
//   v = |y|^2 - 2 <b, c>  (inner product: -<b, c>; uniform kinds: -lb sum(c) - rate <b, c>)
// stands within a bound e of the streaming kernel's distance less the query's constant.  bf16 has the exponent range of
// fp32: no operand needs a scale, and what is below the normal range may be taken as zero.
//
// A flat scan (launch_scan_b16) needs no exact distance before the end:
//   1. a sample of the storage tiles, spread over the store, leaves the least v of every 64 codes; k of those lie at or
//      below the k-th smallest, m;
//   2. whoever is among the k best has v <= m + 2 e: the pass over all codes records (v, slot) of those, a few hundred a
//      query (b16_sample_count says how many are expected);
//   3. of the records only those within 2 e of their own k-th smallest are rescored with the streaming kernel's arithmetic
//      (rescore_kernel): k and a handful, and the result is the streaming result, bit for bit.
// Rows stored in the order of their clusters, or a mask over one run of them, make a poor sample, and more records than there
// is room for: those that found room are a second sample, its k-th smallest a second threshold, and the queries concerned
// pass over the codes once more.  One that overflows again is gated and streams.  A deny mask takes part in 1 and 2 as a |y|^2
// beyond every threshold.  100k x 128 fp32, 1000 queries, k 10 (fp32 matrix cores, an exact prefix and levels before: 460 us): 150 us.
// 100k x 768 fp32, 32 queries (streamed before: 684 us on the device): 141 us.  500k x 100 sq8 under a deny mask, 200
// queries, k 100 (streamed before: 664 us): 157 us.  100k x 128 fp32, 1000 queries, rows in the order of their clusters: 469 us.
//
// What bounds it: with 128 queries per workgroup the matrix cores beside the splitting of the codes and the verdicts (100k x
// 128 fp32, 1000 queries: matrix pipe busy 34 % of the pass, vector instructions issued 38 %, a third of the waves' time spent
// waiting; no bank conflicts to speak of); with few queries the bytes of the codes, each read once per 32, 64 or 128 queries
// (100k x 768 fp32, 32 queries: 6.0 TB/s, matrix pipe 10 %).
//
// Work split: a workgroup of four waves takes 256 codes, a storage tile a wave, and 128, 64 or 32 queries (JB blocks of
// 32), so a code is read by one wave alone and goes from memory into the registers of the lanes that multiply it (lane %
// 32 = code, lane / 32 = which eight of sixteen dimensions): a load instruction covers two runs of 512 bytes.  It is split
// there, a stage of 32 dimensions (sq8, sq4: 64) at a time, while the loads of the next stage are under way.  The queries
// are split once per call into a table of 16-byte slots [eight dimensions][part][row]; a workgroup stages them in LDS
// twice 16 KB at a time (sq8, sq4 with 128 queries: 32), one barrier each.
#include "distance.h"
#include "kth_value.h"
#include "prepare_rows.h"
#include "store.h"
#include "topk.h"

namespace vsag_amd {

void timing_begin(hipStream_t st);
void timing_end(hipStream_t st);

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr uint32_t kB16N = 128;     // most queries per workgroup tile; the rows of the query table are padded to it
constexpr uint32_t kB16Pad = 64;    // the query table covers whole stages of either length
// |y|^2 of a slot that cannot be found: a quiet NaN, which no product carries below a threshold, no minimum takes and four
// other low bits leave a quiet NaN.  (A number above every threshold comes down with a large enough product, and the slots
// past a list's end, which multiply the codes of another, lie outside the store.)
constexpr float kB16Absent = __builtin_nanf("");
constexpr uint32_t kB16CountStride = 32;  // words between the queries' record counters: atomics on one memory line take turns
// Thresholds end at kB16Closed: a code of |y|^2 from 3e38 on (l2) is further than that, with products of 1e37 at most.  Beyond
// it, and where nothing bounds a query, a threshold is kB16Open, and every code that can be found is a candidate.
constexpr float kB16Closed = 2.8e38F;
constexpr float kB16Open = 3.0e38F;
constexpr uint32_t kB16Held = 4096;       // values of the sample that b16_tau_kernel keeps in LDS
constexpr uint32_t kB16Streams = 0x40000000;  // the record counter of a query that streams whatever it finds
// What the two parts of a value can miss of it, and its low part: 2^-17 and 2^-8, and a little for their own rounding.
constexpr double kB16Left = 7.7e-6;
constexpr double kB16Low = 3.92e-3;
constexpr uint32_t kB16Queue = 128; // records a wave gathers in LDS before it asks for room in the queries' lists

constexpr uint32_t kIvfB16ChunkTiles = 32;  // as ivf_i8.hip: kIvfI8ChunkTiles, kIvfI8Chunks
constexpr uint32_t kIvfB16Chunks = 4;

template <int KIND>
struct B16Layout {
    static constexpr bool kSplit = KIND == VSAG_AMD_KIND_FP32;           // the code has a low part too
    static constexpr uint32_t kSlots = kSplit ? 4 : 8;                   // eight dimensions each, per stage
    static constexpr uint32_t kGranules = KIND == VSAG_AMD_KIND_FP32 ? 8 : KIND == VSAG_AMD_KIND_SQ8 ? 4 : 2;  // per stage
};

static bool
b16_uniform(const vsag_amd_store* s) {
    return s->kind == VSAG_AMD_KIND_SQ8_UNIFORM || s->kind == VSAG_AMD_KIND_SQ4_UNIFORM;
}

// Posting lists of sq8 / sq4 / uniform codes and rabitq stores have passes of their own.
bool
prefilter_b16_supports(const vsag_amd_store* s) {
    const bool kind = s->kind == VSAG_AMD_KIND_FP32 || s->kind == VSAG_AMD_KIND_SQ8 || s->kind == VSAG_AMD_KIND_SQ4 ||
                      (b16_uniform(s) && s->nlist == 0 && s->dpad <= kUniformTermDims);
    return kind && s->pf_term != nullptr && s->pf_ymax != nullptr;
}

// Whether a batch takes this route of its own accord, measured on Gaussian mixtures against what served it before (us per
// call, other -> this).
//   Streaming passes serve four or eight queries at a time: fp32 100k x 768, k 10 4 queries 131 -> 140 (cosine; not taken), 5:
//   153 -> 139, 8: 281 -> 141, 32: 686 -> 141; k 100 6: 161 -> 234 (not taken), 8: 294 -> 212; sq8 500k x 100 cosine, k 10
//   2: 62 -> 69 (not taken), 4: 93 -> 68; sq4 100k x 960 cosine, k 100 8: 133 -> 143 (not taken), 64: 543 -> 159; sq8 600k x
//   960 l2, k 100 6: 930 -> 274; 1M x 128 16: 259 -> 87; sq8_uniform (cheap to stream) 200k x 768, k 10 4: 97 -> 102 (not
//   taken), 6: 108 -> 102, 64: 337 -> 116; k 100 8: 121 -> 138 (not taken), 10: 164 -> 139.
//   sq8 / sq4 up to 128 dimensions have the int8 matrix cores, twice as fast a product behind a prefix and four levels: 1M x
//   128, k 10 512 queries 415 -> 362 (not taken from 508 on), 1000 532 -> 653 (not taken); k 100 600 710 -> 568, 1000 802 ->
//   828 (not taken); k 1 600 370 -> 407 (not taken); 300k 1000 318 -> 269 (not taken), 2000 402 -> 456 (not taken); 100k, k 10
//   512 231 -> 112, 2000 300 -> 238 (not taken), 4000 354 -> 410 (not taken), k 100 4000 704 -> 490.
//   Beyond, the fp16 ones, one product where this takes two: sq4 200k x 512 cosine, k 10 1000 508 -> 456, 2000 792 -> 856
//   (not taken); sq8 600k x 960 ip 256 798 -> 629, 1000 1825 -> 2265 (not taken); 200k x 768, k 100 1000 1504 -> 879.
//   The uniform kinds take one product here as well: 1M x 128, k 10 1000 queries 517 -> 507 (not taken from 914 on), 100k x
//   128, 2000 279 -> 172; beyond 128 dimensions they have nothing else (200k x 768, 2000 queries 4221 -> 854; 600k x 960
//   sq4_uniform, 1000 5790 -> 1312).
//   A deny mask leaves the streaming kernel alone as the other side.
// Rows in the order of their clusters take the second pass (us, streaming -> this): fp32 100k x 768 5 queries 178 -> 195, 8: 269
// -> 261, 32: 683 -> 259; 100k x 128 5: 85 -> 90, 1000 (by levels before) 2676 -> 469; sq8 500k x 100, k 100 9: 186 -> 128.
// Thousands of equal distances stream behind the pass: 100k x 128 of 40 distinct rows 8 queries 123 -> 192, 64 578 -> 409.
// Smaller stores than 81920 codes would gain as well (sq8 70000 x 200, 512 queries 263 -> 121; 70000 x 32, 8 60 -> 47), but
// the records of a query take 16 KB, several times the streaming kernel's workspace there: batches of those keep it.
bool
prefilter_b16_pays(const vsag_amd_store* s, uint64_t nq, uint32_t k, bool masked) {
    const bool fp32 = s->kind == VSAG_AMD_KIND_FP32;
    const uint32_t least = fp32             ? (k <= 20 ? 5 : 8)
                           : b16_uniform(s) ? (k <= 20 ? 5 : 9)
                                            : (k <= 20 ? 4 : s->metric == VSAG_AMD_METRIC_L2 ? 6 : 9);
    if (s->ntiles < 1280 || nq < least) {
        return false;
    }
    if (fp32 || masked || nq <= 64) {
        return true;
    }
    if (b16_uniform(s) && s->dpad > 128) {
        return true;
    }
    const double n = static_cast<double>(s->n), work = static_cast<double>(nq) * n * s->dim;
    if (s->dim > 128) {
        return work <= 1.4e11 + 2.0e9 * k;
    }
    return work <= (b16_uniform(s) ? 1.8 : 1.0) * (2.0e10 + 5.0e8 * k + 4.0e10 * log10(n * 1.0e-5));
}

static uint64_t
b16_query_rows(uint64_t nq) {
    return round_up(nq + 1, static_cast<uint64_t>(kB16N));  // (the row of a pair that does not exist is a row of zeros)
}
static uint32_t
b16_slots(const vsag_amd_store* s) {
    return static_cast<uint32_t>(round_up(s->dpad, kB16Pad) / 8);
}
static size_t
b16_plane_bytes(const vsag_amd_store* s, uint64_t nq) {
    return static_cast<size_t>(b16_slots(s)) * 2 * b16_query_rows(nq) * 16;
}

// Eight floats as their two bf16 parts.
__device__ inline void
b16_split8(const float (&x)[8], uint4* hi, uint4* lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bf16x2 hh = __builtin_convertvector((floatx2{x[2 * i], x[2 * i + 1]}), bf16x2);
        h[i] = __builtin_bit_cast(uint32_t, hh);
        const float r0 = x[2 * i] - __uint_as_float(h[i] << 16);
        const float r1 = x[2 * i + 1] - __uint_as_float(h[i] & 0xFFFF0000U);
        l[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{r0, r1}), bf16x2));
    }
    *hi = make_uint4(h[0], h[1], h[2], h[3]);
    *lo = make_uint4(l[0], l[1], l[2], l[3]);
}

// The two low bytes (bits 0..7, 8..15 of w) as bf16: a float of at most eight significant bits is its own upper half.
__device__ inline uint32_t
b16_two_bytes(uint32_t w, int at) {
    const uint32_t a = __float_as_uint(static_cast<float>((w >> (8 * at)) & 0xffU));
    const uint32_t b = __float_as_uint(static_cast<float>((w >> (8 * at + 8)) & 0xffU));
    return __builtin_amdgcn_perm(b, a, 0x07060302U);
}
// An sq4 word (byte b: dimension 2 b in the low, 2 b + 1 in the high nibble) as the slot of its eight dimensions.
__device__ inline uint4
b16_nibbles(uint32_t w) {
    const uint32_t lo = w & 0x0F0F0F0FU, hi = (w >> 4) & 0x0F0F0F0FU;
    uint32_t out[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const uint32_t x = __float_as_uint(static_cast<float>((lo >> (8 * b)) & 0xffU));
        const uint32_t y = __float_as_uint(static_cast<float>((hi >> (8 * b)) & 0xffU));
        out[b] = __builtin_amdgcn_perm(y, x, 0x07060302U);
    }
    return make_uint4(out[0], out[1], out[2], out[3]);
}

// What a query's v can be off by: distance = v + constant, |v + constant - streaming distance| <= fixed + stream(D), with
// stream(D) = root sqrt(D) + slope D the part that grows with the distance.
struct B16Error {
    float constant, fixed, root, slope;
};

struct B16QueryArgs {
    FloatQueryArgs raw;  // raw.q: the queries that `qtab` is made of first, nq_pad rows of it (null: it holds them)
    uint64_t nq_pad;
    const float* qtab;   // processed queries, zero beyond the dimension
    uint32_t qstride;
    uint32_t kdim;
    const float* scale;  // sq8 / sq4 under l2: per dimension; null: ones
    uint64_t nq, rows;
    uint32_t slots;
    uint4* planes;
    const uint32_t* ymax_bits;  // largest |y| of the store (l2: scaled codes; ip: raw codes; fp32: the vectors; uniform kinds:
                                // largest term)
    float cmax;          // largest code value: 255, 15; fp32: 0
    int is_l2;
    // uniform kinds: qtab holds the query's bytes (nibbles: per eight dimensions a word of the even ones, one of the odd)
    int uniform, nibbles;
    float lb, rate;
    const float* qmeta;  // sq8 / sq4, ip: sum q_d lb_d per query
    uint32_t qmeta_stride;
    B16Error* error;     // per query
    // posting lists: thresholds from the queries' bounds
    const uint32_t* bound;
    float* tau;
    // flat scans: what a search starts from, bound0 (and no seeds, unless seed is null), and no query to pass over again
    uint32_t* start;
    uint32_t bound0;
    uint32_t* seed;
    uint32_t* again;
    float* magnitude;    // residual lists: the query's magnitudes (see IvfF32Args in prefilter.hip), or null
    // queries that stream: their flags, then how many; their pairs' first private list of k records is marked as overflowed
    uint32_t* gate;
    uint32_t* partial_cnt;
    uint32_t p0, nprobe;
    uint32_t k;
};

// One workgroup per row of the query table (rows at or beyond nq: zeros).  A flat scan of the float kinds has its queries
// prepared here as well: a launch that returns at once still takes 4.5 us.
__global__ void __launch_bounds__(256)
b16_query_kernel(B16QueryArgs p) {
    __shared__ double part[4][5];
    const uint64_t q = blockIdx.x;
    const uint32_t tid = threadIdx.x;
    if (p.raw.q != nullptr && q < p.nq_pad) {
        prepare_float_row(p.raw, q);
        __syncthreads();
    }
    const bool real = q < p.nq;
    const float* row = p.qtab + q * p.qstride;
    double a2 = 0.0, a1 = 0.0;               // of the processed query
    double r1 = 0.0, r2 = 0.0, l2 = 0.0;     // the remainders and the low parts of b
    for (uint32_t s = tid; s < p.slots; s += blockDim.x) {
        float x[8];
        double exact[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t d = 8 * s + i;
            const bool in = real && d < p.kdim;
            double a = 0.0;
            if (in && p.uniform != 0) {
                const uint32_t* words = reinterpret_cast<const uint32_t*>(row);
                a = p.nibbles != 0 ? (words[2 * (d >> 3) + (d & 1)] >> (8 * ((d >> 1) & 3))) & 255U
                                   : (words[d >> 2] >> (8 * (d & 3))) & 255U;
            } else if (in) {
                a = static_cast<double>(row[d]);
            }
            exact[i] = a * (in && p.scale != nullptr ? static_cast<double>(p.scale[d]) : 1.0);
            x[i] = static_cast<float>(exact[i]);
            a2 += a * a;
            a1 += fabs(a);
        }
        uint4 hi, lo;
        b16_split8(x, &hi, &lo);
        p.planes[(static_cast<uint64_t>(s) * 2) * p.rows + q] = hi;
        p.planes[(static_cast<uint64_t>(s) * 2 + 1) * p.rows + q] = lo;
        const uint32_t hw[4] = {hi.x, hi.y, hi.z, hi.w}, lw[4] = {lo.x, lo.y, lo.z, lo.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float h = __uint_as_float((i & 1) != 0 ? hw[i >> 1] & 0xFFFF0000U : hw[i >> 1] << 16);
            const float l = __uint_as_float((i & 1) != 0 ? lw[i >> 1] & 0xFFFF0000U : lw[i >> 1] << 16);
            const double left = exact[i] - static_cast<double>(h) - static_cast<double>(l);
            r1 += fabs(left);
            r2 += left * left;
            l2 += static_cast<double>(l) * static_cast<double>(l);
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        a2 += __shfl_xor(a2, off);
        a1 += __shfl_xor(a1, off);
        r1 += __shfl_xor(r1, off);
        r2 += __shfl_xor(r2, off);
        l2 += __shfl_xor(l2, off);
    }
    if ((tid & 63) == 0) {
        double* const mine = part[tid >> 6];
        mine[0] = a2;
        mine[1] = a1;
        mine[2] = r1;
        mine[3] = r2;
        mine[4] = l2;
    }
    __syncthreads();
    if (real && p.seed != nullptr) {
        for (uint32_t i = tid; i < p.k; i += blockDim.x) {
            p.seed[q * p.k + i] = 0xFFFFFFFFU;
        }
    }
    if (tid != 0 || !real) {
        return;
    }
    auto total = [&](int i) { return (part[0][i] + part[1][i]) + (part[2][i] + part[3][i]); };
    a2 = total(0);
    a1 = total(1);
    r1 = total(2);
    r2 = total(3);
    l2 = total(4);
    if (p.start != nullptr) {
        p.start[q] = p.bound0;
        p.again[q] = 0;
    }
    constexpr double kU = 5.9604644775390625e-8;  // 2^-24, the unit roundoff of fp32
    const double kd = static_cast<double>(p.kdim);
    if (p.uniform != 0) {
        // No remainders.  l2: v + norm_q is the distance over the rate, whose sign and range keep the order; both forms round
        // a few times at these magnitudes, and the low four bits of v are cut off.
        const double qm = static_cast<double>(p.qmeta[q * p.qmeta_stride]);
        const double term = static_cast<double>(__uint_as_float(*p.ymax_bits)) * (1.0 + 1.0e-6);
        double sums = static_cast<double>(p.cmax) * a1;  // most <b, c>
        if (p.is_l2) {
            sums = fmin(sums, sqrt(a2 * term));  // (|c|^2 is the term)
        }
        const double rate = static_cast<double>(p.rate), lb = static_cast<double>(p.lb);
        const double factor = p.is_l2 ? 2.0 : fabs(rate);
        // (an integer below 2^24 is exact in the accumulator)
        const double rounding = sums < 16777216.0 ? 0.0 : 4.0 * kU * (kd / 16.0 + 4.0) * sums;
        const double magnitude = term + factor * sums + (p.is_l2 ? fabs(qm) : fabs(lb * qm) + lb * lb + 1.0);
        const double fixed = factor * rounding + 48.0 * kU * magnitude;
        const bool ordered = p.is_l2 ? rate > 1.0e-30 && rate < 1.0e28 : true;
        B16Error e;
        e.constant = static_cast<float>(p.is_l2 ? qm : 1.0 - lb * qm - lb * lb);
        e.fixed = ordered && magnitude < 1.0e37 ? static_cast<float>(fixed) * 1.000001F + 1.0e-37F : 1.0e38F;
        e.root = e.slope = 0.0F;
        p.error[q] = e;
        return;
    }
    const double ymax = static_cast<double>(__uint_as_float(*p.ymax_bits)) * (1.0 + 1.0e-6);
    const double an = sqrt(a2);
    const double dots = an * ymax;  // sum |b_d c_d| of any code, by Cauchy and Schwarz
    const bool fp32 = p.cmax == 0.0F;
    const double sums = fp32 || p.is_l2 ? dots : fmin(static_cast<double>(p.cmax) * a1, dots);
    const double factor = p.is_l2 ? 2.0 : 1.0;
    // Left out: the remainders of the query against a code (codes of bytes lie in [0, cmax]); of an fp32 code at most
    // kB16Left of it against the query, and its low part (kB16Low of it) against the query's.
    const double split = fp32 ? ymax * (sqrt(r2) + kB16Left * an + kB16Low * sqrt(l2)) : static_cast<double>(p.cmax) * r1;
    // The accumulation, two or three instructions per sixteen dimensions.  One was measured to lose at most 2 units of 2^-24 of
    // its accumulator and 8 of its largest product (it cuts off what it aligns: one product of 1 and fifteen just below 2^-24
    // lose 7.9; random and crafted inputs): 2 n + 8 of the absolute sum over n instructions.  Twice that.
    const double rounding = 4.0 * kU * ((fp32 ? 3.0 : 2.0) * kd / 16.0 + 4.0) * sums;
    // Operands below the normal range taken as zero; fma(factor, acc, term) and |y|^2 rounded, the low four bits cut off.
    const double flushed = kd * 4.7e-38 * (an + ymax + 1.0);
    const double test = 36.0 * kU * ((p.is_l2 ? ymax * ymax : 0.0) + factor * dots);
    // (Where a product can leave fp32, or with entries that are not finite, the query streams.)
    double fixed = factor * dots < 1.0e37 ? factor * (split + rounding) + flushed + test : 1.0e39;
    double root = 0.0, slope = 0.0;
    double constant = a2;
    if (p.is_l2) {
        // The streaming kernel's fp32 sum of squares: every term (fl(c s) - a)^2 is off by two or three roundings of itself
        // and, for codes of bytes, by the rounding of c s; then kdim roundings of the sum.
        slope = (kd + 4.0) * kU;
        root = fp32 ? 0.0 : 2.0 * kU * ymax;
    } else {
        // 1 - (fl(sum) + qmeta): kdim roundings of sum |terms|, then the closing operations.
        const double qm = p.qmeta != nullptr ? static_cast<double>(p.qmeta[q * p.qmeta_stride]) : 0.0;
        fixed += (kd + 2.0) * kU * sums + 4.0 * kU * (sums + fabs(qm) + 1.0);
        constant = 1.0 - qm;
    }
    B16Error e;
    e.constant = static_cast<float>(constant);
    e.fixed = static_cast<float>(fixed) * 1.000001F + 1.0e-37F;
    e.root = static_cast<float>(root) * 1.000001F;
    e.slope = static_cast<float>(slope) * 1.000001F;
    if (p.error != nullptr) {
        p.error[q] = e;
    }
    if (p.tau == nullptr) {
        return;
    }
    if (!(fixed < 1.0e37)) {
        // Nothing passes, and the query streams.  (A product beyond fp32 would be an infinity with other low bits: a NaN, and
        // the code lost.)
        p.tau[q] = kB16Absent;
        p.gate[q] = 1;
        atomicAdd(&p.gate[p.nq], 1U);
        for (uint32_t c = p.p0; c < p.nprobe; ++c) {
            p.partial_cnt[(q * p.nprobe + c) * 2 * kIvfB16Chunks] = p.k + 1;
        }
        return;
    }
    const uint32_t b = p.bound[q];
    const double bd = static_cast<double>(ordered_to_float(b));
    const double t = bd - constant + fixed + 1.01 * (root * sqrt(fabs(bd)) + slope * fabs(bd)) +
                     1.0e-6 * (fabs(bd) + fabs(constant));
    const float tf = static_cast<float>(t);
    const float up = tf + fabsf(tf) * 1.2e-7F + 1.0e-37F;
    // no bound yet: everything is a candidate (and the query overflows, or its lists are short)
    const bool open = b == 0xFFFFFFFFU || !(up < kB16Closed);
    p.tau[q] = open ? kB16Open : up;
    if (p.magnitude != nullptr) {
        const double magnitude = fabs(bd) + fabs(constant) + (p.is_l2 ? ymax * ymax : 0.0) + factor * dots;
        p.magnitude[q] = open ? 0.0F : static_cast<float>(magnitude) * 1.000001F;
    }
}

struct B16TauArgs {
    const float* least;     // nq x groups: the least v of every group of sampled codes
    uint32_t groups, k;
    const B16Error* error;
    float* tau;
    float* slack;           // twice what v can be off by, at the distances that matter
    uint32_t* cand_cnt;     // zeroed
    uint32_t* gate;         // zeroed
};

struct B16Threshold {
    float tau, slack;  // not below the k best values; twice what a value can be off by there
};

// The k codes at or below kth have distances of at most D; so has whoever is among the k best.
__device__ inline B16Threshold
b16_threshold(const B16Error& e, float kth) {
    const float far = fmaxf(kth + e.constant, 0.0F) * 1.00001F + 2.0F * e.fixed;
    const float slack = 2.0F * e.fixed + 2.05F * (e.root * sqrtf(far) + e.slope * far);
    const float tau = kth + slack;
    return {tau + fabsf(tau) * 2.4e-7F + 1.0e-37F, slack};
}

// One wave per query.
__global__ void __launch_bounds__(64)
b16_tau_kernel(B16TauArgs p) {
    __shared__ uint32_t hist[256];
    __shared__ float held[kB16Held];
    const uint64_t q = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    const float* least = p.least + q * p.groups;
    // (Asked for three times: from LDS as far as they fit, eight loads of a lane under way.  2608 values, k 100: 19.8 -> 12.7 us.)
    const uint32_t nheld = p.groups < kB16Held ? p.groups : kB16Held;
    for (uint32_t i0 = 0; i0 < nheld; i0 += 8 * kWave) {
        float v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            const uint32_t i = i0 + u * kWave + lane;
            v[u] = least[i < nheld ? i : nheld - 1];
        }
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            const uint32_t i = i0 + u * kWave + lane;
            if (i < nheld) {
                held[i] = v[u];
            }
        }
    }
    wave_lds_fence();
    const float kth =
        kth_value_or_above([&](uint32_t i) { return i < kB16Held ? held[i] : least[i]; }, p.groups, p.k, hist, lane);
    if (lane != 0) {
        return;
    }
    const B16Error e = p.error[q];
    const B16Threshold t = b16_threshold(e, kth);
    // fewer than k codes sampled: everything is a candidate
    const bool open = !(kth < 3.0e38F);
    // A query whose sums can leave fp32, with entries that are not finite, or so far out that the threshold is, streams: more
    // records than there is room for, and nothing passes (8 queries of 1e30 against 100k x 128 fp32, every code a record of
    // each: 1367 us a call, now 234).
    const bool streams = !(e.fixed < 1.0e37F) || (!open && !(t.tau < kB16Closed));
    p.cand_cnt[q * kB16CountStride] = streams ? kB16Streams : 0U;
    p.gate[q] = 0;
    p.tau[q] = streams ? kB16Absent : open ? kB16Open : t.tau;
    p.slack[q] = streams || open ? 3.0e38F : t.slack;
}

struct B16AgainArgs {
    const uint64_t* cand;
    uint32_t cap, k;
    const B16Error* error;
    float* tau;
    float* slack;
    uint32_t* cand_cnt;
    uint32_t* again;   // per query tile of `columns`: whether one of its queries passes over the codes once more
    uint32_t columns;
};

// One wave per query, behind the pass: a threshold from the records that found room, where some did not.
__global__ void __launch_bounds__(64)
b16_again_kernel(B16AgainArgs p) {
    __shared__ uint32_t hist[256];
    const uint64_t q = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    const uint32_t count = as_const(p.cand_cnt)[q * kB16CountStride];
    B16Threshold t{kB16Absent, 0.0F};  // nothing passes
    if (count > p.cap && count < kB16Streams) {
        const uint64_t* cand = p.cand + q * p.cap;
        auto value = [&](uint32_t i) { return ordered_to_float(static_cast<uint32_t>(cand[i] >> 32)); };
        // (Once more among what is left: the bins of the first span other clusters, in which the query's own is a bin or two.)
        float kth = kth_value_or_above(value, p.cap, p.k, hist, lane);
        const float first = kth;
        wave_lds_fence();
        kth = kth_value_or_above([&](uint32_t i) { const float v = value(i); return v <= first ? v : __builtin_inff(); }, p.cap, p.k,
                                 hist, lane);
        t = b16_threshold(p.error[q], kth);
        // As many of all as of those here will pass.  (Thousands of equal distances: nothing helps.)
        uint32_t pass = 0;
        for (uint32_t i = lane; i < p.cap; i += kWave) {
            pass += ordered_to_float(static_cast<uint32_t>(cand[i] >> 32)) <= t.tau ? 1U : 0U;
        }
        for (int off = 32; off > 0; off >>= 1) {
            pass += __shfl_xor(pass, off);
        }
        const bool fits = static_cast<uint64_t>(pass) * count <= static_cast<uint64_t>(p.cap) * p.cap;
        t.tau = t.tau < kB16Closed && fits ? t.tau : kB16Absent;
    }
    if (lane == 0) {
        p.tau[q] = t.tau;
        if (t.tau < kB16Closed) {
            p.slack[q] = t.slack;
            p.cand_cnt[q * kB16CountStride] = 0;
            p.again[q / p.columns] = 1;
        }
    }
}

struct PrefilterB16Args {
    const uint4* tiles;
    uint32_t G;
    const uint4* planes;
    uint64_t nq, rows;
    uint32_t slots;
    const float* term;  // per slot |y|^2 (uniform kinds: launch_code_terms)
    int terms;          // whether v has it: l2, uniform kinds
    float factor;       // of <b, c> in v
    const float* tau;
    // flat stores
    uint64_t ntiles, n;
    float* least;       // a sampling pass: nq x groups values, and no records; else null
    uint32_t groups;    // the storage tiles of the sample: tile (i spread) >> 32 for i = 0 .. groups - 1
    uint64_t spread;
    const uint32_t* again;  // a second pass: the query tiles it is for; else null
    uint64_t* cand;     // nq x cap records: v as its ordered bits above the slot
    uint32_t* cand_cnt;
    uint32_t cap;
    const uint32_t* deny;
    // posting lists (as IvfF32Args in prefilter.hip)
    const float* res_bias;
    const float* res_term;
    const float* magnitude;
    const uint32_t* ymax_bits;
    float res_cmax;
    const uint32_t* ids;
    const uint32_t* list_tile;
    const uint32_t* pair_off;
    const uint32_t* item_off;
    const uint32_t* sorted_pair;
    uint32_t nlist, nprobe;
    uint32_t k;
    uint64_t* partial;
    uint32_t* partial_cnt;
    uint32_t* gate;
};

// The codes of one stage of a wave, in registers: of both blocks of 32 codes, the granules this lane multiplies.
template <int KIND>
struct B16Codes {
    static constexpr int kLoads = B16Layout<KIND>::kGranules / 2;  // per block
    uint4 g[2][kLoads];
};

// Granules past a code's end repeat its last one (the query's values there are zeros): no load stands behind a branch.
template <int KIND>
__device__ __forceinline__ void
b16_fetch_codes(B16Codes<KIND>& c, const uint4* tile, uint32_t G, uint32_t st, uint32_t half, uint32_t l32) {
    using L = B16Layout<KIND>;
#pragma unroll
    for (int u = 0; u < B16Codes<KIND>::kLoads; ++u) {
        // fp32: the two granules of the eight dimensions that this half multiplies in step u / 2; sq8, sq4: one granule
        // holds this half's dimensions of two (four) steps
        uint32_t j = L::kGranules * st + (KIND == VSAG_AMD_KIND_FP32 ? 4 * (u / 2) + 2 * half + (u & 1) : 2 * u + half);
        j = j < G ? j : G - 1;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            c.g[i][u] = tile[j * kWave + 32 * i + l32];
        }
    }
}

// The operand of step ks: eight dimensions of the code of this lane.
template <int KIND>
__device__ __forceinline__ void
b16_operand(const B16Codes<KIND>& c, int i, int ks, bf16x8* hi, bf16x8* lo) {
    if constexpr (KIND == VSAG_AMD_KIND_FP32) {
        const uint4 v = c.g[i][2 * ks], w = c.g[i][2 * ks + 1];
        const float x[8] = {__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w),
                            __uint_as_float(w.x), __uint_as_float(w.y), __uint_as_float(w.z), __uint_as_float(w.w)};
        uint4 h, l;
        b16_split8(x, &h, &l);
        *hi = __builtin_bit_cast(bf16x8, h);
        *lo = __builtin_bit_cast(bf16x8, l);
    } else if constexpr (KIND == VSAG_AMD_KIND_SQ8) {
        const uint4 v = c.g[i][ks / 2];
        const uint32_t a = (ks & 1) != 0 ? v.z : v.x, b = (ks & 1) != 0 ? v.w : v.y;
        *hi = __builtin_bit_cast(bf16x8, make_uint4(b16_two_bytes(a, 0), b16_two_bytes(a, 2), b16_two_bytes(b, 0),
                                                    b16_two_bytes(b, 2)));
    } else {
        const uint4 v = c.g[i][0];
        *hi = __builtin_bit_cast(bf16x8, b16_nibbles(ks == 0 ? v.x : ks == 1 ? v.y : ks == 2 ? v.z : v.w));
    }
}

// The slot (eight dimensions) of the query table that lines up with a half's operand of step ks of stage st.
template <int KIND>
__device__ __forceinline__ uint32_t
b16_slot(uint32_t ks, uint32_t half) {
    if constexpr (KIND == VSAG_AMD_KIND_FP32) {
        return 2 * ks + half;
    } else if constexpr (KIND == VSAG_AMD_KIND_SQ8) {
        return 4 * (ks >> 1) + 2 * half + (ks & 1);
    } else {
        return 4 * half + ks;
    }
}

// ONE: the query has no low part (uniform kinds; KIND says how the codes lie).
template <int KIND, bool LISTS, int JB, bool ONE = false>
__global__ void __launch_bounds__(256, JB == 4 || (JB == 2 && KIND == VSAG_AMD_KIND_FP32) ? 2 : 3)
prefilter_b16_kernel(PrefilterB16Args p) {
    using L = B16Layout<KIND>;
    constexpr uint32_t N = JB * 32;
    constexpr uint32_t kSteps = L::kSlots / 2;
    constexpr uint32_t kRound = JB * L::kSlots >= 16 ? 1 : 16 / (JB * L::kSlots);  // stages of codes per stage of queries
    constexpr uint32_t kSlotsB = kRound * L::kSlots;       // slots of a stage of queries
    constexpr uint32_t kQueryRegs = kSlotsB * 2 * N / 256;
    constexpr uint32_t kRowStep = 256 / N;                 // (slot, part) pairs that one round of the workgroup covers
    __shared__ uint4 sb[2][kSlotsB][2][N];
    __shared__ float code_term[4][kWave];
    __shared__ uint64_t queue_key[4][kB16Queue];
    __shared__ uint32_t queue_col[4][kB16Queue];
    __shared__ uint32_t col_count[LISTS ? 1 : 4][LISTS ? 1 : N];
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = tid & 63;
    const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t half = lane >> 5;
    const uint32_t l32 = lane & 31;
    const uint32_t stages = (p.G + L::kGranules - 1) / L::kGranules;

    // What this workgroup walks: code tiles first, first + step, ... below mtiles (of four storage tiles from tile_begin
    // on, one a wave), against the query rows of its N columns.
    uint64_t tile_begin = 0, tile_end, first = 0, step = 1;
    uint64_t q0 = 0;
    uint32_t pbeg = 0, pend = 0, chunk = 0;
    if constexpr (LISTS) {
        const uint32_t item = blockIdx.x;
        const cu32_p ioff = as_const(p.item_off);
        if (item >= ioff[p.nlist]) {
            return;  // the whole workgroup
        }
        uint32_t lo_b = 0, hi_b = p.nlist;
        while (hi_b - lo_b > 1) {
            const uint32_t mid = (lo_b + hi_b) >> 1;
            if (ioff[mid] <= item) {
                lo_b = mid;
            } else {
                hi_b = mid;
            }
        }
        const uint32_t list_begin = as_const(p.list_tile)[2 * lo_b], list_end = as_const(p.list_tile)[2 * lo_b + 1];
        uint32_t chunks = (list_end - list_begin + kIvfB16ChunkTiles - 1) / kIvfB16ChunkTiles;
        chunks = chunks < kIvfB16Chunks ? chunks : kIvfB16Chunks;
        if (chunks == 0) {
            return;
        }
        const uint32_t per = (list_end - list_begin + chunks - 1) / chunks;
        chunk = (item - ioff[lo_b]) % chunks;
        const uint32_t group = (item - ioff[lo_b]) / chunks;
        uint32_t tb = list_begin + chunk * per;
        tb = tb < list_end ? tb : list_end;
        tile_begin = tb;
        tile_end = tb + per < list_end ? tb + per : list_end;
        pbeg = as_const(p.pair_off)[lo_b] + group * N;
        pend = as_const(p.pair_off)[lo_b + 1];
        if (tile_begin >= tile_end || pbeg >= pend) {
            return;
        }
    } else {
        tile_end = p.ntiles;
        first = blockIdx.x;
        step = gridDim.x;
        q0 = static_cast<uint64_t>(blockIdx.y) * N;
        if (p.again != nullptr && as_const(p.again)[blockIdx.y] == 0) {
            return;  // the whole workgroup
        }
    }
    const bool sampling = !LISTS && p.least != nullptr;
    const uint64_t mtiles = sampling ? p.groups / 4 : (tile_end - tile_begin + 3) / 4;
    if (first >= mtiles) {
        return;  // the whole workgroup
    }

    // Verdict side: the columns l32 of the JB blocks.
    float tau_n[JB];
#pragma unroll
    for (int j = 0; j < JB; ++j) {
        const uint32_t col = j * 32 + l32;
        if constexpr (LISTS) {
            const uint32_t at = pbeg + col;
            const uint32_t pair = at < pend ? as_const(p.sorted_pair)[at] : 0U;
            const uint32_t query = pair / p.nprobe;
            tau_n[j] = at < pend ? p.tau[query] : __builtin_nanf("");
            if (p.res_term != nullptr && at < pend) {
                const float rt = p.res_term[pair];
                // |bias| = |2 <c, y> + |c|^2| (l2; inner product has none); five more roundings stand between this test
                // and the streaming result: 2e-6 of the magnitudes is several times their sum
                const float bias_max =
                    p.res_bias != nullptr ? (2.0F * __uint_as_float(*p.ymax_bits) + p.res_cmax) * p.res_cmax : 0.0F;
                tau_n[j] = tau_n[j] + rt + 2.0e-6F * (p.magnitude[query] + fabsf(rt) + bias_max);
            }
        } else {
            tau_n[j] = q0 + col < p.nq && p.least == nullptr ? p.tau[q0 + col] : __builtin_nanf("");  // no verdict passes
        }
    }

    // Query loader: (slot, part) pairs x N rows per stage of queries, consecutive threads on consecutive rows.
    const uint32_t qr = tid % N;
    uint64_t qsrc;
    if constexpr (LISTS) {
        const uint32_t at = pbeg + qr;
        qsrc = at < pend ? as_const(p.sorted_pair)[at] / p.nprobe : p.nq;  // p.nq: a row of zeros
    } else {
        qsrc = q0 + qr;  // below p.rows: the table covers whole tiles of rows
    }
    // (Separate variables, not an array: that ended up in scratch memory.)
    uint4 rq0, rq1, rq2, rq3, rq4, rq5, rq6, rq7;
    static_assert(kQueryRegs == 4 || kQueryRegs == 8, "what the loaders below move");
    auto fetch_queries = [&](uint32_t st) __attribute__((always_inline)) {
        auto slot = [&](uint32_t r) __attribute__((always_inline)) {
            uint32_t sp = st * 2 * L::kSlots + tid / N + kRowStep * r;
            sp = sp < 2 * p.slots ? sp : 2 * p.slots - 1;  // (of no stage that is multiplied)
            return p.planes[static_cast<uint64_t>(sp) * p.rows + qsrc];
        };
        rq0 = slot(0);
        rq1 = slot(1);
        rq2 = slot(2);
        rq3 = slot(3);
        if constexpr (kQueryRegs == 8) {
            rq4 = slot(4);
            rq5 = slot(5);
            rq6 = slot(6);
            rq7 = slot(7);
        }
    };
    auto park_queries = [&](uint32_t buf) __attribute__((always_inline)) {
        auto put = [&](uint32_t r, uint4 v) __attribute__((always_inline)) {
            const uint32_t sp = tid / N + kRowStep * r;
            sb[buf][sp >> 1][sp & 1][qr] = v;
        };
        put(0, rq0);
        put(1, rq1);
        put(2, rq2);
        put(3, rq3);
        if constexpr (kQueryRegs == 8) {
            put(4, rq4);
            put(5, rq5);
            put(6, rq6);
            put(7, rq7);
        }
    };

    // Once a query's list is full, record number pos takes a place with probability cap / (pos + 1): what is there in the end
    // is a sample of all its records, whatever order the codes are in (b16_again_kernel).  (Scrambled twice: places spread as
    // evenly as one product spreads them leave nothing of the first records.)
    auto place = [&](uint64_t q, uint32_t pos, uint64_t key) __attribute__((always_inline)) {
        uint32_t at = pos;
        if (pos >= p.cap) {
            uint32_t h = pos * 0x9E3779B1U;
            h = (h ^ (h >> 15)) * 0x85EBCA77U;
            at = __umulhi(h ^ (h >> 13), pos + 1);
        }
        if (at < p.cap) {
            p.cand[q * p.cap + at] = key;
        }
    };
    auto record = [&](uint32_t col, uint64_t key) __attribute__((always_inline)) {
        if constexpr (LISTS) {
            // private list of the pair: chunk, which half of the 256 codes (the upper word)
            const uint32_t pair = as_const(p.sorted_pair)[pbeg + col];
            const uint64_t list = (static_cast<uint64_t>(pair) * kIvfB16Chunks + chunk) * 2 + static_cast<uint32_t>(key >> 32);
            const uint32_t pos = atomicAdd(&p.partial_cnt[list], 1U);
            if (pos < p.k) {
                p.partial[list * p.k + pos] = static_cast<uint32_t>(key);
            } else if (pos == p.k) {
                if (atomicExch(&p.gate[pair / p.nprobe], 1U) == 0U) {
                    atomicAdd(&p.gate[p.nq], 1U);
                }
            }
        } else {
            const uint64_t q = q0 + col;
            place(q, atomicAdd(&p.cand_cnt[q * kB16CountStride], 1U), key);
        }
    };
    // Records wait in the wave's queue (a query's counter is an atomic a microsecond away: asked for one record at a time it
    // cost half of the pass), until it might overflow or the walk is over.  Flat: the queue asks once for all records of a
    // column, a lane per column (a few queries that admit thousands of codes each otherwise wait for their own counters: 5
    // against 100k x 128 fp32 in the order of its clusters: 147 -> 91 us).
    uint64_t* const keys = queue_key[wave];
    uint32_t* const cols = queue_col[wave];
    uint32_t waiting = 0;
    auto flush = [&]() __attribute__((always_inline)) {
        wave_lds_fence();
        if constexpr (LISTS) {
            for (uint32_t i = lane; i < waiting; i += kWave) {
                record(cols[i], keys[i]);
            }
        } else {
            uint32_t* const counts = col_count[wave];
            for (uint32_t c = lane; c < N; c += kWave) {
                counts[c] = 0;
            }
            wave_lds_fence();
            uint32_t rank[kB16Queue / kWave];
#pragma unroll
            for (uint32_t r = 0; r < kB16Queue / kWave; ++r) {
                const uint32_t i = r * kWave + lane;
                rank[r] = i < waiting ? atomicAdd(&counts[cols[i]], 1U) : 0U;
            }
            wave_lds_fence();
            for (uint32_t c = lane; c < N; c += kWave) {
                if (counts[c] != 0) {
                    counts[c] = atomicAdd(&p.cand_cnt[(q0 + c) * kB16CountStride], counts[c]);
                }
            }
            wave_lds_fence();
#pragma unroll
            for (uint32_t r = 0; r < kB16Queue / kWave; ++r) {
                const uint32_t i = r * kWave + lane;
                if (i < waiting) {
                    place(q0 + cols[i], counts[cols[i]] + rank[r], keys[i]);
                }
            }
        }
        waiting = 0;
        wave_lds_fence();
    };

    auto tile_at = [&](uint64_t mt) __attribute__((always_inline)) {
        const uint64_t i = tile_begin + 4 * mt + wave;
        return sampling ? (i * p.spread) >> 32 : i;
    };
    auto tile_of = [&](uint64_t mt) __attribute__((always_inline)) {
        const uint64_t tile = tile_at(mt);
        return p.tiles + (tile < tile_end ? tile : tile_begin) * p.G * kWave;  // (slots past the end count as absent)
    };
    B16Codes<KIND> codes;
    const uint4* tile = tile_of(first);
    b16_fetch_codes<KIND>(codes, tile, p.G, 0, half, l32);
    fetch_queries(0);
    park_queries(0);
    __syncthreads();
    uint32_t buf = 0;  // where the queries of the current stage are
    for (uint64_t mt = first; mt < mtiles; mt += step) {
        floatx16 acc[2][JB];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int j = 0; j < JB; ++j) {
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    acc[i][j][e] = 0.0F;
                }
            }
        }
        const uint64_t slot0 = tile_at(mt) * kWave;
        const bool more_tiles = mt + step < mtiles;
        float my_term;
        {
            const uint64_t slot = slot0 + lane;
            bool real = tile_at(mt) < tile_end;
            if constexpr (LISTS) {
                // (a padding slot is all zeros: under inner product, and with a residual bias, that is a good distance)
                real = real && p.ids[slot] != VSAG_AMD_INVALID_ID;
            } else {
                real = real && slot < p.n && !denied(p.deny, slot);
            }
            my_term = real ? p.term[slot] : kB16Absent;
            const bool found = my_term < 3.0e38F;
            my_term = !found ? kB16Absent : p.terms == 0 ? 0.0F : my_term;
            if (real && !found && p.least == nullptr) {
                // A code whose squared norm leaves fp32 may have any inner product: a record of every query.  Under l2 it
                // stands behind every threshold but an open one.  Its value is no number, so it is always rescored.
                const uint32_t cols_here =
                    LISTS ? (pend - pbeg < N ? pend - pbeg : N) : static_cast<uint32_t>(p.nq - q0 < N ? p.nq - q0 : N);
                for (uint32_t col = 0; col < cols_here; ++col) {
                    const float limit = p.tau[LISTS ? as_const(p.sorted_pair)[pbeg + col] / p.nprobe : q0 + col];
                    if (!(limit >= (p.terms != 0 ? kB16Open : -kB16Open))) {  // (no number: a query that streams)
                        continue;
                    }
                    record(col, LISTS ? (static_cast<uint64_t>(wave >> 1) << 32) | static_cast<uint32_t>(slot)
                                      : (0xFFFFFFFFULL << 32) | static_cast<uint32_t>(slot));
                }
            }
            if (LISTS && real && p.res_bias != nullptr) {
                my_term -= p.res_bias[slot];
            }
        }
        for (uint32_t st = 0; st < stages; ++st) {
            // The operands of this stage, then the loads of the next one (of the next tile behind the last).
            bf16x8 ah[2][kSteps], al[2][L::kSplit ? kSteps : 1];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (uint32_t ks = 0; ks < kSteps; ++ks) {
                    b16_operand<KIND>(codes, i, static_cast<int>(ks), &ah[i][ks], &al[i][L::kSplit ? ks : 0]);
                }
            }
            const bool last = st + 1 == stages;
            if (last) {
                tile = more_tiles ? tile_of(mt + step) : tile;
            }
            b16_fetch_codes<KIND>(codes, tile, p.G, last ? 0 : st + 1, half, l32);
            // The queries of the next round of stages: fetched as this round begins, parked as it ends.
            const uint32_t within = st % kRound;
            if (within == 0) {
                const uint32_t next = st + kRound;
                fetch_queries(next < stages ? next : 0);
            }
#pragma unroll
            for (uint32_t ks = 0; ks < kSteps; ++ks) {
                const uint32_t slot = within * L::kSlots + b16_slot<KIND>(ks, half);
#pragma unroll
                for (int j = 0; j < JB; ++j) {
                    const bf16x8 bh = __builtin_bit_cast(bf16x8, sb[buf][slot][0][j * 32 + l32]);
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        if constexpr (L::kSplit) {
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i][ks], bh, acc[i][j], 0, 0, 0);
                        }
                        if constexpr (!ONE) {
                            const bf16x8 bl = __builtin_bit_cast(bf16x8, sb[buf][slot][1][j * 32 + l32]);
                            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i][ks], bl, acc[i][j], 0, 0, 0);
                        }
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i][ks], bh, acc[i][j], 0, 0, 0);
                    }
                }
            }
            if (within + 1 == kRound || last) {
                // (the other buffer's readers passed the barrier before this round)
                buf ^= 1;
                park_queries(buf);
                __syncthreads();
            }
        }
        // Nearly nothing passes: sixteen products of a lane share a verdict (their least value).
        code_term[wave][lane] = my_term;
        wave_lds_fence();
        float group_least[JB];
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            group_least[j] = __builtin_inff();
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t m0 = i * 32 + 4 * half;
            float term[16];
#pragma unroll
            for (int e4 = 0; e4 < 4; ++e4) {
                const float4 t4 = *reinterpret_cast<const float4*>(&code_term[wave][m0 + 8 * e4]);
                term[4 * e4] = t4.x;
                term[4 * e4 + 1] = t4.y;
                term[4 * e4 + 2] = t4.z;
                term[4 * e4 + 3] = t4.w;
            }
#pragma unroll
            for (int j = 0; j < JB; ++j) {
                // The low four bits of a value say which of the sixteen it is.
                float v[16];
                float least = __builtin_inff();
#pragma unroll
                for (int e = 0; e < 16; ++e) {
                    const float d = fmaf(p.factor, acc[i][j][e], term[e]);
                    v[e] = __uint_as_float((__float_as_uint(d) & ~15U) | static_cast<uint32_t>(e));
                    least = fminf(least, v[e]);
                }
                group_least[j] = fminf(group_least[j], least);
                while (__ballot(least <= tau_n[j]) != 0) {
                    const bool hit = least <= tau_n[j];
                    const uint64_t mask = __ballot(hit);
                    const uint32_t np = static_cast<uint32_t>(__popcll(mask));
                    if (waiting + np > kB16Queue) {
                        flush();
                    }
                    if (hit) {
                        const uint32_t e = __float_as_uint(least) & 15U;
                        const uint32_t at = waiting + mask_rank(mask);
                        const uint32_t slot = static_cast<uint32_t>(slot0) + m0 + 8 * (e >> 2) + (e & 3);
                        keys[at] = LISTS ? (static_cast<uint64_t>(wave >> 1) << 32) | slot : make_key(least, slot);
                        cols[at] = j * 32 + l32;
                    }
                    waiting += np;
                    // the next of this lane's sixteen (they differ: in the low four bits at least)
                    const float last = least;
                    least = __builtin_inff();
#pragma unroll
                    for (int e = 0; e < 16; ++e) {
                        least = fminf(least, v[e] > last ? v[e] : __builtin_inff());
                    }
                }
            }
        }
        if constexpr (!LISTS) {
            if (p.least != nullptr) {
                // the codes of this wave, one group
#pragma unroll
                for (int j = 0; j < JB; ++j) {
                    const float least = fminf(group_least[j], __shfl_xor(group_least[j], 32));
                    const uint64_t q = q0 + j * 32 + l32;
                    if (half == 0 && q < p.nq) {
                        p.least[q * p.groups + static_cast<uint32_t>(mt) * 4 + wave] = least;
                    }
                }
            }
        }
    }
    if (waiting != 0) {
        flush();
    }
}

static void
b16_query_args(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, B16QueryArgs* qa) {
    const bool l2 = s->metric == VSAG_AMD_METRIC_L2;
    const bool fp32 = s->kind == VSAG_AMD_KIND_FP32;
    *qa = B16QueryArgs{};
    qa->qtab = reinterpret_cast<const float*>(a.qtab);
    qa->qstride = a.qstride;
    qa->kdim = s->dpad;
    qa->scale = !fp32 && l2 ? s->scale_dev : nullptr;
    qa->nq = nq;
    qa->rows = b16_query_rows(nq);
    qa->slots = b16_slots(s);
    qa->ymax_bits = s->pf_ymax;
    qa->cmax = fp32 ? 0.0F : s->kind == VSAG_AMD_KIND_SQ8 || s->kind == VSAG_AMD_KIND_SQ8_UNIFORM ? 255.0F : 15.0F;
    qa->is_l2 = l2 ? 1 : 0;
    qa->uniform = b16_uniform(s) ? 1 : 0;
    qa->nibbles = s->kind == VSAG_AMD_KIND_SQ4_UNIFORM ? 1 : 0;
    qa->lb = s->ulb;
    qa->rate = s->scalar_rate;
    qa->scale = b16_uniform(s) ? nullptr : qa->scale;
    qa->qmeta = (!fp32 && !l2) || b16_uniform(s) ? a.qmeta : nullptr;
    qa->qmeta_stride = a.qmeta_stride;
}

// Queries per workgroup.
static uint32_t
b16_columns(uint64_t nq) {
    return nq <= 32 ? 32 : nq <= 64 ? 64 : kB16N;
}

template <int KIND, bool ONE = false>
static void
launch_b16_flat(uint64_t nq, uint32_t cus, PrefilterB16Args p, hipStream_t st) {
    const uint32_t per = b16_columns(nq);
    const uint64_t qtiles = div_up(nq, static_cast<uint64_t>(per));
    const uint64_t mtiles = p.least != nullptr ? p.groups / 4 : div_up(p.ntiles, 4);
    // Two rounds of the workgroups that fit a compute unit (two or three) and not one more: a few left over would run a
    // third round alone.  A workgroup walks every gridDim.x-th tile.  (One round where most of them return at once.)
    const uint32_t rounds = p.again != nullptr ? 1 : 2;
    uint64_t groups = static_cast<uint64_t>(cus) * rounds * (per == 32 || (per == 64 && KIND != VSAG_AMD_KIND_FP32) ? 3 : 2) / qtiles;
    groups = std::max<uint64_t>(1, std::min<uint64_t>(groups, mtiles));
    const dim3 grid(static_cast<uint32_t>(groups), static_cast<uint32_t>(qtiles));
    if (per == 32) {
        hipLaunchKernelGGL((prefilter_b16_kernel<KIND, false, 1, ONE>), grid, dim3(256), 0, st, p);
    } else if (per == 64) {
        hipLaunchKernelGGL((prefilter_b16_kernel<KIND, false, 2, ONE>), grid, dim3(256), 0, st, p);
    } else {
        hipLaunchKernelGGL((prefilter_b16_kernel<KIND, false, 4, ONE>), grid, dim3(256), 0, st, p);
    }
}

static void
launch_b16_kind(const vsag_amd_store* s, uint64_t nq, const PrefilterB16Args& p, hipStream_t st) {
    const uint32_t cus = static_cast<uint32_t>(device_cu_count());
    if (s->kind == VSAG_AMD_KIND_FP32) {
        launch_b16_flat<VSAG_AMD_KIND_FP32>(nq, cus, p, st);
    } else if (s->kind == VSAG_AMD_KIND_SQ8) {
        launch_b16_flat<VSAG_AMD_KIND_SQ8>(nq, cus, p, st);
    } else if (s->kind == VSAG_AMD_KIND_SQ8_UNIFORM) {
        launch_b16_flat<VSAG_AMD_KIND_SQ8, true>(nq, cus, p, st);
    } else if (s->kind == VSAG_AMD_KIND_SQ4_UNIFORM) {
        launch_b16_flat<VSAG_AMD_KIND_SQ4, true>(nq, cus, p, st);
    } else {
        launch_b16_flat<VSAG_AMD_KIND_SQ4>(nq, cus, p, st);
    }
}

// The sample of a call, in storage tiles spread evenly over the store.  With s of n codes sampled, about k n / s codes lie at or
// below the k-th smallest of the sample: kB16Expect of them (4 k where that is more), a sixteenth of the room a query has (a
// quarter).  Four times as many groups as k keep their k-th least close to the k-th of the sample.
constexpr uint64_t kB16Expect = 128;
constexpr uint32_t kB16Records = 2048;

uint32_t
prefilter_b16_cap(uint32_t k) {
    return std::max<uint32_t>(kB16Records, 16 * k);
}

// A multiple of four, the tiles of whole workgroups.  (A small store's sample is all of its tiles, and up to three behind them
// that hold nothing.)
static uint32_t
b16_sample_groups(const vsag_amd_store* s, uint32_t k) {
    const uint64_t mtiles = div_up(s->ntiles, 4);
    const uint64_t expect = std::max<uint64_t>(kB16Expect, 4ull * k);
    const uint64_t want = std::max<uint64_t>({16, k, div_up(mtiles * k, expect)});
    return static_cast<uint32_t>(4 * div_up(mtiles, std::max<uint64_t>(1, mtiles / want)));
}
// No two of the sample's tiles are the same.
static uint64_t
b16_sample_spread(const vsag_amd_store* s, uint32_t k) {
    const uint64_t groups = b16_sample_groups(s, k);
    return groups < s->ntiles ? (s->ntiles << 32) / groups : 1ull << 32;
}

// Scratch: the queries' parts, then their errors, thresholds, slacks and what the sample leaves.
struct B16Scratch {
    uint4* planes;
    B16Error* error;
    float* tau;
    float* slack;
    uint32_t* again;
    float* least;
};
static size_t
carve_b16(Carver& c, const vsag_amd_store* s, uint64_t nq, uint32_t k, B16Scratch* b) {
    b->planes = reinterpret_cast<uint4*>(c.take<uint8_t>(b16_plane_bytes(s, nq)));
    b->error = c.take<B16Error>(nq);
    b->tau = c.take<float>(nq);
    b->slack = c.take<float>(nq);
    b->again = c.take<uint32_t>(nq);
    b->least = c.take<float>(nq * b16_sample_groups(s, k));
    return c.used;
}
size_t
prefilter_b16_scratch_bytes(const vsag_amd_store* s, uint64_t nq, uint32_t k) {
    Carver c(nullptr, 0);
    B16Scratch b;
    return carve_b16(c, s, nq, k, &b);
}

int launch_rescore_valued(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t k, uint32_t S, uint32_t* bound,
                          const uint64_t* valued, const float* slack, const uint32_t* cand_cnt, uint32_t cap,
                          uint64_t* partial, uint32_t* partial_cnt, uint32_t nslots, uint32_t out_slot, uint32_t* gate,
                          hipStream_t st);

// The flat scan of the header comment: list 0 of every query's nslots partial lists holds its k best, or, where the query has
// to stream, its gate is up and all its lists are empty.  (The other lists of the others hold nothing.)  `bound` and `seed` (or null) are what a search starts from: bound0, and no
// seeds.  raw.q (or null): the queries that the tables of `a` are made of here, nq_pad rows, fewer than 128 above nq.
int
launch_scan_b16(const vsag_amd_store* s, const ScanArgs& a, const FloatQueryArgs& raw, uint64_t nq_pad, uint64_t nq, uint32_t k,
                uint32_t S, uint32_t* bound,
                uint32_t bound0, uint32_t* seed, uint8_t* scratch, uint64_t* cand, uint32_t* cand_cnt, uint32_t cap, const uint32_t* deny, uint64_t* partial,
                uint32_t* partial_cnt, uint32_t nslots, uint32_t* gate, hipStream_t st) {
    Carver c(scratch, ~size_t{0});
    B16Scratch b;
    carve_b16(c, s, nq, k, &b);
    B16QueryArgs qa;
    b16_query_args(s, a, nq, &qa);
    qa.planes = b.planes;
    qa.error = b.error;
    qa.raw = raw;
    qa.nq_pad = nq_pad;
    qa.start = bound;
    qa.bound0 = bound0;
    qa.seed = seed;
    qa.k = k;
    qa.again = b.again;
    hipLaunchKernelGGL(b16_query_kernel, dim3(static_cast<uint32_t>(qa.rows)), dim3(256), 0, st, qa);
    PrefilterB16Args p{};
    p.tiles = s->tiles;
    p.G = s->G;
    p.planes = b.planes;
    p.nq = nq;
    p.rows = qa.rows;
    p.slots = qa.slots;
    p.term = s->pf_term;
    p.terms = qa.is_l2 != 0 || qa.uniform != 0 ? 1 : 0;
    p.factor = qa.is_l2 != 0 ? -2.0F : qa.uniform != 0 ? -qa.rate : -1.0F;
    p.tau = b.tau;
    p.ntiles = s->ntiles;
    p.n = s->n;
    p.deny = deny;
    p.least = b.least;
    p.groups = b16_sample_groups(s, k);
    p.spread = b16_sample_spread(s, k);
    launch_b16_kind(s, nq, p, st);
    B16TauArgs ta{b.least, p.groups, k, b.error, b.tau, b.slack, cand_cnt, gate};
    hipLaunchKernelGGL(b16_tau_kernel, dim3(static_cast<uint32_t>(nq)), dim3(kWave), 0, st, ta);
    p.least = nullptr;
    p.cand = cand;
    p.cand_cnt = cand_cnt;
    p.cap = cap;
    timing_begin(st);
    launch_b16_kind(s, nq, p, st);
    timing_end(st);
    B16AgainArgs aa{cand, cap, k, b.error, b.tau, b.slack, cand_cnt, b.again, b16_columns(nq)};
    hipLaunchKernelGGL(b16_again_kernel, dim3(static_cast<uint32_t>(nq)), dim3(kWave), 0, st, aa);
    p.again = b.again;
    launch_b16_kind(s, nq, p, st);
    VA_HIP(hipGetLastError());
    return launch_rescore_valued(s, a, nq, k, S, bound, cand, b.slack, cand_cnt, cap, partial, partial_cnt, nslots, 0, gate, st);
}

bool
ivf_b16_supports(const vsag_amd_store* s) {
    return s->kind == VSAG_AMD_KIND_FP32 && s->nlist > 0 && s->pf_term != nullptr && s->pf_ymax != nullptr &&
           s->ids_dev != nullptr && (s->residual_centroids_dev == nullptr || s->metric != VSAG_AMD_METRIC_COSINE);
}

uint32_t
ivf_b16_pairs_per_item() {
    return kB16N;
}
size_t
ivf_b16_scratch_bytes(const vsag_amd_store* s, uint64_t nq) {
    return b16_plane_bytes(s, nq);
}

// The candidates of probe columns [p0, nprobe) grouped by list (pair_off, sorted_pair; item_off counted with
// ivf_b16_pairs_per_item() pairs per item) into the private lists (pair * 8 + chunk * 2 + half of the code tile) of
// kcand records in `partial`; partial_cnt and gate zero before.  tau: 2 nq + 1 floats; gate: nq + 2 words.
int
launch_ivf_b16(const vsag_amd_store* s, const ScanArgs& a, uint64_t nq, uint32_t nprobe, uint32_t p0, const uint32_t* pair_off,
               const uint32_t* item_off, const uint32_t* sorted_pair, const uint32_t* bound, uint32_t kcand, float* tau,
               uint8_t* scratch, uint64_t* partial, uint32_t* partial_cnt, uint32_t* gate, const float* res_term,
               hipStream_t st) {
    B16QueryArgs qa;
    b16_query_args(s, a, nq, &qa);
    qa.planes = reinterpret_cast<uint4*>(scratch);
    qa.bound = bound;
    qa.tau = tau;
    qa.gate = gate;
    qa.partial_cnt = partial_cnt;
    qa.p0 = p0;
    qa.nprobe = nprobe;
    qa.k = kcand;
    qa.magnitude = res_term != nullptr ? tau + nq + 1 : nullptr;
    hipLaunchKernelGGL(b16_query_kernel, dim3(static_cast<uint32_t>(qa.rows)), dim3(256), 0, st, qa);
    PrefilterB16Args p{};
    p.tiles = s->tiles;
    p.G = s->G;
    p.planes = qa.planes;
    p.nq = nq;
    p.rows = qa.rows;
    p.slots = qa.slots;
    p.term = s->pf_term;
    p.terms = qa.is_l2;
    p.factor = qa.is_l2 != 0 ? -2.0F : -1.0F;
    p.tau = tau;
    if (res_term != nullptr) {
        p.res_term = res_term;
        p.res_bias = s->residual_bias_dev;
        p.magnitude = qa.magnitude;
        p.ymax_bits = s->pf_ymax;
        p.res_cmax = s->residual_cmax;
    }
    p.ids = s->ids_dev;
    p.list_tile = s->list_tile_dev;
    p.pair_off = pair_off;
    p.item_off = item_off;
    p.sorted_pair = sorted_pair;
    p.nlist = s->nlist;
    p.nprobe = nprobe;
    p.k = kcand;
    p.partial = partial;
    p.partial_cnt = partial_cnt;
    p.gate = gate;
    const uint64_t pairs = nq * (nprobe - p0);
    const uint64_t max_items =
        (div_up(pairs, static_cast<uint64_t>(kB16N)) + std::min<uint64_t>(s->nlist, pairs)) * kIvfB16Chunks;
    timing_begin(st);
    hipLaunchKernelGGL((prefilter_b16_kernel<VSAG_AMD_KIND_FP32, true, 4>), dim3(static_cast<uint32_t>(max_items)),
                       dim3(256), 0, st, p);
    timing_end(st);
    VA_HIP(hipGetLastError());
    return 0;
}

}  // namespace vsag_amd
