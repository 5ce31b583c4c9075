// Quantizer training and encoding on the device: scalar-quantization bounds, sq8/sq4 codes, uniform
// codes, RaBitQ 1-bit codes and processed queries.  These are build-time and per-batch steps, not the
// scan; they are written so that their results equal the reference's scalar arithmetic bit for bit where
// that arithmetic is order-dependent (running fp32 sums are kept in element order, products and sums are
// not fused: this translation unit is compiled with -ffp-contract=off).
#include <cfloat>
#include <type_traits>

#include "common.h"
#include "topk.h"

namespace vsag_amd {

// ------------------------------------------------------------------ helpers
// Sums that must run in element order belong to one thread per row, but a thread that walks a row of its own touches a
// memory line per lane and load (a pass over 1M x 128 rows that way ran at a tenth of the copy rate).  So a wave takes 64
// rows and brings 32 dimensions of all of them at a time into LDS with loads along the rows -- eight lanes a 128-byte run
// -- and every lane then reads its own row there (a stride of 33 words: no bank conflicts).  The next 32 dimensions are
// on their way while a chunk is worked on.
constexpr uint32_t kRowDims = 32;

struct RowTile {
    float v[kWave][kRowDims + 1];
};

// Calls body(d0, m) for every chunk of m <= 32 dimensions with the wave's rows in `t`; row(r) is the address of row r of
// the 64 (null: no such row, its values read as zero).
template <typename Row, typename Body>
__device__ inline void
for_row_chunks(RowTile& t, uint32_t dim, uint32_t lane, Row row, Body body) {
    const bool vec = (dim & 3U) == 0 && (reinterpret_cast<uintptr_t>(row(0)) & 15U) == 0;
    float4 next[8];
    auto load = [&](uint32_t d0) {
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) {
            const float* p = row(8 * i + lane / 8);
            const uint32_t d = d0 + 4 * (lane & 7U);
            next[i] = make_float4(0.0F, 0.0F, 0.0F, 0.0F);
            if (p != nullptr && d < dim) {
                if (vec) {
                    next[i] = *reinterpret_cast<const float4*>(p + d);
                } else {
                    next[i].x = p[d];
                    next[i].y = d + 1 < dim ? p[d + 1] : 0.0F;
                    next[i].z = d + 2 < dim ? p[d + 2] : 0.0F;
                    next[i].w = d + 3 < dim ? p[d + 3] : 0.0F;
                }
            }
        }
    };
    load(0);
    for (uint32_t d0 = 0; d0 < dim; d0 += kRowDims) {
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) {
            float* to = &t.v[8 * i + lane / 8][4 * (lane & 7U)];
            to[0] = next[i].x;
            to[1] = next[i].y;
            to[2] = next[i].z;
            to[3] = next[i].w;
        }
        wave_lds_fence();
        if (d0 + kRowDims < dim) {
            load(d0 + kRowDims);
        }
        body(d0, dim - d0 < kRowDims ? dim - d0 : kRowDims);
        wave_lds_fence();
    }
}

// generic::Normalize (src/simd/generic.cpp:874-878, kernels/scalar_op.h:32-60): ||x|| as a running sum in
// element order; a zero norm divides by one.  A wave per 64 rows.
__global__ void __launch_bounds__(256)
row_norm_kernel(const float* x, uint64_t n, uint32_t dim, float* norms) {
    __shared__ RowTile tiles[4];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t row0 = (static_cast<uint64_t>(blockIdx.x) * 4 + wave) * kWave;
    if (row0 >= n) {
        return;
    }
    RowTile& t = tiles[wave];
    float s = 0.0F;
    for_row_chunks(
        t, dim, lane, [&](uint32_t r) { return row0 + r < n ? x + (row0 + r) * dim : nullptr; },
        [&](uint32_t, uint32_t m) {
            if (m == kRowDims) {
#pragma unroll
                for (uint32_t c = 0; c < kRowDims; ++c) {
                    s = t.v[lane][c] * t.v[lane][c] + s;
                }
            } else {
                for (uint32_t c = 0; c < m; ++c) {
                    s = t.v[lane][c] * t.v[lane][c] + s;
                }
            }
        });
    if (row0 + lane < n) {
        const float norm = sqrtf(s);
        norms[row0 + lane] = norm == 0.0F ? 1.0F : norm;
    }
}

static void
launch_row_norms(const float* x, uint64_t n, uint32_t dim, float* norms, hipStream_t st) {
    hipLaunchKernelGGL(row_norm_kernel, dim3(static_cast<uint32_t>(div_up(n, 4 * kWave))), dim3(256), 0, st, x, n, dim,
                       norms);
}

// ClampScalarQuantizationDelta (scalar_quantization_utils.h:19-30).
__device__ inline float
clamp_delta(float delta) {
    if (!(delta >= 0.0F)) {
        return 0.0F;
    }
    if (delta > 0.999F) {
        return 1.0F;
    }
    return delta;
}

// ------------------------------------------------------------------ sq8 / sq4 encode
// ScalarQuantizer::EncodeOneImpl (scalar_quantizer.cpp:85-112) of one value.
__device__ inline uint32_t
sq_level(float v, float lb, float diff, float levels) {
    float delta;
    if (diff < FLT_EPSILON) {
        delta = 1.0F;
    } else {
        delta = 1.0F * (v - lb) / diff;
    }
    return static_cast<uint8_t>(levels * clamp_delta(delta));
}

// 1 / diff where a division by diff can be replaced: a = v - lb, q = a * inv is two units in the last place off at most, a
// first remainder brings it to within one, and from there a remainder and a correction give the rounded quotient if inv is
// the rounded reciprocal (Markstein, IBM J. Res. Dev. 34, 1990), as long as nothing leaves the normal numbers: diff is held
// to [2^-23, 2^100], and a quotient below 1/256 is level 0 however it is rounded.  0 elsewhere: such a column divides.
__device__ inline float
sq_inverse(float diff) {
    return diff >= FLT_EPSILON && diff <= 0x1p100F ? 1.0F / diff : 0.0F;
}

// sq_level with inv = sq_inverse(diff): the same level for every v.
__device__ inline uint32_t
sq_level_by_inverse(float v, float lb, float diff, float inv, float levels) {
    if (inv == 0.0F) {
        return sq_level(v, lb, diff, levels);
    }
    const float a = v - lb;
    const float q = a * inv;
    float delta = fmaf(fmaf(-q, diff, a), inv, q);
    delta = fmaf(fmaf(-delta, diff, a), inv, delta);
    delta = q < 2.0F ? delta : q;  // (far above the range an infinity has no remainder)
    return static_cast<uint8_t>(levels * clamp_delta(delta));
}

// Rows and codes as two flat arrays: where a row fills whole bytes (sq8; sq4 with an even dimension) neither has a gap, so
// a thread turns 4 (sq8) or 8 (sq4) values in a run, wherever rows begin in it, into one code word: 16-byte loads and 4-byte
// stores at any dimension.  A workgroup of `blockDim` threads takes RUNS x blockDim consecutive runs; with RUNS > 1 blockDim
// runs are whole rows, so a thread meets the same dimensions in each of its runs and keeps their bounds in registers, with
// RUNS loads on their way.  What bounds it is memory: 1M x 128 rows to sq8 466 us with a thread per byte, 138 us with a run
// per thread and a division per value, 132 us without the division, and 102 us with short workgroups of four runs a
// thread that pass the caches by (2048 long-lived ones, loads and stores as they come: 132; the reading alone 72).  Past the
// caches go neither the two loads of a run of sq4, which share their lines (161 -> 148 us), nor rows whose norms were taken just
// before (20 000 x 960 to sq8 under cosine: 60 -> 52 us with the norms).
//
// VEC: the dimension is a multiple of four, so bounds (then on 16 bytes) come four a load and a norm serves four values.  In
// single words they were more loads than the rows: 1M x 128 to sq4 148 us and 101 so (134 with a run per thread), 427k x 300 under
// cosine 302 and 237 with the norms (261).
template <int BITS, bool NORM, bool VEC, int RUNS>
__global__ void __launch_bounds__(1024)
sq_encode_kernel(const float* x, uint64_t total, uint32_t dim, const float* lb, const float* diff, const float* norms,
                 uint8_t* codes) {
    constexpr uint32_t kDims = 32 / BITS;  // per code word
    const uint64_t first = static_cast<uint64_t>(blockIdx.x) * (blockDim.x * RUNS);  // of the workgroup
    const uint64_t whole = total / kDims;
    const uint64_t run = first + threadIdx.x;
    if (run * kDims >= total) {
        return;
    }
    typedef float float4_v __attribute__((ext_vector_type(4)));
    float v[RUNS][kDims];
#pragma unroll
    for (uint32_t r = 0; r < RUNS; ++r) {
        const uint64_t at = run + r * blockDim.x;
#pragma unroll
        for (uint32_t e = 0; e < kDims; e += 4) {
            if (at < whole) {
                const float4_v* from = reinterpret_cast<const float4_v*>(x + at * kDims + e);
                const float4_v a = BITS == 8 && !NORM && RUNS > 1 ? __builtin_nontemporal_load(from) : *from;
                v[r][e] = a.x, v[r][e + 1] = a.y, v[r][e + 2] = a.z, v[r][e + 3] = a.w;
            } else {
#pragma unroll
                for (uint32_t u = e; u < e + 4; ++u) {
                    v[r][u] = at * kDims + u < total ? x[at * kDims + u] : 0.0F;
                }
            }
        }
    }
    // Row and dimension of the first value, from those of the workgroup (wave-uniform).
    const uint64_t row0 = first * kDims / dim;
    const uint32_t off = static_cast<uint32_t>(first * kDims - row0 * dim) + threadIdx.x * kDims;
    const uint64_t row = row0 + off / dim;
    const uint64_t step_rows = static_cast<uint64_t>(blockDim.x) * kDims / dim;
    float lo[kDims], df[kDims], inv[kDims];
    uint32_t row_off[kDims];
    {
        uint32_t d = off % dim, r = 0;
        constexpr uint32_t kStep = VEC ? 4 : 1;
#pragma unroll
        for (uint32_t e = 0; e < kDims; e += kStep) {
            if constexpr (VEC) {
                const float4_v l4 = *reinterpret_cast<const float4_v*>(lb + d), f4 = *reinterpret_cast<const float4_v*>(diff + d);
                lo[e] = l4.x, lo[e + 1] = l4.y, lo[e + 2] = l4.z, lo[e + 3] = l4.w;
                df[e] = f4.x, df[e + 1] = f4.y, df[e + 2] = f4.z, df[e + 3] = f4.w;
            } else {
                lo[e] = lb[d];
                df[e] = diff[d];
            }
            row_off[e] = r;
            d += kStep;
            r += d == dim ? 1 : 0;
            d = d == dim ? 0 : d;
        }
#pragma unroll
        for (uint32_t e = 0; e < kDims; ++e) {
            inv[e] = sq_inverse(df[e]);
        }
    }
    const float levels = static_cast<float>((1 << BITS) - 1);
    float nrm[RUNS][kDims / 4];
    if constexpr (NORM && VEC) {
#pragma unroll
        for (uint32_t r = 0; r < RUNS; ++r) {
#pragma unroll
            for (uint32_t e = 0; e < kDims; e += 4) {
                nrm[r][e / 4] = (run + r * blockDim.x) * kDims + e < total ? norms[row + r * step_rows + row_off[e]] : 1.0F;
            }
        }
    }
#pragma unroll
    for (uint32_t r = 0; r < RUNS; ++r) {
        const uint64_t at = run + r * blockDim.x;
        if (at * kDims >= total) {
            break;
        }
        const uint32_t values = at < whole ? kDims : static_cast<uint32_t>(total - at * kDims);
        float each[kDims];
        if constexpr (NORM && !VEC) {
            if (at < whole) {
#pragma unroll
                for (uint32_t e = 0; e < kDims; ++e) {
                    each[e] = norms[row + r * step_rows + row_off[e]];
                }
            } else {
#pragma unroll
                for (uint32_t e = 0; e < kDims; ++e) {
                    each[e] = e < values ? norms[row + r * step_rows + row_off[e]] : 1.0F;
                }
            }
        }
        uint32_t word = 0;
#pragma unroll
        for (uint32_t e = 0; e < kDims; ++e) {
            float value = v[r][e];
            if constexpr (NORM) {
                value /= VEC ? nrm[r][e / 4] : each[e];
            }
            // (a reciprocal is a division too: with one value to a dimension there is nothing to save)
            const uint32_t level = RUNS > 1 ? sq_level_by_inverse(value, lo[e], df[e], inv[e], levels) : sq_level(value, lo[e], df[e], levels);
            word |= level << (e * BITS);
        }
        if (at < whole) {
            __builtin_nontemporal_store(word, reinterpret_cast<uint32_t*>(codes) + at);
        } else {
            for (uint32_t b = 0; b < values * BITS / 8; ++b) {
                codes[at * kDims * BITS / 8 + b] = static_cast<uint8_t>(word >> (8 * b));
            }
        }
    }
}

// The workgroup of the kernel above: threads, runs per thread.  After `period` runs the dimensions repeat; workgroups are
// multiples of it with four runs where that makes at most 1024 threads and six workgroups a compute unit (twelve under
// cosine, whose divisions make the threads longer), and one run otherwise: odd dimensions beyond 1024, and few rows, which four
// runs leave on a fourth of the chip (20 000 x 128 sq8 6.0 us, 5.0 with one; 99 000 x 128 sq4 under cosine 30.9 and 28.4).
// Workgroups that do not fill their last wave are worth it: 498k x 257 to sq8, 257 threads, 232 -> 128 us.
static void
sq_encode_shape(uint32_t dim, uint32_t kdims, uint64_t words, bool norm, uint32_t* threads, uint32_t* runs) {
    uint32_t g = kdims;
    while (dim % g != 0) {
        g /= 2;
    }
    const uint32_t period = dim / g;
    *threads = period > 1024 || period == 1 ? 256 : period > 256 ? period : 256 / period * period;
    *runs = period <= 1024 && words >= 4ull * *threads * (norm ? 3072 : 1536) ? 4 : 1;
}

// The same with one thread per code byte: sq4 codes of an odd dimension (the last byte of a row holds one value), and
// pointers that the vector form does not take.
__global__ void __launch_bounds__(256)
sq_encode_bytes_kernel(const float* x, uint64_t n, uint32_t dim, int bits, const float* lb, const float* diff,
                       const float* norms, uint32_t code_size, uint8_t* codes) {
    const uint64_t gid = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    const uint64_t i = gid / code_size;
    const uint32_t b = static_cast<uint32_t>(gid % code_size);
    if (i >= n) {
        return;
    }
    const float* r = x + i * dim;
    const float norm = norms != nullptr ? norms[i] : 1.0F;
    const float levels = static_cast<float>((1 << bits) - 1);
    const uint32_t per_byte = 8 / bits;
    uint32_t byte = 0;
    for (uint32_t e = 0; e < per_byte; ++e) {
        const uint32_t d = b * per_byte + e;
        if (d >= dim) {
            break;
        }
        byte |= sq_level(norms != nullptr ? r[d] / norm : r[d], lb[d], diff[d], levels) << (e * bits);
    }
    codes[i * code_size + b] = static_cast<uint8_t>(byte);
}

// ------------------------------------------------------------------ uniform encode
// SQ4UniformQuantizer::EncodeOneImpl / SQ8UniformQuantizer::EncodeOneImpl.  A wave per 64 rows (for_row_chunks): a lane
// encodes its row and adds the two fp32 sums up in element order (with a wave per row, one lane adding what 64 had encoded,
// 432k x 100 rows under inner product took 2.5 ms).  The code words of a chunk leave through LDS, eight lanes a run.
// Code sizes of the uniform kinds are multiples of four bytes.
template <int BITS>
__global__ void __launch_bounds__(256)
squ_encode_kernel(const float* x, uint64_t n, uint32_t dim, int metric, const float* bounds, const float* norms,
                  uint32_t code_size, uint32_t payload, uint32_t off_norm, uint32_t off_sum, uint32_t off_codes_sum,
                  uint8_t* codes) {
    constexpr uint32_t kDims = 32 / BITS;           // per code word
    constexpr uint32_t kWords = kRowDims / kDims;   // per chunk
    __shared__ RowTile tiles[4];
    __shared__ uint32_t outs[4][kWave][kWords + 1];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t row0 = (static_cast<uint64_t>(blockIdx.x) * 4 + wave) * kWave;
    if (row0 >= n) {
        return;
    }
    RowTile& t = tiles[wave];
    auto& out = outs[wave];
    const float lb = bounds[0], diff = bounds[1];
    const float inv_diff = diff == 0.0F ? 0.0F : 1.0F / diff;
    const float levels = BITS == 4 ? 15.0F : 255.0F;
    const bool live = row0 + lane < n;
    const float nrm = norms != nullptr && live ? norms[row0 + lane] : 1.0F;
    const bool aligned = (reinterpret_cast<uintptr_t>(codes) & 3U) == 0;
    auto put = [&](uint8_t* to, uint32_t word) {
        if (aligned) {
            *reinterpret_cast<uint32_t*>(to) = word;
        } else {
            for (uint32_t k = 0; k < 4; ++k) {
                to[k] = static_cast<uint8_t>(word >> (8 * k));
            }
        }
    };
    const uint32_t payload_words = (payload + 3) / 4;
    uint32_t norm_part = 0;
    float sum = 0.0F, codes_sum = 0.0F;
    for_row_chunks(
        t, dim, lane, [&](uint32_t r) { return row0 + r < n ? x + (row0 + r) * dim : nullptr; },
        [&](uint32_t d0, uint32_t m) {
#pragma unroll
            for (uint32_t w = 0; w < kWords; ++w) {
                uint32_t word = 0;
#pragma unroll
                for (uint32_t e = 0; e < kDims; ++e) {
                    const uint32_t c = w * kDims + e;
                    if (c < m) {
                        const float v = norms != nullptr ? t.v[lane][c] / nrm : t.v[lane][c];
                        const float delta = clamp_delta((v - lb) * inv_diff);
                        const uint32_t scaled = static_cast<uint8_t>(levels * delta);
                        word |= scaled << (e * BITS);
                        norm_part += scaled * scaled;
                        sum += v;
                        codes_sum += static_cast<float>(scaled);
                    }
                }
                out[lane][w] = word;
            }
            wave_lds_fence();
            const uint32_t w0 = d0 / kDims;
            for (uint32_t i = lane; i < kWave * kWords; i += kWave) {
                const uint32_t r = i / kWords, w = i % kWords;
                if (row0 + r < n && w0 + w < payload_words) {
                    put(codes + (row0 + r) * code_size + 4 * (w0 + w), out[r][w]);
                }
            }
        });
    if (!live) {
        return;
    }
    uint8_t* c = codes + (row0 + lane) * code_size;
    for (uint32_t b = 4 * payload_words; b < code_size; b += 4) {
        uint32_t word = 0;
        if (metric == VSAG_AMD_METRIC_L2) {
            word = b == off_norm ? norm_part : 0U;  // a u64 whose upper half is zero
        } else if (b == off_sum) {
            word = __float_as_uint(sum);
        } else if (BITS == 4 && b == off_codes_sum) {
            word = __float_as_uint(codes_sum);
        }
        put(c + b, word);
    }
}

// The same for few rows (the queries of a search): a wave per row, which it keeps in LDS, and the norm of a cosine row with
// it.  64 rows per wave would leave most of the machine idle and wait for memory once per chunk (987 queries x 128: 21 us
// against 4 us).  The sums in element order are one lane's chain of adds over LDS; the sum of the codes is a sum of small
// integers, exact in any order.  dim <= kRowEncodeMaxDim.
constexpr uint32_t kRowEncodeMaxDim = 4096;
constexpr uint64_t kRowEncodeMaxRows = 32768;  // 64 rows per wave: one wave per SIMD from twice that on

template <int BITS>
__global__ void __launch_bounds__(256)
squ_encode_row_kernel(const float* x, uint64_t n, uint32_t dim, uint32_t dim_pad, int metric, const float* bounds,
                      uint32_t code_size, uint32_t payload, uint32_t off_norm, uint32_t off_sum, uint32_t off_codes_sum,
                      uint8_t* codes) {
    extern __shared__ __align__(16) float row_lds[];
    constexpr uint32_t kDims = 32 / BITS;  // per code word
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t row = static_cast<uint64_t>(blockIdx.x) * 4 + wave;
    if (row >= n) {
        return;
    }
    float* v = row_lds + wave * dim_pad;  // dim_pad: a multiple of 32
    for (uint32_t d = lane; d < dim_pad; d += kWave) {
        v[d] = d < dim ? x[row * dim + d] : 0.0F;
    }
    wave_lds_fence();
    float nrm = 1.0F;
    if (metric == VSAG_AMD_METRIC_COSINE) {
        float s = 0.0F;  // every lane the same chain (row_norm_kernel's; the zeros behind the row add nothing)
        for (uint32_t d = 0; d < dim_pad; d += 32) {
#pragma unroll
            for (uint32_t u = 0; u < 32; u += 4) {
                const float4 f = *reinterpret_cast<const float4*>(v + d + u);
                s = f.x * f.x + s;
                s = f.y * f.y + s;
                s = f.z * f.z + s;
                s = f.w * f.w + s;
            }
        }
        nrm = sqrtf(s);
        nrm = nrm == 0.0F ? 1.0F : nrm;
        wave_lds_fence();
    }
    const float lb = bounds[0], diff = bounds[1];
    const float inv_diff = diff == 0.0F ? 0.0F : 1.0F / diff;
    const float levels = BITS == 4 ? 15.0F : 255.0F;
    uint8_t* c = codes + row * code_size;
    const bool aligned = (reinterpret_cast<uintptr_t>(codes) & 3U) == 0;
    auto put = [&](uint32_t at, uint32_t word) {
        if (aligned) {
            *reinterpret_cast<uint32_t*>(c + at) = word;
        } else {
            for (uint32_t k = 0; k < 4; ++k) {
                c[at + k] = static_cast<uint8_t>(word >> (8 * k));
            }
        }
    };
    const uint32_t payload_words = (payload + 3) / 4;
    uint32_t norm_part = 0, codes_sum = 0;
    for (uint32_t w = lane; w < payload_words; w += kWave) {
        uint32_t word = 0;
#pragma unroll
        for (uint32_t e = 0; e < kDims; ++e) {
            const uint32_t d = w * kDims + e;
            if (d < dim) {
                const float value = metric == VSAG_AMD_METRIC_COSINE ? v[d] / nrm : v[d];
                v[d] = value;
                const uint32_t scaled = static_cast<uint8_t>(levels * clamp_delta((value - lb) * inv_diff));
                word |= scaled << (e * BITS);
                norm_part += scaled * scaled;
                codes_sum += scaled;
            }
        }
        put(4 * w, word);
    }
    for (int off = 32; off > 0; off >>= 1) {
        norm_part += __shfl_xor(norm_part, off);
        codes_sum += __shfl_xor(codes_sum, off);
    }
    float sum = 0.0F;
    if (metric != VSAG_AMD_METRIC_L2) {
        wave_lds_fence();
        for (uint32_t d = 0; d < dim_pad; d += 32) {
#pragma unroll
            for (uint32_t u = 0; u < 32; u += 4) {
                const float4 f = *reinterpret_cast<const float4*>(v + d + u);
                sum += f.x;
                sum += f.y;
                sum += f.z;
                sum += f.w;
            }
        }
    }
    for (uint32_t b = 4 * (payload_words + lane); b < code_size; b += 4 * kWave) {
        uint32_t word = 0;
        if (metric == VSAG_AMD_METRIC_L2) {
            word = b == off_norm ? norm_part : 0U;  // a u64 whose upper half is zero
        } else if (b == off_sum) {
            word = __float_as_uint(sum);
        } else if (BITS == 4 && b == off_codes_sum) {
            word = __float_as_uint(static_cast<float>(codes_sum));
        }
        put(b, word);
    }
}

// ------------------------------------------------------------------ C = A * B^T, k in element order
// C[i][j] = sum_k A[i][k] * B[j][k], one unfused multiply and add per k in increasing k, so every output
// equals a scalar running-sum dot product (the RowMajor sgemv of random_orthogonal_transformer.cpp:58-77
// restated in element order).  64 x 64 output tile per workgroup, 4 x 4 outputs per thread.
__global__ void __launch_bounds__(256)
gemm_nt_seq_kernel(const float* A, const float* B, float* C, uint64_t M, uint32_t N, uint32_t K) {
    __shared__ float As[16][65];
    __shared__ float Bs[16][65];
    const uint32_t tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const uint64_t row0 = static_cast<uint64_t>(blockIdx.y) * 64;
    const uint32_t col0 = blockIdx.x * 64;
    float acc[4][4] = {};
    for (uint32_t k0 = 0; k0 < K; k0 += 16) {
        for (uint32_t idx = threadIdx.x; idx < 64 * 16; idx += 256) {
            uint32_t r = idx >> 4, kk = idx & 15;
            uint64_t ar = row0 + r;
            uint32_t br = col0 + r;
            As[kk][r] = (ar < M && k0 + kk < K) ? A[ar * K + k0 + kk] : 0.0F;
            Bs[kk][r] = (br < N && k0 + kk < K) ? B[static_cast<uint64_t>(br) * K + k0 + kk] : 0.0F;
        }
        __syncthreads();
        uint32_t kmax = K - k0 < 16 ? K - k0 : 16;
        for (uint32_t kk = 0; kk < kmax; ++kk) {
            float a[4], b[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                a[i] = As[kk][ty * 4 + i];
                b[i] = Bs[kk][tx * 4 + i];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    acc[i][j] = a[i] * b[j] + acc[i][j];
                }
            }
        }
        __syncthreads();
    }
    for (int i = 0; i < 4; ++i) {
        uint64_t r = row0 + ty * 4 + i;
        if (r >= M) {
            continue;
        }
        for (int j = 0; j < 4; ++j) {
            uint32_t cidx = col0 + tx * 4 + j;
            if (cidx < N) {
                C[r * N + cidx] = acc[i][j];
            }
        }
    }
}

static int
gemm_nt_seq(const float* A, const float* B, float* C, uint64_t M, uint32_t N, uint32_t K, hipStream_t st) {
    dim3 grid((N + 63) / 64, static_cast<uint32_t>(div_up(M, 64)));
    hipLaunchKernelGGL(gemm_nt_seq_kernel, grid, dim3(256), 0, st, A, B, C, M, N, K);
    VA_HIP(hipGetLastError());
    return 0;
}

// ------------------------------------------------------------------ RaBitQ
struct RabitqLayout {
    uint32_t dim, code_bytes;
    uint32_t base_bits, offset_norm_code;  // bits per dimension of the base code; |code - centre| where base_bits != 1
    uint32_t offset_norm, offset_error, offset_sum, offset_raw_norm, code_size;
    int has_sum, has_raw_norm;
    uint32_t aligned_dim, plane_bytes;
    uint32_t q_offset_lb, q_offset_delta, q_offset_sum, q_offset_norm, q_offset_raw_norm, query_code_size;
};

// rabitq_quantizer.cpp:102-176 (standard version, no PCA / MRQ / split storage).  `query_bits` is the bits word of the
// C interface: 4 or 32 for the query, plus 256 * base bits for multi-bit base codes (VSAG_AMD_RABITQ_BITS).
__host__ __device__ inline RabitqLayout
rabitq_layout(uint32_t dim, int metric, int query_bits) {
    RabitqLayout l{};
    l.dim = dim;
    l.base_bits = (query_bits >> 8) == 0 ? 1U : static_cast<uint32_t>(query_bits >> 8);
    query_bits &= 255;
    l.code_bytes = (dim + 7) / 8 * l.base_bits;
    uint32_t cs = (l.code_bytes + 3) / 4 * 4;
    if (l.base_bits != 1) {
        l.offset_norm_code = cs;
        cs += 4;
    }
    l.offset_norm = cs;
    cs += 4;
    l.offset_error = cs;
    cs += 4;
    l.has_sum = query_bits != 32;
    if (l.has_sum) {
        l.offset_sum = cs;
        cs += 4;
    }
    l.has_raw_norm = metric != VSAG_AMD_METRIC_L2;
    if (l.has_raw_norm) {
        l.offset_raw_norm = cs;
        cs += 4;
    }
    l.code_size = cs;
    uint32_t qs;
    if (query_bits == 4) {
        l.aligned_dim = (dim + 511) / 512 * 512;
        l.plane_bytes = l.aligned_dim / 8;
        qs = l.plane_bytes * 4;
        l.q_offset_lb = qs;
        qs += 4;
        l.q_offset_delta = qs;
        qs += 4;
        l.q_offset_sum = qs;
        qs += 4;
    } else {
        qs = 4 * dim;
        if (l.base_bits != 1) {
            l.q_offset_sum = qs;
            qs += 4;
        }
    }
    l.q_offset_norm = qs;
    qs += 4;
    if (l.has_raw_norm) {
        l.q_offset_raw_norm = qs;
        qs += 4;
    }
    l.query_code_size = qs;
    return l;
}

uint64_t
rabitq_code_size(uint32_t dim, int metric, int query_bits) {
    return rabitq_layout(dim, metric, query_bits).code_size;
}
uint64_t
rabitq_query_code_size(uint32_t dim, int metric, int query_bits) {
    return rabitq_layout(dim, metric, query_bits).query_code_size;
}

__device__ inline float
load_f32(const uint8_t* p) {
    uint32_t u = 0;
    for (int b = 0; b < 4; ++b) {
        u |= static_cast<uint32_t>(p[b]) << (8 * b);
    }
    return __uint_as_float(u);
}

__device__ inline void
store_f32(uint8_t* p, float v) {
    uint32_t u = __float_as_uint(v);
    for (int b = 0; b < 4; ++b) {
        p[b] = static_cast<uint8_t>(u >> (8 * b));
    }
}

// Column means as running fp32 sums over the rows in order (rabitq_quantizer.cpp:224-241).  A workgroup owns 32
// columns: eight waves stage the next 256 rows of those columns in LDS while a ninth adds the current 256, one column a
// lane, in row order -- the additions stay sequential, the loads do not.
//
// What bounds it is the chain of adds.  Four stages are on their way, so that a memory latency is spread over 1024 rows, and
// the adding wave does nothing else and goes first on its SIMD (168 787 x 128 rows: 849 us with a
// wave that loads as well, 730 now: 4.3 ns a row).
constexpr uint32_t kMeanCols = 32;
constexpr uint32_t kMeanRows = 256;
constexpr uint32_t kMeanAhead = 4;
constexpr uint32_t kMeanLoaders = 512;
constexpr uint32_t kMeanSlots = kMeanLoaders / kMeanCols;   // rows of a load
constexpr uint32_t kMeanLoads = kMeanRows / kMeanSlots;     // loads of a stage

__global__ void __launch_bounds__(kMeanLoaders + kWave)
column_mean_seq_kernel(const float* x, uint64_t n, uint32_t dim, float* mean) {
    __shared__ __align__(16) float stage[2][kMeanCols][kMeanRows + 4];  // a column's rows in a run: four of them a read
    static_assert(kMeanAhead % 2 == 0, "the two LDS buffers alternate within a round");
    if (threadIdx.x < kMeanLoaders) {
        const uint32_t col = threadIdx.x & (kMeanCols - 1);
        const uint32_t slot = threadIdx.x / kMeanCols;
        const uint32_t d = blockIdx.x * kMeanCols + col;
        float regs[kMeanAhead][kMeanLoads];
        // (no branch around a load: the wait for one stage must not become a wait for all that are in flight)
        const uint32_t d_in = d < dim ? d : dim - 1;
        auto fetch = [&](uint64_t row0, float(&to)[kMeanLoads]) {
#pragma unroll
            for (uint32_t u = 0; u < kMeanLoads; ++u) {
                const uint64_t r = row0 + u * kMeanSlots + slot;
                to[u] = x[(r < n ? r : n - 1) * dim + d_in];
            }
        };
#pragma unroll
        for (uint32_t a = 0; a < kMeanAhead; ++a) {
            fetch(static_cast<uint64_t>(a) * kMeanRows, regs[a]);
        }
        for (uint64_t base = 0; base < n; base += kMeanAhead * kMeanRows) {
#pragma unroll
            for (uint32_t a = 0; a < kMeanAhead; ++a) {
                const uint64_t row0 = base + a * kMeanRows;
                if (row0 >= n) {
                    break;
                }
                // Buffer a & 1 was last read two stages ago, a barrier ago.
#pragma unroll
                for (uint32_t u = 0; u < kMeanLoads; ++u) {
                    stage[a & 1U][col][u * kMeanSlots + slot] = regs[a][u];
                }
                fetch(row0 + kMeanAhead * kMeanRows, regs[a]);
                __syncthreads();
            }
        }
        return;
    }
    __builtin_amdgcn_s_setprio(3);
    const uint32_t col = threadIdx.x & (kMeanCols - 1);  // (both halves of the wave add; the first one writes)
    const uint32_t d = blockIdx.x * kMeanCols + col;
    float s = 0.0F;
    uint32_t a = 0;
    for (uint64_t row0 = 0; row0 < n; row0 += kMeanRows, a ^= 1) {  // a barrier per stage, as above
        __syncthreads();
        const uint32_t m = n - row0 < kMeanRows ? static_cast<uint32_t>(n - row0) : kMeanRows;
        const float* rows = stage[a][col];
        if (m == kMeanRows) {
            // the LDS reads of the next 32 rows ahead of the adds of these: only the adds wait for each other
            float4 v[2][8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) {
                v[0][u] = *reinterpret_cast<const float4*>(rows + 4 * u);
            }
#pragma unroll
            for (uint32_t r = 0; r < kMeanRows; r += 32) {
                if (r + 32 < kMeanRows) {
#pragma unroll
                    for (uint32_t u = 0; u < 8; ++u) {
                        v[(r / 32 + 1) & 1][u] = *reinterpret_cast<const float4*>(rows + r + 32 + 4 * u);
                    }
                }
#pragma unroll
                for (uint32_t u = 0; u < 8; ++u) {
                    const float4 w = v[(r / 32) & 1][u];
                    s += w.x;
                    s += w.y;
                    s += w.z;
                    s += w.w;
                }
            }
        } else {
            for (uint32_t r = 0; r < m; ++r) {
                s += rows[r];
            }
        }
    }
    if (threadIdx.x < kMeanLoaders + kMeanCols && d < dim) {
        mean[d] = s / static_cast<float>(n);
    }
}

// Second half of RaBitQuantizer::EncodeOneInternal (rabitq_quantizer.cpp:749-856) for rows already rotated:
// raw norm of the input row, NormalizeWithCentroid (kernels/normalize.h:35-83), sign bits, error =
// RaBitQFloatBinaryIP(normed, bits) (generic.cpp:447-471), bit count.  One thread per row, element order, the rows through
// for_row_chunks.
__global__ void __launch_bounds__(256)
rabitq_finish_encode_kernel(const float* raw, const float* rotated, uint64_t n, uint32_t dim, const float* centroid,
                            int metric, int query_bits, uint8_t* codes) {
    __shared__ RowTile tiles[4];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t row0 = (static_cast<uint64_t>(blockIdx.x) * 4 + wave) * kWave;
    if (row0 >= n) {
        return;
    }
    RowTile& t = tiles[wave];
    const bool live = row0 + lane < n;
    const RabitqLayout l = rabitq_layout(dim, metric, query_bits);
    uint8_t* c = codes + (row0 + lane) * l.code_size;  // code sizes are multiples of four bytes
    auto rows_of = [&](const float* x) {
        return [=](uint32_t r) { return row0 + r < n ? x + (row0 + r) * dim : nullptr; };
    };
    float raw_norm = 0.0F;
    if (l.has_raw_norm) {
        for_row_chunks(t, dim, lane, rows_of(raw), [&](uint32_t, uint32_t m) {
            for (uint32_t e = 0; e < m; ++e) {
                raw_norm += t.v[lane][e] * t.v[lane][e];
            }
        });
    }
    raw_norm = sqrtf(raw_norm);
    float norm_sq = 0.0F;
    for_row_chunks(t, dim, lane, rows_of(rotated), [&](uint32_t d0, uint32_t m) {
        for (uint32_t e = 0; e < m; ++e) {
            const float v = t.v[lane][e] - centroid[d0 + e];
            norm_sq = v * v + norm_sq;
        }
    });
    const float norm = norm_sq < 1e-5F ? 1.0F : sqrtf(norm_sq);
    const float inv_sqrt_d = 1.0F / sqrtf(static_cast<float>(dim));
    float pos, neg;
    if (inv_sqrt_d > 1e-3F) {
        pos = inv_sqrt_d;
        neg = -inv_sqrt_d;
    } else {
        pos = 1.0F;
        neg = 0.0F;
    }
    const bool aligned = (reinterpret_cast<uintptr_t>(codes) & 3U) == 0;
    auto put = [&](uint32_t at, uint32_t word) {
        if (!live) {
            return;
        }
        if (aligned) {
            *reinterpret_cast<uint32_t*>(c + at) = word;
        } else {
            store_f32(c + at, __uint_as_float(word));
        }
    };
    float error = 0.0F;
    uint32_t binary_sum = 0;
    for_row_chunks(t, dim, lane, rows_of(rotated), [&](uint32_t d0, uint32_t m) {
        uint32_t word = 0;
        for (uint32_t e = 0; e < m; ++e) {
            const float nd = (t.v[lane][e] - centroid[d0 + e]) / norm;
            const bool bit = nd >= 0.0F;
            word |= bit ? 1U << e : 0U;
            error += (bit ? pos : neg) * nd;
        }
        binary_sum += __popc(word);
        put(d0 / 8, word);  // 32 dimensions are a code word; behind the last one lie zero bits
    });
    put(l.offset_norm, __float_as_uint(norm));
    put(l.offset_error, __float_as_uint(error));
    if (l.has_sum) {
        put(l.offset_sum, __float_as_uint(static_cast<float>(binary_sum)));
    }
    if (l.has_raw_norm) {
        put(l.offset_raw_norm, __float_as_uint(raw_norm));
    }
}

// ---- multi-bit base codes (rabitq_bits_per_dim_base 2..8) ----
// Norm of (rotated row - centroid) as NormalizeWithCentroid takes it (kernels/normalize.h:35-83).
__device__ inline float
rabitq_row_norm(const float* y, const float* centroid, uint32_t dim) {
    float norm_sq = 0.0F;
    for (uint32_t d = 0; d < dim; ++d) {
        float t = y[d] - centroid[d];
        norm_sq = t * t + norm_sq;
    }
    return norm_sq < 1e-5F ? 1.0F : sqrtf(norm_sq);
}

// RaBitQuantizer::FastEncodeRaBitQ (rabitq_quantizer.cpp:609-704): a floor grid over [-max|o|, max|o|], then `rounds`
// sweeps of one-level moves per coordinate that raise <o, y>^2 / |y|^2 (y = code - centre).  The sweep is sequential
// per row (every move changes the sums the next coordinate is judged by), so one thread owns a row; all sums are
// doubles in the reference's order.  scalar: n x dim code values; norm_code: n floats.
__global__ void __launch_bounds__(64)
rabitq_fast_encode_kernel(const float* rotated, uint64_t n, uint32_t dim, const float* centroid, uint32_t bits,
                          uint32_t rounds, uint8_t* scalar, float* norm_code) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) {
        return;
    }
    const float* y = rotated + i * dim;
    uint8_t* code = scalar + i * dim;
    const float norm = rabitq_row_norm(y, centroid, dim);
    const uint32_t code_max = (1U << bits) - 1U;
    const double center = 0.5 * static_cast<double>(code_max);
    double max_abs = 0.0;
    for (uint32_t d = 0; d < dim; ++d) {
        const float o = (y[d] - centroid[d]) / norm;
        max_abs = fmax(max_abs, fabs(static_cast<double>(o)));
    }
    if (max_abs <= 0.0) {
        for (uint32_t d = 0; d < dim; ++d) {
            code[d] = static_cast<uint8_t>(code_max / 2U);
        }
        norm_code[i] = 1.0F;
        return;
    }
    const double delta = 2.0 * max_abs / static_cast<double>(code_max + 1U);
    const double inv_delta = 1.0 / delta;
    double ip = 0.0, norm_sqr = 0.0;
    for (uint32_t d = 0; d < dim; ++d) {
        const float o = (y[d] - centroid[d]) / norm;
        const double scaled = (static_cast<double>(o) + max_abs) * inv_delta;
        long long q = static_cast<long long>(floor(scaled));
        q = q < 0 ? 0 : (q > static_cast<long long>(code_max) ? static_cast<long long>(code_max) : q);
        code[d] = static_cast<uint8_t>(q);
        const double centered = static_cast<double>(q) - center;
        ip += static_cast<double>(o) * centered;
        norm_sqr += centered * centered;
    }
    for (uint32_t round = 0; round < rounds; ++round) {
        bool adjusted = false;
        for (uint32_t d = 0; d < dim; ++d) {
            const double o = static_cast<double>((y[d] - centroid[d]) / norm);
            const int cur = code[d];
            const double cur_value = static_cast<double>(cur) - center;
            int best_code = cur;
            double best_ip = ip, best_norm = norm_sqr;
            double best_score = norm_sqr > 0.0 ? ip * ip / norm_sqr : 0.0;
#pragma unroll
            for (int dir = -1; dir <= 1; dir += 2) {
                const int cand = cur + dir;
                if (cand < 0 || cand > static_cast<int>(code_max)) {
                    continue;
                }
                const double cand_ip = ip + static_cast<double>(dir) * o;
                if (cand_ip < 0.0) {
                    continue;
                }
                const double cand_norm = norm_sqr + 2.0 * cur_value * static_cast<double>(dir) + 1.0;
                const double cand_score = cand_norm > 0.0 ? cand_ip * cand_ip / cand_norm : 0.0;
                const double tolerance = 1e-8 * fmax(1.0, fabs(best_score));
                if (cand_score > best_score + tolerance) {
                    best_code = cand;
                    best_ip = cand_ip;
                    best_norm = cand_norm;
                    best_score = cand_score;
                }
            }
            if (best_code != cur) {
                code[d] = static_cast<uint8_t>(best_code);
                ip = best_ip;
                norm_sqr = best_norm;
                adjusted = true;
            }
        }
        if (!adjusted) {
            break;
        }
    }
    norm_sqr = 0.0;
    for (uint32_t d = 0; d < dim; ++d) {
        const double centered = static_cast<double>(code[d]) - center;
        norm_sqr += centered * centered;
    }
    float yn = static_cast<float>(sqrt(norm_sqr));
    if (!isfinite(yn) || yn <= 0.0F) {
        yn = 1.0F;
    }
    norm_code[i] = yn;
}

// RaBitQuantizer::EncodeExtendRaBitQ (rabitq_quantizer.cpp:455-607): the scale t walks upwards, one grid step of one
// coordinate per event, events in (t, coordinate) order -- the reference's priority queue always holds at most one
// pending event per coordinate, so "pop" is the minimum over the coordinates' next event times.  One wave per row:
// the lanes share that minimum search, every lane repeats the running sums (doubles, the reference's order).
// LDS per row: dim doubles (next event), dim ints (grid position), dim floats (o).
__global__ void __launch_bounds__(64)
rabitq_extend_encode_kernel(const float* rotated, uint64_t n, uint32_t dim, const float* centroid, uint32_t bits,
                            uint8_t* scalar, float* norm_code) {
    extern __shared__ double ee_lds[];
    double* next_t = ee_lds;
    int* y2_cur = reinterpret_cast<int*>(next_t + dim);
    float* o = reinterpret_cast<float*>(y2_cur + dim);
    const uint64_t i = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    const float* y = rotated + i * dim;
    uint8_t* code = scalar + i * dim;
    float norm = 0.0F;
    if (lane == 0) {
        norm = rabitq_row_norm(y, centroid, dim);
    }
    norm = __shfl(norm, 0);
    const int y2_max = static_cast<int>((1U << bits) - 1U);
    const double c = 0.5 * static_cast<double>(y2_max);
    const double inf = __builtin_huge_val();
    double max_o = 0.0;
    for (uint32_t d = lane; d < dim; d += kWave) {
        const float v = (y[d] - centroid[d]) / norm;
        o[d] = v;
        max_o = fmax(max_o, fabs(static_cast<double>(v)));
    }
    for (int off = 32; off > 0; off >>= 1) {
        max_o = fmax(max_o, __shfl_xor(max_o, off));
    }
    if (max_o <= 0.0) {
        for (uint32_t d = lane; d < dim; d += kWave) {
            code[d] = static_cast<uint8_t>(y2_max / 2);
        }
        if (lane == 0) {
            norm_code[i] = 1.0F;
        }
        return;
    }
    const double t_end = (static_cast<double>(y2_max) + 2.0) / (2.0 * max_o);
    // Next event time of a coordinate at grid position `pos` (compute_next_t_for_dim, :513-531).
    auto next_event = [&](double oi, int pos) {
        if (fabs(oi) < 1e-3) {
            return inf;
        }
        const int sign = (oi > 0.0) ? +1 : -1;
        const int y2_next = pos + sign * 2;
        if (y2_next < -y2_max || y2_next > +y2_max) {
            return inf;
        }
        double t = static_cast<double>(pos + sign) / (2.0 * oi);
        if (t < 0.0) {
            t = 0.0;
        }
        return t;
    };
    for (uint32_t d = lane; d < dim; d += kWave) {
        const double oi = static_cast<double>(o[d]);
        double t0 = inf;
        if (oi != 0.0) {
            t0 = next_event(oi, 0);
            if (!(t0 <= t_end)) {
                t0 = inf;
            }
        }
        next_t[d] = t0;
        y2_cur[d] = 0;
    }
    wave_lds_fence();
    double ip_y2_o = 0.0, norm_y2 = 0.0;
    double best_ip = 1e-12, best_t = 0.0;
    // Every pass retires one event; a coordinate has at most 2^(bits - 1) of them, so the walk ends.
    const uint64_t max_events = static_cast<uint64_t>(dim) << bits;
    for (uint64_t ev = 0; ev < max_events; ++ev) {
        double bt = inf;
        uint32_t bi = 0xFFFFFFFFU;
        for (uint32_t d = lane; d < dim; d += kWave) {
            const double t = next_t[d];
            if (t < bt) {
                bt = t;
                bi = d;
            }
        }
        for (int off = 32; off > 0; off >>= 1) {
            const double ot = __shfl_xor(bt, off);
            const uint32_t oi = __shfl_xor(bi, off);
            if (ot < bt || (ot == bt && oi < bi)) {
                bt = ot;
                bi = oi;
            }
        }
        if (bi == 0xFFFFFFFFU || !(bt < t_end)) {
            break;
        }
        const double cur_t = bt;
        const uint32_t k = bi;
        const double ok = static_cast<double>(o[k]);
        const int sign = (o[k] > 0.0F) ? +1 : -1;
        const int y2_old = y2_cur[k];
        const int y2_new = y2_old + sign * 2;
        wave_lds_fence();
        if (y2_new < -y2_max || y2_new > +y2_max) {
            if (lane == 0) {
                next_t[k] = inf;
            }
            wave_lds_fence();
            continue;
        }
        ip_y2_o += (static_cast<double>(y2_new) - static_cast<double>(y2_old)) * ok;
        norm_y2 += static_cast<double>(y2_new) * static_cast<double>(y2_new) -
                   static_cast<double>(y2_old) * static_cast<double>(y2_old);
        const double cur_ip = (norm_y2 > 0.0) ? (ip_y2_o / sqrt(norm_y2)) : 0.0;
        if (cur_ip > best_ip) {
            best_ip = cur_ip;
            best_t = cur_t;
        }
        double t_next = next_event(ok, y2_new);
        if (t_next <= cur_t) {
            t_next = __longlong_as_double(__double_as_longlong(cur_t) + 1);  // nextafter(cur_t, +inf), cur_t >= 0
        }
        if (lane == 0) {
            y2_cur[k] = y2_new;
            next_t[k] = (t_next < t_end) ? t_next : inf;  // a finite time below the end, else no further event
        }
        wave_lds_fence();
    }
    double sum_y2 = 0.0;  // a sum of k + 0.25 terms: exact in any order
    for (uint32_t d = lane; d < dim; d += kWave) {
        const double val = 2.0 * best_t * static_cast<double>(o[d]);
        const double shifted = val + ((val >= 0) ? 1e-12 : -1e-12);
        long long r = llround(shifted);
        int ri = r < -y2_max ? -y2_max : (r > y2_max ? y2_max : static_cast<int>(r));
        if ((ri & 1) != (y2_max & 1)) {
            const int step = (shifted >= 0.0) ? +1 : -1;
            int cand = ri + step;
            if (cand < -y2_max || cand > y2_max) {
                cand = ri - step;
            }
            ri = cand < -y2_max ? -y2_max : (cand > y2_max ? y2_max : cand);
        }
        int u = (ri + y2_max) / 2;
        u = u < 0 ? 0 : (u > y2_max ? y2_max : u);
        code[d] = static_cast<uint8_t>(u);
        const double yy = static_cast<double>(u) - c;
        sum_y2 += yy * yy;
    }
    for (int off = 32; off > 0; off >>= 1) {
        sum_y2 += __shfl_xor(sum_y2, off);
    }
    if (lane == 0) {
        float yn = static_cast<float>(sqrt(sum_y2));
        if (!isfinite(yn) || yn <= 0.0F) {
            yn = 1.0F;
        }
        norm_code[i] = yn;
    }
}

// Rest of the multi-bit branch of RaBitQuantizer::EncodeOneInternal (rabitq_quantizer.cpp:789-809, 852-855): bit planes
// (PackIntoPlanes, :431-453: plane b holds bit b of every dimension), |code - centre|, the norms, and error =
// ip_obar_q(<o, code>, sum o, |code - centre|) with both sums as running floats in element order.  One thread per row.
__global__ void __launch_bounds__(64)
rabitq_multibit_finish_kernel(const float* raw, const float* rotated, uint64_t n, uint32_t dim, const float* centroid,
                              int metric, int bits_word, const uint8_t* scalar, const float* norm_code,
                              uint8_t* codes) {
    const uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= n) {
        return;
    }
    const RabitqLayout l = rabitq_layout(dim, metric, bits_word);
    const float* y = rotated + i * dim;
    const uint8_t* sc = scalar + i * dim;
    uint8_t* c = codes + i * l.code_size;
    float raw_norm = 0.0F;
    if (l.has_raw_norm) {
        const float* x = raw + i * dim;
        for (uint32_t d = 0; d < dim; ++d) {
            raw_norm += x[d] * x[d];
        }
    }
    raw_norm = sqrtf(raw_norm);
    const float norm = rabitq_row_norm(y, centroid, dim);
    const uint32_t plane_bytes = (dim + 7) / 8;
    float query_sum = 0.0F, scalar_ip = 0.0F;
    for (uint32_t b = 0; b < plane_bytes; ++b) {
        uint32_t plane[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        for (uint32_t e = 0; e < 8; ++e) {
            const uint32_t d = b * 8 + e;
            if (d >= dim) {
                break;
            }
            const float nd = (y[d] - centroid[d]) / norm;
            const uint32_t v = sc[d];
            query_sum += nd;
            scalar_ip += static_cast<float>(v) * nd;
#pragma unroll
            for (uint32_t p = 0; p < 8; ++p) {
                plane[p] |= ((v >> p) & 1U) << e;
            }
        }
#pragma unroll
        for (uint32_t p = 0; p < 8; ++p) {
            if (p < l.base_bits) {
                c[p * plane_bytes + b] = static_cast<uint8_t>(plane[p]);
            }
        }
    }
    for (uint32_t b = l.code_bytes; b < l.offset_norm_code; ++b) {
        c[b] = 0;
    }
    const float yn = norm_code[i];
    // ip_obar_q (rabitq_quantizer.cpp:256-267)
    float error = 0.0F;
    if (yn > 0.0F) {
        error = scalar_ip - 0.5F * static_cast<float>((1U << l.base_bits) - 1U) * query_sum;
        error /= yn;
    }
    store_f32(c + l.offset_norm_code, yn);
    store_f32(c + l.offset_norm, norm);
    store_f32(c + l.offset_error, error);
    if (l.has_raw_norm) {
        store_f32(c + l.offset_raw_norm, raw_norm);
    }
}

// Second half of RaBitQuantizer::ProcessQueryImpl (rabitq_quantizer.cpp:2130-2217) with EncodeSQ and
// ReOrderSQ (:2049-2088) for queries already rotated.  One thread per query.
__global__ void __launch_bounds__(64)
rabitq_finish_query_kernel(const float* raw, const float* rotated, uint64_t nq, uint32_t dim, const float* centroid,
                           int metric, int query_bits, uint8_t* qcodes) {
    uint64_t i = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i >= nq) {
        return;
    }
    RabitqLayout l = rabitq_layout(dim, metric, query_bits);
    const float* y = rotated + i * dim;
    uint8_t* qc = qcodes + i * l.query_code_size;
    float raw_norm = 0.0F;
    if (l.has_raw_norm) {
        const float* x = raw + i * dim;
        for (uint32_t d = 0; d < dim; ++d) {
            raw_norm += x[d] * x[d];
        }
    }
    raw_norm = sqrtf(raw_norm);
    float norm_sq = 0.0F;
    for (uint32_t d = 0; d < dim; ++d) {
        float t = y[d] - centroid[d];
        norm_sq = t * t + norm_sq;
    }
    float norm = norm_sq < 1e-5F ? 1.0F : sqrtf(norm_sq);
    if (l.base_bits != 1) {
        float sum = 0.0F;
        for (uint32_t d = 0; d < dim; ++d) {
            sum += (y[d] - centroid[d]) / norm;
        }
        store_f32(qc + l.q_offset_sum, sum);
    }
    if ((query_bits & 255) == 4) {
        float lb = FLT_MAX, ub = -FLT_MAX;
        for (uint32_t d = 0; d < dim; ++d) {
            float v = (y[d] - centroid[d]) / norm;
            if (v < lb) {
                lb = v;
            }
            if (v > ub) {
                ub = v;
            }
        }
        float delta = (ub - lb) / 15;
        float inv_delta = fabsf(delta) < 1e-5F ? 0.0F : 1.0F / delta;
        float qsum = 0.0F;
        for (uint32_t b = 0; b < l.plane_bytes; ++b) {
            uint32_t plane[4] = {0, 0, 0, 0};
            for (uint32_t e = 0; e < 8; ++e) {
                uint32_t d = b * 8 + e;
                if (d >= dim) {
                    break;
                }
                float v = (y[d] - centroid[d]) / norm;
                float val = roundf((v - lb) * inv_delta);
                uint32_t q = static_cast<uint8_t>(val);
                qsum += static_cast<float>(val);
                for (uint32_t p = 0; p < 4; ++p) {
                    plane[p] |= ((q >> p) & 1U) << e;
                }
            }
            for (uint32_t p = 0; p < 4; ++p) {
                qc[p * l.plane_bytes + b] = static_cast<uint8_t>(plane[p]);
            }
        }
        store_f32(qc + l.q_offset_lb, lb);
        store_f32(qc + l.q_offset_delta, delta);
        store_f32(qc + l.q_offset_sum, qsum);
    } else {
        for (uint32_t d = 0; d < dim; ++d) {
            store_f32(qc + 4 * d, (y[d] - centroid[d]) / norm);
        }
    }
    store_f32(qc + l.q_offset_norm, norm);
    if (l.has_raw_norm) {
        store_f32(qc + l.q_offset_raw_norm, raw_norm);
    }
}

// The same, one wave per query: the loads are coalesced and everything but the two sums whose order matters (the
// squared norms, added dimension by dimension like the reference does) is spread over the lanes.  The sum of the
// quantised values is a sum of small integers, exact in any order.  LDS: dim floats, twice that with a raw norm.
__global__ void __launch_bounds__(64)
rabitq_finish_query_wave_kernel(const float* raw, const float* rotated, uint64_t nq, uint32_t dim, const float* centroid,
                                int metric, int query_bits, uint8_t* qcodes) {
    extern __shared__ float fq_lds[];
    const uint64_t i = blockIdx.x;
    const uint32_t lane = threadIdx.x;
    RabitqLayout l = rabitq_layout(dim, metric, query_bits);
    const float* y = rotated + i * dim;
    uint8_t* qc = qcodes + i * l.query_code_size;
    float* t = fq_lds;        // y - centroid
    float* xx = fq_lds + dim;  // squares of the raw query
    for (uint32_t d = lane; d < dim; d += kWave) {
        t[d] = y[d] - centroid[d];
        if (l.has_raw_norm) {
            const float x = raw[i * dim + d];
            xx[d] = x * x;
        }
    }
    wave_lds_fence();
    float raw_norm = 0.0F, norm_sq = 0.0F;
    if (lane == 0) {
        for (uint32_t d = 0; d < dim; ++d) {
            const float v = t[d];
            norm_sq = v * v + norm_sq;
            if (l.has_raw_norm) {
                raw_norm += xx[d];
            }
        }
    }
    raw_norm = sqrtf(__shfl(raw_norm, 0));
    norm_sq = __shfl(norm_sq, 0);
    const float norm = norm_sq < 1e-5F ? 1.0F : sqrtf(norm_sq);
    if (l.base_bits != 1 && lane == 0) {
        float sum = 0.0F;  // in element order, like the reference (rabitq_quantizer.cpp:2199-2205)
        for (uint32_t d = 0; d < dim; ++d) {
            sum += t[d] / norm;
        }
        store_f32(qc + l.q_offset_sum, sum);
    }
    if ((query_bits & 255) == 4) {
        float lb = FLT_MAX, ub = -FLT_MAX;
        for (uint32_t d = lane; d < dim; d += kWave) {
            const float v = t[d] / norm;
            if (v < lb) {
                lb = v;
            }
            if (v > ub) {
                ub = v;
            }
        }
        for (int off = 32; off > 0; off >>= 1) {
            const float ol = __shfl_xor(lb, off), ou = __shfl_xor(ub, off);
            if (ol < lb) {
                lb = ol;
            }
            if (ou > ub) {
                ub = ou;
            }
        }
        const float delta = (ub - lb) / 15;
        const float inv_delta = fabsf(delta) < 1e-5F ? 0.0F : 1.0F / delta;
        float qsum = 0.0F;
        for (uint32_t b = lane; b < l.plane_bytes; b += kWave) {
            uint32_t plane[4] = {0, 0, 0, 0};
            for (uint32_t e = 0; e < 8; ++e) {
                const uint32_t d = b * 8 + e;
                if (d >= dim) {
                    break;
                }
                const float v = t[d] / norm;
                const float val = roundf((v - lb) * inv_delta);
                const uint32_t q = static_cast<uint8_t>(val);
                qsum += static_cast<float>(val);
                for (uint32_t p = 0; p < 4; ++p) {
                    plane[p] |= ((q >> p) & 1U) << e;
                }
            }
            for (uint32_t p = 0; p < 4; ++p) {
                qc[p * l.plane_bytes + b] = static_cast<uint8_t>(plane[p]);
            }
        }
        for (int off = 32; off > 0; off >>= 1) {
            qsum += __shfl_xor(qsum, off);
        }
        if (lane == 0) {
            store_f32(qc + l.q_offset_lb, lb);
            store_f32(qc + l.q_offset_delta, delta);
            store_f32(qc + l.q_offset_sum, qsum);
        }
    } else {
        for (uint32_t d = lane; d < dim; d += kWave) {
            store_f32(qc + 4 * d, t[d] / norm);
        }
    }
    if (lane == 0) {
        store_f32(qc + l.q_offset_norm, norm);
        if (l.has_raw_norm) {
            store_f32(qc + l.q_offset_raw_norm, raw_norm);
        }
    }
}

int
squ_encode_launch(const float* x, uint64_t n, uint32_t dim, int bits, int metric, const float* bounds, uint8_t* codes,
                  hipStream_t st, float* norm_scratch) {
    if (n == 0) {
        return 0;
    }
    int kind = bits == 4 ? VSAG_AMD_KIND_SQ4_UNIFORM : VSAG_AMD_KIND_SQ8_UNIFORM;
    uint32_t code_size = static_cast<uint32_t>(vsag_amd_code_size(kind, metric, dim, 0));
    uint32_t payload = bits == 4 ? (dim + 1) / 2 : dim;
    bool norm = metric == VSAG_AMD_METRIC_L2 || (bits == 4 && metric == VSAG_AMD_METRIC_COSINE);
    uint32_t align = norm ? 8 : 4;
    uint32_t off = static_cast<uint32_t>(round_up(payload, align));
    uint32_t off_norm = off;
    uint32_t off_sum = off + (norm ? 8 : 0);
    uint32_t off_codes_sum = off_sum + align;
    if (n <= kRowEncodeMaxRows && dim <= kRowEncodeMaxDim) {
        const uint32_t dim_pad = static_cast<uint32_t>(round_up(dim, 32));
        const dim3 grid(static_cast<uint32_t>(div_up(n, 4)));
        auto kernel = bits == 4 ? squ_encode_row_kernel<4> : squ_encode_row_kernel<8>;
        hipLaunchKernelGGL(kernel, grid, dim3(256), 4ull * dim_pad * 4, st, x, n, dim, dim_pad, metric, bounds, code_size,
                           payload, off_norm, off_sum, off_codes_sum, codes);
        VA_HIP(hipGetLastError());
        return 0;
    }
    // Cosine needs a float per row; a caller that must not allocate brings them (norm_scratch, n floats).
    float* norms = nullptr;
    if (metric == VSAG_AMD_METRIC_COSINE) {
        norms = norm_scratch;
        if (norms == nullptr) {
            VA_HIP(hipMallocAsync(reinterpret_cast<void**>(&norms), n * 4, st));
        }
        launch_row_norms(x, n, dim, norms, st);
    }
    const dim3 grid(static_cast<uint32_t>(div_up(n, 4 * kWave)));
    if (bits == 4) {
        hipLaunchKernelGGL(squ_encode_kernel<4>, grid, dim3(256), 0, st, x, n, dim, metric, bounds, norms, code_size,
                           payload, off_norm, off_sum, off_codes_sum, codes);
    } else {
        hipLaunchKernelGGL(squ_encode_kernel<8>, grid, dim3(256), 0, st, x, n, dim, metric, bounds, norms, code_size,
                           payload, off_norm, off_sum, off_codes_sum, codes);
    }
    VA_HIP(hipGetLastError());
    if (norms != nullptr && norms != norm_scratch) {
        VA_HIP(hipFreeAsync(norms, st));
    }
    return 0;
}

// Rotates rows in slabs so that the temporary stays bounded, then runs `finish` on each slab.  The temporary
// (min(n, kRotateSlabRows) x dim floats) is `scratch` when the caller brings one, else allocated on the stream.
template <typename Finish>
static int
rabitq_rotate_slabs(const float* x, uint64_t n, uint32_t dim, const float* rot, hipStream_t st, float* scratch,
                    Finish finish) {
    const uint64_t slab = kRotateSlabRows;
    uint64_t rows = n < slab ? n : slab;
    float* tmp = scratch;
    if (tmp == nullptr) {
        VA_HIP(hipMallocAsync(reinterpret_cast<void**>(&tmp), rows * dim * 4, st));
    }
    int rc = 0;
    for (uint64_t s = 0; s < n && rc == 0; s += slab) {
        uint64_t m = n - s < slab ? n - s : slab;
        rc = gemm_nt_seq(x + s * dim, rot, tmp, m, dim, dim, st);
        if (rc == 0) {
            rc = finish(s, m, tmp);
        }
    }
    if (tmp != scratch) {
        hipError_t e = hipFreeAsync(tmp, st);
        if (rc == 0 && e != hipSuccess) {
            return fail(VSAG_AMD_INTERNAL_ERROR, "hipFreeAsync failed: %s", hipGetErrorString(e));
        }
    }
    return rc;
}

int
rabitq_process_query_launch(const float* q, uint64_t nq, uint32_t dim, const float* rot, const float* centroid,
                            int metric, int query_bits, uint8_t* qcodes, hipStream_t st, float* scratch) {
    if (nq == 0) {
        return 0;
    }
    uint64_t qsize = rabitq_query_code_size(dim, metric, query_bits);
    return rabitq_rotate_slabs(q, nq, dim, rot, st, scratch, [&](uint64_t s, uint64_t m, const float* rotated) {
        const size_t lds = static_cast<size_t>(dim) * 4 * (rabitq_layout(dim, metric, query_bits).has_raw_norm ? 2 : 1);
        if (lds <= 48 * 1024) {
            hipLaunchKernelGGL(rabitq_finish_query_wave_kernel, dim3(static_cast<uint32_t>(m)), dim3(64), lds, st,
                               q + s * dim, rotated, m, dim, centroid, metric, query_bits, qcodes + s * qsize);
        } else {
            hipLaunchKernelGGL(rabitq_finish_query_kernel, dim3(static_cast<uint32_t>(div_up(m, 64))), dim3(64), 0, st,
                               q + s * dim, rotated, m, dim, centroid, metric, query_bits, qcodes + s * qsize);
        }
        VA_HIP(hipGetLastError());
        return 0;
    });
}

// ------------------------------------------------------------------ scalar-quantization trainer
// Sample gather (scalar_quantization_trainer.cpp:125-146): row j of the sample is row (j * step) % n,
// written transposed (sample_t[d][j]) so that the per-dimension selection reads contiguously.  A wave per 64 sample rows,
// turned round in LDS: runs of 128 bytes in, of 256 bytes out (100 000 x 128: 128 us with scattered stores, 24 us).
__global__ void __launch_bounds__(256)
sq_sample_kernel(const float* x, uint64_t n, uint32_t dim, uint64_t step, uint64_t sample_count, const float* norms,
                 float* sample_t) {
    __shared__ RowTile tiles[4];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t j0 = (static_cast<uint64_t>(blockIdx.x) * 4 + wave) * kWave;
    if (j0 >= sample_count) {
        return;
    }
    RowTile& t = tiles[wave];
    const bool live = j0 + lane < sample_count;
    // The source rows of the wave's samples, one per lane, handed round by shuffles (a 64-bit modulo each).
    const uint64_t mine = live ? (j0 + lane) * step % n : 0;
    const uint32_t mine_lo = static_cast<uint32_t>(mine), mine_hi = static_cast<uint32_t>(mine >> 32);
    const float norm = norms != nullptr ? norms[mine] : 1.0F;
    for_row_chunks(
        t, dim, lane,
        [&](uint32_t r) {
            const uint64_t idx = (static_cast<uint64_t>(__shfl(mine_hi, static_cast<int>(r))) << 32) |
                                 __shfl(mine_lo, static_cast<int>(r));
            return x + idx * dim;
        },
        [&](uint32_t d0, uint32_t m) {
            for (uint32_t e = 0; e < m; ++e) {
                const float v = t.v[lane][e];
                if (live) {
                    sample_t[static_cast<uint64_t>(d0 + e) * sample_count + j0 + lane] = norms != nullptr ? v / norm : v;
                }
            }
        });
}

// f(value) for every value of a column, by all threads of the workgroup: eight loads go out before the first value is
// looked at (a load at a time, the workgroup waits for memory a hundred times per pass).
template <typename F>
__device__ inline void
for_column(const float* vals, uint64_t count, F f) {
    for (uint64_t i0 = threadIdx.x; i0 < count; i0 += 8ULL * blockDim.x) {
        float v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            const uint64_t i = i0 + u * blockDim.x;
            v[u] = vals[i < count ? i : count - 1];
        }
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
            if (i0 + u * blockDim.x < count) {
                f(v[u]);
            }
        }
    }
}

// The values of a column, thread t of 1024 holding t, t + 1024, ...: REGS of them in registers, or none (0), where they are
// read again for every pass over them.
constexpr uint32_t kBoundThreads = 1024;

template <uint32_t REGS>
struct ColumnValues {
    const float* vals;
    uint64_t count;
    float v[REGS > 0 ? REGS : 1];

    __device__ inline void
    load() {
        if constexpr (REGS > 0) {
            const uint32_t end = static_cast<uint32_t>(count);
#pragma unroll
            for (uint32_t u0 = 0; u0 < REGS; u0 += 16) {
                if (u0 == 0 || u0 * kBoundThreads < end) {  // (the same for all threads)
#pragma unroll
                    for (uint32_t u = u0; u < u0 + 16 && u < REGS; ++u) {
                        const uint32_t i = threadIdx.x + u * kBoundThreads;
                        v[u] = vals[i < end ? i : end - 1];
                    }
                }
            }
        }
    }

    template <typename F>
    __device__ inline void
    each(F f) {
        if constexpr (REGS > 0) {
            uint32_t end = static_cast<uint32_t>(count);
            asm volatile("" : "+s"(end));
#pragma unroll
            for (uint32_t u = 0; u < REGS; ++u) {
                // (opaque to the compiler, which would keep a mask and a key of every value from one pass to the next: more
                // than there are registers)
                asm volatile("" : "+v"(v[u]));
                if (threadIdx.x + u * kBoundThreads < end) {
                    f(v[u]);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            for_column(vals, count, f);
        }
    }
};

constexpr uint32_t kBins = 1024;
constexpr uint32_t kFewKeys = 2048;

struct BoundScratch {
    uint32_t hist[kBins];
    uint32_t keys[2][kFewKeys];
    uint32_t fill[2];
    uint32_t bin, before, answer, lo, hi;
};

// Which bin of sc.hist holds rank `kth` and how many keys lie before it (sc.bin, sc.before); one wave does it.
__device__ inline void
find_bin(BoundScratch& sc, uint64_t kth) {
    if (threadIdx.x < kWave) {
        const uint32_t lane = threadIdx.x;
        uint32_t sum = 0;
        for (uint32_t i = 0; i < kBins / kWave; ++i) {
            sum += sc.hist[lane * (kBins / kWave) + i];
        }
        uint32_t incl = sum;
        for (int off = 1; off < kWave; off <<= 1) {
            const uint32_t o = __shfl_up(incl, off);
            incl += static_cast<int>(lane) >= off ? o : 0U;
        }
        uint32_t before = incl - sum;
        if (before < kth && kth <= incl) {
            uint32_t b = lane * (kBins / kWave);
            while (before + sc.hist[b] < kth) {
                before += sc.hist[b];
                ++b;
            }
            sc.bin = b;
            sc.before = before;
        }
    }
    __syncthreads();
}

// The kth smallest (1-based) of sc.keys[s][0, sc.fill[s]), every key ranked against all.
__device__ inline uint32_t
kth_of_few(BoundScratch& sc, int s, uint64_t kth) {
    const uint32_t m = sc.fill[s];
    for (uint32_t i = threadIdx.x; i < m; i += blockDim.x) {
        const uint32_t mine = sc.keys[s][i];
        uint32_t less = 0, equal = 0;
        for (uint32_t j = 0; j < m; ++j) {
            const uint32_t o = sc.keys[s][j];
            less += o < mine ? 1U : 0U;
            equal += o == mine ? 1U : 0U;
        }
        if (less < kth && kth <= less + equal) {
            sc.answer = mine;  // equal keys write the same value
        }
    }
    __syncthreads();
    const uint32_t key = sc.answer;
    __syncthreads();
    return key;
}

// The kth smallest (1-based) among the `population` values of a column whose ordered keys lie in [base, last]: round by
// round the interval is cut into bins of the keys and the one that holds the rank is kept, until few keys are left (or one).
__device__ inline uint32_t
kth_key_in(const float* vals, uint64_t count, uint32_t base, uint32_t last, uint64_t population, uint64_t kth,
           BoundScratch& sc) {
    while (base < last) {
        if (population <= kFewKeys) {
            if (threadIdx.x == 0) {
                sc.fill[0] = 0;
            }
            __syncthreads();
            for_column(vals, count, [&](float v) {
                const uint32_t key = float_to_ordered(v);
                if (key >= base && key <= last) {
                    const uint32_t at = atomicAdd(&sc.fill[0], 1U);
                    if (at < kFewKeys) {
                        sc.keys[0][at] = key;
                    }
                }
            });
            __syncthreads();
            return kth_of_few(sc, 0, kth);
        }
        const uint32_t bits = 32 - __clz(last - base);
        const uint32_t shift = bits > 10 ? bits - 10 : 0;
        for (uint32_t i = threadIdx.x; i < kBins; i += blockDim.x) {
            sc.hist[i] = 0;
        }
        __syncthreads();
        for_column(vals, count, [&](float v) {
            const uint32_t key = float_to_ordered(v);
            if (key >= base && key <= last) {
                atomicAdd(&sc.hist[(key - base) >> shift], 1U);
            }
        });
        __syncthreads();
        find_bin(sc, kth);
        base += sc.bin << shift;
        const uint32_t width = (1U << shift) - 1U;
        last = last - base < width ? last : base + width;
        kth -= sc.before;
        population = sc.hist[sc.bin];
        __syncthreads();
    }
    return base;
}

// trunc_bound_train / classic_train (scalar_quantization_trainer.cpp:72-122): the bounded heaps keep the
// ignore_count largest and smallest sample values of a dimension; their tops are the ignore_count-th
// largest and smallest.  CLASSIC is the same with ignore_count = 1.  Writes lower bound and diff.
//
// One workgroup per dimension.  The range of the column's values is cut into 1024 equal bins -- any map that keeps the order
// serves, and bins of the float's bits put nearly all values of a column into a few of them, where the atomics of a wave
// wait for each other --; that one histogram places both order statistics in bins of a few hundred values, which are ranked
// in LDS: three passes over the column, whose values stay in registers where 1024 threads hold them (up to REGS each: 98
// for the default sample of 100 000, of which six spill) -- a workgroup per column leaves every second compute unit idle at
// 128 dimensions, and the other half waited for the same 400 KB three times.  100 000 x 128: 980 us with eight reads by 256
// threads, 50 us with three reads by 1024, 37 us now.  REGS that a sample leaves unused cost as much as used ones, so there is a
// form for every few thousand rows (training on 33 000 x 960 with 64 of them for 33: 175 us, three reads 166, with 48 165; 3000 x
// 960 with 32 for 3: 132, three reads 123, with 8 120).
// A column with values beyond any such range (NaN, infinities) takes bins of the ordered bits.
template <uint32_t REGS>
__global__ void __launch_bounds__(kBoundThreads)
sq_bounds_kernel(const float* sample_t, uint64_t count, uint64_t ignore_count, float* lb, float* diff, float* upper_out,
                 float* lower_out) {
    __shared__ BoundScratch sc;
    const uint32_t d = blockIdx.x;
    const float* col = sample_t + static_cast<uint64_t>(d) * count;
    const uint64_t k = ignore_count < count ? ignore_count : count;
    ColumnValues<REGS> column{col, count, {}};
    column.load();
    // Smallest and largest ordered bits of the values of `values` that `in` admits, in sc.lo / sc.hi.
    auto range_of = [&](auto&& values, auto in) {
        if (threadIdx.x == 0) {
            sc.lo = 0xFFFFFFFFU;
            sc.hi = 0;
        }
        __syncthreads();
        uint32_t lo = 0xFFFFFFFFU, hi = 0;
        values.each([&](float v) {
            if (in(v)) {
                const uint32_t key = float_to_ordered(v);
                lo = key < lo ? key : lo;
                hi = key > hi ? key : hi;
            }
        });
        lo = wave_min_u32(lo);
        hi = wave_max_u32(hi);
        if ((threadIdx.x & 63U) == 0) {
            atomicMin(&sc.lo, lo);
            atomicMax(&sc.hi, hi);
        }
        __syncthreads();
    };
    for (uint32_t i = threadIdx.x; i < kBins; i += blockDim.x) {
        sc.hist[i] = 0;
    }
    if (threadIdx.x < 2) {
        sc.fill[threadIdx.x] = 0;
    }
    range_of(column, [](float) { return true; });
    const uint32_t kmin = sc.lo, kmax = sc.hi;
    const float vmin = ordered_to_float(kmin), vmax = ordered_to_float(kmax);
    const float scale = static_cast<float>(kBins) / (vmax - vmin);
    const bool linear = vmax - vmin < 1.0e30F && scale < 1.0e30F;  // neither with NaN, an infinity or a range of zero
    const uint32_t spread = kmax - kmin;
    const uint32_t bits = spread == 0 ? 0 : 32 - __clz(spread);
    const uint32_t shift = bits > 10 ? bits - 10 : 0;
    auto bin_of = [&](float v) {
        if (linear) {
            const float f = (v - vmin) * scale;
            return f < static_cast<float>(kBins - 1) ? static_cast<uint32_t>(f) : kBins - 1;
        }
        return (float_to_ordered(v) - kmin) >> shift;
    };
    column.each([&](float v) { atomicAdd(&sc.hist[bin_of(v)], 1U); });
    __syncthreads();
    uint32_t bin[2], population[2];
    uint64_t rank[2] = {k, count - k + 1};
    for (int s = 0; s < 2; ++s) {
        find_bin(sc, rank[s]);
        bin[s] = sc.bin;
        rank[s] -= sc.before;
        population[s] = sc.hist[sc.bin];
        __syncthreads();
    }
    if (population[0] <= kFewKeys || population[1] <= kFewKeys) {
        column.each([&](float v) {
            const uint32_t b = bin_of(v);
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (b == bin[s] && population[s] <= kFewKeys) {
                    sc.keys[s][atomicAdd(&sc.fill[s], 1U)] = float_to_ordered(v);
                }
            }
        });
        __syncthreads();
    }
    float bound[2];
    for (int s = 0; s < 2; ++s) {  // (kth_key_in collects in list 0, which is done with when bin 1 is looked at)
        uint32_t key;
        if (population[s] <= kFewKeys) {
            key = kth_of_few(sc, s, rank[s]);
        } else {
            const uint32_t want = bin[s];
            range_of(ColumnValues<0>{col, count, {}}, [&](float v) { return bin_of(v) == want; });
            const uint32_t from = sc.lo, to = sc.hi;
            __syncthreads();
            key = kth_key_in(col, count, from, to, population[s], rank[s], sc);
            __syncthreads();
        }
        bound[s] = ordered_to_float(key);
    }
    const float lower = bound[0], upper = bound[1];
    if (threadIdx.x == 0) {
        if (lb != nullptr) {
            lb[d] = lower;
            diff[d] = upper - lower;
        }
        if (upper_out != nullptr) {
            upper_out[d] = upper;
            lower_out[d] = lower;
        }
    }
}

// TrainUniform (scalar_quantization_trainer.cpp:47-70): CLASSIC -> max of uppers / min of lowers;
// TRUNC_BOUND -> min of uppers / max of lowers, swapped when inverted.  out = {lb, diff}.
__global__ void __launch_bounds__(64)
sq_uniform_reduce_kernel(const float* upper, const float* lower, uint32_t dim, int mode, float* out) {
    const uint32_t lane = threadIdx.x;
    float ub = upper[0], lb = lower[0];
    const bool classic = mode == VSAG_AMD_SQ_TRAIN_CLASSIC;
    for (uint32_t d = lane; d < dim; d += kWave) {
        ub = classic ? fmaxf(ub, upper[d]) : fminf(ub, upper[d]);
        lb = classic ? fminf(lb, lower[d]) : fmaxf(lb, lower[d]);
    }
    for (int off = 32; off > 0; off >>= 1) {
        const float u = __shfl_xor(ub, off), l = __shfl_xor(lb, off);
        ub = classic ? fmaxf(ub, u) : fminf(ub, u);
        lb = classic ? fminf(lb, l) : fmaxf(lb, l);
    }
    if (lane != 0) {
        return;
    }
    if (!classic && lb > ub) {
        float t = lb;
        lb = ub;
        ub = t;
    }
    out[0] = lb;
    out[1] = ub - lb;
}

struct TrainPlan {
    uint64_t sample_count, step, ignore_count;
};

static TrainPlan
train_plan(uint64_t n, int bits, int mode, float trunc_rate, uint64_t max_sample) {
    TrainPlan p{};
    if (max_sample == 0) {
        max_sample = 100000;
    }
    p.step = 2147483647ULL % n;
    p.sample_count = max_sample;
    if (n <= max_sample) {
        p.step = 1;
        p.sample_count = n;
    }
    if (mode == VSAG_AMD_SQ_TRAIN_CLASSIC) {
        p.ignore_count = 1;
    } else {
        double rate = bits == 4 ? static_cast<double>(trunc_rate) : 0.001;
        auto ic = static_cast<uint64_t>(static_cast<double>(p.sample_count - 1) * rate);
        p.ignore_count = ic < 1 ? 1 : ic;
    }
    return p;
}

static int
sq_train_common(const float* x, uint64_t n, uint32_t dim, int bits, int metric, int mode, float trunc_rate,
                uint64_t max_sample, float* lb, float* diff, float* uniform_out, void* ws, size_t ws_bytes,
                hipStream_t st) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG(x != nullptr && n >= 1, "sq_train needs at least one row");
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    VA_CHECK_ARG(bits == 4 || bits == 8, "bits must be 4 or 8, got %d", bits);
    VA_CHECK_ARG(mode == VSAG_AMD_SQ_TRAIN_CLASSIC || mode == VSAG_AMD_SQ_TRAIN_TRUNC_BOUND, "unknown train mode %d",
                 mode);
    TrainPlan p = train_plan(n, bits, mode, trunc_rate, max_sample);
    Carver c(ws, ws_bytes);
    float* sample_t = c.take<float>(p.sample_count * dim);
    float* norms = c.take<float>(metric == VSAG_AMD_METRIC_COSINE ? n : 0);
    float* upper = c.take<float>(dim);
    float* lower = c.take<float>(dim);
    VA_CHECK_ARG(c.ok(), "workspace too small: need %zu bytes, got %zu", c.used, ws_bytes);
    if (metric == VSAG_AMD_METRIC_COSINE) {
        launch_row_norms(x, n, dim, norms, st);
    } else {
        norms = nullptr;
    }
    hipLaunchKernelGGL(sq_sample_kernel, dim3(static_cast<uint32_t>(div_up(p.sample_count, 4 * kWave))), dim3(256), 0, st,
                       x, n, dim, p.step, p.sample_count, norms, sample_t);
    const uint64_t each = div_up(p.sample_count, kBoundThreads);
    auto bounds = each <= 8 ? sq_bounds_kernel<8> : each <= 16 ? sq_bounds_kernel<16> : each <= 32 ? sq_bounds_kernel<32>
                  : each <= 48 ? sq_bounds_kernel<48> : each <= 64 ? sq_bounds_kernel<64>
                  : each <= 80 ? sq_bounds_kernel<80> : each <= 98 ? sq_bounds_kernel<98> : sq_bounds_kernel<0>;
    hipLaunchKernelGGL(bounds, dim3(dim), dim3(kBoundThreads), 0, st, sample_t, p.sample_count, p.ignore_count, lb, diff,
                       upper, lower);
    if (uniform_out != nullptr) {
        hipLaunchKernelGGL(sq_uniform_reduce_kernel, dim3(1), dim3(64), 0, st, upper, lower, dim, mode, uniform_out);
    }
    VA_HIP(hipGetLastError());
    return 0;
}

}  // namespace vsag_amd

using namespace vsag_amd;

extern "C" size_t
vsag_amd_sq_train_workspace_bytes(uint64_t n, uint32_t dim, uint64_t max_sample) {
    if (n == 0) {
        return 0;
    }
    TrainPlan p = train_plan(n, 8, VSAG_AMD_SQ_TRAIN_TRUNC_BOUND, 0.05F, max_sample);
    return round_up(p.sample_count * dim * 4, 256) + round_up(n * 4, 256) + 2 * round_up(dim * 4ull, 256) + 256;
}

extern "C" int
vsag_amd_sq_train(const float* x_dev, uint64_t n, uint32_t dim, int bits, int metric, int mode, float trunc_rate,
                  uint64_t max_sample, float* lower_bound_dev, float* diff_dev, void* workspace_dev,
                  size_t workspace_bytes, void* stream) {
    VA_CHECK_ARG(lower_bound_dev && diff_dev, "null output");
    return sq_train_common(x_dev, n, dim, bits, metric, mode, trunc_rate, max_sample, lower_bound_dev, diff_dev,
                           nullptr, workspace_dev, workspace_bytes, static_cast<hipStream_t>(stream));
}

extern "C" int
vsag_amd_sq_train_uniform(const float* x_dev, uint64_t n, uint32_t dim, int bits, int metric, int mode,
                          float trunc_rate, uint64_t max_sample, float* out_dev, void* workspace_dev,
                          size_t workspace_bytes, void* stream) {
    VA_CHECK_ARG(out_dev, "null output");
    return sq_train_common(x_dev, n, dim, bits, metric, mode, trunc_rate, max_sample, nullptr, nullptr, out_dev,
                           workspace_dev, workspace_bytes, static_cast<hipStream_t>(stream));
}

extern "C" int
vsag_amd_sq_encode(const float* x_dev, uint64_t n, uint32_t dim, int bits, int metric, const float* lower_bound_dev,
                   const float* diff_dev, uint8_t* codes_dev, void* stream) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG(bits == 4 || bits == 8, "bits must be 4 or 8, got %d", bits);
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    if (n == 0) {
        return 0;
    }
    VA_CHECK_ARG(x_dev && lower_bound_dev && diff_dev && codes_dev, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint32_t code_size = (dim * bits + 7) / 8;
    float* norms = nullptr;
    if (metric == VSAG_AMD_METRIC_COSINE) {
        VA_HIP(hipMallocAsync(reinterpret_cast<void**>(&norms), n * 4, st));
        launch_row_norms(x_dev, n, dim, norms, st);
    }
    const uint64_t total = n * dim;
    const bool flat = (dim * bits) % 8 == 0 && (reinterpret_cast<uintptr_t>(x_dev) & 15U) == 0 &&
                      (reinterpret_cast<uintptr_t>(codes_dev) & 3U) == 0;
    const uint64_t threads = flat ? div_up(total, static_cast<uint64_t>(32 / bits)) : n * code_size;
    VA_CHECK_ARG(div_up(threads, 256) < (1ull << 31), "too many rows for one encode call");
    if (!flat) {
        hipLaunchKernelGGL(sq_encode_bytes_kernel, dim3(static_cast<uint32_t>(div_up(threads, 256))), dim3(256), 0, st, x_dev,
                           n, dim, bits, lower_bound_dev, diff_dev, norms, code_size, codes_dev);
    } else {
        uint32_t block = 0, runs = 0;
        sq_encode_shape(dim, 32U / bits, threads, norms != nullptr, &block, &runs);
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(static_cast<uint32_t>(div_up(threads, static_cast<uint64_t>(block) * runs))),
                               dim3(block), 0, st, x_dev, total, dim, lower_bound_dev, diff_dev, norms, codes_dev);
        };
        const bool vec = (dim & 3U) == 0 && ((reinterpret_cast<uintptr_t>(lower_bound_dev) |
                                              reinterpret_cast<uintptr_t>(diff_dev)) & 15U) == 0;
        auto pick = [&](auto bits_c, auto runs_c) {
            constexpr int kBits = decltype(bits_c)::value, kRuns = decltype(runs_c)::value;
            if (norms != nullptr) {
                launch(vec ? sq_encode_kernel<kBits, true, true, kRuns> : sq_encode_kernel<kBits, true, false, kRuns>);
            } else {
                launch(vec ? sq_encode_kernel<kBits, false, true, kRuns> : sq_encode_kernel<kBits, false, false, kRuns>);
            }
        };
        if (bits == 8) {
            runs == 4 ? pick(std::integral_constant<int, 8>{}, std::integral_constant<int, 4>{})
                      : pick(std::integral_constant<int, 8>{}, std::integral_constant<int, 1>{});
        } else {
            runs == 4 ? pick(std::integral_constant<int, 4>{}, std::integral_constant<int, 4>{})
                      : pick(std::integral_constant<int, 4>{}, std::integral_constant<int, 1>{});
        }
    }
    VA_HIP(hipGetLastError());
    if (norms != nullptr) {
        VA_HIP(hipFreeAsync(norms, st));
    }
    return 0;
}

extern "C" int
vsag_amd_squ_encode(const float* x_dev, uint64_t n, uint32_t dim, int bits, int metric, const float* bounds_dev,
                    uint8_t* codes_dev, void* stream) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG(bits == 4 || bits == 8, "bits must be 4 or 8, got %d", bits);
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    VA_CHECK_ARG(n == 0 || (x_dev && bounds_dev && codes_dev), "null pointer");
    return squ_encode_launch(x_dev, n, dim, bits, metric, bounds_dev, codes_dev, static_cast<hipStream_t>(stream),
                             nullptr);
}

extern "C" int
vsag_amd_rabitq_train(const float* x_dev, uint64_t n, uint32_t dim, const float* rotation_dev, float* centroid_dev,
                      void* stream) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG(x_dev && rotation_dev && centroid_dev && n >= 1, "null pointer or empty data");
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    hipStream_t st = static_cast<hipStream_t>(stream);
    float* mean = nullptr;
    VA_HIP(hipMallocAsync(reinterpret_cast<void**>(&mean), dim * 4, st));
    hipLaunchKernelGGL(column_mean_seq_kernel, dim3((dim + kMeanCols - 1) / kMeanCols), dim3(kMeanLoaders + kWave), 0,
                       st, x_dev, n, dim, mean);
    int rc = gemm_nt_seq(mean, rotation_dev, centroid_dev, 1, dim, dim, st);
    VA_HIP(hipFreeAsync(mean, st));
    return rc;
}

extern "C" int
vsag_amd_rabitq_encode(const float* x_dev, uint64_t n, uint32_t dim, const float* rotation_dev,
                       const float* centroid_dev, int metric, int query_bits, uint8_t* codes_dev, void* stream) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG(query_bits == 4 || query_bits == 32, "query_bits must be 4 or 32, got %d", query_bits);
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    if (n == 0) {
        return 0;
    }
    VA_CHECK_ARG(x_dev && rotation_dev && centroid_dev && codes_dev, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    uint64_t csize = rabitq_code_size(dim, metric, query_bits);
    return rabitq_rotate_slabs(x_dev, n, dim, rotation_dev, st, nullptr, [&](uint64_t s, uint64_t m, const float* rotated) {
        hipLaunchKernelGGL(rabitq_finish_encode_kernel, dim3(static_cast<uint32_t>(div_up(m, 4 * kWave))), dim3(256), 0, st,
                           x_dev + s * dim, rotated, m, dim, centroid_dev, metric, query_bits, codes_dev + s * csize);
        VA_HIP(hipGetLastError());
        return 0;
    });
}

// FhtKacRotator (impl/transform/fht_kac_rotate_transformer.cpp:64-96, rabitq_use_fht) as the dense matrix the rabitq
// entry points take: y = R x with R[i][j] = Transform(e_j)[i].  The rotator is a product of sign flips, Hadamard
// butterflies on a power-of-two block, Kac walks and scalings, all of them row operations on the matrix of the
// transformed basis vectors (one column per basis vector), which starts as the identity.  Host memory on both sides.
extern "C" int
vsag_amd_fht_kac_matrix(const uint8_t* flip, uint32_t dim, float* rotation) {
    VA_CHECK_ARG(flip != nullptr && rotation != nullptr, "null pointer");
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    const size_t d = dim;
    const size_t flip_bytes = (d + 7) / 8;
    size_t block = 1;  // the largest power of two within dim
    while (block * 2 <= d) {
        block *= 2;
    }
    const float scale = 1.0F / std::sqrt(static_cast<float>(block));
    std::fill(rotation, rotation + d * d, 0.0F);
    for (size_t i = 0; i < d; ++i) {
        rotation[i * d + i] = 1.0F;
    }
    auto row = [&](size_t i) { return rotation + i * d; };
    auto flip_rows = [&](int round) {
        const uint8_t* f = flip + static_cast<size_t>(round) * flip_bytes;
        for (size_t i = 0; i < d; ++i) {
            if ((f[i >> 3] >> (i & 7)) & 1) {
                float* r = row(i);
                for (size_t j = 0; j < d; ++j) {
                    r[j] = -r[j];
                }
            }
        }
    };
    auto pair_rows = [&](size_t a, size_t b) {  // (a, b) <- (a + b, a - b)
        float* ra = row(a);
        float* rb = row(b);
        for (size_t j = 0; j < d; ++j) {
            const float x = ra[j], y = rb[j];
            ra[j] = x + y;
            rb[j] = x - y;
        }
    };
    auto scale_rows = [&](size_t first, size_t count, float v) {
        for (size_t i = first; i < first + count; ++i) {
            float* r = row(i);
            for (size_t j = 0; j < d; ++j) {
                r[j] *= v;
            }
        }
    };
    auto hadamard = [&](size_t first) {
        for (size_t step = 1; step < block; step *= 2) {
            for (size_t i = 0; i < block; i += 2 * step) {
                for (size_t j = 0; j < step; ++j) {
                    pair_rows(first + i + j, first + i + j + step);
                }
            }
        }
        scale_rows(first, block, scale);
    };
    auto kac_walk = [&]() {
        const size_t half = d / 2, offset = half + d % 2;
        for (size_t i = 0; i < half; ++i) {
            pair_rows(i, i + offset);
        }
        if (d % 2 != 0) {
            scale_rows(half, 1, std::sqrt(2.0F));
        }
    };
    if (block == d) {
        for (int round = 0; round < 4; ++round) {
            flip_rows(round);
            hadamard(0);
        }
        return 0;
    }
    for (int round = 0; round < 4; round += 2) {
        flip_rows(round);
        hadamard(0);
        kac_walk();
        flip_rows(round + 1);
        hadamard(d - block);
        kac_walk();
    }
    scale_rows(0, d, 0.25F);  // four Kac walks, each of which doubles the squared length
    return 0;
}

// RaBitQuantizer::DecodeOneImpl (rabitq_quantizer.cpp:871-899), 1-bit codes: y = (+-1 / sqrt(d)) * norm + centroid
// per dimension (InverseNormalizeWithCentroid, simd/kernels/normalize.h:88-119), x = R^T y.  A workgroup per code, a
// thread per output dimension, the rows of R summed in order.
__global__ void __launch_bounds__(256)
rabitq_decode_kernel(const uint8_t* codes, uint32_t dim, const float* rot, const float* centroid, uint32_t code_size,
                     uint32_t offset_norm, float* out) {
    const uint64_t i = blockIdx.x;
    const uint8_t* c = codes + i * code_size;
    const float norm = load_f32(c + offset_norm);
    const float inv_sqrt_d = 1.0F / sqrtf(static_cast<float>(dim));
    for (uint32_t j = threadIdx.x; j < dim; j += blockDim.x) {
        float acc = 0.0F;
        for (uint32_t r = 0; r < dim; ++r) {
            const bool bit = ((c[r >> 3] >> (r & 7)) & 1) != 0;
            const float y = (bit ? inv_sqrt_d : -inv_sqrt_d) * norm + centroid[r];
            acc += rot[static_cast<uint64_t>(r) * dim + j] * y;
        }
        out[i * dim + j] = acc;
    }
}

extern "C" int
vsag_amd_rabitq_decode(const uint8_t* codes_dev, uint64_t n, uint32_t dim, const float* rotation_dev,
                       const float* centroid_dev, int metric, int bits_word, float* out_dev, void* stream) {
    VA_TRY(ensure_init());
    const int query_bits = bits_word & 255;
    VA_CHECK_ARG(query_bits == 4 || query_bits == 32, "query_bits must be 4 or 32, got %d", query_bits);
    VA_CHECK_ARG((bits_word >> 8) <= 1, "only 1-bit codes decode (RaBitQuantizer::DecodeOneImpl returns false for the others)");
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    if (n == 0) {
        return 0;
    }
    VA_CHECK_ARG(codes_dev && rotation_dev && centroid_dev && out_dev, "null pointer");
    VA_CHECK_ARG(n < (1ull << 31), "n must be below 2^31");
    const RabitqLayout l = rabitq_layout(dim, metric, query_bits);
    hipLaunchKernelGGL(rabitq_decode_kernel, dim3(static_cast<uint32_t>(n)), dim3(256), 0, static_cast<hipStream_t>(stream),
                       codes_dev, dim, rotation_dev, centroid_dev, l.code_size, l.offset_norm, out_dev);
    VA_HIP(hipGetLastError());
    return 0;
}

extern "C" int
vsag_amd_rabitq_encode_multibit(const float* x_dev, uint64_t n, uint32_t dim, const float* rotation_dev,
                                const float* centroid_dev, int metric, int bits_word, int fast_encode,
                                uint32_t fast_encode_rounds, uint8_t* codes_dev, void* stream) {
    VA_TRY(ensure_init());
    const int base_bits = bits_word >> 8;
    VA_CHECK_ARG((bits_word & 255) == 32, "multi-bit base codes need fp32 queries (query bits 32), got %d", bits_word & 255);
    VA_CHECK_ARG(base_bits >= 2 && base_bits <= 8, "base bits must be in [2, 8], got %d", base_bits);
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    VA_CHECK_ARG(!fast_encode || (fast_encode_rounds >= 1 && fast_encode_rounds <= 32),
                 "fast_encode_rabitq_rounds must be in [1, 32], but got %u", fast_encode_rounds);
    VA_CHECK_ARG(fast_encode || dim <= 3072, "the exhaustive encoder supports at most 3072 dimensions, got %u", dim);
    if (n == 0) {
        return 0;
    }
    VA_CHECK_ARG(x_dev && rotation_dev && centroid_dev && codes_dev, "null pointer");
    hipStream_t st = static_cast<hipStream_t>(stream);
    const uint64_t csize = rabitq_code_size(dim, metric, bits_word);
    const uint64_t rows = n < kRotateSlabRows ? n : kRotateSlabRows;
    uint8_t* scalar = nullptr;
    float* norm_code = nullptr;
    VA_HIP(hipMallocAsync(reinterpret_cast<void**>(&scalar), rows * dim, st));
    hipError_t e = hipMallocAsync(reinterpret_cast<void**>(&norm_code), rows * 4, st);
    if (e != hipSuccess) {
        (void)hipFreeAsync(scalar, st);
        return fail(VSAG_AMD_NO_ENOUGH_MEMORY, "hipMallocAsync failed: %s", hipGetErrorString(e));
    }
    int rc = rabitq_rotate_slabs(x_dev, n, dim, rotation_dev, st, nullptr, [&](uint64_t s, uint64_t m, const float* rotated) {
        if (fast_encode) {
            hipLaunchKernelGGL(rabitq_fast_encode_kernel, dim3(static_cast<uint32_t>(div_up(m, 64))), dim3(64), 0, st,
                               rotated, m, dim, centroid_dev, static_cast<uint32_t>(base_bits), fast_encode_rounds, scalar,
                               norm_code);
        } else {
            const size_t lds = static_cast<size_t>(dim) * 16;
            hipLaunchKernelGGL(rabitq_extend_encode_kernel, dim3(static_cast<uint32_t>(m)), dim3(64), lds, st, rotated, m,
                               dim, centroid_dev, static_cast<uint32_t>(base_bits), scalar, norm_code);
        }
        VA_HIP(hipGetLastError());
        hipLaunchKernelGGL(rabitq_multibit_finish_kernel, dim3(static_cast<uint32_t>(div_up(m, 64))), dim3(64), 0, st,
                           x_dev + s * dim, rotated, m, dim, centroid_dev, metric, bits_word, scalar, norm_code,
                           codes_dev + s * csize);
        VA_HIP(hipGetLastError());
        return 0;
    });
    (void)hipFreeAsync(scalar, st);
    (void)hipFreeAsync(norm_code, st);
    return rc;
}

extern "C" uint64_t
vsag_amd_rabitq_query_code_size(uint32_t dim, int metric, int query_bits) {
    return rabitq_query_code_size(dim, metric, query_bits);
}

extern "C" int
vsag_amd_rabitq_process_query(const float* q_dev, uint64_t nq, uint32_t dim, const float* rotation_dev,
                              const float* centroid_dev, int metric, int query_bits, uint8_t* qcodes_dev,
                              void* stream) {
    VA_TRY(ensure_init());
    VA_CHECK_ARG((query_bits & 255) == 4 || (query_bits & 255) == 32, "query_bits must be 4 or 32, got %d",
                 query_bits & 255);
    VA_CHECK_ARG((query_bits >> 8) == 0 || ((query_bits & 255) == 32 && (query_bits >> 8) <= 8),
                 "multi-bit base codes (%d bits) need fp32 queries and at most 8 bits", query_bits >> 8);
    VA_CHECK_ARG(dim >= 1 && dim <= 65536, "dim must be in [1, 65536], got %u", dim);
    VA_CHECK_ARG(nq == 0 || (q_dev && rotation_dev && centroid_dev && qcodes_dev), "null pointer");
    return rabitq_process_query_launch(q_dev, nq, dim, rotation_dev, centroid_dev, metric, query_bits, qcodes_dev,
                                       static_cast<hipStream_t>(stream), nullptr);
}
