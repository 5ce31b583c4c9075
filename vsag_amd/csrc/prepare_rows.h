// The query rows of the fp32, sq8 and sq4 kinds, as the scans (prepare.hip) and the bf16 pre-selection (prefilter_b16.hip) make
// them.
#pragma once

#include "store.h"

namespace vsag_amd {

// The sum over a workgroup of at most four waves.
__device__ inline float
block_sum(float v, float* red) {
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_down(v, off);
    }
    uint32_t wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
        red[wave] = v;
    }
    __syncthreads();
    float s = 0;
    for (uint32_t i = 0; i < (blockDim.x >> 6); ++i) {
        s += red[i];
    }
    __syncthreads();
    return s;
}

struct FloatQueryArgs {
    const float* q;  // nq x dim
    uint64_t nq;
    uint32_t dim;
    int kind, metric;
    const float* scale;
    const float* lb;
    float* qtab;
    uint32_t qstride;
    float* qmeta;
    uint32_t qmeta_stride;
};

// One workgroup of 256 threads per row; rows at or beyond nq are written as zeros.
// (ProcessQueryImpl of fp32_quantizer.cpp:216-233 and scalar_quantizer.cpp:154-171 keep the query in fp32, normalised for
// cosine; the per-dimension constants are folded in here.)
__device__ inline void
prepare_float_row(const FloatQueryArgs& p, uint64_t row) {
    __shared__ float red[4];
    float* out = p.qtab + row * p.qstride;
    if (row >= p.nq) {
        for (uint32_t d = threadIdx.x; d < p.qstride; d += blockDim.x) {
            out[d] = 0.0F;
        }
        if (threadIdx.x < p.qmeta_stride) {
            p.qmeta[row * p.qmeta_stride + threadIdx.x] = 0.0F;
        }
        return;
    }
    const float* src = p.q + row * p.dim;
    float inv_norm = 1.0F;
    bool cosine = p.metric == VSAG_AMD_METRIC_COSINE;
    if (cosine) {
        float s = 0;
        for (uint32_t d = threadIdx.x; d < p.dim; d += blockDim.x) {
            s += src[d] * src[d];
        }
        s = block_sum(s, red);
        inv_norm = sqrtf(s);
        if (inv_norm == 0.0F) {
            inv_norm = 1.0F;  // DivScalarImpl (src/simd/kernels/scalar_op.h:40-42): a zero norm divides by 1
        }
    }
    float bias = 0;
    for (uint32_t d = threadIdx.x; d < p.qstride; d += blockDim.x) {
        float v = 0.0F;
        if (d < p.dim) {
            float x = cosine ? src[d] / inv_norm : src[d];
            if (p.kind == VSAG_AMD_KIND_FP32) {
                v = x;
            } else if (p.metric == VSAG_AMD_METRIC_L2) {
                v = x - p.lb[d];
            } else {
                v = x * p.scale[d];
                bias += x * p.lb[d];
            }
        }
        out[d] = v;
    }
    if (p.kind != VSAG_AMD_KIND_FP32 && p.metric != VSAG_AMD_METRIC_L2) {
        bias = block_sum(bias, red);
        if (threadIdx.x == 0) {
            p.qmeta[row * p.qmeta_stride] = bias;
        }
    } else if (threadIdx.x < p.qmeta_stride) {
        p.qmeta[row * p.qmeta_stride + threadIdx.x] = 0.0F;
    }
}

inline FloatQueryArgs
float_query_args(const vsag_amd_store* s, const float* queries, uint64_t nq, const QueryLayout& ql, uint32_t* qtab, float* qmeta) {
    return {queries, nq, s->dim, s->kind, s->metric, s->scale_dev, s->lb_dev, reinterpret_cast<float*>(qtab), ql.qstride, qmeta,
            ql.qmeta};
}

}  // namespace vsag_amd
