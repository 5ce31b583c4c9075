// The k-th smallest of many floats, near enough from above, by one wave.
#pragma once

#include "topk.h"

namespace vsag_amd {

// Any value with at least k of the `count` (>= k) values at or below it, by one wave: 256 bins between the smallest and
// the largest value, the first bin at which the running count reaches k, and two bins more for the rounding of the
// binning itself.  Values that are no numbers, or from 3e38 on, do not count; infinity where fewer than k are left.
// value(i) is asked for three times.
template <typename F>
__device__ inline float
kth_value_or_above(F value, uint32_t count, uint32_t k, uint32_t* hist, uint32_t lane) {
    const float inf = __builtin_inff();
    auto counts = [](float v) { return v > -3.0e38F && v < 3.0e38F; };
    float vmin = inf, vmax = -inf;
    uint32_t left = 0;
    for (uint32_t i = lane; i < count; i += kWave) {
        const float v = value(i);
        if (counts(v)) {
            vmin = fminf(vmin, v);
            vmax = fmaxf(vmax, v);
            ++left;
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        vmin = fminf(vmin, __shfl_xor(vmin, off));
        vmax = fmaxf(vmax, __shfl_xor(vmax, off));
        left += __shfl_xor(left, off);
    }
    if (left < k) {
        return inf;
    }
    const float width = (vmax - vmin) * (1.0F / 256.0F);
    if (!(width > 1.0e-30F) || !(width < 1.0e30F)) {
        return vmax;
    }
    const float inv_width = 1.0F / width;
    for (uint32_t b = lane; b < 256; b += kWave) {
        hist[b] = 0;
    }
    wave_lds_fence();
    for (uint32_t i = lane; i < count; i += kWave) {
        const float v = value(i);
        if (counts(v)) {
            const float f = (v - vmin) * inv_width;
            atomicAdd(&hist[f < 255.0F ? static_cast<uint32_t>(f) : 255U], 1U);
        }
    }
    wave_lds_fence();
    const uint32_t h[4] = {hist[4 * lane], hist[4 * lane + 1], hist[4 * lane + 2], hist[4 * lane + 3]};
    uint32_t incl = h[0] + h[1] + h[2] + h[3];
    const uint32_t mine = incl;
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t o = __shfl_up(incl, off);
        incl += lane >= static_cast<uint32_t>(off) ? o : 0U;
    }
    uint32_t before = incl - mine, bin = 4 * lane;
#pragma unroll
    for (int b = 0; b < 3; ++b) {
        if (before + h[b] >= k) {
            break;
        }
        before += h[b];
        ++bin;
    }
    bin = __shfl(bin, static_cast<int>(__builtin_ctzll(__ballot(incl >= k))));
    const float edge = vmin + static_cast<float>(bin + 3) * width;
    return edge < vmax ? edge : vmax;
}

}  // namespace vsag_amd
