// kvq_attention.hpp -- what the dense-attention kernels share.
#pragma once

#include <limits.h>
#include <math.h>

#include "kvq_device.hpp"
#include "kvq_internal.hpp"

namespace kvq {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// One query row over keys [k0, k1) by one wave in fp32 FMAs: scores of 64 keys
// per step, one per lane (dot over d), online softmax over the steps, the
// unnormalised accumulator in LDS (d floats at acc).  Sets the row's max m
// (log2 units) and denominator l.
__device__ __forceinline__ void attention_row(const AttnArgs& a, int row, int k0, int k1, float* acc, float& m, float& l) {
    const int lane = threadIdx.x & (kWave - 1);
    const int d = a.d;
    for (int j = lane; j < d; j += kWave) acc[j] = 0.0f;
    const float* q = a.q + static_cast<size_t>(row) * d;
    m = -INFINITY;
    l = 0.0f;
    for (int t0 = k0; t0 < k1; t0 += kWave) {
        const int t = t0 + lane;
        float s = -INFINITY;
        if (t < k1) {
            const float* k = a.k + static_cast<size_t>(t) * d;
            float dot = 0.0f;
            for (int j = 0; j < d; j++) dot = fmaf(q[j], k[j], dot);
            s = dot * a.scale_log2;
        }
        const float mn = fmaxf(m, wave_max(s));
        const float ms = mn == -INFINITY ? 0.0f : mn;  // no key with a score above -inf so far: weights 0
        const float alpha = fast_exp2(m - ms);
        const float p = fast_exp2(s - ms);
        l = l * alpha + wave_sum(p);
        m = mn;
        const int nt = min(kWave, k1 - t0);
        // Dims in passes of 64 with every lane active, so the shuffles read
        // live lanes; lanes past d carry zeros and store nothing.
        for (int j0 = 0; j0 < d; j0 += kWave) {
            const int j = j0 + lane;
            const bool in = j < d;
            float x = in ? acc[j] * alpha : 0.0f;
            for (int u = 0; u < nt; u++) {
                const float pu = __shfl(p, u);
                x = fmaf(pu, in ? a.v[static_cast<size_t>(t0 + u) * d + j] : 0.0f, x);
            }
            if (in) acc[j] = x;
        }
    }
}

}  // namespace kvq
