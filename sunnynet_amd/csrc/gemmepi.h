// Row addressing and output epilogues shared by the product kernels.
#pragma once

#include "gemm.h"

namespace snhip {

__device__ __forceinline__ const float* gemm_xrow(const GemmArgs& g, int m) {
    if (g.shift_T > 0) {
        const int t = m % g.shift_T;
        return t == 0 ? g.X0 + (long)(m / g.shift_T) * g.ldx0 : g.X + (long)(m - 1) * g.ldx;
    }
    return g.X + (long)m * g.ldx;
}

__device__ __forceinline__ void gemm_epilogue(const GemmArgs& g, int m, int n, float acc) {
    float* y = g.Y + (long)m * g.ldy + n;
    if (g.epi == GEPI_STORE) {
        *y = acc;
    } else if (g.epi == GEPI_WEDGE) {
        *y = acc * (1.0f + 0.5f * g.a_tanh / (1.0f + fabsf(acc)));       // sunnynet.c:270-271
    } else if (g.epi == GEPI_RESID) {
        *y = acc + (g.b_gain * g.s[(long)m * g.lds + n] + g.sfb[(long)m * g.ldf + n] + *y);  // :276
    } else if (g.epi == GEPI_ADD) {
        *y = *y + acc;                                                    // rwkv7.c:300,314
    } else {
        const float t = acc > 0.0f ? acc : 0.0f;                          // rwkv7.c:308-312
        *y = t * t;
    }
}

// Sums `splits` split-K partials of (M, N) in split order into g's epilogue.
snhip_status launch_gemm_reduce(const GemmArgs& g, int splits, const float* part, hipStream_t st);

}  // namespace snhip
