// The LayerNorm epilogue that takes any row (width, type, alignment).
#pragma once
#include "ob_common.h"

// LayerNorm epilogue, one 256-thread workgroup per token.  Three passes over the (L2-resident)
// row: mean, centred variance, normalise -- the biased-variance / eps form of
// nn.LayerNorm(elementwise_affine=False) (bitnet.py:86,118), then the optional bias (:119-120).
//   FROM_Z: input is fp32 z (pre-g); u = g * z with the dtype's rounding points.
//   else   : input is u already (TD), normalised in place or into y.
template <typename TD, bool FROM_Z>
__global__ __launch_bounds__(256) void ob_layernorm_kernel(
    const float *z, const TD *uin, const TD *__restrict__ g, const TD *__restrict__ bias, TD *y,
    TD *uout, int N, float eps, int skip_ln)   // y may alias uin (in-place), so no restrict there
{
    __shared__ float red[8];
    const int64_t t = blockIdx.x;
    const float *zr = FROM_Z ? z + t * N : nullptr;
    const TD *ur = FROM_Z ? nullptr : uin + t * N;
    auto load_u = [&](int n) -> float {
        if (FROM_Z) {
            if (sizeof(TD) == 2) return ob_round_h(ob_round_h(zr[n]) * (float)g[n]);
            return zr[n] * (float)g[n];
        }
        return (float)ur[n];
    };
    if (skip_ln) {
        for (int n = threadIdx.x; n < N; n += 256) {
            const float v = load_u(n);
            y[t * N + n] = (TD)v;
            if (uout) uout[t * N + n] = (TD)v;
        }
        return;
    }
    float s = 0.f;
    for (int n = threadIdx.x; n < N; n += 256) s += load_u(n);
    const float mean = ob_block_sum(s, red) / (float)N;
    float v = 0.f;
    for (int n = threadIdx.x; n < N; n += 256) {
        const float d = load_u(n) - mean;
        v += d * d;
    }
    const float var = ob_block_sum(v, red) / (float)N;
    const float rstd = 1.0f / sqrtf(var + eps);
    for (int n = threadIdx.x; n < N; n += 256) {
        const float uu = load_u(n);
        float o = (uu - mean) * rstd;
        if (sizeof(TD) == 2) o = ob_round_h(o);
        if (bias) {
            o += (float)bias[n];
            if (sizeof(TD) == 2) o = ob_round_h(o);
        }
        if (uout) uout[t * N + n] = (TD)uu;
        y[t * N + n] = (TD)o;
    }
}
