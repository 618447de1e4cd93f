// The end of a sequential layer with many rows (a prompt), bf16: the row kernel behind its feed-forward, the token input's gate and output products and the row
// kernel that ends the layer, in one launch.
//
// A workgroup has up to 16 rows and keeps them in registers in the LANE ORDER OF THE MATRIX OPERAND from the first load to the last store: a lane holds columns
// (lane >> 4) * 8 .. + 7 of row lane & 15 of its wave's k tiles.  The row is the gate product's operand as it stands; the output product's weight rows are
// fetched in the order that makes its results come out in that same layout.  LDS holds the gate product's partial sums and the rows' square sums only.  What
// stays away is the row's way out and back between the four launches (fp32 residual once more each way, its bf16 copy, the output product's fp32 sums, the
// gate's): 250 of 850 MB of 6100 rows of 2048 columns.
// Bound by memory, and by what one CU takes from it: 16 rows fill a CU's registers, so the rows are dealt out evenly over the fewest rounds of one workgroup
// a CU (ob_side_rows_of; always 16: 6080 rows 153 us instead of 136, 1024 66 instead of 45).  6080 rows of 2048 columns, six choices, two to eight results
// averaged: 104 .. 155 us, for launches of 57 + 11 + 5 + 11 + 65 .. 95.  Eight rows a workgroup and two workgroups a CU: 172-185 (registers spilled).
#pragma once
#include "ob_few.h"

typedef float ObSideF8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ ObSideF8 ob_side_load(const float *p)
{
    const ob_float4 a = reinterpret_cast<const ob_float4 *>(p)[0], b = reinterpret_cast<const ob_float4 *>(p)[1];
    return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ void ob_side_store(float *p, ObSideF8 v)
{
    reinterpret_cast<ob_float4 *>(p)[0] = __builtin_shufflevector(v, v, 0, 1, 2, 3);
    reinterpret_cast<ob_float4 *>(p)[1] = __builtin_shufflevector(v, v, 4, 5, 6, 7);
}

// Sum over the row of a lane's `ss` (lanes 16 apart, 16 waves).  red: [16][16] floats, one per use
__device__ __forceinline__ float ob_side_row_sum(float ss, float *red, int wave, int lane)
{
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (lane < 16) red[wave * 16 + lane] = ss;
    __syncthreads();
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) s += red[(4 * (lane >> 4) + w) * 16 + (lane & 15)];
    s += __shfl_xor(s, 16);
    return s + __shfl_xor(s, 32);
}

// rows of a workgroup
static inline int ob_side_rows_of(int rows, int cus) { const int rounds = (rows + 16 * cus - 1) / (16 * cus), wgs = rounds * cus; return (rows + wgs - 1) / wgs; }
static inline int ob_side_rows_lds(int nt) { return nt * 16 * 1024 + 16 * 16 * nt * 2 + 3 * 16 * 16 * 4; }
// grid (rows / wg_rows), 1024 threads; W % 32 == 0, W <= 512 NV: wave w has the k tiles w NV ..  NT: n tiles of the gate product
template <int KIND, int NT, int NV>
__global__ __launch_bounds__(1024) void ob_side_rows_kernel(const ObFewSideArgs A, int n_rows, int wg_rows)
{
    constexpr int KQ = NT / 2, EC = NV == 4 ? 2 : 4;                   // EC: choices in flight
    typedef ObSideF8 f8;
    extern __shared__ __attribute__((aligned(16))) char smem[];        // [16][NT][64] x 4 partial sums | formed [KQ] operand tiles bf16 | [3][16][16] reductions
    ob_float4 *part = reinterpret_cast<ob_float4 *>(smem);
    __bf16 *formed = reinterpret_cast<__bf16 *>(smem + NT * 16 * 1024);
    float *red = reinterpret_cast<float *>(smem + NT * 16 * 1024 + 16 * 16 * NT * 2);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4, nkt = A.p.nkt;
    const int row0 = blockIdx.x * wg_rows, mine = min(wg_rows, n_rows - row0), t = row0 + min(lane & 15, mine - 1), kt0 = wave * NV;
    const bool live = (lane & 15) < mine;                              // (lanes beyond the workgroup's rows: its last row again, not written)
    const auto there = [&](int i) { return kt0 + i < nkt; };           // (wave-uniform)
    const auto col = [&](int i) { return (kt0 + i) * 32 + g * 8; };
    float *xr = A.x + (size_t)t * A.W, *hr = A.hist + (size_t)t * A.W;
    // the token input's entry of the sum that is this thread's (below)
    const int fr = (tid >> 2) & 15, fn = (tid >> 8) * 16 + ((tid >> 6) & 3) * 4 + (tid & 3);
    float entry = 0.f;
    if (fn < A.dim) entry = (float)((const __bf16 *)A.table)[(size_t)A.tokens[row0 + min(fr, mine - 1)] * A.ld_table + fn];
    f8 x[NV], s[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) s[i] = x[i] = (f8)0.f;
    for (int k = 0; k < (A.z ? A.n_split : 0); ++k)                    // splits in order
#pragma unroll
        for (int i = 0; i < NV; ++i) if (there(i)) s[i] += ob_side_load(A.z + k * A.z_split + (size_t)t * A.ldz + col(i));
    if constexpr (KIND == OB_X_EXPERTS) {
#pragma unroll 1
        for (int k0 = 0; k0 < A.top; k0 += EC) {                       // choices in order
            ob_bf8 y[EC][NV];
            float w[EC];
#pragma unroll
            for (int j = 0; j < EC; ++j) {
                const size_t k = (size_t)t * A.top + min(k0 + j, A.top - 1);
                const int at = A.tok_row[k];                           // (-1: none)
                w[j] = k0 + j < A.top && at >= 0 ? A.tok_w[k] : 0.f;
                const __bf16 *p = (const __bf16 *)A.eo + (size_t)max(at, 0) * A.ld_ez;
#pragma unroll
                for (int i = 0; i < NV; ++i) if (there(i)) y[j][i] = *reinterpret_cast<const ob_bf8 *>(p + col(i));
            }
#pragma unroll
            for (int j = 0; j < EC; ++j)
                if (w[j] != 0.f) {                                     // (the row of a choice that is no expert's holds anything)
#pragma unroll
                    for (int i = 0; i < NV; ++i)
                        if (there(i)) {
#pragma unroll
                            for (int e = 0; e < 8; ++e) s[i][e] = __builtin_fmaf(w[j], (float)y[j][i][e], s[i][e]);
                        }
                }
        }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) if (there(i)) x[i] = ob_side_load(xr + col(i));
    if (KIND == OB_X_EXPERTS && A.id_w) {                              // (uniform)
        const float w = A.id_w[t];
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (there(i)) {
                f8 h = x[i];
                if (A.idh) {
                    const ob_bf8 b = *reinterpret_cast<const ob_bf8 *>((const __bf16 *)A.idh + (size_t)t * A.ld_idh + col(i));
#pragma unroll
                    for (int e = 0; e < 8; ++e) h[e] = (float)b[e];
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) s[i][e] = __builtin_fmaf(w, h[e], s[i][e]);
            }
    }
    const auto rms = [&](const f8 (&v)[NV], float *r) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = __builtin_fmaf(v[i][e], v[i][e], ss);
        return 1.0f / sqrtf(ob_side_row_sum(ss, r, wave, lane) / (float)A.W + A.eps);
    };
    if (A.post_w) {                                                    // (uniform)
        const float r = rms(s, red);
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if (there(i)) {
                const f8 pw = ob_side_load(A.post_w + col(i));
#pragma unroll
                for (int e = 0; e < 8; ++e) s[i][e] = s[i][e] * r * pw[e];
            }
    }
    ob_float4 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = (ob_float4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if (there(i)) {
            ob_bf8 b;
#pragma unroll
            for (int e = 0; e < 8; ++e) { x[i][e] += A.mult * s[i][e]; b[e] = (__bf16)x[i][e]; }
#pragma unroll
            for (int n = 0; n < NT; ++n)
                acc[n] = ObElem<__bf16>::mma(*reinterpret_cast<const ob_bf8 *>((const char *)A.p.w + (size_t)(uint32_t)(n * nkt + kt0 + i) * 1024 + lane * 16), b, acc[n]);
        }
#pragma unroll
    for (int n = 0; n < NT; ++n) part[(wave * NT + n) * 64 + lane] = acc[n];
    // the depth average's earlier results meanwhile, added in order
    const bool depth = A.hist && A.dwa;                                // (uniform)
#pragma unroll
    for (int i = 0; i < NV; ++i) s[i] = (f8)0.f;
    if (depth) {
#pragma unroll 1
        for (int j = 0; j < A.hist_i; ++j) {
            const float d = A.dwa[j];
            f8 v[NV];
#pragma unroll
            for (int i = 0; i < NV; ++i) if (there(i)) v[i] = ob_side_load(hr + (size_t)j * A.hist_stride + col(i));
#pragma unroll
            for (int i = 0; i < NV; ++i)
                if (there(i)) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) s[i][e] = __builtin_fmaf(d, v[i][e], s[i][e]);
                }
        }
    }
    __syncthreads();
    if (tid < NT * 256) {                                              // sum `tid` of the workgroup's: lane tid / 4 % 64 of n tile tid / 256, element tid % 4
        const float *pp = reinterpret_cast<const float *>(part) + tid;
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < 16; ++w) v += pp[w * NT * 256];
        formed[ob_frag<__bf16>(fr, fn, KQ)] = (__bf16)(fn < A.dim ? ob_gelu_tanh<__bf16>(v) * entry : 0.f);
    }
    __syncthreads();
    ob_bf8 f[KQ];
#pragma unroll
    for (int k = 0; k < KQ; ++k) f[k] = *reinterpret_cast<const ob_bf8 *>(formed + (k * 64 + lane) * 8);
    // Output product: a k tile's 32 columns are two n tiles' weight rows.  Result e of lane group g is weight row 4 g + e of the instruction's 16; fetched from
    // row 8 g + 4 p + e of the 32 by instruction p, it is column 8 g + 4 p + e, where the lane has it.
    f8 y[NV];
    const int wr = 8 * ((lane & 15) >> 2) + (lane & 3);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        y[i] = (f8)0.f;
        if (there(i)) {
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const int r = wr + 4 * p;
                const char *w = (const char *)A.q.w + (size_t)(uint32_t)((2 * (kt0 + i) + (r >> 4)) * KQ) * 1024 + (g * 16 + (r & 15)) * 16;
                ob_float4 o = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < KQ; ++k) o = ObElem<__bf16>::mma(*reinterpret_cast<const ob_bf8 *>(w + k * 1024), f[k], o);
#pragma unroll
                for (int e = 0; e < 4; ++e) y[i][4 * p + e] = o[e];
            }
        }
    }
    const float r = rms(y, red + 256), di = depth ? A.dwa[A.hist_i] : 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if (there(i)) {
            const f8 sw = ob_side_load(A.side_w + col(i));
#pragma unroll
            for (int e = 0; e < 8; ++e) x[i][e] += y[i][e] * r * sw[e];
            if (A.hist && live) ob_side_store(hr + A.hist_i * A.hist_stride + col(i), x[i]);
            if (depth) {
#pragma unroll
                for (int e = 0; e < 8; ++e) x[i][e] = __builtin_fmaf(di, x[i][e], s[i][e]);
            }
            if (live) ob_side_store(xr + col(i), x[i]);
        }
    if (!A.out) return;                                                // (uniform: the last layer's row goes through the final norm)
    const float r2 = A.w ? rms(x, red + 512) : 1.f;                    // (uniform)
    if (!live) return;
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if (there(i)) {
            f8 v = x[i];
            if (A.w) {
                const f8 nw = ob_side_load(A.w + col(i));
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = v[e] * r2 * (A.off + nw[e]);
            }
            ob_bf8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = (__bf16)v[e];
            *reinterpret_cast<ob_bf8 *>((__bf16 *)A.out + ob_frag<__bf16>(t, col(i), A.out_nkt)) = o;
        }
}
