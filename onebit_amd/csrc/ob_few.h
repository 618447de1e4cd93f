// Few rows (a decode step): what would otherwise be launches of four microseconds with next to nothing to do, merged.  bf16.
//   ob_few_route_kernel  a sequential layer's row kernel behind its mixer, with the router's product and the choice of experts of its row
//   ob_few_side_kernel   the row kernel behind its feed-forward, the token input's two products and the row kernel that ends the layer
//   ob_few_expert_kernel expert products, gate / up or down, of the routed experts and the shared one in one launch; a workgroup finds its expert's
//                        rows in the choices by itself (no row lists, no block table, no launch that makes them)
//   ob_few_query_kernel  latent attention from its input product to the absorbed queries: both norms, the cache's new entry, query product, absorbing product
//   ob_few_value_kernel  the splits of its context together, and the product that makes the heads' outputs of them
//   ob_few_gated_out_kernel  the output product behind a state-space mixer, with the mixer's norm
// Rows of the experts' space here are the choices themselves: row t * top + k is choice k of token t.
#pragma once
#include "ob_hrows.h"
#include "ob_latent.h"
#include "ob_moe.h"

// A row's product with NT n tiles (16 NT <= 64 columns).  The weights depend on nothing: a wave requests its k tiles (nkt / 16 of them, four at a time) before
// the row is there; the row comes through LDS.  Every lane column multiplies the same row (the matrix instruction has 16 of them).
struct ObFewProduct { const void *w; int nkt; };
template <int NT> struct ObFewWeights { ob_bf8 w[4 * NT]; };
template <int NT, int I0 = 0, int I1 = 4> __device__ __forceinline__ void ob_few_fetch(ObFewWeights<NT> &W, const ObFewProduct &P, int k0, int lane)
{                                                                      // (k tiles there are not: the last one again)
#pragma unroll
    for (int i = I0; i < I1; ++i)
#pragma unroll
        for (int n = 0; n < NT; ++n)
            W.w[NT * i + n] = *reinterpret_cast<const ob_bf8 *>((const char *)P.w + (size_t)(uint32_t)(n * P.nkt + min(k0 + i, P.nkt - 1)) * 1024 + lane * 16);
}
// sums of all 16 waves: column `tid` of the product in thread tid < 16 NT.  row: P.nkt k tiles in LDS; part: [16][64] floats of LDS.  Whole workgroup of 1024.
template <int NT> __device__ __forceinline__ float ob_few_multiply(ObFewWeights<NT> &W, const ObFewProduct &P, const __bf16 *row, float *part, int tid)
{
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), per = (P.nkt + 15) >> 4, k1 = min(P.nkt, (wave + 1) * per);
    ob_float4 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = (ob_float4){0.f, 0.f, 0.f, 0.f};
    for (int k0 = wave * per; k0 < k1; k0 += 4) {                      // (wave-uniform)
        if (k0 > wave * per) ob_few_fetch(W, P, k0, lane);
#pragma unroll
        for (int i = 0; i < 4; ++i) {                                  // (k tiles beyond the wave's: times zero)
            const ob_bf8 x = k0 + i < k1 ? *reinterpret_cast<const ob_bf8 *>(row + (k0 + i) * 32 + (lane >> 4) * 8) : (ob_bf8)(__bf16)0.f;
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[n] = ObElem<__bf16>::mma(W.w[NT * i + n], x, acc[n]);
        }
    }
    if ((lane & 15) == 0) {
#pragma unroll
        for (int n = 0; n < NT; ++n) *reinterpret_cast<ob_float4 *>(part + wave * 64 + n * 16 + (lane >> 4) * 4) = acc[n];
    }
    __syncthreads();
    float s = 0.f;
    if (tid < 16 * NT) {
#pragma unroll
        for (int w = 0; w < 16; ++w) s += part[w * 64 + tid];
    }
    return s;
}

// Both row kernels below: one workgroup of 16 waves per row, four columns per thread; what bounds them is instructions (four waves share a SIMD: 100 of them
// in every wave are 0.7 us) and the chain of fetches, so waves beyond the row's columns only multiply, and nothing is computed twice.
// The partial sums of four columns of a row, its first four splits: all requested at once, with nothing between them and the row's other requests.
struct ObFewSplits { ob_float4 v[4]; };
__device__ __forceinline__ ObFewSplits ob_few_splits(const ObXRowArgs &A, int t, int c)
{
    ObFewSplits r;
    const float *p = A.z ? A.z + (size_t)t * A.ldz + c : A.x + (size_t)t * A.W + c;      // (no product pending: anything, added as zeros)
#pragma unroll
    for (int j = 0; j < 4; ++j) r.v[j] = *reinterpret_cast<const ob_float4 *>(p + (size_t)max(min(j, A.n_split - 1), 0) * A.z_split);
    return r;
}
__device__ __forceinline__ void ob_few_sum(float (&s)[4], const ObFewSplits &r, const ObXRowArgs &A, int t, int c)
{
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if (j < A.n_split) {                                           // (uniform)
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] += r.v[j][e];
        }
    for (int k = 4; k < A.n_split; k += 4) ob_sum_splits_u<4, 4>(s, A.z + (size_t)t * A.ldz + c, A.z_split, k, A.n_split);
}
// 1 / rms of a row whose waves hold four columns a thread; waves beyond the row bring nothing and leave behind the barrier.  red: [16], one per use
__device__ __forceinline__ float ob_few_rms(const float (&v)[4], float *red, bool mine, int waves, int lane, int wave, int W, float eps)
{
    if (mine) {                                                        // (wave-uniform)
        float ss = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = __builtin_fmaf(v[e], v[e], ss);
        ss = ob_wave_sum(ss);
        if (lane == 0) red[wave] = ss;
    }
    __syncthreads();
    if (!mine) return 0.f;
    float ss = (lane & 15) < waves ? red[lane & 15] : 0.f;
    ss += OB_DPP_F(ss, 0xB1, 0xF);
    ss += OB_DPP_F(ss, 0x4E, 0xF);
    ss += OB_DPP_F(ss, 0x141, 0xF);
    ss += OB_DPP_F(ss, 0x140, 0xF);                                    // (every lane of 16 holds the sum)
    return 1.0f / sqrtf(ss / (float)W + eps);
}

struct ObFewRowArgs : ObXRowArgs {
    ObFewProduct p;                    // router
    ObRouteArgs route;                 // (its table of blocks unused)
    int32_t *sel;                      // [T][top] expert of every choice, -1: none (an identity expert, an idle row)
};
// grid (rows), 1024 threads; W <= 4096, W % 4 == 0; experts + identity experts <= 64.  s, post norm and residual as ob_xrow_kernel's plain form, output
// row-major; then the row's experts.  12 rows of 2048 columns, 40 router columns: 7.6 us, for a row kernel of 4.6, the router's 6.1 (with the shared expert's
// gate and up, now with the experts') and its launch of 6.6.
static inline int ob_few_row_lds(const ObFewRowArgs &A) { return A.p.nkt * 64 + (16 * 64 + 2 * 16 + A.route.groups + A.route.top) * 4; }
template <int NT>                                                      // n tiles of the router
__global__ __launch_bounds__(1024) void ob_few_route_kernel(const ObFewRowArgs A)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];        // row [nkt 32] bf16 | [16][64] partial sums | [2][16] reductions | group maxima | choices
    __bf16 *row = reinterpret_cast<__bf16 *>(smem);
    float *part = reinterpret_cast<float *>(smem + A.p.nkt * 64), *red = part + 16 * 64;
    uint32_t *gs = reinterpret_cast<uint32_t *>(red + 32);
    int *slots = reinterpret_cast<int *>(gs + A.route.groups);
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = 4 * tid, per = (A.p.nkt + 15) >> 4;
    const int waves = (A.W + 255) >> 8;
    const bool mine = wave < waves, on = c < A.W;                      // (mine: wave-uniform)
    const int slot = A.row_slot[t], pos = A.row_pos[t], cc = on ? c : 0;       // (a last wave's threads beyond the row: its first columns again, times zero)
    float corr[1] = {0.f}, s[4] = {0.f, 0.f, 0.f, 0.f};
    float *xr = A.x + (size_t)t * A.W + cc;
    ob_float4 x, pw, nw, bias;
    ObFewSplits z4;
    if (mine) {
        x = *reinterpret_cast<const ob_float4 *>(xr);
        z4 = ob_few_splits(A, t, cc);
        if (A.post_w) pw = *reinterpret_cast<const ob_float4 *>(A.post_w + cc);
        if (A.w) nw = *reinterpret_cast<const ob_float4 *>(A.w + cc);
        if (A.bias) bias = *reinterpret_cast<const ob_float4 *>(A.bias + cc);
        if (wave == 0 && lane < A.route.experts + A.route.identity) corr[0] = A.route.correction[lane];
    }
    // (the weights behind the row's own requests, those of all waves: a CU's requests are served in order, 256 KB take 2 us)
    asm volatile("s_barrier" ::: "memory");
    ObFewWeights<NT> w;
    ob_few_fetch(w, A.p, wave * per, lane);
    if (mine) {
        ob_few_sum(s, z4, A, t, cc);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (A.bias) s[e] += bias[e];
            s[e] = on ? s[e] : 0.f;
            x[e] = on ? x[e] : 0.f;
        }
    }
    if (A.post_w) {                                                    // (uniform)
        const float r = ob_few_rms(s, red, mine, waves, lane, wave, A.W, A.eps);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = s[e] * r * pw[e];
    }
    if (mine) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] += A.mult * s[e];
        if (on) *reinterpret_cast<ob_float4 *>(xr) = x;
    }
    if (A.w) {                                                         // (uniform)
        const float v[4] = {x[0], x[1], x[2], x[3]}, r = ob_few_rms(v, red + 16, mine, waves, lane, wave, A.W, A.eps);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = x[e] * r * (A.off + nw[e]);
    }
    if (c < A.p.nkt * 32) {                                            // (zeros behind the row, by waves without columns of it too)
        const ob_bf4 h = on ? ob_to_v4<__bf16>(x) : (ob_bf4)(__bf16)0.f;
        *reinterpret_cast<ob_bf4 *>(row + c) = h;
        if (on) *reinterpret_cast<ob_bf4 *>((__bf16 *)A.out_rm + (size_t)t * A.ld_rm + c) = h;
    }
    __syncthreads();
    const float logit = ob_few_multiply(w, A.p, row, part, tid);
    if (wave) return;
    const int N = A.route.experts + A.route.identity;
    const float z[1] = {lane < N ? logit : -INFINITY};
    ob_route_token<1>(A.route, t, z, corr, gs, slots, lane);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                 // (this wave's own choices)
    const bool live = slot >= 0 && slot < A.n_slots && pos >= 0 && pos < A.max_len;
    for (int k = lane; k < A.route.top; k += 64) {
        const int e = live ? slots[k] : -1, at = t * A.route.top + k;
        A.sel[at] = e;
        A.route.tok_row[at] = e < 0 ? -1 : at;
    }
}

struct ObFewSideArgs : ObXRowArgs {
    ObFewProduct p, q;                 // gate product [16 NT columns], output product [rup(W, 16) columns, NT / 2 k tiles]
    const void *table; int ld_table, dim;          // entry (tokens[t], n), n < dim
    const float *side_w;
};
// grid (rows), 1024 threads; W <= 2048 (eight n tiles of the output product a wave), W % 4 == 0, top <= 64.  The row kernel behind a feed-forward (KIND: with
// experts or not), the token's own input (gate product, gelu times the token's table row, output product, its norm, residual) and the row kernel behind that
// (depth average, next norm): what the row leaves for the next layer, in one launch.  12 rows of 2048 columns, 64 of the token input (256 KB of weights for
// either product, a CU takes them at 64 bytes a clock): 11.4 us, for launches of 6.6 + 4.6 + 4.7 + 5.0.
static inline int ob_few_side_lds(const ObFewSideArgs &A) { return A.p.nkt * 64 + 128 + (16 * 64 + 3 * 16 + 16 * ((A.W + 15) / 16)) * 4; }
template <int KIND, int NT>
__global__ __launch_bounds__(1024) void ob_few_side_kernel(const ObFewSideArgs A)
{
    constexpr int NH = 8, KQ = NT / 2;
    extern __shared__ __attribute__((aligned(16))) char smem[];        // row [nkt 32] bf16 | formed [64] bf16 | [16][64] partial sums | [3][16] reductions | [W] output
    __bf16 *row = reinterpret_cast<__bf16 *>(smem), *formed = reinterpret_cast<__bf16 *>(smem + A.p.nkt * 64);
    float *part = reinterpret_cast<float *>(smem + A.p.nkt * 64 + 128), *red = part + 16 * 64, *out = red + 3 * 16;
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), c = 4 * tid, per = (A.p.nkt + 15) >> 4, nq = (A.W + 15) >> 4;
    const int waves = (A.W + 255) >> 8;
    const bool mine = wave < waves, on = c < A.W;                      // (mine: wave-uniform)
    const int cc = on ? c : 0;                                         // (a last wave's threads beyond the row: its first columns again, times zero)
    float *xr = A.x + (size_t)t * A.W + cc, *hr = A.hist + (size_t)t * A.W + cc;
    float s[4] = {0.f, 0.f, 0.f, 0.f}, tw = 0.f, idw = 0.f, entry = 0.f;
    ob_float4 x, pw, y[8];
    ObFewSplits z4;
    if (mine) {
        x = *reinterpret_cast<const ob_float4 *>(xr);
        if (KIND == OB_X_EXPERTS) {                                    // a choice's row is its own number: eight of the first split in flight
            const int at = t * A.top + min(lane, A.top - 1), tr = A.tok_row[at];
            const float v = A.tok_w[at];
            tw = tr >= 0 && lane < A.top ? v : 0.f;
#pragma unroll
            for (int j = 0; j < 8; ++j) y[j] = *reinterpret_cast<const ob_float4 *>(A.ez + (size_t)(t * A.top + min(j, A.top - 1)) * A.ld_ez + cc);
            if (A.id_w) idw = A.id_w[t];
        }
        z4 = ob_few_splits(A, t, cc);
        if (A.post_w) pw = *reinterpret_cast<const ob_float4 *>(A.post_w + cc);
        if (wave == 0 && lane < A.dim) entry = (float)((const __bf16 *)A.table)[(size_t)A.tokens[t] * A.ld_table + lane];
    }
    // (the weights behind the row's own requests, those of all waves: a CU's requests are served in order, 256 KB take 2 us)
    asm volatile("s_barrier" ::: "memory");
    ObFewWeights<NT> w;
    ob_few_fetch<NT, 0, KIND == OB_X_EXPERTS ? 1 : 4>(w, A.p, wave * per, lane);
    if (mine) {
        ob_few_sum(s, z4, A, t, cc);
        if (KIND == OB_X_EXPERTS) {                                    // choices, then their further splits, added in order
            const auto add = [&](float wj, ob_float4 v) {
                if (wj == 0.f) return;                                 // (uniform; the row of a choice that is no expert's holds anything)
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = __builtin_fmaf(wj, v[e], s[e]);
            };
            const auto weight = [&](int k) { return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, tw), k)); };
#pragma unroll
            for (int j = 0; j < 8; ++j) if (j < A.top) add(weight(j), y[j]);
            for (int sp = 0; sp < A.ez_n; ++sp)
                for (int k = sp ? 0 : 8; k < A.top; ++k) add(weight(k), *reinterpret_cast<const ob_float4 *>(A.ez + sp * A.ez_split + (size_t)(t * A.top + k) * A.ld_ez + cc));
            if (A.id_w) {
#pragma unroll
                for (int e = 0; e < 4; ++e) s[e] = __builtin_fmaf(idw, A.idh ? (float)((const __bf16 *)A.idh)[(size_t)t * A.ld_idh + cc + e] : x[e], s[e]);
            }
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s[e] = on ? s[e] : 0.f;
            x[e] = on ? x[e] : 0.f;
        }
    }
    if (KIND == OB_X_EXPERTS) ob_few_fetch<NT, 1, 4>(w, A.p, wave * per, lane);        // (their registers held the choices)
    if (A.post_w) {                                                    // (uniform)
        const float r = ob_few_rms(s, red, mine, waves, lane, wave, A.W, A.eps);
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] = s[e] * r * pw[e];
    }
    if (mine) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] += A.mult * s[e];
        if (c < A.p.nkt * 32) *reinterpret_cast<ob_bf4 *>(row + c) = on ? ob_to_v4<__bf16>(x) : (ob_bf4)(__bf16)0.f;
    }
    __syncthreads();
    const float pre = ob_few_multiply(w, A.p, row, part, tid);
    // the output product's tiles: n tiles wave, wave + 16, .. of this wave and all their k tiles (n tiles there are not: the last one again)
    ob_bf8 wq[8 * KQ];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int k = 0; k < KQ; ++k) wq[i * KQ + k] = *reinterpret_cast<const ob_bf8 *>((const char *)A.q.w + (size_t)(uint32_t)(min(wave + 16 * i, nq - 1) * KQ + k) * 1024 + lane * 16);
    if (wave == 0) formed[lane] = (__bf16)(lane < A.dim ? ob_gelu_tanh<__bf16>(pre) * entry : 0.f);
    __syncthreads();
    ob_bf8 f[KQ];
#pragma unroll
    for (int k = 0; k < KQ; ++k) f[k] = *reinterpret_cast<const ob_bf8 *>(formed + k * 32 + (lane >> 4) * 8);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        ob_float4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < KQ; ++k) acc = ObElem<__bf16>::mma(wq[i * KQ + k], f[k], acc);
        if (wave + 16 * i < nq && (lane & 15) == 0) *reinterpret_cast<ob_float4 *>(out + (wave + 16 * i) * 16 + (lane >> 4) * 4) = acc;
    }
    const bool depth = A.hist && A.dwa;                                // (uniform)
    ob_float4 sw, nw, h[NH];
    if (mine) {
        sw = *reinterpret_cast<const ob_float4 *>(A.side_w + cc);
        if (A.w) nw = *reinterpret_cast<const ob_float4 *>(A.w + cc);
        if (depth) {
#pragma unroll
            for (int j = 0; j < NH; ++j) h[j] = *reinterpret_cast<const ob_float4 *>(hr + (size_t)min(j, A.hist_i - 1) * A.hist_stride);
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = on ? out[c + e] : 0.f;
    const float r = ob_few_rms(s, red + 16, mine, waves, lane, wave, A.W, A.eps);
    if (mine) {
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] += s[e] * r * sw[e];
        if (A.hist && on) *reinterpret_cast<ob_float4 *>(hr + A.hist_i * A.hist_stride) = x;
        if (depth) {
            ob_float4 a = {0.f, 0.f, 0.f, 0.f};
            for (int j = 0; j < A.hist_i; j += NH) {                   // eight results in flight, added in order
                if (j) {
#pragma unroll
                    for (int q = 0; q < NH; ++q) h[q] = *reinterpret_cast<const ob_float4 *>(hr + (size_t)min(j + q, A.hist_i - 1) * A.hist_stride);
                }
#pragma unroll
                for (int q = 0; q < NH; ++q)
                    if (j + q < A.hist_i) {                            // (uniform)
                        const float d = A.dwa[j + q];
#pragma unroll
                        for (int e = 0; e < 4; ++e) a[e] = __builtin_fmaf(d, h[q][e], a[e]);
                    }
            }
            const float d = A.dwa[A.hist_i];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = __builtin_fmaf(d, x[e], a[e]);
        }
        if (on) *reinterpret_cast<ob_float4 *>(xr) = x;
    }
    if (!A.out) return;                                                // (uniform: the last layer's row goes through the final norm)
    if (A.w) {                                                         // (uniform)
        const float v[4] = {on ? x[0] : 0.f, on ? x[1] : 0.f, on ? x[2] : 0.f, on ? x[3] : 0.f}, r2 = ob_few_rms(v, red + 32, mine, waves, lane, wave, A.W, A.eps);
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = x[e] * r2 * (A.off + nw[e]);
    }
    if (on) *reinterpret_cast<ob_bf4 *>((__bf16 *)A.out + ob_frag<__bf16>(t, c, A.out_nkt)) = ob_to_v4<__bf16>(x);
}

// Expert products of few rows.  Workgroup = 2 n tiles x one K split of one expert (of the shared one: of all rows), four waves with a quarter of the
// split's k tiles each, as ob_dense_skinny_kernel; operands row-major.  Workgroups [0, ns): the shared expert.  Bound by the weights' way from HBM: 12 rows,
// 2048 columns, six of 32 experts of 704, shared 1408: 26.7 + 16.4 us (gate / up 160 MB, down 80), for 22.5 + 13.2 of the experts' alone, 4.3 of the shared
// output product and 6.6 of the launch that made row lists.
struct ObFewExpert { const void *w; int n_tiles, nkt, kt_split, n_split; const void *a; int lda; void *act; int ld_act; float *z; size_t z_split; };
struct ObFewExpertArgs {
    ObFewExpert e, s;                  // routed, shared (n_tiles 0: none)
    size_t w_group;
    const int32_t *sel; int T, top, by_choice;     // by_choice: one workgroup row per choice (the first of its expert works), else one per expert
    int ldz;
};
template <int MT, bool UP, bool DEEP>
__global__ __launch_bounds__(256, MT >= 4 ? 2 : MT == 1 && !DEEP ? 4 : 3) void ob_few_expert_kernel(const ObFewExpertArgs A)
{
    __shared__ ob_float4 red[4][2][MT][64];
    __shared__ int list[64], info[2];                                  // an expert's choices; their number, the first of them
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4;
    const int ns = ((A.s.n_tiles + 1) >> 1) * A.s.n_split;
    const bool shared = (int)blockIdx.x < ns;                          // (uniform)
    const ObFewExpert &P = shared ? A.s : A.e;
    int id = shared ? blockIdx.x : blockIdx.x - ns, expert = 0, rows = A.T;
    const int pairs = (P.n_tiles + 1) >> 1, per_e = pairs * P.n_split;
    if (!shared) {
        const int b = id / per_e, n = A.T * A.top;
        id -= b * per_e;
        expert = A.by_choice ? A.sel[b] : b;
        if (expert < 0) return;                                        // (uniform)
        if (wave == 0) {
            int cnt = 0, first = -1;
            for (int i0 = 0; i0 < n; i0 += 256) {
                int v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = i0 + 64 * j + lane < n ? A.sel[i0 + 64 * j + lane] : -1;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const uint64_t m = __builtin_amdgcn_ballot_w64(v[j] == expert);
                    if (v[j] == expert) list[cnt + __popcll(m & ((1ull << lane) - 1))] = i0 + 64 * j + lane;       // (a token has an expert once: at most 64)
                    if (m && first < 0) first = i0 + 64 * j + __builtin_ctzll(m);
                    cnt += __popcll(m);
                }
            }
            if (lane == 0) { info[0] = cnt; info[1] = first; }
        }
        __syncthreads();
        rows = info[0];
        if (rows == 0 || (A.by_choice && info[1] != b)) return;        // (uniform)
    }
    const int nt = 2 * (id % pairs), split = id / pairs, k_lo = split * P.kt_split, k_hi = min(P.nkt, k_lo + P.kt_split), per = (k_hi - k_lo + 3) >> 2;
    const int k0 = k_lo + wave * per, k1 = min(k0 + per, k_hi);
    const ob_bf8 *wp = (const ob_bf8 *)P.w + (size_t)expert * A.w_group * 64 + lane;
    const ob_bf8 *ap[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int i = min(m * 16 + (lane & 15), rows - 1), c = shared ? i : list[i];
        ap[m] = (const ob_bf8 *)((const __bf16 *)P.a + (size_t)(UP && !shared ? c / A.top : c) * P.lda) + g;
    }
    ob_float4 acc[2][MT];
    ob_skinny_stream<__bf16, MT, 4, DEEP>(wp + (size_t)nt * P.nkt * 64, wp + (size_t)min(nt + 1, P.n_tiles - 1) * P.nkt * 64, ap, k0, k1, acc);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m) red[wave][h][m][lane] = acc[h][m];
    __syncthreads();
    for (int m = wave; m < MT; m += 4) {
        ob_float4 v[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) v[h] = (red[0][h][m][lane] + red[1][h][m][lane]) + (red[2][h][m][lane] + red[3][h][m][lane]);
        const int i = m * 16 + (lane & 15);
        if (i >= rows) continue;
        const size_t c = shared ? i : list[i];
        if constexpr (UP) {
            ob_float4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = ob_silu<__bf16>(v[0][e]) * v[1][e];
            *reinterpret_cast<ob_bf4 *>((__bf16 *)P.act + c * P.ld_act + 8 * nt + 4 * g) = ob_to_v4<__bf16>(o);
        } else {
            float *z = P.z + (size_t)split * P.z_split + c * A.ldz + 16 * nt + 4 * g;
            *reinterpret_cast<ob_float4 *>(z) = v[0];
            if (nt + 1 < P.n_tiles) *reinterpret_cast<ob_float4 *>(z + 16) = v[1];
        }
    }
}

// Up to 32 rows of latent attention.  Workgroups [0, 4 H): head b % H, a quarter of its absorbed columns (a head's four on one XCD where H % 8 == 0: they read
// the same rows of W_uq, and q is computed in all of them: less of a CU's work than two launches); then one per row: the cache's new entry.
// Eight waves; a wave takes the n tiles wave, wave + 8 .. of the query product and requests its first 24 k tiles before the normalised row is there.
// 12 rows, 16 heads of 128, ranks 768 and 256: 7.6 us behind an input product of one split (9.9 behind four: every workgroup adds them), for launches of
// 4.5 (norms) + 4.7 + 4.7.  A head's weights of 384 KB (rank 1536) take longer than the launches: 0.97 of a step.
struct ObFewQueryArgs : ObLatPrepArgs {
    int T, H;
    const void *w_uq, *w_uk;           // [H][kp / 16][cq_nkt] and [H][rp / 16][kp / 32] tiles
    int kp;
    void *heads; int d_shift, head_rows;
};
static inline int ob_few_query_ld(int cols) { return (cols + 31) / 32 * 32 + 8; }       // elements of a row in LDS: rows in different banks
static inline int ob_few_query_lds(const ObFewQueryArgs &A, int mt) { return 16 * mt * (ob_few_query_ld(A.q_rank) + ob_few_query_ld(A.kp)) * 2; }
template <int MT>
__global__ __launch_bounds__(512) void ob_few_query_kernel(const ObFewQueryArgs A, int ldc, int ldq)
{
    constexpr int U = 12;
    extern __shared__ __attribute__((aligned(16))) char smem[];        // c_q [16 MT][ldc] | q [16 MT][ldq], bf16
    __bf16 *cq = reinterpret_cast<__bf16 *>(smem), *qs = cq + 16 * MT * ldc;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, g = lane >> 4;
    // norm of `cols` columns (a multiple of 4) from column c0 of a row, by one wave; the first 1024 columns wait in registers: request, then finish with
    // piece(column, four values)
    struct Row { ob_float4 v[4]; };
    const auto at = [&](int t, int c) {
        float s[4] = {0.f, 0.f, 0.f, 0.f};
        ob_sum_splits<4>(s, A.z + (size_t)t * A.ldz + c, A.z_split, A.n_split);
        return (ob_float4){s[0], s[1], s[2], s[3]};
    };
    const auto request = [&](Row &x, int t, int c0, int cols) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = (i * 64 + lane) * 4;
            x.v[i] = (ob_float4){0.f, 0.f, 0.f, 0.f};
            if (i * 256 < cols) {                                      // (uniform)
                if (A.n_split == 1) x.v[i] = *reinterpret_cast<const ob_float4 *>(A.z + (size_t)t * A.ldz + c0 + min(c, cols - 4));
                else x.v[i] = at(t, c0 + min(c, cols - 4));
            }
        }
    };
    const auto finish = [&](const Row &x, int t, int c0, int cols, const float *w, auto piece) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if ((i * 64 + lane) * 4 < cols) {
#pragma unroll
                for (int e = 0; e < 4; ++e) ss = __builtin_fmaf(x.v[i][e], x.v[i][e], ss);
            }
        for (int c = 1024 + lane * 4; c < cols; c += 256) {
            const ob_float4 u = at(t, c0 + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) ss = __builtin_fmaf(u[e], u[e], ss);
        }
        const float r = 1.0f / sqrtf(ob_wave_sum(ss) / (float)cols + A.eps);
        const auto out = [&](int c, ob_float4 u) {
            const ob_float4 wv = *reinterpret_cast<const ob_float4 *>(w + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) u[e] = u[e] * r * wv[e];
            piece(c, ob_to_v4<__bf16>(u));
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) if ((i * 64 + lane) * 4 < cols) out((i * 64 + lane) * 4, x.v[i]);
        for (int c = 1024 + lane * 4; c < cols; c += 256) out(c, at(t, c0 + c));
    };
    if ((int)blockIdx.x >= 4 * A.H) {                                  // the cache's new entry, columns beyond kv_rank zero
        const int t = blockIdx.x - 4 * A.H;
        if (wave) return;
        const int slot = A.row_slot[t], pos = A.row_pos[t];
        if (slot < 0 || slot >= A.n_slots || pos < 0 || pos >= A.max_len) return;      // idle row
        const int nkt = A.rp / 32;
        __bf16 *dst = (__bf16 *)A.cache + (size_t)slot * A.bands * nkt * 512;
        Row x;
        request(x, t, A.c0, A.kv_rank);
        finish(x, t, A.c0, A.kv_rank, A.kvn_w, [&](int c, ob_bf4 v) { *reinterpret_cast<ob_bf4 *>(dst + ob_frag<__bf16>(pos, c, nkt)) = v; });
        for (int c = A.kv_rank + lane * 4; c < A.rp; c += 256) *reinterpret_cast<ob_bf4 *>(dst + ob_frag<__bf16>(pos, c, nkt)) = (ob_bf4)(__bf16)0.f;
        return;
    }
    const int h = blockIdx.x % A.H, part = blockIdx.x / A.H, nt = A.kp >> 4, kts = A.kp >> 5, rt = A.rp >> 6;      // n tiles, k tiles of the absorbing product, its n tiles here
    const ob_bf8 *wq = (const ob_bf8 *)A.w_uq + (size_t)h * nt * A.cq_nkt * 64 + lane;
    ob_bf8 w[2 * U];
    const auto fetch = [&](int b, int n, int k0) {                     // (tiles there are not: the last one again)
#pragma unroll
        for (int u = 0; u < U; ++u) w[b * U + u] = wq[((size_t)n * A.cq_nkt + min(k0 + u, A.cq_nkt - 1)) * 64];
    };
    Row x[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) if (wave + 8 * q < A.T) request(x[q], wave + 8 * q, 0, A.q_rank);
    // (the weights behind the rows, those of all waves: a CU's requests are served in order, the head's part of W_uq takes 1.3 us)
    asm volatile("s_barrier" ::: "memory");
    if (wave < nt) { fetch(0, wave, 0); fetch(1, wave, U); }
#pragma unroll
    for (int q = 0; q < 2 * MT; ++q) {
        const int t = wave + 8 * q;
        if (t >= A.T) break;
        if (q >= 2) request(x[q & 1], t, 0, A.q_rank);
        finish(x[q & 1], t, 0, A.q_rank, A.qn_w, [&](int c, ob_bf4 v) { *reinterpret_cast<ob_bf4 *>(cq + t * ldc + c) = v; });
        for (int c = A.q_rank + lane * 4; c < A.cq_nkt * 32; c += 256) *reinterpret_cast<ob_bf4 *>(cq + t * ldc + c) = (ob_bf4)(__bf16)0.f;
    }
    __syncthreads();
    int row[MT];                                                       // (rows beyond the last: the last one again, not written)
#pragma unroll
    for (int m = 0; m < MT; ++m) row[m] = min(m * 16 + lr, A.T - 1);
    for (int n = wave; n < nt; n += 8) {                               // (wave-uniform)
        if (n != wave) { fetch(0, n, 0); fetch(1, n, U); }
        ob_float4 acc[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m] = (ob_float4){0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < A.cq_nkt; k0 += 2 * U) {
#pragma unroll
            for (int b = 0; b < 2; ++b) {
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int k = k0 + b * U + u;
                    if (k < A.cq_nkt) {                                // (uniform)
#pragma unroll
                        for (int m = 0; m < MT; ++m) acc[m] = ObElem<__bf16>::mma(w[b * U + u], *reinterpret_cast<const ob_bf8 *>(cq + row[m] * ldc + k * 32 + g * 8), acc[m]);
                    }
                }
                if (k0 + 2 * U + b * U < A.cq_nkt) fetch(b, n, k0 + 2 * U + b * U);
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m) if (m * 16 + lr < A.T) *reinterpret_cast<ob_bf4 *>(qs + (m * 16 + lr) * ldq + n * 16 + 4 * g) = ob_to_v4<__bf16>(acc[m]);
    }
    // this quarter's tiles of the absorbing product: wave, wave + 8 ..
    const ob_bf8 *wk = (const ob_bf8 *)A.w_uk + ((size_t)h * (A.rp >> 4) + part * rt) * kts * 64 + lane;
    ob_bf8 wa[4];
    const auto absorb = [&](int n, int k0) {
#pragma unroll
        for (int k = 0; k < 4; ++k) wa[k] = wk[(size_t)(n * kts + min(k0 + k, kts - 1)) * 64];
    };
    if (wave < rt) absorb(wave, 0);
    __syncthreads();
    for (int n = wave; n < rt; n += 8) {
        if (n != wave) absorb(n, 0);
        ob_float4 acc[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m] = (ob_float4){0.f, 0.f, 0.f, 0.f};
        for (int k0 = 0; k0 < kts; k0 += 4) {
            if (k0) absorb(n, k0);
#pragma unroll
            for (int k = 0; k < 4; ++k)
                if (k0 + k < kts) {                                    // (uniform)
#pragma unroll
                    for (int m = 0; m < MT; ++m) acc[m] = ObElem<__bf16>::mma(wa[k], *reinterpret_cast<const ob_bf8 *>(qs + row[m] * ldq + (k0 + k) * 32 + g * 8), acc[m]);
                }
        }
        const int r = (part * rt + n) * 16 + 4 * g;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int t = m * 16 + lr;
            if (t < A.T) *reinterpret_cast<ob_bf4 *>((__bf16 *)A.heads + ((((size_t)t * A.head_rows + (h >> 4)) << (A.d_shift + 4)) + ob_frag<__bf16>(h & 15, r, 0))) = ob_to_v4<__bf16>(acc[m]);
        }
    }
}

// Up to 32 rows.  Workgroup = (head, two n tiles of its outputs), eight waves: the splits of all rows' contexts of this head together (as
// ob_lat_combine_kernel, every workgroup of the head again: 18 KB at 12 rows of three live splits), in LDS, then the product with W_uv: a wave takes one n tile
// and every fourth k tile, all requested before the splits are there.  12 rows, 16 heads of 128, rank 256: 4.8 us for launches of 4.7 + 4.7.
struct ObFewValueArgs : ObLatArgs {
    int T;
    const void *w; int nt, nkt;        // [H][nt][nkt] tiles
    void *act; int act_nkt;
};
static inline int ob_few_value_lds(const ObFewValueArgs &A, int mt) { return 16 * mt * (A.rp + 8) * 2; }
template <int MT>
__global__ __launch_bounds__(512) void ob_few_value_kernel(const ObFewValueArgs A)
{
    extern __shared__ __attribute__((aligned(16))) char smem[];        // [16 MT][rp + 8] bf16
    __shared__ ob_float4 red[6][MT][64];
    __bf16 *ctx = reinterpret_cast<__bf16 *>(smem);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, g = lane >> 4, ld = A.rp + 8, pieces = A.rp >> 3;
    const int h = blockIdx.x, n = blockIdx.y * 2 + (wave & 1), k0 = wave >> 1;
    const ob_bf8 *wp = (const ob_bf8 *)A.w + ((size_t)h * A.nt + min(n, A.nt - 1)) * A.nkt * 64 + lane;
    ob_bf8 w[4];                                                       // (at most rank 512: 16 k tiles; tiles there are not: the last one again)
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] = wp[(size_t)min(k0 + 4 * u, A.nkt - 1) * 64];
    for (int i = tid; i < A.T * pieces; i += 512) {
        const int t = i / pieces, d = (i - t * pieces) * 8, slot = A.row_slot[t], pos = A.row_pos[t];
        float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (slot >= 0 && slot < A.n_slots && pos >= 0 && pos < A.max_len) {
            const int nlive = (pos + A.chunk) / A.chunk;
            if (nlive == 1) {                                          // (written by the attention itself)
                const ob_bf8 v = *reinterpret_cast<const ob_bf8 *>((const __bf16 *)A.ctx + (size_t)t * A.ldq + (size_t)h * A.rp + d);
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] = (float)v[e];
            } else {
                const size_t at = (size_t)t * A.nsplit * A.H + h;
                const float *ml = A.ml + 2 * at;
                const __bf16 *part = (const __bf16 *)A.part + at * A.rp + d;
                float m = -INFINITY, l = 0.f;                          // four splits in flight
                for (int s0 = 0; s0 < nlive; s0 += 4) {
                    ob_bf8 v[4];
                    float ms[4], ls[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const size_t sp = (size_t)min(s0 + j, nlive - 1) * A.H;
                        v[j] = *reinterpret_cast<const ob_bf8 *>(part + sp * A.rp);
                        ms[j] = ml[2 * sp]; ls[j] = ml[2 * sp + 1];
                    }
                    float mx = fmaxf(fmaxf(m, fmaxf(ms[0], ms[1])), fmaxf(ms[2], ms[3]));
                    const float keep = __builtin_amdgcn_exp2f(m - mx);         // (a split's maximum is finite)
                    l *= keep;
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] *= keep;
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float f = s0 + j < nlive ? ls[j] * __builtin_amdgcn_exp2f(ms[j] - mx) : 0.f;
                        l += f;
#pragma unroll
                        for (int e = 0; e < 8; ++e) o[e] = __builtin_fmaf(f, (float)v[j][e], o[e]);
                    }
                    m = mx;
                }
                const float inv = 1.0f / l;
#pragma unroll
                for (int e = 0; e < 8; ++e) o[e] *= inv;
            }
        }
        ob_bf8 r;
#pragma unroll
        for (int e = 0; e < 8; ++e) r[e] = (__bf16)o[e];
        *reinterpret_cast<ob_bf8 *>(ctx + t * ld + d) = r;
    }
    __syncthreads();
    ob_float4 acc[MT];
    const __bf16 *xr[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        acc[m] = (ob_float4){0.f, 0.f, 0.f, 0.f};
        xr[m] = ctx + min(m * 16 + lr, A.T - 1) * ld + g * 8;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (k0 + 4 * u < A.nkt) {                                      // (wave-uniform)
#pragma unroll
            for (int m = 0; m < MT; ++m) acc[m] = ObElem<__bf16>::mma(w[u], *reinterpret_cast<const ob_bf8 *>(xr[m] + (k0 + 4 * u) * 32), acc[m]);
        }
    if (k0) {
#pragma unroll
        for (int m = 0; m < MT; ++m) red[wave - 2][m][lane] = acc[m];
    }
    __syncthreads();
    if (k0 || n >= A.nt) return;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        const int t = m * 16 + lr;
        if (t < A.T) *reinterpret_cast<ob_bf4 *>((__bf16 *)A.act + ob_frag<__bf16>(t, (h * A.nt + n) * 16 + 4 * g, A.act_nkt)) = ob_to_v4<__bf16>((acc[m] + red[wave][m][lane]) + (red[wave + 2][m][lane] + red[wave + 4][m][lane]));
    }
}

// Up to 32 rows.  The output product of a layer with a state-space mixer, the mixer's norm (one group) in it: its columns, the first mix_nkt k tiles, come as
// y silu(gate) w without the factor 1 / rms, which a row's sums take after them (the rounding to bf16 is relative: of either product the same).  Else as
// ob_dense_skinny_kernel.  Takes the norm's launch of 4.6 us off a decode step's layer; 12 rows, 2048 columns of 4096 + 5632: 9.4 us for 8.4 of the product
// alone, the state-space step 13.0 for 12.2; 24 rows 12.4 for 9.7 and 24.8 for 23.1.
struct ObFewGatedOutArgs : ObDenseArgs { const float *sq; int n_sq, mix_nkt; float inner, eps; };
template <int MT>
__global__ __launch_bounds__(256, MT >= 2 ? 2 : 3) void ob_few_gated_out_kernel(const ObFewGatedOutArgs A)
{
    __shared__ ob_float4 red[4][2][MT][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), nt = blockIdx.x * 2, split = blockIdx.y;
    const int k_lo = split * A.kt_split, k_hi = min(A.nkt, k_lo + A.kt_split), per = (k_hi - k_lo + 3) >> 2, k0 = k_lo + wave * per, k1 = min(k0 + per, k_hi);
    const ob_bf8 *w0 = (const ob_bf8 *)A.w + (size_t)nt * A.nkt * 64 + lane, *w1 = (const ob_bf8 *)A.w + (size_t)min(nt + 1, A.n_tiles - 1) * A.nkt * 64 + lane;
    const ob_bf8 *ap[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) ap[m] = (const ob_bf8 *)A.a + lane + (size_t)m * A.nkt * 64;
    ob_float4 acc[2][MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[0][m] = acc[1][m] = (ob_float4){0.f, 0.f, 0.f, 0.f};
    const int mid = max(k0, min(k1, A.mix_nkt));
    constexpr int SU = MT == 1 ? 8 : 2;
#pragma unroll 1
    for (int part = 0; part < 2; ++part) {                             // the mixer's k tiles, the others (a wave mostly has one of them)
        const int a = part ? mid : k0, b = part ? k1 : mid;
        if (a >= b) continue;                                          // (wave-uniform)
        float s[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            s[m] = 1.f;
            if (part == 0) {                                           // 1 / rms of row lane & 15 of the token tile
                const float *p = A.sq + (size_t)min(m * 16 + (lane & 15), A.T - 1) * A.n_sq;
                ob_float4 q = {0.f, 0.f, 0.f, 0.f};
#pragma unroll SU
                for (int j = 4 * (lane >> 4); j < A.n_sq; j += 16) q += *reinterpret_cast<const ob_float4 *>(p + j);
                float v = (q[0] + q[1]) + (q[2] + q[3]);
                v += __shfl_xor(v, 16);
                v += __shfl_xor(v, 32);
                s[m] = 1.0f / sqrtf(v / A.inner + A.eps);
            }
        }
        ob_float4 c[2][MT];
        ob_skinny_stream<__bf16, MT, 64, false>(w0, w1, ap, a, b, c);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[h][m][e] += s[m] * c[h][m][e];
    }
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < MT; ++m) red[wave][h][m][lane] = acc[h][m];
    __syncthreads();
    for (int m = wave; m < MT; m += 4) {
        ob_float4 v[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) v[h] = (red[0][h][m][lane] + red[1][h][m][lane]) + (red[2][h][m][lane] + red[3][h][m][lane]);
        const int t = m * 16 + (lane & 15);
        ob_dense_epilogue<__bf16, OB_EPI_PART>(A, nt, t, t < A.T, lane >> 4, v[0], v[1], split);
    }
}
