// The float32 train-mode layer on bf16 matrix products (arithmetic: ob_train.h; tiles, loops and numbering: ob_train16.h, ob_mm.h).
//
// A float32 is the sum of three bf16 (each the nearest to what the ones before leave: 8 + 8 + 8 bits), a sign is exact in one:
//   z  = a S^T      three products, the parts of a = x h against S
//   ga = gz S       three, the parts of gz
//   gS = gz^T a     six: gz0 a0, gz0 a1, gz1 a0, gz0 a2, gz1 a1, gz2 a0; of the other three the largest is 2^-26 of its term, either sign (a float32 rounding: 2^-25)
// added into one set of float32 sums, smallest terms first.  The parts are the numbers themselves (exactly, from 2^-110 on), and a K step adds 32 products for one
// rounding where v_mfma_f32_16x16x4_f32 adds four, so z, ga and gS are closer to the 64-bit sums than with that instruction.  An infinite gz or x h gives NaN where
// one float32 product would be infinite (inf * 0 of the lower parts): either is a row that LayerNorm has made NaN already, or a gradient beyond float32.
// What bounds it: the matrix cores, 3 or 6 products for one, and below some 500 rows the length of the sums that a workgroup takes (the few tiles leave CUs idle).
// Forward + backward, v_mfma_f32_16x16x4_f32 products (at 84-97 TFLOP/s) -> these: 3600 rows 4096 -> 4096 4336 us -> 1141 (in a trace z 1397 -> 218, ga 1243 -> 250,
// gS 1562 -> 478), 1000 rows 1371 -> 464, 64 rows 554 -> 327, 512 rows 4096 -> 11008 1995 -> 883, 3600 rows 1376 -> 4100 1774 -> 581, 64 rows 1024 -> 2816 250 -> 170.
// Off the 64-bit results, norms, before / now: y 1.2e-6 / 9e-8, gx 1.1e-6 / 9e-8, gW 1.1e-6 / 3.8e-7 (3600 rows; 64 rows 4096 -> 1000 2.1e-7 / 9.5e-8, 2 rows 1024 -> 1000 1.23e-7 / 1.18e-7), the scales' 1.2e-6 / 1.6e-7.
#pragma once
#include "ob_train16.h"

#define OB_T32_PARTS 3

// eight floats -> their parts
__device__ __forceinline__ void ob_t32_split(const float (&v)[8], ob_u32x4 (&out)[OB_T32_PARTS])
{
    uint32_t w[OB_T32_PARTS][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        float r = v[e];
#pragma unroll
        for (int p = 0; p < OB_T32_PARTS; ++p) {
            const uint32_t b = __float_as_uint(r);
            // to nearest, but for those that would become infinite, infinities and NaN (cut off)
            const uint32_t q = (b & 0x7fffffffu) >= 0x7f7f8000u ? b : b + 0x8000u;
            w[p][e] = q & 0xffff0000u;
            const bool inf = (b & 0x7fffffffu) == 0x7f800000u;
            r = inf ? 0.f : r - __uint_as_float(w[p][e]);
        }
    }
#pragma unroll
    for (int p = 0; p < OB_T32_PARTS; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) out[p][e] = __builtin_amdgcn_perm(w[p][2 * e + 1], w[p][2 * e], 0x07060302u);
}
// 8 floats at p, those from `n` on zero
__device__ __forceinline__ void ob_t32_load(const float *p, int n, float (&v)[8])
{
    if (n >= 8 && ((uintptr_t)p & 15) == 0) {
        const ob_float4 a = reinterpret_cast<const ob_float4 *>(p)[0], b = reinterpret_cast<const ob_float4 *>(p)[1];
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[e] = a[e]; v[4 + e] = b[e]; }
        return;
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = e < n ? p[e] : 0.f;
}

// x -> parts of a = x h, [part][16-row band][column tile]; W -> S.  A wave takes four column tiles of a band.
struct ObT32Tiles { const float *p, *vec; char *out; size_t part; int rows, cols, bands, ct; };
template <int TX>
__global__ __launch_bounds__(256) void ob_t32_tiles_kernel(const ObT32Tiles A)
{
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, cg = (A.ct + 3) >> 2;
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6), band = unit / cg, c0 = (unit - band * cg) * 4, row = band * 16 + r;
    if (band >= A.bands) return;
    float v[4][8];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int col = (c0 + c) * 32 + 8 * g;
        ob_t32_load(A.p + (size_t)row * A.cols + col, row < A.rows ? A.cols - col : 0, v[c]);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c0 + c >= A.ct) return;                                    // (wave-uniform)
        const int col = (c0 + c) * 32 + 8 * g;
        char *out = A.out + ((size_t)band * A.ct + c0 + c) * 1024 + ob_t16_place(r, g);
        if (TX == OB_T16_SCALE) {
            float h[8];
            ob_t32_load(A.vec + col, A.cols - col, h);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] *= h[e];
            ob_u32x4 w[OB_T32_PARTS];
            ob_t32_split(v[c], w);
#pragma unroll
            for (int p = 0; p < OB_T32_PARTS; ++p) *reinterpret_cast<ob_u32x4 *>(out + p * A.part) = w[p];
        } else {
            ob_u32x4 w;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t lo = v[c][2 * e] > 0.f ? 0x3F80u : v[c][2 * e] < 0.f ? 0xBF80u : 0u, hi = v[c][2 * e + 1] > 0.f ? 0x3F80u : v[c][2 * e + 1] < 0.f ? 0xBF80u : 0u;      // NaN -> 0
                w[e] = lo | hi << 16;
            }
            *reinterpret_cast<ob_u32x4 *>(out) = w;
        }
    }
}

// x -> parts of (x h)^T: [16-column band][part, the lowest first][32-row tile] (ob_t16_turn_kernel; the LDS holds one part at a time)
struct ObT32Turn { const float *p, *vec; char *out; int rows, cols, rt, ct; };
__global__ __launch_bounds__(256) void ob_t32_turn_kernel(const ObT32Turn A)
{
    __shared__ __attribute__((aligned(16))) char smem[4][8 * 1024];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4, cg = (A.ct + 3) >> 2;
    const int unit = blockIdx.x * 4 + wave, tt = unit % A.rt, c0 = unit / A.rt * 4;
    if (c0 >= 4 * cg) return;                                          // (wave-uniform; no barrier below)
    ob_u32x4 w[4][2][OB_T32_PARTS];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int col = (c0 + c) * 32 + 8 * g;
        float h[8];
        ob_t32_load(A.vec + col, A.cols - col, h);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int row = tt * 32 + b * 16 + r;
            float v[8];
            ob_t32_load(A.p + (size_t)row * A.cols + col, row < A.rows ? A.cols - col : 0, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= h[e];
            ob_t32_split(v, w[c][b]);
        }
    }
    char *base = smem[wave];
#pragma unroll
    for (int p = 0; p < OB_T32_PARTS; ++p) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int b = 0; b < 2; ++b) *reinterpret_cast<ob_u32x4 *>(base + (2 * c + b) * 1024 + ob_t16_place(r, g)) = w[c][b][p];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        ob_u32x4 t[4][2];
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int i = 0; i < 2; ++i) t[c][i] = ob_t16_turned(base + 2 * c * 1024, i, r, g);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");             // (the next part goes where this one was read)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c0 + c < A.ct) {                                       // (wave-uniform)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    *reinterpret_cast<ob_u32x4 *>(A.out + (((size_t)(2 * (c0 + c) + i) * OB_T32_PARTS + OB_T32_PARTS - 1 - p) * A.rt + tt) * 1024 + ob_t16_place(r, g)) = t[c][i];
            }
    }
}

// C[t][n] = sum_r a(t, r) w(n, r) in segments: wofs[s] / aofs[s] = bytes from w / a to the segment's first tiles, nk[s] steps
struct ObT32Mm {
    const char *w, *a;
    int nw, na, wld, ald;          // groups of 16 outputs, tiles per band
    int nk[OB_T32_PARTS];
    size_t wofs[OB_T32_PARTS], aofs[OB_T32_PARTS];
    float *C; int rows, cols;
    const float *vec;              // OB_T16_GX: h;  OB_T16_GW: latent W, laid out as C
    const float *x; float *part;   // OB_T16_GX: [rows][cols]; sums of ga x over half a block's rows, [2 token blocks][cols]
    int vec4;                      // rows of C, vec and x in 16-byte pieces
    float *zp; size_t zld; int ns; // OB_T16_PART: as in ObT16Mm; the parts have as many steps
};

// 1.001 - tanh(w)^2 (bitnet.py:22-23), no farther from 64 bits anywhere than 1.001f - tanhf(w)^2, whose 1.001f alone is 4.7e-8 off: 0.001 is added last.  Below 0.8, with
// latent weights, 1 - w^2 P(w^2), P fitted to tanh(w)^2 / w^2 (4.3e-9 of 1 left); above 4 e / (1 + e)^2, e = exp(-2 |w|), where nothing cancels.  Root mean square and
// largest error at |w| in 0-0.02, 0.25-0.5, 0.5-0.8, 0.8-1, 2.5-4: 1.001f - tanhf(w)^2 5.8e-8 / 1.1e-7, 5.2e-8 / 1.2e-7, 6.7e-8 / 2.1e-7, 7.5e-8 / 2.2e-7, 9e-8 / 2.5e-7; the last
// form everywhere 7.1e-8 / 3.3e-7, 7.1e-8 / 2.8e-7, 6.0e-8 / 2.6e-7, 4.9e-8 / 2.1e-7, 2e-9 / 1e-8; the two 3.9e-8 / 7.7e-8, 2.2e-8 / 5.6e-8, 2.5e-8 / 8.4e-8, as it, as it.
__device__ __forceinline__ float ob_t32_ste_small(float w)
{
    const float q = w * w;
    float p = __builtin_fmaf(0.00799220707f, q, -0.0359845459f);
    p = __builtin_fmaf(p, q, 0.0928287283f);
    p = __builtin_fmaf(p, q, -0.195705429f);
    p = __builtin_fmaf(p, q, 0.377643019f);
    p = __builtin_fmaf(p, q, -0.666660547f);
    p = __builtin_fmaf(p, q, 1.0f);
    return __builtin_fmaf(-q, p, 1.0f) + 0.001f;
}
__device__ __forceinline__ float ob_t32_ste(float w)
{
    const float a = fabsf(w), e = __builtin_amdgcn_exp2f(-2.8853900817779268f * a), d = 1.0f + e;
    return a < 0.8f ? ob_t32_ste_small(w) : 4.0f * e * __builtin_amdgcn_rcpf(d * d) + 0.001f;
}

// as ob_t16_epilogue; x / W beside an output are requested 8 tiles ahead
template <int EPI, int MN, int MT, typename ACC>
__device__ __forceinline__ void ob_t32_epilogue(const ObT32Mm &A, int n0, int t0, int half, int lane, ACC acc)
{
    if constexpr (EPI == OB_T16_PART) { ob_t16_part<MN, MT>(A.zp + blockIdx.y * A.zld, A.rows, A.cols, n0, t0, lane, acc); return; }
    constexpr int JB = MT < 8 ? MT : 8, NB = MN * (MT / JB);           // batches of row tiles of one column tile
    static_assert(MT % JB == 0, "whole batches");
    const int lr = lane & 15, lg = lane >> 4;
    const float *q = EPI == OB_T16_GX ? A.x : A.vec;
    ob_float4 p[2][JB];
    const auto fetch = [&](int b) __attribute__((always_inline)) {
        const int n = n0 + b / (MT / JB) * 16 + 4 * lg, left = A.cols - n;
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            const int t = t0 + (b % (MT / JB) * JB + j) * 16 + lr;
            ob_float4 v = {0.f, 0.f, 0.f, 0.f};
            if (t < A.rows && left > 0) {
                if (A.vec4 && left >= 4) v = *reinterpret_cast<const ob_float4 *>(q + (size_t)t * A.cols + n);
                else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) if (e < left) v[e] = q[(size_t)t * A.cols + n + e];
                }
            }
            p[b & 1][j] = v;
        }
    };
    if (EPI != OB_T16_Z) fetch(0);
    float sum[4];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        if (EPI != OB_T16_Z && b + 1 < NB) fetch(b + 1);
        const int i = b / (MT / JB), jb = b % (MT / JB) * JB;
        const int n = n0 + i * 16 + 4 * lg, left = A.cols - n;         // four columns, `left` of them inside
        const bool v4 = A.vec4 && left >= 4;
        ob_float4 h4 = {0.f, 0.f, 0.f, 0.f};
        if (EPI == OB_T16_GX) {
#pragma unroll
            for (int e = 0; e < 4; ++e) { if (e < left) h4[e] = A.vec[n + e]; if (jb == 0) sum[e] = 0.f; }
        }
        if (EPI == OB_T16_GW) {                                        // W -> its factors
            float most = 0.f;
#pragma unroll
            for (int j = 0; j < 4 * JB; ++j) most = fmaxf(most, fabsf(p[b & 1][j >> 2][j & 3]));
            if (__builtin_amdgcn_ballot_w64(most >= 0.8f)) {           // (uniform)
#pragma unroll
                for (int j = 0; j < 4 * JB; ++j) p[b & 1][j >> 2][j & 3] = ob_t32_ste(p[b & 1][j >> 2][j & 3]);
            } else {
#pragma unroll
                for (int j = 0; j < 4 * JB; ++j) p[b & 1][j >> 2][j & 3] = ob_t32_ste_small(p[b & 1][j >> 2][j & 3]);
            }
        }
#pragma unroll
        for (int j = 0; j < JB; ++j) {
            const int t = t0 + (jb + j) * 16 + lr;
            if (t >= A.rows || left <= 0) continue;
            const size_t o = (size_t)t * A.cols + n;
            ob_float4 c = acc(i, jb + j);
            const ob_float4 d = p[b & 1][j];
            if (EPI == OB_T16_GX) {
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] += c[e] * d[e];
                c = c * h4;
            }
            if (EPI == OB_T16_GW) c = c * d;
            if (v4) *reinterpret_cast<ob_float4 *>(A.C + o) = c;
            else {
#pragma unroll
                for (int e = 0; e < 4; ++e) if (e < left) A.C[o + e] = c[e];
            }
        }
        if (EPI == OB_T16_GX && jb + JB == MT) {                       // over the 16 rows of the lane group
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[e] += OB_DPP_F(sum[e], 0xB1, 0xF);
                sum[e] += OB_DPP_F(sum[e], 0x4E, 0xF);
                sum[e] += OB_DPP_F(sum[e], 0x141, 0xF);
                sum[e] += OB_DPP_F(sum[e], 0x140, 0xF);
                if (lr == 0 && e < left && half < 2 * ((A.rows + 127) >> 7)) A.part[(size_t)half * A.cols + n + e] = sum[e];
            }
        }
    }
}

// both operands through the LDS (ob_mm_loop), 128 x 128 outputs: few tiles
template <int EPI, bool TRW, bool TRA>
__global__ __launch_bounds__(256, 2) void ob_t32_mm_kernel(const ObT32Mm A)
{
    constexpr int NB = 8, TB = 8, NST = 4, TILES = NB + TB, PER = TILES / 4, MN = NB / 2, MT = TB / 2;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wn = wave & 1, wt = wave >> 1, lr = lane & 15, lg = lane >> 4;
    int nb, tb;
    if (!ob_tile_of(blockIdx.x, (A.nw + NB - 1) / NB, (A.na + TB - 1) / TB, nb, tb)) return;      // (uniform)
    const char *src[PER];
    size_t step[PER];
    bool isw[PER];
#pragma unroll
    for (int d = 0; d < PER; ++d) {
        const int j = wave * PER + d;
        const bool w = j < NB, tr = w ? TRW : TRA;
        const int o = w ? j : j - NB, ld = w ? A.wld : A.ald, n = w ? A.nw : A.na, b0 = w ? nb * NB : tb * TB;
        const char *m = w ? A.w : A.a;
        isw[d] = w;
        if (tr) { src[d] = m + ((size_t)(o & 1) * ld + min(b0 / 2 + (o >> 1), ld - 1)) * 1024; step[d] = (size_t)ld * 2048; }
        else { src[d] = m + (size_t)min(b0 + o, n - 1) * ld * 1024; step[d] = 1024; }
    }
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char *)smem;
    const int plain = ob_t16_place(lr, lg);
    const auto frag = [&](bool tr, int buf, int t0, int i) -> ob_u32x4 {
        const char *base = smem + (buf * TILES + t0) * 1024;
        if (!tr) return *reinterpret_cast<const ob_u32x4 *>(base + i * 1024 + plain);
        return ob_t16_turned(base + (i >> 1) * 2048, i & 1, lr, lg);
    };
    ob_float4 acc[MN][MT];
    const auto segment = [&]<bool CONT>(int s) __attribute__((always_inline)) {
        int k0;
        const int nk = ob_t16_slice<EPI>(A.nk[s], A.ns, k0);
        const char *at[PER];
#pragma unroll
        for (int d = 0; d < PER; ++d) at[d] = src[d] + (isw[d] ? A.wofs[s] : A.aofs[s]) + (size_t)k0 * step[d];
        ob_mm_loop<true, MN, MT, PER, NST, CONT>(acc, nk, [&](int buf, int i) { return frag(TRW, buf, 0, wn * MN + i); },
            [&](int buf, int j) { return frag(TRA, buf, NB, wt * MT + j); },
            [&](int d, int k, int buf) { ob_dma_1k(at[d] + (size_t)min(k, nk - 1) * step[d], lane * 16, lds0 + (uint32_t)(buf * TILES + wave * PER + d) * 1024); });
    };
    segment.template operator()<false>(0);
    segment.template operator()<true>(1);
    segment.template operator()<true>(2);
    ob_t32_epilogue<EPI, MN, MT>(A, (nb * NB + wn * MN) * 16, (tb * TB + wt * MT) * 16, tb * 2 + wt, lane, [&](int i, int j) -> const ob_float4 & { return acc[i][j]; });
}

// ... with one operand straight into registers (ob_t16_wr_kernel)
template <int EPI, bool TRL, bool SWAP, int MT>
__global__ __launch_bounds__(256, MT > 8 ? 1 : 2) void ob_t32_wr_kernel(const ObT32Mm A)
{
    constexpr int MN = 4, PER = MT / 4, NST = ob_wr_steps(MT);
    static_assert(MT % 4 == 0, "pairs of tiles, as many transfers in every wave");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lr = lane & 15, lg = lane >> 4;
    const char *dm = SWAP ? A.a : A.w, *lm = SWAP ? A.w : A.a;
    const int nd = SWAP ? A.na : A.nw, dld = SWAP ? A.ald : A.wld, nl = SWAP ? A.nw : A.na, lld = SWAP ? A.wld : A.ald;
    int nb, tb;
    if (!ob_tile_of(blockIdx.x, SWAP ? (nl + MT - 1) / MT : (nd + 15) / 16, SWAP ? (nd + 15) / 16 : (nl + MT - 1) / MT, nb, tb)) return;      // (uniform)
    const int d0 = (SWAP ? tb : nb) * 16 + wave * MN, l0 = (SWAP ? nb : tb) * MT;
    const char *lsrc[PER], *dsrc[MN];
    uint32_t ldst[PER];
    const size_t step = TRL ? (size_t)lld * 2048 : 1024;
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char *)smem;
#pragma unroll
    for (int d = 0; d < PER; ++d) {
        const int o = wave * PER + d;
        lsrc[d] = lm + (TRL ? (size_t)(o & 1) * lld + min(l0 / 2 + (o >> 1), lld - 1) : (size_t)min(l0 + o, nl - 1) * lld) * 1024;
        ldst[d] = lds0 + (uint32_t)o * 1024;
    }
#pragma unroll
    for (int i = 0; i < MN; ++i) dsrc[i] = dm + (size_t)min(d0 + i, nd - 1) * dld * 1024;
    const int plain = ob_t16_place(lr, lg);
    ob_float4 acc[MN][MT];
    const auto segment = [&]<bool CONT>(int s) __attribute__((always_inline)) {
        const char *src[PER], *nxt[PER], *wb[MN];
        int k0;
        const int nk = ob_t16_slice<EPI>(A.nk[s], A.ns, k0);
#pragma unroll
        for (int d = 0; d < PER; ++d) { src[d] = lsrc[d] + (SWAP ? A.wofs[s] : A.aofs[s]) + (size_t)k0 * step; nxt[d] = src[d] + (NST - 1) * step; }
#pragma unroll
        for (int i = 0; i < MN; ++i) wb[i] = dsrc[i] + (SWAP ? A.aofs[s] : A.wofs[s]) + (size_t)k0 * 1024;
        ob_wr_loop<true, SWAP, MT, PER, NST, CONT>(acc, nk, wb, plain,
            [&](int buf, int j) -> ob_u32x4 {
                if constexpr (TRL) return ob_t16_turned(smem + (buf * MT + (j & ~1)) * 1024, j & 1, lr, lg);
                else return *reinterpret_cast<const ob_u32x4 *>(smem + (buf * MT + j) * 1024 + plain);
            },
            [&](int d, int k, int buf) { ob_dma_1k(src[d] + (size_t)k * step, lane * 16, ldst[d] + buf * MT * 1024); },
            [&](int d, int, int buf) { ob_dma_1k(nxt[d], lane * 16, ldst[d] + buf * MT * 1024); nxt[d] += step; });
    };
    segment.template operator()<false>(0);
    segment.template operator()<true>(1);
    segment.template operator()<true>(2);
    if constexpr (SWAP) ob_t32_epilogue<EPI, MT, MN>(A, l0 * 16, d0 * 16, tb * 4 + wave, lane, [&](int i, int j) -> const ob_float4 & { return acc[j][i]; });
    else ob_t32_epilogue<EPI, MN, MT>(A, d0 * 16, l0 * 16, 0, lane, [&](int i, int j) -> const ob_float4 & { return acc[i][j]; });
}

// LayerNorm of z g, rows up to 16384 wide in registers (N % 4 == 0, 16-byte aligned): ob_train_ln_fwd_kernel's arithmetic, z read once
template <int NV>
__global__ __launch_bounds__(256) void ob_t32_ln_kernel(const float *__restrict__ z, const float *__restrict__ g, const float *__restrict__ bias, float *__restrict__ y,
                                                        float *__restrict__ stats, int N, float eps)
{
    __shared__ float red[2][4];
    const int tid = threadIdx.x;
    const size_t row = (size_t)blockIdx.x * N;
    ob_float4 u[NV];
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int n = (v * 256 + tid) * 4;
        u[v] = (ob_float4){0.f, 0.f, 0.f, 0.f};
        if (n < N) u[v] = *reinterpret_cast<const ob_float4 *>(z + row + n) * *reinterpret_cast<const ob_float4 *>(g + n);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) s += (u[v][0] + u[v][1]) + (u[v][2] + u[v][3]);
    const float mean = ob_block_sum(s, red[0]) / (float)N;
#pragma unroll
    for (int v = 0; v < NV; ++v)
        if ((v * 256 + tid) * 4 < N) {
#pragma unroll
            for (int e = 0; e < 4; ++e) { const float d = u[v][e] - mean; q += d * d; }
        }
    const float rstd = 1.0f / sqrtf(ob_block_sum(q, red[1]) / (float)N + eps);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int n = (v * 256 + tid) * 4;
        if (n >= N) break;
        ob_float4 o = (u[v] - mean) * rstd;
        if (bias) o += *reinterpret_cast<const ob_float4 *>(bias + n);
        *reinterpret_cast<ob_float4 *>(y + row + n) = o;
    }
    if (tid == 0) { stats[2 * blockIdx.x] = mean; stats[2 * blockIdx.x + 1] = rstd; }
}

// backward through the LayerNorm: the rows' means {gy, gy uh}, then the parts of gz, [part][16-row band][column tile], 16 rows and a column tile at a time, with
// the column sums of gu z and gy over a slice of the bands: part[slice][2][N]
struct ObT32Gz { const float *gy, *z, *g, *stats; float *rowc, *part; char *gz; size_t gz_part; int T, N, bands, ct, per; };
__global__ __launch_bounds__(256) void ob_t32_rowc_kernel(const ObT32Gz A)
{
    __shared__ float red[2][4];
    const int t = blockIdx.x;
    const float mean = A.stats[2 * t], rstd = A.stats[2 * t + 1];
    const float *zr = A.z + (size_t)t * A.N, *gr = A.gy + (size_t)t * A.N;
    float s1 = 0.f, s2 = 0.f;
    for (int n = threadIdx.x * 8; n < A.N; n += 2048) {
        float z[8], g[8], d[8];
        ob_t32_load(zr + n, A.N - n, z);
        ob_t32_load(A.g + n, A.N - n, g);
        ob_t32_load(gr + n, A.N - n, d);
#pragma unroll
        for (int e = 0; e < 8; ++e) { s1 += d[e]; s2 += d[e] * ((z[e] * g[e] - mean) * rstd); }      // (d = 0 beyond the row)
    }
    const float c1 = ob_block_sum(s1, red[0]) / (float)A.N, c2 = ob_block_sum(s2, red[1]) / (float)A.N;
    if (threadIdx.x == 0) { A.rowc[2 * t] = c1; A.rowc[2 * t + 1] = c2; }
}
__global__ __launch_bounds__(256) void ob_t32_gz_kernel(const ObT32Gz A)
{
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, c = blockIdx.x * 4 + (threadIdx.x >> 6), n = c * 32 + 8 * g;
    if (c >= A.ct) return;
    const int b0 = blockIdx.y * A.per, b1 = min(A.bands, b0 + A.per);
    float gn[8], sg[8], sb[8];
    ob_t32_load(A.g + n, A.N - n, gn);
#pragma unroll
    for (int e = 0; e < 8; ++e) sg[e] = sb[e] = 0.f;
    for (int b = b0; b < b1; ++b) {
        const int t = b * 16 + r, left = t < A.T ? A.N - n : 0;
        float zz[8], d[8], o[8];
        ob_t32_load(A.z + (size_t)t * A.N + n, left, zz);
        ob_t32_load(A.gy + (size_t)t * A.N + n, left, d);
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = 0.f;
        if (t < A.T) {
            const float mean = A.stats[2 * t], rstd = A.stats[2 * t + 1], c1 = A.rowc[2 * t], c2 = A.rowc[2 * t + 1];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float uh = (zz[e] * gn[e] - mean) * rstd, gu = rstd * (d[e] - c1 - uh * c2);
                sg[e] += gu * zz[e];
                sb[e] += d[e];
                if (e < left) o[e] = gu * gn[e];
            }
        }
        ob_u32x4 w[OB_T32_PARTS];
        ob_t32_split(o, w);
#pragma unroll
        for (int p = 0; p < OB_T32_PARTS; ++p) *reinterpret_cast<ob_u32x4 *>(A.gz + p * A.gz_part + ((size_t)b * A.ct + c) * 1024 + ob_t16_place(r, g)) = w[p];
    }
    float *p = A.part + (size_t)blockIdx.y * 2 * A.N + n;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            float v = k ? sb[e] : sg[e];
            v += OB_DPP_F(v, 0xB1, 0xF);
            v += OB_DPP_F(v, 0x4E, 0xF);
            v += OB_DPP_F(v, 0x141, 0xF);
            v += OB_DPP_F(v, 0x140, 0xF);
            if (r == 0 && n + e < A.N) p[(size_t)k * A.N + e] = v;
        }
    }
}

// out_j[c] = sum over the slices, in order, of part[s][j][c]; out_1 may be null
template <int NOUT>
__global__ __launch_bounds__(256) void ob_t32_cols_kernel(const float *__restrict__ part, float *__restrict__ out0, float *__restrict__ out1, int C, int slices)
{
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
#pragma unroll
    for (int j = 0; j < NOUT; ++j) {
        float *o = j == 0 ? out0 : out1;
        if (!o) continue;
        float a = 0.f;
#pragma unroll 8
        for (int s = 0; s < slices; ++s) a += part[((size_t)s * NOUT + j) * C + c];
        o[c] = a;
    }
}
