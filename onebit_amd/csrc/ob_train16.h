// The float16 train-mode layer on LDS-DMA matrix products (arithmetic and rounding points: ob_train.h).
//
// The three products read three matrices, each formed once by an elementwise pass, both ways:
//   a = fp16(x h) [T][K]     z = a S^T (reduced over K)      gS = gz^T a (reduced over T)
//   S = sign(W)   [N][K]     z = a S^T                       ga = gz S   (reduced over N)
//   gz            [T][N]     ga = gz S                       gS = gz^T a
// stored as 1 KB tiles of 16 rows x 32 columns, [16-row band][column tile], zero beyond the matrix up to 32 rows and columns.  Reduced over its
// columns, a tile is an MFMA operand as it lies (one ds_read_b128); reduced over its rows, two tiles are two operands through the transposing
// read (ds_read_b64_tr_b16).  The 16-byte piece (row, g = column / 8) sits at place 16 g + (row ^ 4 (g & 1)): both reads are free of bank
// conflicts.  Loop, tile shapes and numbering: ob_mm.h.
// What bounds it: the matrix cores for the products (the kernel that transformed operands on their way from registers to LDS reached 430-510
// TFLOP/s), memory for the passes.  T = 4096, 4096 -> 11008, forward + backward: 2496 us before, 1227 now; in a trace the products 309-342 (z), 376-410
// (ga) and 406-446 us (gS) = 1.2 / 0.98 / 0.91 PFLOP/s at best, the passes 215 us at 4-5 TB/s.  64 rows: 811 us before, 320 now.
#pragma once
#include "ob_mm.h"

struct ObT16Tiles { const _Float16 *p, *vec; char *out; int rows, cols, bands, ct; };
enum { OB_T16_SCALE = 0, OB_T16_SIGN = 1 };

// 8 elements at p, those from `n` on zero
__device__ __forceinline__ ob_half8 ob_t16_load(const _Float16 *p, int n)
{
    ob_half8 v = (ob_half8)(_Float16)0;
    if (n >= 8 && ((uintptr_t)p & 15) == 0) return *reinterpret_cast<const ob_half8 *>(p);
#pragma unroll
    for (int e = 0; e < 8; ++e) if (e < n) v[e] = p[e];
    return v;
}
__device__ __forceinline__ int ob_t16_place(int row, int g) { return (16 * g + (row ^ ((g & 1) << 2))) * 16; }

// x -> a, W -> S: a wave takes four column tiles of a band (256 bytes of each of its 16 rows)
template <int TX>
__global__ __launch_bounds__(256) void ob_t16_tiles_kernel(const ObT16Tiles A)
{
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, cg = (A.ct + 3) >> 2;
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6), band = unit / cg, c0 = (unit - band * cg) * 4, row = band * 16 + r;
    if (band >= A.bands) return;
    ob_half8 v[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int col = (c0 + c) * 32 + 8 * g;
        v[c] = ob_t16_load(A.p + (size_t)row * A.cols + col, row < A.rows ? A.cols - col : 0);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c0 + c >= A.ct) return;                                    // (wave-uniform)
        const int col = (c0 + c) * 32 + 8 * g;
        if (TX == OB_T16_SCALE) v[c] = v[c] * ob_t16_load(A.vec + col, A.cols - col);
        else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[c][e] = (_Float16)(v[c][e] > (_Float16)0 ? 1.0f : v[c][e] < (_Float16)0 ? -1.0f : 0.0f);      // NaN -> 0
        }
        *reinterpret_cast<ob_half8 *>(A.out + ((size_t)band * A.ct + c0 + c) * 1024 + ob_t16_place(r, g)) = v[c];
    }
}

// C[t][n] = sum_r a(t, r) w(n, r).  TRW / TRA: the operand's tiles are reduced over their rows (nw / na count its 16-element groups either way).
enum { OB_T16_Z = 0, OB_T16_GX = 1, OB_T16_GW = 2 };
struct ObT16Mm {
    const char *w, *a;
    int nw, na, wld, ald, nk;      // groups of 16 outputs, tiles per band, steps of 32
    _Float16 *C; int rows, cols;
    const _Float16 *vec;           // OB_T16_GX: h;  OB_T16_GW: latent W, laid out as C
    const _Float16 *x; float *part;      // OB_T16_GX: [rows][cols]; sums of ga x over half a block's rows, [2 token blocks][cols]
    int vec4;                      // rows of C, vec and x in 8-byte pieces
};

// 1.001 - tanh(w)^2 with the tensor ops' roundings (SignSTEFunc.backward, bitnet.py:22-23; ob_train.h); tanh = 1 - 2 / (1 + e^2|w|) from the exp2
// and reciprocal instructions: 2e-7 absolute before its rounding to 11 bits, and it enters as 1.001 - t^2
__device__ __forceinline__ float ob_t16_ste(float w)
{
    const float t = 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(2.8853900817779268f * fabsf(w)));
    const float t1 = ob_round_h(t), t2 = ob_round_h(t1 * t1);
    return ob_round_h((float)(_Float16)1.001f - t2);
}

template <int EPI, bool TRW, bool TRA, int NB, int TB, int NST>
__global__ __launch_bounds__(256, 2) void ob_t16_mm_kernel(const ObT16Mm A)
{
    constexpr int TILES = NB + TB, PER = TILES / 4, MN = NB / 2, MT = TB / 2;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wn = wave & 1, wt = wave >> 1, lr = lane & 15, lg = lane >> 4;
    int nb, tb;
    if (!ob_tile_of(blockIdx.x, (A.nw + NB - 1) / NB, (A.na + TB - 1) / TB, nb, tb)) return;      // (uniform)
    const char *src[PER];
    size_t step[PER];
#pragma unroll
    for (int d = 0; d < PER; ++d) {
        const int j = wave * PER + d;
        const bool w = j < NB, tr = w ? TRW : TRA;
        const int o = w ? j : j - NB, ld = w ? A.wld : A.ald, n = w ? A.nw : A.na, b0 = w ? nb * NB : tb * TB;
        const char *m = w ? A.w : A.a;
        if (tr) { src[d] = m + ((size_t)(o & 1) * ld + min(b0 / 2 + (o >> 1), ld - 1)) * 1024; step[d] = (size_t)ld * 2048; }
        else { src[d] = m + (size_t)min(b0 + o, n - 1) * ld * 1024; step[d] = 1024; }
    }
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char *)smem;
    const auto dma = [&](int d, int k, int buf) {
        ob_dma_1k(src[d] + (size_t)min(k, A.nk - 1) * step[d], lane * 16, lds0 + (uint32_t)(buf * TILES + wave * PER + d) * 1024);
    };
    // operand i of a side whose tiles start at tile t0 of the step's buffer
    const int plain = ob_t16_place(lr, lg);
    const auto frag = [&](bool tr, int buf, int t0, int i) -> ob_u32x4 {
        const char *base = smem + (buf * TILES + t0) * 1024;
        if (!tr) return *reinterpret_cast<const ob_u32x4 *>(base + i * 1024 + plain);
        typedef short v4s __attribute__((ext_vector_type(4)));
        typedef short v8s __attribute__((ext_vector_type(8)));
        typedef __attribute__((address_space(3))) v4s lds_v4s;
        // rows 8 lg .. + 7 of the 32 (two bands), columns 16 (i & 1) .. of the 32-column tile i / 2: this lane's piece of a 4-row x 16-column block
        const int g = 2 * (i & 1) + ((lr & 3) >> 1), row = 8 * (lg & 1) + (lr >> 2);
        const char *p = base + ((i >> 1) * 2 + (lg >> 1)) * 1024 + 8 * (lr & 1);
        const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(p + ob_t16_place(row, g)));
        const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(p + ob_t16_place(row + 4, g)));
        return __builtin_bit_cast(ob_u32x4, (v8s){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
    };
    ob_float4 acc[MN][MT];
    ob_mm_loop<false, MN, MT, PER, NST>(acc, A.nk, [&](int buf, int i) { return frag(TRW, buf, 0, wn * MN + i); },
                                        [&](int buf, int j) { return frag(TRA, buf, NB, wt * MT + j); }, dma);
#pragma unroll
    for (int i = 0; i < MN; ++i) {
        const int n = (nb * NB + wn * MN + i) * 16 + 4 * lg, left = A.cols - n;      // four columns, `left` of them inside
        const bool v4 = A.vec4 && left >= 4;
        ob_half4 h4 = (ob_half4)(_Float16)0;
        float sum[4] = {0.f, 0.f, 0.f, 0.f};                           // (scalars: OB_DPP_F of a vector's element reads element 0)
        if (EPI == OB_T16_GX) {
#pragma unroll
            for (int e = 0; e < 4; ++e) if (e < left) h4[e] = A.vec[n + e];
        }
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int t = (tb * TB + wt * MT + j) * 16 + lr;
            if (t >= A.rows || left <= 0) continue;
            const size_t o = (size_t)t * A.cols + n;
            ob_half4 c, p = (ob_half4)(_Float16)0;
#pragma unroll
            for (int e = 0; e < 4; ++e) c[e] = (_Float16)acc[i][j][e];
            const _Float16 *q = EPI == OB_T16_GX ? A.x : A.vec;
            if (EPI != OB_T16_Z) {
                if (v4) p = *reinterpret_cast<const ob_half4 *>(q + o);
                else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) if (e < left) p[e] = q[o + e];
                }
            }
            if (EPI == OB_T16_GX) {
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] += (float)(_Float16)(c[e] * p[e]);
                c = c * h4;
            }
            if (EPI == OB_T16_GW) {
#pragma unroll
                for (int e = 0; e < 4; ++e) c[e] = (_Float16)((float)c[e] * ob_t16_ste((float)p[e]));
            }
            if (v4) *reinterpret_cast<ob_half4 *>(A.C + o) = c;
            else {
#pragma unroll
                for (int e = 0; e < 4; ++e) if (e < left) A.C[o + e] = c[e];
            }
        }
        if (EPI == OB_T16_GX) {                                        // over the 16 rows of the lane group
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                sum[e] += OB_DPP_F(sum[e], 0xB1, 0xF);
                sum[e] += OB_DPP_F(sum[e], 0x4E, 0xF);
                sum[e] += OB_DPP_F(sum[e], 0x141, 0xF);
                sum[e] += OB_DPP_F(sum[e], 0x140, 0xF);
                if (lr == 0 && e < left) A.part[(size_t)(tb * 2 + wt) * A.cols + n + e] = sum[e];
            }
        }
    }
}

// LayerNorm of z g, rows up to 16384 wide in registers (N % 8 == 0, 16-byte aligned): ob_train_ln_fwd_kernel's arithmetic, z read once
template <int NV>
__global__ __launch_bounds__(256) void ob_t16_ln_kernel(const _Float16 *__restrict__ z, const _Float16 *__restrict__ g, const _Float16 *__restrict__ bias,
                                                        _Float16 *__restrict__ y, float *__restrict__ stats, int N, float eps)
{
    __shared__ float red[2][4];
    const int tid = threadIdx.x;
    const size_t row = (size_t)blockIdx.x * N;
    ob_half8 u[NV];
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int n = (v * 256 + tid) * 8;
        u[v] = (ob_half8)(_Float16)0;
        if (n < N) u[v] = *reinterpret_cast<const ob_half8 *>(z + row + n) * *reinterpret_cast<const ob_half8 *>(g + n);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v)
#pragma unroll
        for (int e = 0; e < 8; ++e) s += (float)u[v][e];
    const float mean = ob_block_sum(s, red[0]) / (float)N;
#pragma unroll
    for (int v = 0; v < NV; ++v)
        if ((v * 256 + tid) * 8 < N) {
#pragma unroll
            for (int e = 0; e < 8; ++e) { const float d = (float)u[v][e] - mean; q += d * d; }
        }
    const float rstd = 1.0f / sqrtf(ob_block_sum(q, red[1]) / (float)N + eps);
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int n = (v * 256 + tid) * 8;
        if (n >= N) break;
        ob_half8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = (_Float16)(((float)u[v][e] - mean) * rstd);
        if (bias) o = o + *reinterpret_cast<const ob_half8 *>(bias + n);
        *reinterpret_cast<ob_half8 *>(y + row + n) = o;
    }
    if (tid == 0) { stats[2 * blockIdx.x] = mean; stats[2 * blockIdx.x + 1] = rstd; }
}

// backward through the LayerNorm, first the rows' means {gy, gy uh} (ob_train_ln_bwd_kernel), then gz, 16 rows and a column tile at a time, with the
// column sums of gu z and gy over a slice of the bands: part[slice][2][N]
struct ObT16Gz { const _Float16 *gy, *z, *g; const float *stats; float *rowc, *part; char *gz; int T, N, bands, ct, per; };
__global__ __launch_bounds__(256) void ob_t16_rowc_kernel(const ObT16Gz A)
{
    __shared__ float red[2][4];
    const int t = blockIdx.x;
    const float mean = A.stats[2 * t], rstd = A.stats[2 * t + 1];
    const _Float16 *zr = A.z + (size_t)t * A.N, *gr = A.gy + (size_t)t * A.N;
    float s1 = 0.f, s2 = 0.f;
    for (int n = threadIdx.x * 8; n < A.N; n += 2048) {
        const ob_half8 u = ob_t16_load(zr + n, A.N - n) * ob_t16_load(A.g + n, A.N - n), d = ob_t16_load(gr + n, A.N - n);
#pragma unroll
        for (int e = 0; e < 8; ++e) { s1 += (float)d[e]; s2 += (float)d[e] * (((float)u[e] - mean) * rstd); }      // (d = 0 beyond the row)
    }
    const float c1 = ob_block_sum(s1, red[0]) / (float)A.N, c2 = ob_block_sum(s2, red[1]) / (float)A.N;
    if (threadIdx.x == 0) { A.rowc[2 * t] = c1; A.rowc[2 * t + 1] = c2; }
}
__global__ __launch_bounds__(256) void ob_t16_gz_kernel(const ObT16Gz A)
{
    const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4, c = blockIdx.x * 4 + (threadIdx.x >> 6), n = c * 32 + 8 * g;
    if (c >= A.ct) return;
    const int b0 = blockIdx.y * A.per, b1 = min(A.bands, b0 + A.per);
    const ob_half8 gn = ob_t16_load(A.g + n, A.N - n);
    float sg[8], sb[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) sg[e] = sb[e] = 0.f;
    for (int b = b0; b < b1; ++b) {
        const int t = b * 16 + r, left = t < A.T ? A.N - n : 0;
        const ob_half8 zz = ob_t16_load(A.z + (size_t)t * A.N + n, left), d = ob_t16_load(A.gy + (size_t)t * A.N + n, left), u = zz * gn;
        ob_half8 o = (ob_half8)(_Float16)0;
        if (t < A.T) {
            const float mean = A.stats[2 * t], rstd = A.stats[2 * t + 1], c1 = A.rowc[2 * t], c2 = A.rowc[2 * t + 1];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float uh = ((float)u[e] - mean) * rstd;
                const _Float16 gu = (_Float16)(rstd * ((float)d[e] - c1 - uh * c2));
                sg[e] += (float)gu * (float)zz[e];
                sb[e] += (float)d[e];
                if (e < left) o[e] = gu * gn[e];
            }
        }
        *reinterpret_cast<ob_half8 *>(A.gz + ((size_t)b * A.ct + c) * 1024 + ob_t16_place(r, g)) = o;
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

// out_j[c] = fp16(sum over the slices, in order, of part[s][j][c]); out_1 may be null
template <int NOUT>
__global__ __launch_bounds__(256) void ob_t16_cols_kernel(const float *__restrict__ part, _Float16 *__restrict__ out0, _Float16 *__restrict__ out1, int C, int slices)
{
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
#pragma unroll
    for (int j = 0; j < NOUT; ++j) {
        _Float16 *o = j == 0 ? out0 : out1;
        if (!o) continue;
        float a = 0.f;
#pragma unroll 8
        for (int s = 0; s < slices; ++s) a += part[((size_t)s * NOUT + j) * C + c];
        o[c] = (_Float16)a;
    }
}
