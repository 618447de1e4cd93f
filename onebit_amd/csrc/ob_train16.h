// The float16 train-mode layer on LDS-DMA matrix products (arithmetic and rounding points: ob_train.h).
//
// The three products read three matrices that elementwise passes form, each both ways (S and x h by the forward and again by the backward, which is handed no
// tiles: 32 and 14 us at the size below):
//   a = fp16(x h) [T][K]     z = a S^T (reduced over K)      gS = gz^T a (reduced over T)
//   S = sign(W)   [N][K]     z = a S^T                       ga = gz S   (reduced over N)
//   gz            [T][N]     ga = gz S                       gS = gz^T a
// stored as 1 KB tiles of 16 rows x 32 columns, [16-row band][column tile], zero beyond the matrix up to 32 rows and columns.  Reduced over its
// columns, a tile is an MFMA operand as it lies (16 bytes a lane); reduced over its rows, two tiles are two operands through the transposing
// read (ds_read_b64_tr_b16).  The 16-byte piece (row, g = column / 8) sits at place 16 g + (row ^ 4 (g & 1)): both reads are free of bank
// conflicts.  Every product has one operand that lies as it is reduced, and goes straight to registers with it: S for z, gz for ga, and for gS a^T, whose tiles
// their pass turns.  Loops, tile shapes and numbering: ob_mm.h.
// What bounds it: the chip's power for the products, memory for the passes.  T = 4096, 4096 -> 11008, forward + backward: 1217 us with both operands through the
// LDS, 1037 with one of them straight to registers, 972 now that outputs go through the LDS; in a trace the products 343 -> 296 (z), 408 -> 286 (ga) and 441 -> 310 us
// (gS) = 1.25, 1.29 and 1.19 PFLOP/s, the passes 205 us at 4-5 TB/s.  Each product alone in a loop, at 1.39 kW of the 1.4 that the chip is given: 251 us at 2.08 GHz, 222 at 2.19 and 338 at 1.61 (gS multiplies full-range values by full-range
// values, the others by signs).
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

// MFMA operand i (of two) of a pair of tiles (32 rows x 32 columns at p) reduced over its rows, through the transposing read: this lane's 8 of the rows,
// column 16 i + lr
__device__ __forceinline__ ob_u32x4 ob_t16_turned(const char *p, int i, int lr, int lg)
{
    typedef short v4s __attribute__((ext_vector_type(4)));
    typedef short v8s __attribute__((ext_vector_type(8)));
    typedef __attribute__((address_space(3))) v4s lds_v4s;
    // rows 8 lg .. + 7 of the 32 (two bands), columns 16 i ..: this lane's piece of a 4-row x 16-column block
    const int g = 2 * i + ((lr & 3) >> 1), row = 8 * (lg & 1) + (lr >> 2);
    p += (lg >> 1) * 1024 + 8 * (lr & 1);
    const v4s lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(p + ob_t16_place(row, g)));
    const v4s hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s *)(p + ob_t16_place(row + 4, g)));
    return __builtin_bit_cast(ob_u32x4, (v8s){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]});
}

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

// x -> (x h)^T: tiles of 16 columns x 32 rows of x, [16-column band][32-row tile], the operand's transposing read done here once.  A wave takes 32 rows x four
// column tiles (256 bytes of each row), lays them into the LDS as the pass above lays them into memory and reads them back turned.
struct ObT16Turn { const _Float16 *p, *vec; char *out; int rows, cols, rt, ct; };      // rt, ct: tiles of 32 rows / columns
__global__ __launch_bounds__(256) void ob_t16_turn_kernel(const ObT16Turn A)
{
    __shared__ __attribute__((aligned(16))) char smem[4][8 * 1024];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, r = lane & 15, g = lane >> 4, cg = (A.ct + 3) >> 2;
    const int unit = blockIdx.x * 4 + wave, tt = unit % A.rt, c0 = unit / A.rt * 4;
    if (c0 >= 4 * cg) return;                                          // (wave-uniform; no barrier below)
    ob_half8 v[2][4], h[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int col = (c0 + c) * 32 + 8 * g;
        h[c] = ob_t16_load(A.vec + col, A.cols - col);
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int row = tt * 32 + b * 16 + r;
            v[b][c] = ob_t16_load(A.p + (size_t)row * A.cols + col, row < A.rows ? A.cols - col : 0);
        }
    }
    char *base = smem[wave];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int b = 0; b < 2; ++b) *reinterpret_cast<ob_half8 *>(base + (2 * c + b) * 1024 + ob_t16_place(r, g)) = v[b][c] * h[c];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        if (c0 + c >= A.ct) return;                                    // (wave-uniform)
#pragma unroll
        for (int i = 0; i < 2; ++i)
            *reinterpret_cast<ob_u32x4 *>(A.out + ((size_t)(2 * (c0 + c) + i) * A.rt + tt) * 1024 + ob_t16_place(r, g)) = ob_t16_turned(base + 2 * c * 1024, i, r, g);
    }
}

// The lane's number, made here: the products' loop has no register left for what only stands behind it
__device__ __forceinline__ int ob_t16_lane()
{
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}

// C[t][n] = sum_r a(t, r) w(n, r).  TRW / TRA: the operand's tiles are reduced over their rows (nw / na count its 16-element groups either way).
enum { OB_T16_Z = 0, OB_T16_GX = 1, OB_T16_GW = 2, OB_T16_PART = 3 };      // PART: a slice of the steps, its float32 sums to zp
struct ObT16Mm {
    const char *w, *a;
    int nw, na, wld, ald, nk;      // groups of 16 outputs, tiles per band, steps of 32
    _Float16 *C; int rows, cols;
    const _Float16 *vec;           // OB_T16_GX: h;  OB_T16_GW: latent W, laid out as C
    const _Float16 *x; float *part;      // OB_T16_GX: [rows][cols]; sums of ga x over half a block's rows, [2 token blocks][cols]
    int vec4;                      // rows of C, vec and x in 8-byte pieces
    float *zp; size_t zld; int ns; // OB_T16_PART: slice blockIdx.y of ns, its sums from zp + zld * slice on
};
// this workgroup's steps [k0, k0 + nk) of A's
template <int EPI> __device__ __forceinline__ int ob_t16_slice(int nk, int ns, int &k0)
{
    if (EPI != OB_T16_PART) { k0 = 0; return nk; }
    k0 = (int)((int64_t)nk * blockIdx.y / ns);
    return (int)((int64_t)nk * (blockIdx.y + 1) / ns) - k0;
}
template <int MN, int MT, typename ACC>
__device__ __forceinline__ void ob_t16_part(float *zp, int rows, int cols, int n0, int t0, int lane, ACC acc)
{
    const int lr = lane & 15, lg = lane >> 4;
#pragma unroll
    for (int i = 0; i < MN; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int n = n0 + i * 16 + 4 * lg, t = t0 + j * 16 + lr;
            if (t >= rows || n >= cols) continue;
            float *o = zp + (size_t)t * cols + n;
            if ((cols & 3) == 0) *reinterpret_cast<ob_float4 *>(o) = acc(i, j);
            else {
#pragma unroll
                for (int e = 0; e < 4; ++e) if (n + e < cols) o[e] = acc(i, j)[e];
            }
        }
}

// 1.001 - tanh(w)^2 with the tensor ops' roundings (SignSTEFunc.backward, bitnet.py:22-23; ob_train.h); tanh = 1 - 2 / (1 + e^2|w|) from the exp2
// and reciprocal instructions: 2e-7 absolute before its rounding to 11 bits, and it enters as 1.001 - t^2
__device__ __forceinline__ float ob_t16_ste(float w)
{
    const float t = 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(2.8853900817779268f * fabsf(w)));
    const float t1 = ob_round_h(t), t2 = ob_round_h(t1 * t1);
    return ob_round_h((float)(_Float16)1.001f - t2);
}

// MN x MT tiles of outputs from column n0, row t0 on: a lane has four columns n0 + 16 i + 4 lg .. of row t0 + 16 j + lr.  `half`: the rows' place in A.part.
// x / W beside an output are requested 16 tiles ahead: stores lie between the loads, and hipcc leaves them in order (one at a time, the weight gradient's
// epilogue took 38 us a 256 x 256 tile).
template <int EPI, int MN, int MT, typename ACC>
__device__ __forceinline__ void ob_t16_epilogue(const ObT16Mm &A, int n0, int t0, int half, int lane, ACC acc)
{
    if constexpr (EPI == OB_T16_PART) { ob_t16_part<MN, MT>(A.zp + blockIdx.y * A.zld, A.rows, A.cols, n0, t0, lane, acc); return; }
    constexpr int IB = MT >= 16 ? 1 : 16 / MT < MN ? 16 / MT : MN;     // column tiles of a batch
    const int lr = lane & 15, lg = lane >> 4;
    const _Float16 *q = EPI == OB_T16_GX ? A.x : A.vec;
    ob_half4 p[2][IB][MT];
    const auto fetch = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int ii = 0; ii < IB; ++ii)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                const int n = n0 + (b * IB + ii) * 16 + 4 * lg, left = A.cols - n, t = t0 + j * 16 + lr;
                ob_half4 v = (ob_half4)(_Float16)0;
                if (t < A.rows && left > 0) {
                    if (A.vec4 && left >= 4) v = *reinterpret_cast<const ob_half4 *>(q + (size_t)t * A.cols + n);
                    else {
#pragma unroll
                        for (int e = 0; e < 4; ++e) if (e < left) v[e] = q[(size_t)t * A.cols + n + e];
                    }
                }
                p[b & 1][ii][j] = v;
            }
    };
    if (EPI != OB_T16_Z) fetch(0);
#pragma unroll
    for (int i = 0; i < MN; ++i) {
        if (EPI != OB_T16_Z && i % IB == 0 && i + IB < MN) fetch(i / IB + 1);
        const int n = n0 + i * 16 + 4 * lg, left = A.cols - n;         // four columns, `left` of them inside
        const bool v4 = A.vec4 && left >= 4;
        ob_half4 h4 = (ob_half4)(_Float16)0;
        float sum[4] = {0.f, 0.f, 0.f, 0.f};                           // (scalars: OB_DPP_F of a vector's element reads element 0)
        if (EPI == OB_T16_GX) {
#pragma unroll
            for (int e = 0; e < 4; ++e) if (e < left) h4[e] = A.vec[n + e];
        }
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            const int t = t0 + j * 16 + lr;
            if (t >= A.rows || left <= 0) continue;
            const size_t o = (size_t)t * A.cols + n;
            ob_half4 c;
#pragma unroll
            for (int e = 0; e < 4; ++e) c[e] = (_Float16)acc(i, j)[e];
            const ob_half4 b = p[i / IB & 1][i % IB][j];
            if (EPI == OB_T16_GX) {
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] += (float)(_Float16)(c[e] * b[e]);
                c = c * h4;
            }
            if (EPI == OB_T16_GW) {
#pragma unroll
                for (int e = 0; e < 4; ++e) c[e] = (_Float16)((float)c[e] * ob_t16_ste((float)b[e]));
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
                if (lr == 0 && e < left && half < 2 * ((A.rows + 127) >> 7)) A.part[(size_t)half * A.cols + n + e] = sum[e];
            }
        }
    }
}

// The same for z and the weight gradient where the rows of C (and W) are in 8-byte pieces: a wave's 64 columns x 16 MT rows go through its 9 KB of LDS, 64 rows at a
// time, so that a load or store is 8 rows of 128 bytes, 16 a lane, instead of 16 of 32; the next 64 rows of W are requested in front of a store.  For waves of a
// workgroup together (the LDS is the loop's).  The weight gradient of 64 rows, 4096 -> 11008, is 180 MB: 67 -> 39 us (2.7 -> 4.6 TB/s); whole backward, 64 / 300 / 700
// rows 142 -> 115, 194 -> 160, 255 -> 219.
#define OB_T16_ROWS_PITCH 144
#define OB_T16_ROWS_LDS (4 * 64 * OB_T16_ROWS_PITCH)
template <int EPI, int MT, typename ACC>
__device__ __forceinline__ void ob_t16_rows(const ObT16Mm &A, int n0, int t0, int lane, char *lds, ACC acc)
{
    static_assert(MT % 4 == 0 && (EPI == OB_T16_Z || EPI == OB_T16_GW));
    const int lr = lane & 15, lg = lane >> 4, n = n0 + (lane & 7) * 8, left = A.cols - n;        // (left % 4 == 0)
    const int t1 = t0 + (lane >> 3);
    ob_half8 p[2][8];
    const auto fetch = [&](int c) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int t = t1 + c * 64 + q * 8;
            const _Float16 *w = A.vec + (size_t)t * A.cols + n;
            ob_half8 v = (ob_half8)(_Float16)0;
            if (t < A.rows && left >= 8) v = *reinterpret_cast<const ob_half8a *>(w);
            else if (t < A.rows && left > 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = w[e];
            }
            p[c & 1][q] = v;
        }
    };
    if (EPI == OB_T16_GW) fetch(0);
    asm volatile("s_barrier" ::: "memory");                            // (every wave's reads of the loop's buffers have returned)
#pragma unroll
    for (int c = 0; c < MT / 4; ++c) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const ob_float4 &z = acc(i, 4 * c + j);
                *reinterpret_cast<ob_half4 *>(lds + (j * 16 + lr) * OB_T16_ROWS_PITCH + (i * 16 + 4 * lg) * 2) =
                    (ob_half4){(_Float16)z[0], (_Float16)z[1], (_Float16)z[2], (_Float16)z[3]};
            }
        if (EPI == OB_T16_GW && c + 1 < MT / 4) fetch(c + 1);
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int t = t1 + c * 64 + q * 8;
            ob_half8 v = *reinterpret_cast<const ob_half8 *>(lds + (q * 8 + (lane >> 3)) * OB_T16_ROWS_PITCH + (lane & 7) * 16);
            if (EPI == OB_T16_GW) {
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = (_Float16)((float)v[e] * ob_t16_ste((float)p[c & 1][q][e]));
            }
            _Float16 *o = A.C + (size_t)t * A.cols + n;
            if (t < A.rows && left >= 8) *reinterpret_cast<ob_half8a *>(o) = v;
            else if (t < A.rows && left > 0) *reinterpret_cast<ob_half4 *>(o) = (ob_half4){v[0], v[1], v[2], v[3]};
        }
    }
}

// ... and for the input gradient: a wave's 64 rows x 16 CT columns, 64 columns at a time, x likewise; its sums of ga x over the rows end in the lanes of
// the first row.  Whole backward with it, 2000 rows 4096 -> 11008 399 -> 378 us, 4096 rows 4096 -> 4096 289 -> 268, 11008 -> 4096 764 -> 710.
template <int CT, typename ACC>
__device__ __forceinline__ void ob_t16_gx_rows(const ObT16Mm &A, int n0, int t0, int half, int lane, char *lds, ACC acc)
{
    static_assert(CT % 4 == 0);
    const int lr = lane & 15, lg = lane >> 4, t1 = t0 + (lane >> 3), c8 = (lane & 7) * 8;
    ob_half8 p[2][8], h[2];
    const auto fetch = [&](int c) __attribute__((always_inline)) {
        const int n = n0 + c * 64 + c8, left = A.cols - n;                               // (left % 4 == 0)
        h[c & 1] = (ob_half8)(_Float16)0;
#pragma unroll
        for (int e = 0; e < 8; ++e) if (e < left) h[c & 1][e] = A.vec[n + e];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int t = t1 + q * 8;
            const _Float16 *x = A.x + (size_t)t * A.cols + n;
            ob_half8 v = (ob_half8)(_Float16)0;
            if (t < A.rows && left >= 8) v = *reinterpret_cast<const ob_half8a *>(x);
            else if (t < A.rows && left > 0) {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = x[e];
            }
            p[c & 1][q] = v;
        }
    };
    fetch(0);
    asm volatile("s_barrier" ::: "memory");                            // (every wave's reads of the loop's buffers have returned)
#pragma unroll
    for (int c = 0; c < CT / 4; ++c) {
        const int n = n0 + c * 64 + c8, left = A.cols - n;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const ob_float4 &z = acc(4 * c + i, j);
                *reinterpret_cast<ob_half4 *>(lds + (j * 16 + lr) * OB_T16_ROWS_PITCH + (i * 16 + 4 * lg) * 2) =
                    (ob_half4){(_Float16)z[0], (_Float16)z[1], (_Float16)z[2], (_Float16)z[3]};
            }
        if (c + 1 < CT / 4) fetch(c + 1);
        float sum[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) sum[e] = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int t = t1 + q * 8;
            const ob_half8 v = *reinterpret_cast<const ob_half8 *>(lds + (q * 8 + (lane >> 3)) * OB_T16_ROWS_PITCH + c8 * 2);
            const ob_half8 vx = v * p[c & 1][q], o = v * h[c & 1];
            if (t >= A.rows) continue;
#pragma unroll
            for (int e = 0; e < 8; ++e) sum[e] += (float)vx[e];
            _Float16 *d = A.C + (size_t)t * A.cols + n;
            if (left >= 8) *reinterpret_cast<ob_half8a *>(d) = o;
            else if (left > 0) *reinterpret_cast<ob_half4 *>(d) = (ob_half4){o[0], o[1], o[2], o[3]};
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            sum[e] += OB_DPP_F(sum[e], 0x128, 0xF);                                      // row_ror:8
            sum[e] += __shfl_xor(sum[e], 16);
            sum[e] += __shfl_xor(sum[e], 32);
            if (lane < 8 && e < left && half < 2 * ((A.rows + 127) >> 7)) A.part[(size_t)half * A.cols + n + e] = sum[e];
        }
    }
}

// both operands through the LDS (ob_mm_loop), 128 x 128 outputs: few tiles
template <int EPI, bool TRW, bool TRA>
__global__ __launch_bounds__(256, 2) void ob_t16_mm_kernel(const ObT16Mm A)
{
    constexpr int NB = 8, TB = 8, NST = 4, TILES = NB + TB, PER = TILES / 4, MN = NB / 2, MT = TB / 2;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wn = wave & 1, wt = wave >> 1, lr = lane & 15, lg = lane >> 4;
    int nb, tb;
    if (!ob_tile_of(blockIdx.x, (A.nw + NB - 1) / NB, (A.na + TB - 1) / TB, nb, tb)) return;      // (uniform)
    int k0;
    const int nk = ob_t16_slice<EPI>(A.nk, A.ns, k0);
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
        src[d] += (size_t)k0 * step[d];
    }
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char *)smem;
    const auto dma = [&](int d, int k, int buf) {
        ob_dma_1k(src[d] + (size_t)min(k, nk - 1) * step[d], lane * 16, lds0 + (uint32_t)(buf * TILES + wave * PER + d) * 1024);
    };
    // operand i of a side whose tiles start at tile t0 of the step's buffer
    const int plain = ob_t16_place(lr, lg);
    const auto frag = [&](bool tr, int buf, int t0, int i) -> ob_u32x4 {
        const char *base = smem + (buf * TILES + t0) * 1024;
        if (!tr) return *reinterpret_cast<const ob_u32x4 *>(base + i * 1024 + plain);
        return ob_t16_turned(base + (i >> 1) * 2048, i & 1, lr, lg);
    };
    ob_float4 acc[MN][MT];
    ob_mm_loop<false, MN, MT, PER, NST>(acc, nk, [&](int buf, int i) { return frag(TRW, buf, 0, wn * MN + i); },
                                        [&](int buf, int j) { return frag(TRA, buf, NB, wt * MT + j); }, dma);
    if constexpr (EPI == OB_T16_Z || EPI == OB_T16_GW) if (A.vec4) {
        ob_t16_rows<EPI, MT>(A, (nb * NB + wn * MN) * 16, (tb * TB + wt * MT) * 16, lane, smem + wave * 64 * OB_T16_ROWS_PITCH, [&](int i, int j) -> const ob_float4 & { return acc[i][j]; });
        return;
    }
    if constexpr (EPI == OB_T16_GX) if (A.vec4) {
        ob_t16_gx_rows<MN>(A, (nb * NB + wn * MN) * 16, (tb * TB + wt * MT) * 16, tb * 2 + wt, lane, smem + wave * 64 * OB_T16_ROWS_PITCH,
                           [&](int i, int j) -> const ob_float4 & { return acc[i][j]; });
        return;
    }
    ob_t16_epilogue<EPI, MN, MT>(A, (nb * NB + wn * MN) * 16, (tb * TB + wt * MT) * 16, tb * 2 + wt, lane, [&](int i, int j) -> const ob_float4 & { return acc[i][j]; });
}

// ... with one operand straight into registers (ob_mm.h, ob_wr_loop): the one that lies as it is reduced, gz for the input gradient (SWAP: it is the MFMA's
// second operand, so that a lane still has four columns of a row), S and (x h)^T for the others.  TRL: the other one's tiles are reduced over their rows.
template <int EPI, bool TRL, bool SWAP, int MT>
__global__ __launch_bounds__(256, MT > 8 ? 1 : 2) void ob_t16_wr_kernel(const ObT16Mm A)
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
    int k0;
    const int nk = ob_t16_slice<EPI>(A.nk, A.ns, k0);
    const char *src[PER], *nxt[PER], *wb[MN];
    uint32_t ldst[PER];
    const size_t step = TRL ? (size_t)lld * 2048 : 1024;
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char *)smem;
#pragma unroll
    for (int d = 0; d < PER; ++d) {
        const int o = wave * PER + d;
        src[d] = lm + (TRL ? (size_t)(o & 1) * lld + min(l0 / 2 + (o >> 1), lld - 1) : (size_t)min(l0 + o, nl - 1) * lld) * 1024 + (size_t)k0 * step;
        nxt[d] = src[d] + (NST - 1) * step;
        ldst[d] = lds0 + (uint32_t)o * 1024;
    }
#pragma unroll
    for (int i = 0; i < MN; ++i) wb[i] = dm + ((size_t)min(d0 + i, nd - 1) * dld + k0) * 1024;
    const int plain = ob_t16_place(lr, lg);
    ob_float4 acc[MN][MT];
    ob_wr_loop<false, SWAP, MT, PER, NST>(acc, nk, wb, plain,
        [&](int buf, int j) -> ob_u32x4 {
            if constexpr (TRL) return ob_t16_turned(smem + (buf * MT + (j & ~1)) * 1024, j & 1, lr, lg);
            else return *reinterpret_cast<const ob_u32x4 *>(smem + (buf * MT + j) * 1024 + plain);
        },
        [&](int d, int k, int buf) { ob_dma_1k(src[d] + (size_t)k * step, lane * 16, ldst[d] + buf * MT * 1024); },
        [&](int d, int, int buf) { ob_dma_1k(nxt[d], lane * 16, ldst[d] + buf * MT * 1024); nxt[d] += step; });
    const int le = ob_t16_lane();
    if constexpr (!SWAP && (EPI == OB_T16_Z || EPI == OB_T16_GW)) if (A.vec4) {
        ob_t16_rows<EPI, MT>(A, d0 * 16, l0 * 16, le, smem + wave * 64 * OB_T16_ROWS_PITCH, [&](int i, int j) -> const ob_float4 & { return acc[i][j]; });
        return;
    }
    if constexpr (SWAP && EPI == OB_T16_GX) if (A.vec4) {
        ob_t16_gx_rows<MT>(A, l0 * 16, d0 * 16, tb * 4 + wave, le, smem + wave * 64 * OB_T16_ROWS_PITCH, [&](int i, int j) -> const ob_float4 & { return acc[j][i]; });
        return;
    }
    if constexpr (SWAP) ob_t16_epilogue<EPI, MT, MN>(A, l0 * 16, d0 * 16, tb * 4 + wave, le, [&](int i, int j) -> const ob_float4 & { return acc[j][i]; });
    else ob_t16_epilogue<EPI, MN, MT>(A, d0 * 16, l0 * 16, 0, le, [&](int i, int j) -> const ob_float4 & { return acc[i][j]; });
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

// The slices' sums put together, in order.  z = fp16(sum), or float32: four values a thread ...
template <typename T>
__global__ __launch_bounds__(256) void ob_train_zsum_kernel(const float *__restrict__ zp, size_t zld, int ns, T *__restrict__ z, size_t n, int vec)
{
    typedef T T4 __attribute__((ext_vector_type(4)));
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i + 4 <= n) {
        ob_float4 a = *reinterpret_cast<const ob_float4 *>(zp + i);
#pragma unroll 4
        for (int j = 1; j < ns; ++j) a = a + *reinterpret_cast<const ob_float4 *>(zp + j * zld + i);
        const T4 o = {(T)a[0], (T)a[1], (T)a[2], (T)a[3]};
        if (vec) *reinterpret_cast<T4 *>(z + i) = o;
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e) z[i + e] = o[e];
        }
    } else {
        for (size_t e = i; e < n; ++e) {
            float a = zp[e];
            for (int j = 1; j < ns; ++j) a += zp[j * zld + e];
            z[e] = (T)a;
        }
    }
}
// ... and the input gradient's: ga = T(sum), gx = ga h and, over 64 rows, the sums of ga x (the epilogue's rounding points): 64 columns x 64 rows a workgroup, four
// columns and every 16th row a thread
template <typename T>
struct ObTrainGxSum { const float *zp; size_t zld; int ns; const T *h, *x; T *gx; float *part; int rows, cols, vec; };      // vec: x, gx in pieces of four
template <typename T>
__global__ __launch_bounds__(256) void ob_train_gxsum_kernel(const ObTrainGxSum<T> A)
{
    typedef T T4 __attribute__((ext_vector_type(4)));
    __shared__ float red[16][64];
    const int cg = threadIdx.x & 15, rl = threadIdx.x >> 4, n = blockIdx.x * 64 + 4 * cg, left = A.cols - n;
    T h4[4];
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 4; ++e) h4[e] = e < left ? A.h[n + e] : (T)0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int t = blockIdx.y * 64 + r * 16 + rl;
        if (t >= A.rows || left <= 0) continue;
        const size_t o = (size_t)t * A.cols + n;
        float a[4] = {0.f, 0.f, 0.f, 0.f};
        if ((A.cols & 3) == 0) {
#pragma unroll 4
            for (int j = 0; j < A.ns; ++j) {
                const ob_float4 v = *reinterpret_cast<const ob_float4 *>(A.zp + j * A.zld + o);
#pragma unroll
                for (int e = 0; e < 4; ++e) a[e] += v[e];
            }
        } else {
            for (int j = 0; j < A.ns; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) if (e < left) a[e] += A.zp[j * A.zld + o + e];
        }
        T4 x4, o4;
        if (A.vec) x4 = *reinterpret_cast<const T4 *>(A.x + o);
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e) x4[e] = e < left ? A.x[o + e] : (T)0.f;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const T c = (T)a[e];
            if (e < left) sum[e] += (float)(T)(c * x4[e]);
            o4[e] = c * h4[e];
        }
        if (A.vec) *reinterpret_cast<T4 *>(A.gx + o) = o4;
        else {
#pragma unroll
            for (int e = 0; e < 4; ++e) if (e < left) A.gx[o + e] = o4[e];
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) red[rl][4 * cg + e] = sum[e];
    __syncthreads();
    const int c = threadIdx.x;
    if (c >= 64 || (int)(blockIdx.x * 64) + c >= A.cols) return;
    float s = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) s += red[r][c];
    A.part[(size_t)blockIdx.y * A.cols + blockIdx.x * 64 + c] = s;
}
