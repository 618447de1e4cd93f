// Train-mode 1-bit linear layer: forward and backward of the reference's
// BitLinear + SignSTE (transformers/src/transformers/models/bitnet.py:14-28, 58-68) on LATENT full-precision
// weights, for knowledge-distillation training on MI355X.
//
//   forward   a = x * h;  S = sign(W) (sign(0) = 0, :18);  z = a . S^T;  u = z * g;  y = LayerNorm(u) (+ bias)
//   backward  gu = LayerNorm'(gy);  gz = gu * g;  gg = sum_t gu * z;  gbias = sum_t gy
//             ga = gz . S;  gx = ga * h;  gh = sum_t ga * x
//             gS = gz^T . a;  gW = gS * (1.001 - tanh(W)^2)                       (the STE of :21-23)
//
// float16: ob_train16.h, float32: ob_train32.h.  Here: the forward passes without a workspace and the float32 backward pass with as little of one as it can do with (product
// kernels whose operand loaders apply x * h and sign(W) on the way into LDS and whose epilogues apply what follows: * h for gx, the STE factor for gW), and the
// LayerNorm that takes any row.  Accumulation is fp32 in both.  In fp16 every tensor-level op of the reference rounds
// once to fp16 (x * h, z, u, gz, ga, gx, gW), as the torch ops do.
#pragma once
#include "ob_common.h"

enum { OB_TX_NONE = 0, OB_TX_SCALE_R = 1, OB_TX_SCALE_I = 2, OB_TX_SIGN = 3 };
enum { OB_TE_PLAIN = 0, OB_TE_GX = 1, OB_TE_STE = 2 };

#define OB_TG_BM 64
#define OB_TG_BN 64
#define OB_TG_BR 32
#define OB_TG_THREADS 256

struct ObTGemmArgs {
    const void *A, *B;        // C[m, n] = sum_r A(m, r) * B(n, r)
    long long lda, ldb;       // leading dimension of the operand's storage (elements)
    const void *va, *vb;      // transform vectors, or null
    void *C;                  // [M, N] row-major, pitch ldc
    void *C2;                 // OB_TE_GX: C2 = C * vc[n]
    const void *vc;           // OB_TE_GX: vector [N];  OB_TE_STE: latent W [M, N] (pitch ldc)
    long long ldc;
    int M, N, R;
};

#define OB_TG_PITCH (OB_TG_BR + 4)        // 144-byte rows

template <typename TI>
__device__ __forceinline__ TI ob_tg_sign(TI v)
{
    return (TI)((v > (TI)0) ? 1.0f : ((v < (TI)0) ? -1.0f : 0.0f));      // NaN -> 0, as (v > 0) - (v < 0)
}

// One 64 x 32 operand tile into LDS as S[i][r].  RC: the reduction index r is the contiguous one in memory
// (element (i, r) at P[i * ld + r]); otherwise the output index i is (element at P[r * ld + i]) and the tile is
// transposed on its way in.  8 contiguous elements per thread, two 16-byte loads when the run is inside the matrix and aligned.  (Forms are compiled in: chosen by
// whether there is a vec, both transforms are computed, 65 rows 12544 -> 8 877 us instead of 745.)
template <bool RC, int TX>
__device__ __forceinline__ void ob_tg_load(float (*S)[OB_TG_PITCH], const float *__restrict__ P, long long ld, const float *__restrict__ vec,
                                           int i0, int r0, int I, int R, int tid)
{
    float v[8];
    int gi, gr;
    if (RC) { gi = i0 + (tid >> 2); gr = r0 + (tid & 3) * 8; }
    else { gr = r0 + (tid >> 3); gi = i0 + (tid & 7) * 8; }
    const float *p = RC ? P + (long long)gi * ld + gr : P + (long long)gr * ld + gi;
    const bool inside = RC ? (gi < I && gr + 8 <= R) : (gr < R && gi + 8 <= I);
    if (inside && ((uintptr_t)p % 16) == 0) {
        reinterpret_cast<ob_u32x4 *>(v)[0] = reinterpret_cast<const ob_u32x4 *>(p)[0];
        reinterpret_cast<ob_u32x4 *>(v)[1] = reinterpret_cast<const ob_u32x4 *>(p)[1];
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const bool ok = RC ? (gi < I && gr + e < R) : (gr < R && gi + e < I);
            v[e] = ok ? p[e] : 0.f;
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int ei = RC ? gi : gi + e, er = RC ? gr + e : gr;
        if (TX == OB_TX_SIGN) v[e] = ob_tg_sign<float>(v[e]);
        if (TX == OB_TX_SCALE_R) v[e] = (ei < I && er < R) ? v[e] * vec[er] : 0.f;
        if (TX == OB_TX_SCALE_I) v[e] = (ei < I && er < R) ? v[e] * vec[ei] : 0.f;
    }
    if (RC) {
        float *d = &S[tid >> 2][(tid & 3) * 8];
        reinterpret_cast<ob_u32x4 *>(d)[0] = reinterpret_cast<ob_u32x4 *>(v)[0];
        reinterpret_cast<ob_u32x4 *>(d)[1] = reinterpret_cast<ob_u32x4 *>(v)[1];
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) S[(tid & 7) * 8 + e][tid >> 3] = v[e];
    }
}

template <bool RCA, bool RCB, int TXA, int TXB, int EPI>
__global__ __launch_bounds__(OB_TG_THREADS) void ob_tgemm_kernel(const ObTGemmArgs a)
{
    __shared__ __attribute__((aligned(16))) float As[OB_TG_BM][OB_TG_PITCH];
    __shared__ __attribute__((aligned(16))) float Bs[OB_TG_BN][OB_TG_PITCH];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    const int i0 = blockIdx.y * OB_TG_BM, j0 = blockIdx.x * OB_TG_BN;
    const int lr = lane & 15, lg = lane >> 4;
    ob_float4 acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y) acc[x][y] = (ob_float4){0.f, 0.f, 0.f, 0.f};
    const float *A = (const float *)a.A, *B = (const float *)a.B;
    for (int r0 = 0; r0 < a.R; r0 += OB_TG_BR) {
        ob_tg_load<RCA, TXA>(As, A, a.lda, (const float *)a.va, i0, r0, a.M, a.R, tid);
        ob_tg_load<RCB, TXB>(Bs, B, a.ldb, (const float *)a.vb, j0, r0, a.N, a.R, tid);
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < OB_TG_BR; kk += 4) {
            float fa[2], fb[2];
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                fa[x] = As[wm * 32 + x * 16 + lr][kk + lg];
                fb[x] = Bs[wn * 32 + x * 16 + lr][kk + lg];
            }
#pragma unroll
            for (int x = 0; x < 2; ++x)
#pragma unroll
                for (int y = 0; y < 2; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[y], fa[x], acc[x][y], 0, 0, 0);
        }
        __syncthreads();
    }
    float *C = (float *)a.C, *C2 = (float *)a.C2;
    const float *vc = (const float *)a.vc;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const int m = i0 + wm * 32 + x * 16 + lr;
        if (m >= a.M) continue;
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            const int n = j0 + wn * 32 + y * 16 + 4 * lg;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (n + e >= a.N) continue;
                const long long o = (long long)m * a.ldc + n + e;
                const float c = acc[x][y][e];
                if (EPI == OB_TE_PLAIN) C[o] = c;
                if (EPI == OB_TE_GX) { C[o] = c; C2[o] = c * vc[n + e]; }
                if (EPI == OB_TE_STE) {                                // SignSTEFunc.backward (bitnet.py:22-23): grad * (1.001 - tanh(w) ** 2)
                    const float w = tanhf(vc[o]);
                    C[o] = c * (1.001f - w * w);
                }
            }
        }
    }
}

// ---- float16 product of a forward call without a workspace: 128 x 128 x 32 tiles, v_mfma_f32_16x16x32_f16, double-buffered LDS ----------------
// z = (x h) sign(W)^T with the operands transformed on their way from registers into LDS: the next tile's are fetched before this tile's MFMAs and
// written to the other buffer after them, one barrier per 32-deep step; 4 waves as 2 x 2, 64 x 64 sums each.  470 TFLOP/s at T = 4096,
// 4096 -> 11008 (ob_train16.h, with a workspace: 1080-1200).
#define OB_TG2_B 128
#define OB_TG2_PITCH 40
#define OB_TG2_TILE (OB_TG2_B * OB_TG2_PITCH)            // halves per operand buffer
#define OB_TG2_LDS (4 * OB_TG2_TILE * 2)                 // two operands x two buffers, bytes

// this thread's 8 contiguous elements of a half-tile: row i0 + tid / 4, columns r0 + 8 (tid & 3)
__device__ __forceinline__ ob_half8 ob_tg2_fetch(const _Float16 *__restrict__ P, long long ld, int i0, int r0, int I, int R, int tid)
{
    const int gi = i0 + (tid >> 2), gr = r0 + (tid & 3) * 8;
    const _Float16 *p = P + (long long)gi * ld + gr;
    if (gi < I && gr + 8 <= R && ((uintptr_t)p % 16) == 0) return *reinterpret_cast<const ob_half8 *>(p);
    ob_half8 v;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = gi < I && gr + e < R ? p[e] : (_Float16)0;
    return v;
}

__global__ __launch_bounds__(OB_TG_THREADS, 2) void ob_tgemm128_f16_kernel(const ObTGemmArgs a)
{
    extern __shared__ __attribute__((aligned(16))) _Float16 ob_tg2_smem[];
    _Float16 *const As = ob_tg2_smem, *const Bs = ob_tg2_smem + 2 * OB_TG2_TILE;     // [2][OB_TG2_TILE] each
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave & 1, wn = wave >> 1, lr = lane & 15, lg = lane >> 4;
    const int i0 = blockIdx.y * OB_TG2_B, j0 = blockIdx.x * OB_TG2_B;
    ob_float4 acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = (ob_float4){0.f, 0.f, 0.f, 0.f};
    const _Float16 *A = (const _Float16 *)a.A, *B = (const _Float16 *)a.B, *h = (const _Float16 *)a.va;
    ob_half8 ra[2], rb[2];
    auto fetch = [&](int r0) {
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            ra[hf] = ob_tg2_fetch(A, a.lda, i0 + 64 * hf, r0, a.M, a.R, tid);
            rb[hf] = ob_tg2_fetch(B, a.ldb, j0 + 64 * hf, r0, a.N, a.R, tid);
        }
    };
    auto put = [&](int buf, int r0) {
        const int gr = r0 + (tid & 3) * 8;
        ob_half8 f;
        if (gr + 8 <= a.R && ((uintptr_t)(h + gr) % 16) == 0) f = *reinterpret_cast<const ob_half8 *>(h + gr);
        else {
#pragma unroll
            for (int e = 0; e < 8; ++e) f[e] = gr + e < a.R ? h[gr + e] : (_Float16)0;
        }
#pragma unroll
        for (int hf = 0; hf < 2; ++hf) {
            const int o = buf * OB_TG2_TILE + (64 * hf + (tid >> 2)) * OB_TG2_PITCH + (tid & 3) * 8;
            *reinterpret_cast<ob_half8 *>(As + o) = ra[hf] * f;                       // fp16 products, rounded once (bitnet.py:62)
#pragma unroll
            for (int e = 0; e < 8; ++e) rb[hf][e] = ob_tg_sign<_Float16>(rb[hf][e]);
            *reinterpret_cast<ob_half8 *>(Bs + o) = rb[hf];
        }
    };
    fetch(0);
    put(0, 0);
    __syncthreads();
    int buf = 0;
    for (int r0 = 0; r0 < a.R; r0 += 32, buf ^= 1) {
        const bool more = r0 + 32 < a.R;
        if (more) fetch(r0 + 32);                       // in flight underneath this step's MFMAs
        ob_half8 fa[4], fb[4];
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            fa[x] = *reinterpret_cast<const ob_half8 *>(As + buf * OB_TG2_TILE + (wm * 64 + x * 16 + lr) * OB_TG2_PITCH + 8 * lg);
            fb[x] = *reinterpret_cast<const ob_half8 *>(Bs + buf * OB_TG2_TILE + (wn * 64 + x * 16 + lr) * OB_TG2_PITCH + 8 * lg);
        }
        // the N side is the MFMA's row operand: a lane ends up with 4 consecutive n of one m
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[y], fa[x], acc[x][y], 0, 0, 0);
        if (more) put(buf ^ 1, r0 + 32);                // (its last readers passed the barrier that ended the previous step)
        __syncthreads();
    }
    _Float16 *C = (_Float16 *)a.C;
#pragma unroll
    for (int x = 0; x < 4; ++x) {
        const int m = i0 + wm * 64 + x * 16 + lr;
        if (m >= a.M) continue;
#pragma unroll
        for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int n = j0 + wn * 64 + y * 16 + 4 * lg + e;
                if (n < a.N) C[(long long)m * a.ldc + n] = (_Float16)acc[x][y][e];
            }
    }
}

// ---- LayerNorm of the train-mode layer, one workgroup per token row ---------------------------------------------
// forward: u = z * g (rounded to the tensor dtype, bitnet.py:64), y = (u - mean) * rstd (+ bias) (:66-68), biased
// variance, statistics in fp32 (two-pass); stats[t] = {mean, rstd} for the backward pass.
template <typename TI>
__global__ __launch_bounds__(256) void ob_train_ln_fwd_kernel(const TI *__restrict__ z, const TI *__restrict__ g, const TI *__restrict__ bias,
                                                              TI *__restrict__ y, float *__restrict__ stats, int N, float eps)
{
    __shared__ float red[8];
    const int t = blockIdx.x;
    const TI *zr = z + (long long)t * N;
    float s = 0.f;
    for (int n = threadIdx.x; n < N; n += 256) s += (float)(TI)(zr[n] * g[n]);
    const float mean = ob_block_sum(s, red) / (float)N;
    float q = 0.f;
    for (int n = threadIdx.x; n < N; n += 256) { const float d = (float)(TI)(zr[n] * g[n]) - mean; q += d * d; }
    const float var = ob_block_sum(q, red) / (float)N;
    const float rstd = 1.0f / sqrtf(var + eps);
    for (int n = threadIdx.x; n < N; n += 256) {
        TI o = (TI)(((float)(TI)(zr[n] * g[n]) - mean) * rstd);
        if (bias) o = (TI)(o + bias[n]);
        y[(long long)t * N + n] = o;
    }
    if (threadIdx.x == 0) { stats[2 * t] = mean; stats[2 * t + 1] = rstd; }
}

// backward through the LayerNorm and the * g: with uh = (u - mean) * rstd,
//   gu = rstd * (gy - mean_n(gy) - uh * mean_n(gy * uh));   gz = gu * g
// rowc[t] = {mean_n(gy), mean_n(gy * uh)} is kept for the column reductions (gg needs gu again).
__global__ __launch_bounds__(256) void ob_train_ln_bwd_kernel(const float *__restrict__ gy, const float *__restrict__ z, const float *__restrict__ g,
                                                              const float *__restrict__ stats, float *__restrict__ gz, float *__restrict__ rowc, int N)
{
    __shared__ float red[8];
    const int t = blockIdx.x;
    const float *zr = z + (long long)t * N, *gr = gy + (long long)t * N;
    const float mean = stats[2 * t], rstd = stats[2 * t + 1];
    float s1 = 0.f, s2 = 0.f;
    for (int n = threadIdx.x; n < N; n += 256) {
        const float uh = (zr[n] * g[n] - mean) * rstd, d = gr[n];
        s1 += d; s2 += d * uh;
    }
    const float c1 = ob_block_sum(s1, red) / (float)N;
    const float c2 = ob_block_sum(s2, red) / (float)N;
    for (int n = threadIdx.x; n < N; n += 256) {
        const float uh = (zr[n] * g[n] - mean) * rstd;
        const float gu = rstd * (gr[n] - c1 - uh * c2);
        gz[(long long)t * N + n] = gu * g[n];
    }
    if (threadIdx.x == 0) { rowc[2 * t] = c1; rowc[2 * t + 1] = c2; }
}

// Column sums over the tokens, in two deterministic stages (one 64-column block walking all T rows took 0.45 / 0.30 ms of a
// 3.3 ms layer step): stage 1 -- block (column block, token slice s of OB_TC_SLICES) accumulates its rows in fp32 and writes
// part[s][column]; stage 2 -- one thread per column adds the slices in order.
//   gg[n] = sum_t gu[t, n] * z[t, n], gbias[n] = sum_t gy[t, n]      (gu: the LayerNorm backward of ob_train_ln_bwd_kernel, recomputed)
//   gh[k] = sum_t ga[t, k] * x[t, k]
#define OB_TC_SLICES 32                  // (also: bands of rows of ob_train16.h's and ob_train32.h's column sums, at most)
__global__ __launch_bounds__(256) void ob_train_cols_ln_kernel(const float *__restrict__ gy, const float *__restrict__ z, const float *__restrict__ g,
                                                               const float *__restrict__ stats, const float *__restrict__ rowc,
                                                               float *__restrict__ part, int T, int N)
{
    __shared__ float sm[2][4][64];
    const int c = threadIdx.x & 63, rl = threadIdx.x >> 6, n = blockIdx.x * 64 + c;
    const int per = (T + OB_TC_SLICES - 1) / OB_TC_SLICES, t0 = blockIdx.y * per, t1 = min(T, t0 + per);
    float a0 = 0.f, a1 = 0.f;
    if (n < N) {
        const float gn = g[n];
        for (int t = t0 + rl; t < t1; t += 4) {
            const float mean = stats[2 * t], rstd = stats[2 * t + 1], c1 = rowc[2 * t], c2 = rowc[2 * t + 1];
            const float zz = z[(long long)t * N + n];
            const float uh = (zz * gn - mean) * rstd, d = gy[(long long)t * N + n];
            const float gu = rstd * (d - c1 - uh * c2);
            a0 += gu * zz;
            a1 += d;
        }
    }
    sm[0][rl][c] = a0; sm[1][rl][c] = a1;
    __syncthreads();
    if (rl == 0 && n < N) {
        part[((size_t)blockIdx.y * 2 + 0) * N + n] = (sm[0][0][c] + sm[0][1][c]) + (sm[0][2][c] + sm[0][3][c]);
        part[((size_t)blockIdx.y * 2 + 1) * N + n] = (sm[1][0][c] + sm[1][1][c]) + (sm[1][2][c] + sm[1][3][c]);
    }
}

__global__ __launch_bounds__(256) void ob_train_cols_gh_kernel(const float *__restrict__ ga, const float *__restrict__ x, float *__restrict__ part, int T, int K)
{
    __shared__ float sm[4][64];
    const int c = threadIdx.x & 63, rl = threadIdx.x >> 6, k = blockIdx.x * 64 + c;
    const int per = (T + OB_TC_SLICES - 1) / OB_TC_SLICES, t0 = blockIdx.y * per, t1 = min(T, t0 + per);
    float a0 = 0.f;
    if (k < K)
        for (int t = t0 + rl; t < t1; t += 4) a0 += ga[(long long)t * K + k] * x[(long long)t * K + k];
    sm[rl][c] = a0;
    __syncthreads();
    if (rl == 0 && k < K) part[(size_t)blockIdx.y * K + k] = (sm[0][c] + sm[1][c]) + (sm[2][c] + sm[3][c]);
}

// stage 2: out_j[c] = sum over slices of part[s][j][c], j < NOUT (out_1 may be null)
template <int NOUT>
__global__ __launch_bounds__(256) void ob_train_cols_finish_kernel(const float *__restrict__ part, float *__restrict__ out0, float *__restrict__ out1, int C)
{
    const int c = blockIdx.x * 256 + threadIdx.x;
    if (c >= C) return;
#pragma unroll
    for (int j = 0; j < NOUT; ++j) {
        float a = 0.f;
        for (int sl = 0; sl < OB_TC_SLICES; ++sl) a += part[((size_t)sl * NOUT + j) * C + c];
        float *o = j == 0 ? out0 : out1;
        if (o) o[c] = a;
    }
}
