// Row kernels of the hybrid decoders: the residual stream in fp32 between the two matrix products of a layer, the gated group norm
// behind a recurrent mixer, and the greedy token.
#pragma once
#include "ob_dense.h"

// s += sum of n partial sums `stride` apart, added in order, up to eight in flight.  (Splits there are not are fetched again and added as zeros: with a branch
// around each addition, as below, the compiler fetches the last ones behind it, a second trip to memory.  12 rows of 2048 columns: a decode step's norms
// 4.7 -> 4.4 us.)
template <int VEC, int U>
__device__ __forceinline__ void ob_sum_splits_u(float (&s)[VEC], const float *p, size_t stride, int k, int n)
{
    float zv[U][VEC];
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
        for (int e = 0; e < VEC; ++e) zv[j][e] = p[(size_t)min(k + j, n - 1) * stride + e];
#pragma unroll
    for (int j = 0; j < U; ++j)
#pragma unroll
        for (int e = 0; e < VEC; ++e) s[e] += k + j < n ? zv[j][e] : 0.f;
}
template <int VEC>
__device__ __forceinline__ void ob_sum_splits(float (&s)[VEC], const float *p, size_t stride, int n)
{
    if (n == 1) {                                                     // (uniform)
#pragma unroll
        for (int e = 0; e < VEC; ++e) s[e] += p[e];
    } else if (n > 4) {
        for (int k = 0; k < n; k += 8) ob_sum_splits_u<VEC, 8>(s, p, stride, k, n);
    } else if (n > 0) ob_sum_splits_u<VEC, 4>(s, p, stride, 0, n);
}
// ... of many rows: mostly one split, and other rows fill the waits
template <int VEC>
__device__ __forceinline__ void ob_sum_splits_rows(float (&s)[VEC], const float *p, size_t stride, int n)
{
    for (int k = 0; k < n; k += 4) {
        float zv[4][VEC];
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < VEC; ++e) zv[j][e] = p[(size_t)min(k + j, n - 1) * stride + e];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (k + j < n) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) s[e] += zv[j][e];
            }
    }
}

// r = residual row, formed one of two ways; x (fragment-major, the next product's operand) = r / sqrt(mean r^2 + eps) * (off + w)
//   embed != NULL   r = embed[token] (+ pos_embed[position]); copied to emb_save when given
//   else            r = x_in + mult * (sum of the splits of the output product + bias) (+ emb_add: a looped stretch starting over)
// `rows` gathers (the final norm runs on the sampling rows only; the residual is then not written back).
struct ObHNormArgs {
    const void *embed, *pos_embed; const int32_t *tokens, *row_pos;
    float *x; const float *z; size_t z_split; int n_split, ldz; const float *bias; float mult;
    const float *emb_add; float *emb_save;
    const float *w; float off, eps;
    void *out; int out_nkt;
    const int32_t *rows;
    int W;
};

// (the workgroup is as wide as the row allows, up to 1024 threads: at one to 64 rows its few dependent passes ARE the launch's time.  Eight waves a SIMD, that
// is two workgroups a CU, here and in ob_xrow_kernel's plain form: with a scalar register too many there is room for seven, one workgroup at a time.  Plain form
// of 4096 columns, 300 / 500 / 900 rows: 11.9 / 14.3 / 20.0 -> 9.9 / 11.5 / 16.9 us; here 900 rows of 2048 columns 9.7 -> 8.6)
template <typename E, int VEC>
__global__ __launch_bounds__(1024, 8) void ob_hnorm_kernel(const ObHNormArgs A)
{
    extern __shared__ __attribute__((aligned(16))) float sm[];        // [W] row | [16] reduction
    float *red = sm + ((A.W + 3) & ~3);
    const int t = blockIdx.x, tid = threadIdx.x, stride = blockDim.x * VEC;
    const int src = A.rows ? A.rows[t] : t;
    float *xr = A.x + (size_t)src * A.W;
    const E *er = nullptr, *pr = nullptr;
    if (A.embed) {
        er = (const E *)A.embed + (size_t)A.tokens[src] * A.W;
        if (A.pos_embed) pr = (const E *)A.pos_embed + (size_t)max(A.row_pos[src], 0) * A.W;
    }
    float ss = 0.f;
    for (int c = tid * VEC; c < A.W; c += stride) {
        float r[VEC];
        if (er) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) r[e] = (float)er[c + e] + (pr ? (float)pr[c + e] : 0.f);
        } else {
            float s[VEC], xv[VEC];
#pragma unroll
            for (int e = 0; e < VEC; ++e) { s[e] = 0.f; xv[e] = xr[c + e]; }
            ob_sum_splits<VEC>(s, A.z + (size_t)src * A.ldz + c, A.z_split, A.n_split);
#pragma unroll
            for (int e = 0; e < VEC; ++e) r[e] = xv[e] + A.mult * (A.bias ? s[e] + A.bias[c + e] : s[e]);
            if (A.emb_add) {
                const float *ea = A.emb_add + (size_t)src * A.W + c;
#pragma unroll
                for (int e = 0; e < VEC; ++e) r[e] += ea[e];
            }
        }
        if (!A.rows) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) xr[c + e] = r[e];
        }
        if (A.emb_save) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) A.emb_save[(size_t)src * A.W + c + e] = r[e];
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) { sm[c + e] = r[e]; ss = __builtin_fmaf(r[e], r[e], ss); }
    }
    ss = ob_block_sum(ss, red);
    const float rs = 1.0f / sqrtf(ss / (float)A.W + A.eps);
    E *out = (E *)A.out;
    for (int c = tid * VEC; c < A.W; c += stride) {
        ob_float4 v;
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = sm[c + e] * rs * (A.off + A.w[c + e]);
        if constexpr (VEC == 4) *reinterpret_cast<typename ObElem<E>::V4 *>(out + ob_frag<E>(t, c, A.out_nkt)) = ob_to_v4<E>(v);
        else out[ob_frag<E>(t, c, A.out_nkt)] = (E)v[0];
    }
}

// Sum of a row that four of the workgroup's waves share (row q of four, thread tid of its 256), in the order of ob_block_sum over 256 NS threads: v[i] is
// what thread 256 i + tid would have.  `red`: 16 NS floats of its own.
template <int NS> __device__ __forceinline__ float ob_rows4_sum(const float (&v)[NS], float *red, int q, int tid)
{
    float *rq = red + 4 * NS * q;
#pragma unroll
    for (int i = 0; i < NS; ++i) {
        const float w = ob_wave_sum(v[i]);
        if ((tid & 63) == 0) rq[4 * i + (tid >> 6)] = w;
    }
    __syncthreads();
    if (NS == 1) return (rq[0] + rq[1]) + (rq[2] + rq[3]);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4 * NS; ++i) s += rq[i];
    return s;
}

// ... of many rows: four rows a workgroup, four waves each (1024 NV columns, W % 4 == 0, no embedding row), the row in registers.  The four rows' pieces
// of the fragment-major output lie next to each other and leave as whole sectors from one L2 (ob_gated_norm_rows_kernel):
// 6100 rows of 2048 columns 46 -> 42 us.  A row's squares are added in ob_hnorm_kernel's order: a row's result does not depend on the others' number.
template <typename E, int NV>
__global__ __launch_bounds__(1024) void ob_hnorm_rows_kernel(const ObHNormArgs A, int n_rows)
{
    constexpr int NS = NV < 2 ? NV : 2;                                // (ob_hnorm_kernel has 512 threads here: pieces i and i + 2 are one thread's)
    __shared__ float red[16 * NS];
    const int tid = threadIdx.x & 255, q = threadIdx.x >> 8, t = min((int)blockIdx.x * 4 + q, n_rows - 1);
    const bool live = (int)blockIdx.x * 4 + q < n_rows;                // (a row beyond the last: read again, not written)
    const int src = A.rows ? A.rows[t] : t;
    float *xr = A.x + (size_t)src * A.W;
    ob_float4 r[NV];
    float ss[NS] = {};
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 256 + tid) * 4;
        if (c < A.W) {
            r[i] = *reinterpret_cast<const ob_float4 *>(xr + c);
            float s[4] = {0.f, 0.f, 0.f, 0.f};
            ob_sum_splits_rows<4>(s, A.z + (size_t)src * A.ldz + c, A.z_split, A.n_split);
#pragma unroll
            for (int e = 0; e < 4; ++e) r[i][e] += A.mult * (A.bias ? s[e] + A.bias[c + e] : s[e]);
            if (A.emb_add) r[i] += *reinterpret_cast<const ob_float4 *>(A.emb_add + (size_t)src * A.W + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) ss[i % NS] = __builtin_fmaf(r[i][e], r[i][e], ss[i % NS]);
        }
    }
    const float rs = 1.0f / sqrtf(ob_rows4_sum<NS>(ss, red, q, tid) / (float)A.W + A.eps);      // (every read of the residual row is done)
    if (!live) return;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 256 + tid) * 4;
        if (c >= A.W) break;
        if (!A.rows) *reinterpret_cast<ob_float4 *>(xr + c) = r[i];
        const ob_float4 w = *reinterpret_cast<const ob_float4 *>(A.w + c);
        ob_float4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = r[i][e] * rs * (A.off + w[e]);
        *reinterpret_cast<typename ObElem<E>::V4 *>((E *)A.out + ob_frag<E>(t, c, A.out_nkt)) = ob_to_v4<E>(v);
    }
}

// The same row with everything a sequential layer adds to it:
//   s = sum of the splits (+ bias) + sum_k tok_w[k] ez[tok_row[k]] (experts; eo: their outputs in the work type) + id_w h (identity experts; h = idh or the residual itself)
//   r = x + mult * (post_w ? s / sqrt(mean s^2 + eps) * post_w : s) (+ emb_add)
//     or, embed != NULL: r = embed[token] * embed_scale (+ bigram[row of (previous token, token)]) (+ pos_embed[position])
//   hist: X_i = r is kept (i = hist_i), and with dwa the stream goes on as sum_j dwa[j] X_j, j = 0 .. hist_i
//   output: r / sqrt(mean r^2 + eps) * (off + w), or r itself (w == NULL); fragment-major and, out_rm, also row-major
// The previous token of an item's first row comes from tok_hist [slots][max_len], where every row leaves its token.
struct ObXRowArgs : ObHNormArgs {
    float embed_scale; const void *bigram; int buckets, mul_prev, mul_cur;
    int32_t *tok_hist; const int32_t *row_slot, *row_off; int n_slots, max_len;
    const float *post_w;
    const float *ez; const void *eo; size_t ez_split; int ez_n, ld_ez, top; const int32_t *tok_row; const float *tok_w, *id_w; const void *idh; int ld_idh;
    float *hist; size_t hist_stride; int hist_i; const float *dwa;
    void *out_rm; int ld_rm;
};
// ONE: a thread has one piece of the row (W <= threads * VEC); everything that does not depend on the first reduction is then requested before it.
// KIND: what can be there besides the sum of splits (smaller code: at a few rows a launch's time is its chain of fetches, instructions included)
enum ObXKind { OB_X_PLAIN = 0, OB_X_EXPERTS = 1, OB_X_DEPTH = 2, OB_X_BOTH = 3, OB_X_EMBED = 4 };
template <typename E, int VEC, bool ONE, int KIND>
__global__ __launch_bounds__(1024, KIND == OB_X_PLAIN ? 8 : 4) void ob_xrow_kernel(const ObXRowArgs A)
{
    constexpr int NH = 8;
    constexpr bool EMB = KIND == OB_X_EMBED, EXP = (KIND & 1) != 0, DEP = (KIND & 2) != 0;
    extern __shared__ __attribute__((aligned(16))) float sm[];        // [W] row | [16] reduction
    float *red = sm + ((A.W + 3) & ~3);
    const int t = blockIdx.x, tid = threadIdx.x, stride = blockDim.x * VEC;
    const int src = A.rows ? A.rows[t] : t;
    float *xr = A.x + (size_t)src * A.W;
    float *hr = A.hist + (size_t)src * A.W;                           // (DEP, and EMB where the embedding is kept)
    const E *er = nullptr, *pr = nullptr, *br = nullptr;
    if constexpr (EMB) {
        const int tok = A.tokens[src], pos = A.row_pos[src], slot = A.row_slot[src];
        er = (const E *)A.embed + (size_t)tok * A.W;
        if (A.pos_embed) pr = (const E *)A.pos_embed + (size_t)max(pos, 0) * A.W;
        if (A.bigram) {
            const bool live = slot >= 0 && slot < A.n_slots && pos >= 0 && pos < A.max_len;
            int b = A.buckets;                                        // (a sequence's first token)
            if (live && pos > 0) {
                const int prev = A.row_off[src] > 0 ? A.tokens[src - 1] : A.tok_hist[(size_t)slot * A.max_len + pos - 1];
                b = (int)(((long long)prev * A.mul_prev + (long long)tok * A.mul_cur) % A.buckets);
            }
            br = (const E *)A.bigram + (size_t)b * A.W;
            if (live && tid == 0 && !A.rows) A.tok_hist[(size_t)slot * A.max_len + pos] = tok;
        }
    }
    float x1[VEC], h1[DEP ? NH : 1][VEC];                             // ONE: the residual and the first results X_j
    if (ONE && !EMB && tid * VEC < A.W) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) x1[e] = xr[tid * VEC + e];
        if (DEP && A.dwa) {
#pragma unroll
            for (int j = 0; j < NH; ++j)
#pragma unroll
                for (int e = 0; e < VEC; ++e) h1[DEP ? j : 0][e] = hr[(size_t)min(j, A.hist_i - 1) * A.hist_stride + tid * VEC + e];
        }
    }
    float ss = 0.f;
    if (!EMB) {
        for (int c = tid * VEC; c < A.W; c += stride) {
            float s[VEC];
#pragma unroll
            for (int e = 0; e < VEC; ++e) s[e] = 0.f;
            if (A.z) {
                // (with experts the loop: mostly one split, and the larger code costs more than the trip: float32, 1024 columns, 12 rows 6.4 us, 7.2 with
                // ob_sum_splits)
                if constexpr (EXP) ob_sum_splits_rows<VEC>(s, A.z + (size_t)src * A.ldz + c, A.z_split, A.n_split);
                else ob_sum_splits<VEC>(s, A.z + (size_t)src * A.ldz + c, A.z_split, A.n_split);
            }
            if (A.bias) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) s[e] += A.bias[c + e];
            }
            if (EXP && A.eo) {                                        // four experts in flight, added in order
#pragma unroll 1
                for (int k0 = 0; k0 < A.top; k0 += 4) {
                    float y[4][VEC], w[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const size_t k = (size_t)src * A.top + min(k0 + j, A.top - 1);
                        const int row = A.tok_row[k];                 // (uniform; row 0 where there is none)
                        w[j] = k0 + j < A.top && row >= 0 ? A.tok_w[k] : 0.f;
                        const E *p = (const E *)A.eo + (size_t)max(row, 0) * A.ld_ez + c;
#pragma unroll
                        for (int e = 0; e < VEC; ++e) y[j][e] = (float)p[e];
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int e = 0; e < VEC; ++e) s[e] = w[j] != 0.f ? __builtin_fmaf(w[j], y[j][e], s[e]) : s[e];
                }
            } else if (EXP) {
#pragma unroll 1
                for (int k0 = 0; k0 < A.top * A.ez_n; k0 += 4) {      // (choice, split) pairs
                    float y[4][VEC], w[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int kk = min(k0 + j, A.top * A.ez_n - 1), sp = A.ez_n == 1 ? 0 : kk / A.top;
                        const size_t k = (size_t)src * A.top + kk - sp * A.top;
                        const int row = A.tok_row[k];
                        w[j] = k0 + j < A.top * A.ez_n && row >= 0 ? A.tok_w[k] : 0.f;
                        const float *p = A.ez + sp * A.ez_split + (size_t)max(row, 0) * A.ld_ez + c;
#pragma unroll
                        for (int e = 0; e < VEC; ++e) y[j][e] = p[e];
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int e = 0; e < VEC; ++e) s[e] = w[j] != 0.f ? __builtin_fmaf(w[j], y[j][e], s[e]) : s[e];
                }
            }
            if (EXP && A.id_w) {
                const float w = A.id_w[src];
#pragma unroll
                for (int e = 0; e < VEC; ++e)
                    s[e] = __builtin_fmaf(w, A.idh ? (float)((const E *)A.idh)[(size_t)src * A.ld_idh + c + e] : ONE ? x1[e] : xr[c + e], s[e]);
            }
#pragma unroll
            for (int e = 0; e < VEC; ++e) { sm[c + e] = s[e]; ss = __builtin_fmaf(s[e], s[e], ss); }
        }
    }
    float rp = 1.f;
    if (!EMB && A.post_w) rp = 1.0f / sqrtf(ob_block_sum(ss, red) / (float)A.W + A.eps);          // (uniform)
    ss = 0.f;
    for (int c = tid * VEC; c < A.W; c += stride) {
        float r[VEC];
        if (EMB) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) r[e] = (float)er[c + e] * A.embed_scale + (br ? (float)br[c + e] : 0.f) + (pr ? (float)pr[c + e] : 0.f);
        } else {
#pragma unroll
            for (int e = 0; e < VEC; ++e) r[e] = (ONE ? x1[e] : xr[c + e]) + A.mult * (A.post_w ? sm[c + e] * rp * A.post_w[c + e] : sm[c + e]);
            if (A.emb_add) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) r[e] += A.emb_add[(size_t)src * A.W + c + e];
            }
        }
        if (DEP || (EMB && A.hist)) {
            if (!A.rows) {
#pragma unroll
                for (int e = 0; e < VEC; ++e) hr[A.hist_i * A.hist_stride + c + e] = r[e];
            }
            if (DEP && A.dwa) {
                float a[VEC];
#pragma unroll
                for (int e = 0; e < VEC; ++e) a[e] = 0.f;
                for (int j = 0; j < A.hist_i; j += NH) {              // eight results in flight, added in order
                    float v[NH][VEC];
#pragma unroll
                    for (int q = 0; q < NH; ++q)
#pragma unroll
                        for (int e = 0; e < VEC; ++e) v[q][e] = ONE && j == 0 ? h1[DEP ? q : 0][e] : hr[(size_t)min(j + q, A.hist_i - 1) * A.hist_stride + c + e];
#pragma unroll
                    for (int q = 0; q < NH; ++q)
                        if (j + q < A.hist_i) {
#pragma unroll
                            for (int e = 0; e < VEC; ++e) a[e] = __builtin_fmaf(A.dwa[j + q], v[q][e], a[e]);
                        }
                }
#pragma unroll
                for (int e = 0; e < VEC; ++e) r[e] = __builtin_fmaf(A.dwa[A.hist_i], r[e], a[e]);
            }
        }
        if (!A.rows) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) xr[c + e] = r[e];
        }
        if (A.emb_save) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) A.emb_save[(size_t)src * A.W + c + e] = r[e];
        }
#pragma unroll
        for (int e = 0; e < VEC; ++e) { sm[c + e] = r[e]; ss = __builtin_fmaf(r[e], r[e], ss); }
    }
    float rs = 1.f;
    if (A.w) rs = 1.0f / sqrtf(ob_block_sum(ss, red) / (float)A.W + A.eps);               // (uniform)
    E *out = (E *)A.out;
    for (int c = tid * VEC; c < A.W; c += stride) {
        ob_float4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = A.w ? sm[c + e] * rs * (A.off + A.w[c + e]) : sm[c + e];
        if constexpr (VEC == 4) {
            const typename ObElem<E>::V4 o = ob_to_v4<E>(v);
            *reinterpret_cast<typename ObElem<E>::V4 *>(out + ob_frag<E>(t, c, A.out_nkt)) = o;
            if (A.out_rm) *reinterpret_cast<typename ObElem<E>::V4 *>((E *)A.out_rm + (size_t)t * A.ld_rm + c) = o;
        } else {
            out[ob_frag<E>(t, c, A.out_nkt)] = (E)v[0];
            if (A.out_rm) ((E *)A.out_rm)[(size_t)t * A.ld_rm + c] = (E)v[0];
        }
    }
}

// ... of many rows, as ob_hnorm_rows_kernel: four rows a workgroup, four waves each (1024 NV columns, W % 4 == 0; no embedding row, experts' outputs in the
// work type), the row in registers.  Memory bounds it: the four rows write whole sectors of the fragment-major output, a row's pieces are all requested at
// once, and a row takes 56 registers of 256 threads instead of 512 threads and two barriers of its own.  6100 rows of 2048 columns, against
// ob_xrow_kernel: plain 53.8 -> 39.9 us, experts (six a token) 85.3 -> 62.3, depth average (one to eight results) 105 -> 90 = 4.9 TB/s; 1024 columns
// 21.1 -> 16.7, 33.2 -> 27.4, 36.1 -> 28.4; 4096 columns 85.7 -> 68.8, 165.7 -> 115.9, 157.6 -> 127.4.
template <typename E, int NV, int KIND>
__global__ __launch_bounds__(1024) void ob_xrow_rows_kernel(const ObXRowArgs A, int n_rows)
{
    constexpr int NH = 8;
    constexpr bool EXP = (KIND & 1) != 0, DEP = (KIND & 2) != 0;
    typedef typename ObElem<E>::V4 V4;
    __shared__ float red[2][16 * NV];
    const int tid = threadIdx.x & 255, q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8), t = min((int)blockIdx.x * 4 + q, n_rows - 1);
    const bool live = (int)blockIdx.x * 4 + q < n_rows;                // (a row beyond the last: read again, not written)
    const int src = A.rows ? A.rows[t] : t;
    float *xr = A.x + (size_t)src * A.W, *hr = A.hist + (size_t)src * A.W;
    ob_float4 x[NV], s[NV];
    float ss[NV] = {};                                                 // (ob_xrow_kernel has a thread for every piece)
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 256 + tid) * 4;
        x[i] = s[i] = (ob_float4){0.f, 0.f, 0.f, 0.f};
        if (c < A.W) {
            x[i] = *reinterpret_cast<const ob_float4 *>(xr + c);
            float z[4] = {0.f, 0.f, 0.f, 0.f};
            if (A.z) ob_sum_splits_rows<4>(z, A.z + (size_t)src * A.ldz + c, A.z_split, A.n_split);
            if (A.bias) {
#pragma unroll
                for (int e = 0; e < 4; ++e) z[e] += A.bias[c + e];
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) s[i][e] = z[e];
        }
    }
    if constexpr (EXP) {
#pragma unroll 1
        for (int k0 = 0; k0 < A.top; k0 += 4) {                        // four experts in flight, added in order
            V4 y[4][NV];
            float w[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const size_t k = (size_t)src * A.top + min(k0 + j, A.top - 1);
                const int row = A.tok_row[k];                          // (uniform; row 0 where there is none)
                w[j] = k0 + j < A.top && row >= 0 ? A.tok_w[k] : 0.f;
                const E *p = (const E *)A.eo + (size_t)max(row, 0) * A.ld_ez;
#pragma unroll
                for (int i = 0; i < NV; ++i) if ((i * 256 + tid) * 4 < A.W) y[j][i] = *reinterpret_cast<const V4 *>(p + (i * 256 + tid) * 4);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (w[j] != 0.f) {
#pragma unroll
                    for (int i = 0; i < NV; ++i)
                        if ((i * 256 + tid) * 4 < A.W) {
#pragma unroll
                            for (int e = 0; e < 4; ++e) s[i][e] = __builtin_fmaf(w[j], (float)y[j][i][e], s[i][e]);
                        }
                }
        }
        if (A.id_w) {
            const float w = A.id_w[src];
#pragma unroll
            for (int i = 0; i < NV; ++i) {
                const int c = (i * 256 + tid) * 4;
                if (c < A.W) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[i][e] = __builtin_fmaf(w, A.idh ? (float)((const E *)A.idh)[(size_t)src * A.ld_idh + c + e] : x[i][e], s[i][e]);
                }
            }
        }
    }
    float rp = 1.f;
    if (A.post_w) {                                                    // (uniform)
#pragma unroll
        for (int i = 0; i < NV; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) ss[i] = __builtin_fmaf(s[i][e], s[i][e], ss[i]);
        rp = 1.0f / sqrtf(ob_rows4_sum<NV>(ss, red[0], q, tid) / (float)A.W + A.eps);
#pragma unroll
        for (int i = 0; i < NV; ++i) ss[i] = 0.f;
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 256 + tid) * 4;
        if (c < A.W) {
            ob_float4 r;
            const ob_float4 pw = A.post_w ? *reinterpret_cast<const ob_float4 *>(A.post_w + c) : s[i];
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = x[i][e] + A.mult * (A.post_w ? s[i][e] * rp * pw[e] : s[i][e]);
            if (A.emb_add) r += *reinterpret_cast<const ob_float4 *>(A.emb_add + (size_t)src * A.W + c);
            if constexpr (DEP) {
                if (!A.rows && live) *reinterpret_cast<ob_float4 *>(hr + A.hist_i * A.hist_stride + c) = r;
                if (A.dwa) {
                    ob_float4 a = {0.f, 0.f, 0.f, 0.f};
                    for (int j = 0; j < A.hist_i; j += NH) {           // eight results in flight, added in order
                        ob_float4 v[NH];
#pragma unroll
                        for (int u = 0; u < NH; ++u) v[u] = *reinterpret_cast<const ob_float4 *>(hr + (size_t)min(j + u, A.hist_i - 1) * A.hist_stride + c);
#pragma unroll
                        for (int u = 0; u < NH; ++u)
                            if (j + u < A.hist_i) {
#pragma unroll
                                for (int e = 0; e < 4; ++e) a[e] = __builtin_fmaf(A.dwa[j + u], v[u][e], a[e]);
                            }
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) r[e] = __builtin_fmaf(A.dwa[A.hist_i], r[e], a[e]);
                }
            }
            if (!A.rows && live) *reinterpret_cast<ob_float4 *>(xr + c) = r;
#pragma unroll
            for (int e = 0; e < 4; ++e) ss[i] = __builtin_fmaf(r[e], r[e], ss[i]);
            s[i] = r;
        }
    }
    float rs = 1.f;
    if (A.w) rs = 1.0f / sqrtf(ob_rows4_sum<NV>(ss, red[1], q, tid) / (float)A.W + A.eps);       // (uniform)
    if (!live) return;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 256 + tid) * 4;
        if (c >= A.W) break;
        ob_float4 v = s[i];
        if (A.w) {
            const ob_float4 w = *reinterpret_cast<const ob_float4 *>(A.w + c);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = v[e] * rs * (A.off + w[e]);
        }
        const V4 o = ob_to_v4<E>(v);
        *reinterpret_cast<V4 *>((E *)A.out + ob_frag<E>(t, c, A.out_nkt)) = o;
        if (A.out_rm) *reinterpret_cast<V4 *>((E *)A.out_rm + (size_t)t * A.ld_rm + c) = o;
    }
}

// grid (norm groups, rows): v = y * silu(gate); out[k0 + i] = v / sqrt(mean over the group v^2 + eps) * w
struct ObGatedNormArgs {
    const void *y; int ldy; const void *gate; int ldg;       // row-major; the gate is the leading columns of the input product
    const float *w; float eps; int gsize;
    void *out; int out_nkt;
};
template <typename E, int VEC>                                 // VEC = 16 bytes of elements, or 1
__global__ __launch_bounds__(256) void ob_gated_norm_kernel(const ObGatedNormArgs A)
{
    typedef typename ObElem<E>::V16 V16;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float *red = sm + ((A.gsize + 3) & ~3);
    const int t = blockIdx.y, c0 = blockIdx.x * A.gsize, tid = threadIdx.x, stride = blockDim.x * VEC;
    const E *y = (const E *)A.y + (size_t)t * A.ldy + c0, *z = (const E *)A.gate + (size_t)t * A.ldg + c0;
    float ss = 0.f;
    for (int c = tid * VEC; c < A.gsize; c += stride) {
        V16 yv, zv;
        if constexpr (VEC > 1) { yv = *reinterpret_cast<const V16 *>(y + c); zv = *reinterpret_cast<const V16 *>(z + c); }
        else { yv[0] = y[c]; zv[0] = z[c]; }
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float v = (float)yv[e] * ob_silu<E>((float)zv[e]);
            sm[c + e] = v;
            ss = __builtin_fmaf(v, v, ss);
        }
    }
    ss = ob_block_sum(ss, red);
    const float rs = 1.0f / sqrtf(ss / (float)A.gsize + A.eps);
    E *out = (E *)A.out;
    for (int c = tid * VEC; c < A.gsize; c += stride) {
        V16 v;
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] = (E)(sm[c + e] * rs * A.w[c0 + c + e]);
        if constexpr (VEC > 1) *reinterpret_cast<V16 *>(out + ob_frag<E>(t, c0 + c, A.out_nkt)) = v;       // (16 bytes of a row are contiguous)
        else out[ob_frag<E>(t, c0 + c, A.out_nkt)] = v[0];
    }
}

// ... of many rows: a wave per row, four rows a workgroup.  A row's 16-byte pieces of the fragment-major output then leave as whole 64-byte sectors (four
// rows of a tile lie next to each other) from one L2: 6100 rows of 4096 columns 62 us one row a workgroup,
// partial sectors from four XCDs -> 48.
// The row stays in registers (NV 16-byte pieces per lane); groups of up to 512 NV columns, whole pieces.
template <typename E, int NV>
__global__ __launch_bounds__(256) void ob_gated_norm_rows_kernel(const ObGatedNormArgs A, int rows)
{
    typedef typename ObElem<E>::V16 V16;
    constexpr int VEC = ObElem<E>::EPL;
    const int lane = threadIdx.x & 63, t = blockIdx.y * 4 + (threadIdx.x >> 6), c0 = blockIdx.x * A.gsize;
    if (t >= rows) return;
    const E *y = (const E *)A.y + (size_t)t * A.ldy + c0, *z = (const E *)A.gate + (size_t)t * A.ldg + c0;
    V16 yv[NV], zv[NV];
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 64 + lane) * VEC;
        if (c < A.gsize) { yv[i] = *reinterpret_cast<const V16 *>(y + c); zv[i] = *reinterpret_cast<const V16 *>(z + c); }
    }
    constexpr int NS = NV < 4 ? NV : 4;                                // (added in ob_gated_norm_kernel's order: 256 threads, pieces i and i + 4 are one's)
    float v[NV][VEC], ss[NS] = {};
#pragma unroll
    for (int i = 0; i < NV; ++i)
        if ((i * 64 + lane) * VEC < A.gsize) {
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                v[i][e] = (float)yv[i][e] * ob_silu<E>((float)zv[i][e]);
                ss[i % NS] = __builtin_fmaf(v[i][e], v[i][e], ss[i % NS]);
            }
        }
#pragma unroll
    for (int i = 0; i < NS; ++i) ss[i] = ob_wave_sum(ss[i]);
    const float rs = 1.0f / sqrtf((NS == 1 ? ss[0] : (ss[0] + ss[1 % NS]) + (ss[2 % NS] + ss[3 % NS])) / (float)A.gsize + A.eps);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
        const int c = (i * 64 + lane) * VEC;
        if (c >= A.gsize) break;
        V16 o;
#pragma unroll
        for (int e = 0; e < VEC; ++e) o[e] = (E)(v[i][e] * rs * A.w[c0 + c + e]);
        *reinterpret_cast<V16 *>((E *)A.out + ob_frag<E>(t, c0 + c, A.out_nkt)) = o;
    }
}

// greedy token: the smallest index of the largest logit of every row
__global__ __launch_bounds__(1024) void ob_argmax_rows_kernel(const float *__restrict__ logits, int32_t *__restrict__ next, int V)
{
    __shared__ float bv[16];
    __shared__ int bi[16];
    const float *l = logits + (size_t)blockIdx.x * V;
    const int tid = threadIdx.x;
    float best = -INFINITY;
    int idx = 0x7fffffff;
    if ((V & 3) == 0) {
        for (int i0 = tid; i0 < V / 4; i0 += 4096) {                  // four 16-byte loads in flight
            ob_float4 v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = reinterpret_cast<const ob_float4 *>(l)[min(i0 + 1024 * j, V / 4 - 1)];
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e)                           // (ascending indices; a clamped repeat is not larger)
                    if (v[j][e] > best) { best = v[j][e]; idx = 4 * min(i0 + 1024 * j, V / 4 - 1) + e; }
        }
    } else {
        for (int i = tid; i < V; i += 1024) {
            const float v = l[i];
            if (v > best) { best = v; idx = i; }
        }
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        const float ov = __shfl_xor(best, s);
        const int oi = __shfl_xor(idx, s);
        if (ov > best || (ov == best && oi < idx)) { best = ov; idx = oi; }
    }
    if ((tid & 63) == 0) { bv[tid >> 6] = best; bi[tid >> 6] = idx; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; ++w)
            if (bv[w] > best || (bv[w] == best && bi[w] < idx)) { best = bv[w]; idx = bi[w]; }
        next[blockIdx.x] = idx == 0x7fffffff ? 0 : idx;
    }
}
