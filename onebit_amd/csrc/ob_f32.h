// float32 layer on the matrix cores, exactly split: z[t][n] = sum_k s[n][k] a[t][k], a = fp32(x h), s = +-1 (bitnet.py:113-115 in float32).
//
// The signs are exact in bf16, and a float32 IS the sum of three bf16: its upper 8 significant bits, the next 8 of what is left, the last 8
// (truncation, so every remainder is exact).  Three bf16 products with fp32 accumulation therefore multiply the same numbers that a float32
// product multiplies, at a third of the bf16 rate instead of the vector units': nothing of the inputs is rounded away.  The upper parts add
// up in accumulators of their own: 8-bit addends against a 24-bit sum leave almost no rounding error there, and the error of the two
// lower parts is 2^-8 smaller, so the sum is closer to the 64-bit one than 64 lanes' float32 chains are (731 rows, 4096 -> 11008: the layer's
// output is 9.6e-8 off instead of 1.8e-7).  Infinities stay infinite (lower parts zero), NaN stays NaN.  Exact down to |x h| = 2^-110: smaller
// ones lose what lies below the smallest bf16, 2^-133 (2e-6 of an activation of 2^-115), which a LayerNorm with eps 1e-5 takes away anyway.
//
// What bounds it: the matrix cores, three products for one (whole call at 731 rows, 4096 -> 11008: 7371 us with ob_simple_kernel, 162 with a stage's operands read
// in front of its products, 154 with everything placed behind single products, as below; 2000 rows 460 -> 445, 1300 rows 4096 -> 4096 151 -> 141, 300 rows
// 11008 -> 4096 83.5 -> 79, 50 rows 22.4 -> 21.6; the same bits).  In a trace the split takes 8 and the row pass 13.
//
//   ob_f32_split_kernel    x, h -> planes: 1 KB tiles [16-row band][k step][part], a tile in MFMA operand order (one wave, 16 bytes a lane).
//                          Step s of the 256-column quad q holds, for lane group gq, columns 256 q + 64 gq + 8 s ..: a lane's sign bytes of
//                          the quad's eight steps are then 8 ADJACENT bytes of its packed row, one ds_read_b64 per row tile and quad
//   ob_f32_gemm_kernel     128 output columns x 16 TB rows per workgroup, four waves; planes and packed rows through LDS by 1 KB DMAs, NST
//                          stages of 12 or 24 KB, one raw barrier per stage behind a counted wait
//   ob_f32_ln_kernel       one workgroup per row: sums of the K splits, * g, LayerNorm, bias; the row stays in registers
#pragma once
#include "ob_common.h"
#include <type_traits>

struct ObF32Split { const float *x; long long ldx; const float *h; char *planes; int T, K, quads; };

__global__ __launch_bounds__(256) void ob_f32_split_kernel(const ObF32Split A)
{
    const int lane = threadIdx.x & 63, r = lane & 15, gq = lane >> 4;
    const int unit = blockIdx.x * 4 + (threadIdx.x >> 6);              // (band, quad)
    const int band = unit / A.quads, q = unit - band * A.quads;
    if (band * 16 >= A.T) return;
    const int t = band * 16 + r, k0 = 256 * q + 64 * gq;
    const float *xr = A.x + (long long)t * A.ldx + k0;
    char *out = A.planes + ((size_t)band * A.quads + q) * (8 * 3072) + lane * 16;
#pragma unroll
    for (int s = 0; s < 8; ++s) {
        float a[8];
        if (t < A.T && k0 + 8 * s < A.K) {                             // K % 8 == 0: a piece is inside or outside
            const ob_float4 x0 = *reinterpret_cast<const ob_float4 *>(xr + 8 * s), x1 = *reinterpret_cast<const ob_float4 *>(xr + 8 * s + 4);
            const ob_float4 h0 = *reinterpret_cast<const ob_float4 *>(A.h + k0 + 8 * s), h1 = *reinterpret_cast<const ob_float4 *>(A.h + k0 + 8 * s + 4);
#pragma unroll
            for (int i = 0; i < 4; ++i) { a[i] = x0[i] * h0[i]; a[i + 4] = x1[i] * h1[i]; }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) a[i] = 0.f;
        }
        uint32_t hi[8], mid[8], lo[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            hi[i] = __float_as_uint(a[i]);
            const bool inf = (hi[i] & 0x7fffffffu) == 0x7f800000u;
            const float r1 = inf ? 0.f : a[i] - __uint_as_float(hi[i] & 0xffff0000u);
            mid[i] = __float_as_uint(r1);
            lo[i] = __float_as_uint(r1 - __uint_as_float(mid[i] & 0xffff0000u));
        }
        ob_u32x4 w[3];
#pragma unroll
        for (int p = 0; p < 4; ++p) {                                  // upper halves of two floats
            w[0][p] = __builtin_amdgcn_perm(hi[2 * p + 1], hi[2 * p], 0x07060302u);
            w[1][p] = __builtin_amdgcn_perm(mid[2 * p + 1], mid[2 * p], 0x07060302u);
            w[2][p] = __builtin_amdgcn_perm(lo[2 * p + 1], lo[2 * p], 0x07060302u);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<ob_u32x4 *>(out + s * 3072 + p * 1024) = w[p];
    }
}

// packed rows with K % 256 columns left over (of any pitch and address): rows of `quads` x 32 bytes, zeros behind K (their planes are zero)
__global__ __launch_bounds__(256) void ob_f32_rows_kernel(const uint8_t *__restrict__ W, long long ldw, uint32_t *__restrict__ out, int N, int kb, int quads)
{
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    const int per = quads * 8, n = (int)(i / per), j = (int)(i - (long long)n * per) * 4;
    if (n >= N) return;
    const uint8_t *p = W + (long long)n * ldw + j;
    uint32_t v = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) if (j + b < kb) v |= (uint32_t)p[b] << (8 * b);
    out[i] = v;
}

// Tiles: n blocks [0, nb_full) x tb token blocks multiply all of K into z [T][N]; n blocks [nb_full, nb_all) do it in S splits of K whose sums
// go to zt[split][T][ld_t] (columns counted from 128 nb_full): the last round of workgroups, which whole tiles would leave partly empty.
struct ObF32Gemm {
    const char *W; long long ldw;              // packed rows: 16-byte aligned, N * ldw < 4 GB
    const char *planes;
    float *z, *zt; long long zt_split; int ld_t;
    int T, N, quads, tb, nb_full, nb_all, S;
    int columns;                               // whole tiles numbered columns first
};

template <int WN, int WT, int NW, int TW, int KS, int NST>
__global__ __launch_bounds__(256, 2) void ob_f32_gemm_kernel(const ObF32Gemm A)
{
    constexpr int TB = WT * TW, TILES = TB * 3 * KS, PER = TILES / 4, SQ = 8 / KS;      // 1 KB tiles of a stage, per wave; stages of a quad
    static_assert(WN * WT == 4 && WN * NW == 8 && TILES % 4 == 0 && SQ >= NST - 2, "tile shape");
    extern __shared__ __attribute__((aligned(16))) char smem[];
    constexpr int WBUF = NST * TILES * 1024;                                            // two 4 KB buffers of packed rows behind the stages
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave % WN, wt = wave / WN, r = lane & 15, gq = lane >> 4;
    // whole tiles first, then the splits; each part dealt to the 8 XCDs in contiguous ranges.  A column block's packed rows are 1/48 of a token block's parts: the
    // tiles in flight on an XCD are all the columns of a token block or two.  The token blocks come first, so that an XCD reads its own columns' packed rows alone, among
    // the splits, up to 8 token blocks (whose parts its range needs anyway), and where all tiles run at once and the parts are 9 MB at most, little enough for the L2s.
    // Token blocks first -> columns first, whole call: 5500 rows 4096 -> 4096 750 -> 452 us (2.9 GB of parts through the L2s, 0.13 now), 16000 rows 1024 -> 2816 453 -> 312,
    // 2000 rows 4096 -> 11008 446 -> 413, 1300 rows 4096 -> 4096 (11 blocks) 141 -> 136, 9000 rows 64 -> 1024 (568 tiles) 50.4 -> 44.8; 731 rows 4096 -> 11008 (6) 152.4 either
    // way, 130 rows (3) 74.0 -> 75.3; splits alone, 1100 rows 1024 -> 2816, 40.4 -> 41.3; 2000 rows 64 -> 4096 (512 tiles, 0.8 MB) 38.1 -> 44.0, 2871 rows 256 -> 2048
    // (368, 4.4 MB) 34.4 -> 37.9, 1409 rows 512 -> 4096 (384, 4.3 MB) 38.7 -> 42.3.
    const int nfull = A.nb_full * A.tb;
    const bool tail = (int)blockIdx.x >= nfull;
    const int nwg = tail ? (int)gridDim.x - nfull : nfull, orig = (int)blockIdx.x - (tail ? nfull : 0);
    const int xcd = orig & 7, q8 = nwg >> 3, rem = nwg & 7;
    int bid = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + (orig >> 3);
    int tblk, nblk, split = 0;
    if (!tail && A.columns) { nblk = bid % A.nb_full; tblk = bid / A.nb_full; }
    else {
        tblk = bid % A.tb;
        bid /= A.tb;
        const int ntail = A.nb_all - A.nb_full;
        split = tail ? bid / ntail : 0;
        nblk = tail ? A.nb_full + bid % ntail : bid;
    }
    const int n0 = nblk * 128, band0 = tblk * TB, bands = (A.T + 15) >> 4;
    int q_lo = 0, nq = A.quads;
    if (tail) {
        const int b = A.quads / A.S, m = A.quads - b * A.S;
        q_lo = split * b + min(split, m);
        nq = b + (split < m ? 1 : 0);
    }
    const char *src[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int j = wave * PER + i, ks = j / (3 * TB), tt = j / 3 % TB, p = j % 3;
        src[i] = A.planes + (((size_t)min(band0 + tt, bands - 1) * A.quads + q_lo) * 8 + ks) * 3072 + p * 1024;
    }
    const uint32_t woff = (uint32_t)min(n0 + 32 * wave + (lane >> 1), A.N - 1) * (uint32_t)A.ldw + (lane & 1) * 16;
    const char *wsrc = A.W + q_lo * 32;
    const uint32_t lds0 = (uint32_t)(size_t)(__attribute__((address_space(3))) char *)smem;
    const int nst = nq * SQ;
    auto dma = [&](int st, int buf) {
        const size_t o = (size_t)min(st, nst - 1) * (KS * 3072);
#pragma unroll
        for (int i = 0; i < PER; ++i) ob_dma_1k(src[i] + o, lane * 16, lds0 + (uint32_t)(buf * TILES + wave * PER + i) * 1024);
    };
    auto wdma = [&](int q) { ob_dma_1k(wsrc + min(q, nq - 1) * 32, woff, lds0 + WBUF + (uint32_t)(q & 1) * 4096 + wave * 1024); };
    ob_float4 hi[NW][TW], lo[NW][TW];
#pragma unroll
    for (int i = 0; i < NW; ++i)
#pragma unroll
        for (int j = 0; j < TW; ++j) hi[i][j] = lo[i][j] = (ob_float4){0.f, 0.f, 0.f, 0.f};
    if constexpr (KS == 1) {
        // A step's products by part (upper, middle, lower), each part's operands read while the part before is multiplied, a sign operand's words, the reads and the
        // transfers one behind each product (sched_barrier keeps them there).  The wait and barrier stand behind the upper part: stage st + 1 has landed for everyone,
        // and everyone has read stage st, whose buffer takes stage st + NST.
        ob_bf8 a[TW][3];
        ob_u32x4 w[NW];
        ob_u32x2 wq[NW];
        uint32_t c = 0, mask = 0x80008000u, one = 0x3F803F80u;
        asm("" : "+s"(mask));
        asm("" : "+v"(one));
        const char *lane0 = smem + lane * 16 + wt * (TW * 3072), *wrow = smem + WBUF + (wn * NW * 16 + r) * 32 + gq * 8;
        const auto rd = [&](int b, int j, int p) { return *reinterpret_cast<const ob_bf8 *>(lane0 + b * (TILES * 1024) + (j * 3 + p) * 1024); };
        // words 4 j / TW .. of row tile i's sign operand in step st of its quad, behind product j of another row tile
        const auto make = [&](int i, int st, int j) __attribute__((always_inline)) {
            if (j == 0) { const uint32_t b = wq[i][st >> 2] >> (8 * (st & 3)); c = (b & 0x55u) | ((b & 0xAAu) << 15); }
#pragma unroll
            for (int p = 4 * j / TW; p < 4 * (j + 1) / TW; ++p) w[i][p] = ((c << (15 - 2 * p)) & mask) | one;
        };
        wdma(0);
#pragma unroll
        for (int s = 0; s < NST; ++s) dma(s, s);
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#pragma unroll
        for (int i = 0; i < NW; ++i) wq[i] = *reinterpret_cast<const ob_u32x2 *>(wrow + i * 512);
#pragma unroll
        for (int i = 0; i < (NW - 1) * TW; ++i) make(i / TW, 0, i % TW);
#pragma unroll
        for (int j = 0; j < TW; ++j) { a[j][0] = rd(0, j, 0); a[j][1] = rd(0, j, 1); }
        int buf = 0;
        const auto step = [&](auto sqc, int q) __attribute__((always_inline)) {
            constexpr int sq = decltype(sqc)::value, PN = NW * TW;
            static_assert(PN >= 5 + PER && NW >= 2, "room behind the products");
            // (step 7 reads the next quad's packed rows, requested in step 0: six stages of transfers are younger by then, of which the wait may leave NST - 2)
            static_assert(NST >= 2 && NST <= 7, "the next quad's packed rows have landed");
            const int next = buf + 1 == NST ? 0 : buf + 1;
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                // (the younger stages may be outstanding, and the next quad's packed rows where they were requested behind stage st + 1)
                if (p == 1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((NST - 2) * PER + (sq >= 1 && sq <= NST - 1 ? 1 : 0)) : "memory");
#pragma unroll
                for (int m = 0; m < PN; ++m) {
                    const int i = m / TW, j = m % TW;
                    ob_float4 &z = p ? lo[i][j] : hi[i][j];
                    z = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ob_bf8, w[i]), a[j][p], z, 0, 0, 0);
                    if (p == 0 && m < TW) a[m][2] = rd(buf, m, 2);
                    if (p == 1) {
                        if (m < TW) a[m][0] = rd(next, m, 0);
                        if (sq == 7 && m < NW) wq[m] = *reinterpret_cast<const ob_u32x2 *>(wrow + ((q + 1) & 1) * 4096 + m * 512);
                        if (m >= 4 && m < 4 + PER) {
                            const int d = m - 4;
                            ob_dma_1k(src[d] + (size_t)min(q * 8 + sq + NST, nst - 1) * 3072, lane * 16, lds0 + (uint32_t)(buf * TILES + wave * PER + d) * 1024);
                        }
                        if (sq == 0 && m == 4 + PER) wdma(q + 1);
                    }
                    if (p == 2 && m < TW) a[m][1] = rd(next, m, 1);
                    // a row tile's operand makes room for the next step's when its last product has it; the last one's is made in that step
                    if (p == 0 && i == 0) make(NW - 1, sq, j);
                    if (p == 2 && i > 0) make(i - 1, (sq + 1) & 7, j);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            buf = next;
        };
        for (int q = 0; q < nq; ++q) {
            step(std::integral_constant<int, 0>(), q); step(std::integral_constant<int, 1>(), q); step(std::integral_constant<int, 2>(), q);
            step(std::integral_constant<int, 3>(), q); step(std::integral_constant<int, 4>(), q); step(std::integral_constant<int, 5>(), q);
            step(std::integral_constant<int, 6>(), q); step(std::integral_constant<int, 7>(), q);
        }
    } else {
    wdma(0);
#pragma unroll
    for (int s = 0; s < NST - 1; ++s) dma(s, s);
    int buf = 0;
    ob_u32x2 wq[NW];
    for (int q = 0; q < nq; ++q) {
#pragma unroll
        for (int sq = 0; sq < SQ; ++sq) {
            // stage q SQ + sq has landed (at most the NST - 2 younger ones are outstanding; the packed rows of quad q were requested a whole quad
            // ago, SQ >= NST - 2), everyone is done with the stage before it, whose buffer takes the stage NST - 1 ahead
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"((NST - 2) * PER) : "memory");
            if (sq == 0) wdma(q + 1);
            dma(q * SQ + sq + NST - 1, buf == 0 ? NST - 1 : buf - 1);
            const char *base = smem + buf * (TILES * 1024) + lane * 16;
            if (sq == 0) {
#pragma unroll
                for (int i = 0; i < NW; ++i)
                    wq[i] = *reinterpret_cast<const ob_u32x2 *>(smem + WBUF + (q & 1) * 4096 + ((wn * NW + i) * 16 + r) * 32 + gq * 8);
            }
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                ob_bf8 a[TW][3];
#pragma unroll
                for (int j = 0; j < TW; ++j)
#pragma unroll
                    for (int p = 0; p < 3; ++p) a[j][p] = *reinterpret_cast<const ob_bf8 *>(base + ((ks * TB + wt * TW + j) * 3 + p) * 1024);
                const int s = sq * KS + ks;
                uint32_t mask = 0x80008000u;
                asm("" : "+s"(mask));
                __builtin_amdgcn_s_setprio(1);
#pragma unroll
                for (int i = 0; i < NW; ++i) {
                    const uint32_t b = wq[i][s >> 2] >> (8 * (s & 3));
                    const uint32_t c = (b & 0x55u) | ((b & 0xAAu) << 15);
                    ob_u32x4 e;
#pragma unroll
                    for (int p = 0; p < 4; ++p) e[p] = ((c << (15 - 2 * p)) & mask) | (0x3F803F80u & ~mask);
                    const ob_bf8 w = __builtin_bit_cast(ob_bf8, e);
#pragma unroll
                    for (int j = 0; j < TW; ++j) hi[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a[j][0], hi[i][j], 0, 0, 0);
#pragma unroll
                    for (int p = 1; p < 3; ++p)
#pragma unroll
                        for (int j = 0; j < TW; ++j) lo[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, a[j][p], lo[i][j], 0, 0, 0);
                }
                __builtin_amdgcn_s_setprio(0);
            }
            buf = buf + 1 == NST ? 0 : buf + 1;
        }
    }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                   // no transfer may land after the workgroup's LDS is released
    float *out = tail ? A.zt + (size_t)split * A.zt_split - A.nb_full * 128 : A.z;
    const int ld = tail ? A.ld_t : A.N;
#pragma unroll
    for (int j = 0; j < TW; ++j) {
        const int t = (band0 + wt * TW + j) * 16 + r;
        if (t >= A.T) continue;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const int n = n0 + (wn * NW + i) * 16 + 4 * gq;
            if (n < A.N) *reinterpret_cast<ob_float4 *>(out + (size_t)t * ld + n) = hi[i][j] + lo[i][j];      // (N % 4 == 0)
        }
    }
}

// rows of z (columns below n_tail) and zt (S partial sums from there on): u = z g, y = LayerNorm(u) (+ bias); z may be y.  ob_layernorm_kernel's
// arithmetic (mean, centred sum of squares, 1 / sqrt); NV x 4 columns per thread.
struct ObF32Ln {
    const float *z, *zt; long long zt_split; int ld_t, S, n_tail;
    const float *g, *bias; float *y, *u; int N, skip; float eps;
};
// SPLIT: all columns are split ones (the other form keeps twice as many waves on a CU)
template <int NV, int THREADS, bool SPLIT>
__global__ __launch_bounds__(THREADS, 4) void ob_f32_ln_kernel(const ObF32Ln A)
{
    __shared__ float red[2][THREADS / 64];
    const int tid = threadIdx.x;
    const size_t t = blockIdx.x, row = t * A.N;
    ob_float4 u[NV];
    float s = 0.f;
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int n = (v * THREADS + tid) * 4;
        u[v] = !SPLIT && n < A.n_tail && n < A.N ? *reinterpret_cast<const ob_float4 *>(A.z + row + n) : (ob_float4){0.f, 0.f, 0.f, 0.f};
    }
    if constexpr (SPLIT) {
        // the splits in order, G of them in flight for all of a thread's columns (column by column, as below, the way there is made NV S / 4 times: one row of
        // 11008 columns, five splits 9.8 -> 6.7 us)
        constexpr int G = NV >= 4 ? 2 : 4;
        const float *p = A.zt + t * A.ld_t;
#pragma unroll 1
        for (int k = 0; k < A.S; k += G) {
            ob_float4 e[G][NV];
#pragma unroll
            for (int i = 0; i < G; ++i)
#pragma unroll
                for (int v = 0; v < NV; ++v) {
                    const int n = (v * THREADS + tid) * 4;
                    e[i][v] = *reinterpret_cast<const ob_float4 *>(p + min(k + i, A.S - 1) * A.zt_split + (n < A.N ? n : 0));
                }
#pragma unroll
            for (int i = 0; i < G; ++i)
#pragma unroll
                for (int v = 0; v < NV; ++v) if (k + i < A.S) u[v] += e[i][v];
        }
#pragma unroll
        for (int v = 0; v < NV; ++v) if ((v * THREADS + tid) * 4 >= A.N) u[v] = (ob_float4){0.f, 0.f, 0.f, 0.f};
    } else if (A.n_tail < A.N) {                                       // (uniform)
        const float *p = A.zt + t * A.ld_t - A.n_tail;
#pragma unroll
        for (int v = 0; v < NV; ++v) {
            const int n = (v * THREADS + tid) * 4;
            if (n >= A.n_tail && n < A.N) {
                const float *pn = p + n;
#pragma unroll 1
                for (int k = 0; k < A.S; k += 4, pn += 4 * A.zt_split) {                // the splits in order, four in flight
                    ob_float4 e[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = *reinterpret_cast<const ob_float4 *>(pn + min(i, A.S - 1 - k) * A.zt_split);
#pragma unroll
                    for (int i = 0; i < 4; ++i) if (k + i < A.S) u[v] += e[i];
                }
            }
        }
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int n = (v * THREADS + tid) * 4;
        if (n < A.N) u[v] *= *reinterpret_cast<const ob_float4 *>(A.g + n);
    }
    float mean = 0.f, rstd = 1.f;
    if (!A.skip) {                                                     // (uniform)
#pragma unroll
        for (int v = 0; v < NV; ++v) s += (u[v][0] + u[v][1]) + (u[v][2] + u[v][3]);
        mean = ob_block_sum(s, red[0]) / (float)A.N;
        float q = 0.f;
#pragma unroll
        for (int v = 0; v < NV; ++v)
            if ((v * THREADS + tid) * 4 < A.N) {
#pragma unroll
                for (int i = 0; i < 4; ++i) { const float d = u[v][i] - mean; q += d * d; }
            }
        rstd = 1.0f / sqrtf(ob_block_sum(q, red[1]) / (float)A.N + A.eps);
    }
#pragma unroll
    for (int v = 0; v < NV; ++v) {
        const int n = (v * THREADS + tid) * 4;
        if (n < A.N) {
            if (A.u) *reinterpret_cast<ob_float4 *>(A.u + row + n) = u[v];
            ob_float4 o = u[v];
            if (!A.skip) {
                o = (o - mean) * rstd;
                if (A.bias) o += *reinterpret_cast<const ob_float4 *>(A.bias + n);
            }
            *reinterpret_cast<ob_float4 *>(A.y + row + n) = o;
        }
    }
}
