// float32 1-bit layer of libonebit_hip.so: launches of ob_f32.h.
#include <algorithm>
#include "ob_host.h"
#include "ob_ln.h"
#include "ob_f32.h"

// Token block: the smallest of 16 / 32 / 64 that holds all rows, else 128, or 64 where 128 would pad a tenth more rows.  Whole 128-column blocks
// fill whole rounds of two workgroups per CU; the blocks left over split K so that they fill one more (at most 8 ways: the row pass reads every
// split's sums).  731 rows, 4096 -> 11008: 510 whole tiles + 6 x 8 pieces instead of a second round of 4 tiles.
// Products below 24 M (36 M where the packed rows are copied first) stay with ob_simple_kernel: three or four launches and their host work cost more
// than they save there (1 row of 4096 -> 4096: 18.2 us a call against 19.8; 2 rows: 21.3 / 20.4; 4 rows of 4064 -> 1000: 16.8 / 23.0, 16 rows:
// 22.8 / 22.6).  Larger ones: 16 rows of 4096 -> 11008 188 us -> 26, 731 rows 7371 -> 165 (1.2 PFLOP/s of bf16 products), 2048 rows 20.6 ms -> 483 us.
static bool ob_f32_takes(int64_t T, int64_t K, int64_t N)
{
    return T >= 1 && K >= 8 && N >= 4 && N % 4 == 0 && T <= (1 << 24) && K <= (1 << 24) && N <= (1 << 24) && T * N >= (K % 256 == 0 ? 24000000 : 36000000) / K &&
           (size_t)N * ((K + 255) / 256) * 32 < ((size_t)1 << 32);
}
// Rows whose parts the scratch memory holds at once (6 bytes per activation, at most OB_F32_PLANES of them): all, or as few equal portions as fit.
// (16384 rows of 4096 columns fit; 30000 in two portions 9.64 ms to 11008 columns, at once 9.51.)
#define OB_F32_PLANES ((size_t)512 << 20)
static int64_t ob_f32_portion(int64_t T, int64_t K)
{
    const size_t band = (size_t)((K + 255) / 256) * (8 * 3072);
    const int64_t fit = (int64_t)std::max<size_t>(1, OB_F32_PLANES / band) * 16;
    if (T <= fit) return T;
    const int64_t n = (T + fit - 1) / fit, even = (T + n - 1) / n, up = (even + 127) / 128 * 128;
    return up <= fit ? up : fit >= 128 ? fit / 128 * 128 : fit;
}
struct ObF32Plan { int bt, tb, quads, nb, nb_full, S, ld_t; size_t planes, rows, zt; };
static void ob_f32_plan(int64_t T, int64_t K, int64_t N, ObF32Plan &p)
{
    const auto align = [](size_t b) { return (b + 255) & ~(size_t)255; };
    p.quads = (int)((K + 255) / 256);
    const int64_t t64 = (T + 63) / 64 * 64, t128 = (T + 127) / 128 * 128;
    p.bt = T <= 16 ? 16 : T <= 32 ? 32 : T <= 64 || 10 * t128 > 11 * t64 ? 64 : 128;
    p.tb = (int)((T + p.bt - 1) / p.bt);
    p.nb = (int)((N + 127) / 128);
    const int64_t slots = 2 * (int64_t)ob_cu_count(), tiles = (int64_t)p.nb * p.tb;
    p.nb_full = (int)(tiles / slots * slots / p.tb);
    const int64_t left = (int64_t)(p.nb - p.nb_full) * p.tb;
    p.S = left > 0 ? (int)(slots / left) : 1;
    if (p.S > 8) p.S = 8;
    if (p.S > p.quads) p.S = p.quads;
    if (p.S <= 1 || N > 16384) { p.S = 1; p.nb_full = p.nb; }          // (wider rows: ob_layernorm_kernel, z whole in y)
    p.ld_t = (p.nb - p.nb_full) * 128;
    p.planes = align((size_t)((T + 15) / 16) * p.quads * (8 * 3072));
    p.rows = K % 256 == 0 ? 0 : align((size_t)N * p.quads * 32);
    p.zt = (size_t)p.S * T * p.ld_t * 4;
}
size_t ob_f32_workspace(int64_t T, int64_t K, int64_t N)
{
    if (!ob_f32_takes(T, K, N)) return 0;
    const int64_t Tp = ob_f32_portion(T, K), rest = T % Tp;            // (the last portion, if shorter, may split K further)
    ObF32Plan p, q;
    ob_f32_plan(Tp, K, N, p);
    ob_f32_plan(rest ? rest : Tp, K, N, q);
    return p.rows + std::max(p.planes + p.zt, q.planes + q.zt);
}

template <int WN, int WT, int NW, int TW, int KS, int NST>
static void ob_launch_f32_gemm(const ObF32Gemm &a, hipStream_t s)
{
    constexpr int lds = NST * WT * TW * 3 * KS * 1024 + 8192;
    static bool attr_set[OB_MAX_DEVICES] = {};
    ob_set_max_lds_once(ob_f32_gemm_kernel<WN, WT, NW, TW, KS, NST>, attr_set, lds);
    const int grid = a.nb_full * a.tb + (a.nb_all - a.nb_full) * a.tb * a.S;
    hipLaunchKernelGGL((ob_f32_gemm_kernel<WN, WT, NW, TW, KS, NST>), dim3((unsigned)grid), dim3(256), lds, s, a);
}

// the rows of one portion
static void ob_f32_rows(const ObF32Plan &p, const void *packed, int64_t ldw_bytes, const float *x, const float *h, const float *g, const float *bias, float *y,
                        float *u, char *planes, int64_t T, int64_t K, int64_t N, float eps, int skip, hipStream_t s)
{
    float *zt = (float *)(planes + p.planes);
    ObF32Split sp = {x, K, h, planes, (int)T, (int)K, p.quads};
    const int64_t units = (T + 15) / 16 * p.quads;
    hipLaunchKernelGGL(ob_f32_split_kernel, dim3((unsigned)((units + 3) / 4)), dim3(256), 0, s, sp);
    ObF32Gemm a = {};
    a.W = (const char *)packed; a.ldw = ldw_bytes;
    a.planes = planes; a.z = y; a.zt = zt; a.zt_split = (long long)T * p.ld_t; a.ld_t = p.ld_t;
    a.T = (int)T; a.N = (int)N; a.quads = p.quads; a.tb = p.tb; a.nb_full = p.nb_full; a.nb_all = p.nb; a.S = p.S;
    a.columns = p.tb > 8 && ((int64_t)p.nb * p.tb > 2 * (int64_t)ob_cu_count() || T * K * 6 > 9000000);
    if (p.bt == 16) ob_launch_f32_gemm<4, 1, 2, 1, 4, 4>(a, s);
    else if (p.bt == 32) ob_launch_f32_gemm<4, 1, 2, 2, 2, 4>(a, s);
    else if (p.bt == 64) ob_launch_f32_gemm<2, 2, 4, 2, 1, 4>(a, s);
    else ob_launch_f32_gemm<2, 2, 4, 4, 1, 3>(a, s);
    if (N > 16384) {
        hipLaunchKernelGGL((ob_layernorm_kernel<float, true>), dim3((unsigned)T), dim3(256), 0, s, (const float *)y, (const float *)nullptr, g, bias, y, u,
                           (int)N, eps, skip);
        return;
    }
    ObF32Ln l = {y, zt, a.zt_split, p.ld_t, p.S, p.nb_full * 128, g, bias, y, u, (int)N, skip, eps};
#define OB_F32_LN(NV_, TH_) do { if (p.nb_full == 0) hipLaunchKernelGGL((ob_f32_ln_kernel<NV_, TH_, true>), dim3((unsigned)T), dim3(TH_), 0, s, l); \
                                 else hipLaunchKernelGGL((ob_f32_ln_kernel<NV_, TH_, false>), dim3((unsigned)T), dim3(TH_), 0, s, l); } while (0)
    if (N <= 1024) OB_F32_LN(1, 256);
    else if (N <= 2048) OB_F32_LN(1, 512);
    else if (N <= 4096) OB_F32_LN(2, 512);
    else if (N <= 8192) OB_F32_LN(4, 512);
    else if (N <= 12288) OB_F32_LN(6, 512);
    else OB_F32_LN(8, 512);
#undef OB_F32_LN
}

bool ob_f32_forward(const void *packed, int64_t ldw_bytes, const float *x, const float *h, const float *g, const float *bias, float *y, float *u,
                    void *workspace, size_t workspace_bytes, int64_t T, int64_t K, int64_t N, float eps, int skip, hipStream_t s)
{
    if (!ob_f32_takes(T, K, N) || !workspace || !ob_aligned(workspace, 16) || workspace_bytes < ob_f32_workspace(T, K, N)) return false;
    const int64_t Tp = ob_f32_portion(T, K);
    ObF32Plan p;
    ob_f32_plan(Tp, K, N, p);
    // packed rows that are not whole 16-byte pieces of whole quads are copied so first
    if (!p.rows && (ldw_bytes % 16 != 0 || !ob_aligned(packed, 16) || N * ldw_bytes >= ((int64_t)1 << 32))) return false;
    if (!ob_aligned(g, 16) || (bias && !ob_aligned(bias, 16)) || (u && !ob_aligned(u, 16))) return false;
    char *planes = (char *)workspace + p.rows;
    if (p.rows) {
        const int64_t words = N * p.quads * 8;
        hipLaunchKernelGGL(ob_f32_rows_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, s, (const uint8_t *)packed, (long long)ldw_bytes,
                           (uint32_t *)workspace, (int)N, (int)(K / 8), p.quads);
        packed = workspace; ldw_bytes = p.quads * 32;
    }
    for (int64_t t0 = 0; t0 < T; t0 += Tp) {
        const int64_t n = std::min(Tp, T - t0);
        ob_f32_plan(n, K, N, p);
        ob_f32_rows(p, packed, ldw_bytes, x + t0 * K, h, g, bias, y + t0 * N, u ? u + t0 * N : nullptr, planes, n, K, N, eps, skip, s);
    }
    return true;
}
