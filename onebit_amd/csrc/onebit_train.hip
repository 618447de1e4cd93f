// Train-mode 1-bit linear layer of libonebit_hip.so (include/onebit.h): launches of ob_train.h.
#include <algorithm>
#include <type_traits>
#include "ob_host.h"
#include "ob_train.h"
#include "ob_train16.h"
#include "ob_train32.h"

// onebit_train_forward / onebit_train_backward: bitnet.py:14-28 (SignSTE) and :58-68 (BitLinear.forward)
template <bool RCA, bool RCB, int TXA, int TXB, int EPI>
static void ob_launch_tgemm(const ObTGemmArgs &a, hipStream_t s)
{
    const dim3 grid((unsigned)((a.N + OB_TG_BN - 1) / OB_TG_BN), (unsigned)((a.M + OB_TG_BM - 1) / OB_TG_BM));
    hipLaunchKernelGGL((ob_tgemm_kernel<RCA, RCB, TXA, TXB, EPI>), grid, dim3(OB_TG_THREADS), 0, s, a);
}

static size_t ob_train_align(size_t b) { return (b + 255) & ~(size_t)255; }

// ---- float16 (ob_train16.h) ---------------------------------------------------------------------------------------------
static int64_t ob_t16_up32(int64_t n) { return (n + 31) / 32 * 32; }
static size_t ob_t16_bytes(int64_t rows, int64_t cols) { return (size_t)ob_t16_up32(rows) * ob_t16_up32(cols) * 2; }
// band slices of the column sums, and the sums' bytes ([slices][2][N]; the input gradient's: two per block of 128 rows, [..][K])
static int ob_t16_slices(int64_t T) { const int64_t bands = ob_t16_up32(T) / 16; return (int)(bands < OB_TC_SLICES ? bands : OB_TC_SLICES); }
static size_t ob_t16_part_bytes(int64_t T, int64_t K, int64_t N)
{
    const size_t a = (size_t)ob_t16_slices(T) * 2 * N * 4, b = (size_t)((T + 127) / 128) * 2 * K * 4;
    return ob_train_align(a > b ? a : b);
}

// z [T][N] (gx = false) and the input gradient [T][K] of few rows are few tiles with a long sum: their steps of 32 in ns slices, one workgroup a CU, whose float32 sums
// a pass adds.  128 x 128 outputs a workgroup, beyond 128 rows (wide) 128 x 256.  By what it gives: a step takes 0.26 us (float32: three products, 0.75), the pass 4.5 us
// and the sums' way out and back at 5 TB/s.  From 600 launches, whole passes, unsliced -> sliced: forward 64 rows 11008 -> 4096 114 -> 56 us, 300 rows 119 -> 74, 700 rows
// 4096 -> 4096 56 -> 53; backward 64 rows 4096 -> 11008 220 -> 142, 300 rows 258 -> 194, 700 rows 293 -> 255; float32 64 rows 515 -> 280, 700 rows 770 -> 673.  More
// workgroups than 256, two a CU: 1-4 % either way.  (256: the chip's CUs, as a constant, so that what a workspace was asked for with holds on every device.)
struct ObTrainPlan { int ns; bool wide; };
static ObTrainPlan ob_train_plan(int dtype, bool gx, int64_t T, int64_t C, int64_t R)
{
    const int nk = (int)std::min<int64_t>(ob_t16_up32(R) / 32, 1 << 26);
    ObTrainPlan best = {1, T > 128};
    const int64_t tiles = !best.wide ? (C + 127) / 128 : gx ? ((T + 255) / 256) * ((C + 127) / 128) : ((T + 127) / 128) * ((C + 255) / 256);
    double most = 0;
    for (int ns = 2; ns <= 16 && ns * tiles <= 256 && ns * 8 <= nk; ++ns) {
        const double gain = (dtype == ONEBIT_F16 ? 0.26 : 0.75) * nk * (1.0 - 1.0 / ns) - 4.5 - 8.0 * ns * (double)T * (double)C / 5e6;
        if (gain > most) { most = gain; best.ns = ns; }
    }
    return best;
}
static ObTrainPlan ob_train_plan(int dtype, bool gx, int64_t T, int64_t C, int64_t R, bool slices)
{
    ObTrainPlan p = ob_train_plan(dtype, gx, T, C, R);
    if (!slices) p.ns = 1;
    return p;
}
static size_t ob_train_zld(int64_t T, int64_t C) { return ob_train_align((size_t)T * C * 4) / 4; }
static size_t ob_train_slice_bytes(const ObTrainPlan &p, int64_t T, int64_t C) { return p.ns > 1 ? p.ns * ob_train_zld(T, C) * 4 : 0; }
template <typename T>
static void ob_train_zsum(const float *zp, size_t zld, int ns, T *z, size_t n, hipStream_t s)
{
    hipLaunchKernelGGL(ob_train_zsum_kernel<T>, dim3((unsigned)((n + 1023) / 1024)), dim3(256), 0, s, zp, zld, ns, z, n, ob_aligned(z, 4 * sizeof(T)));
}
template <typename T>
static void ob_train_gxsum(const float *zp, int ns, const void *h, const void *x, void *gx, float *part, int64_t rows, int64_t cols, hipStream_t s)
{
    ObTrainGxSum<T> a = {zp, ob_train_zld(rows, cols), ns, (const T *)h, (const T *)x, (T *)gx, part, (int)rows, (int)cols, cols % 4 == 0 && ob_aligned(x, 4 * sizeof(T)) && ob_aligned(gx, 4 * sizeof(T))};
    hipLaunchKernelGGL(ob_train_gxsum_kernel<T>, dim3((unsigned)((cols + 63) / 64), (unsigned)(2 * ((rows + 127) / 128))), dim3(256), 0, s, a);
}

static void ob_t16_tiles(bool sign, const void *p, const void *vec, char *out, int64_t rows, int64_t cols, hipStream_t s)
{
    ObT16Tiles a = {(const _Float16 *)p, (const _Float16 *)vec, out, (int)rows, (int)cols, (int)(ob_t16_up32(rows) / 16), (int)(ob_t16_up32(cols) / 32)};
    const unsigned grid = (unsigned)(((int64_t)a.bands * ((a.ct + 3) / 4) + 3) / 4);
    if (sign) hipLaunchKernelGGL(ob_t16_tiles_kernel<OB_T16_SIGN>, dim3(grid), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(ob_t16_tiles_kernel<OB_T16_SCALE>, dim3(grid), dim3(256), 0, s, a);
}

static void ob_t16_turn(const void *p, const void *vec, char *out, int64_t rows, int64_t cols, hipStream_t s)
{
    ObT16Turn a = {(const _Float16 *)p, (const _Float16 *)vec, out, (int)rows, (int)cols, (int)(ob_t16_up32(rows) / 32), (int)(ob_t16_up32(cols) / 32)};
    hipLaunchKernelGGL(ob_t16_turn_kernel, dim3((unsigned)(((int64_t)a.rt * ((a.ct + 3) / 4) + 3) / 4)), dim3(256), 0, s, a);
}

static int ob_t16_wr_lds(int mt) { return std::max(ob_wr_steps(mt) * mt * 1024, OB_T16_ROWS_LDS); }
// One operand straight into registers from more 128 x 128 outputs than CUs on, with 128 or 256 of the other operand's, whichever costs less by its rounds.  The
// weight gradient's epilogue reads W: with 128, whose second workgroup's products run meanwhile.
// Both operands through the LDS -> now, 4096 and 1024 rows: z 343 -> 316, 95 -> 89 us, input gradient 408 -> 282, 131 -> 130 (few tiles: as before), weight
// gradient 441 -> 376, 163 -> 130.
template <int EPI, bool TRW, bool TRA>
static void ob_t16_mm(const ObT16Mm &a, const ObTrainPlan &p, hipStream_t s)
{
    constexpr bool SWAP = TRW, TRL = TRW || TRA;
    static_assert(!(TRW && TRA), "one operand lies as it is reduced");
    const int64_t cus = ob_cu_count(), narrow = (int64_t)((a.nw + 7) / 8) * ((a.na + 7) / 8), nd = ((SWAP ? a.na : a.nw) + 15) / 16, nl = SWAP ? a.nw : a.na;
    const auto go = [&](auto kern, int64_t grid, int lds, bool (&attr_set)[OB_MAX_DEVICES], int ns = 1) {
        ob_set_max_lds_once(kern, attr_set, lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)grid, (unsigned)ns), dim3(256), lds, s, a);
    };
    static bool attr_set[5][OB_MAX_DEVICES] = {};
    const int64_t t8 = nd * ((nl + 7) / 8), t16 = nd * ((nl + 15) / 16);
    if constexpr (EPI != OB_T16_GW) if (p.ns > 1) {
        if (p.wide) go(ob_t16_wr_kernel<OB_T16_PART, TRL, SWAP, 8>, t8, ob_t16_wr_lds(8), attr_set[3], p.ns);
        else go(ob_t16_mm_kernel<OB_T16_PART, TRW, TRA>, narrow, 4 * 16 * 1024, attr_set[4], p.ns);
        return;
    }
    if (narrow <= cus) go(ob_t16_mm_kernel<EPI, TRW, TRA>, narrow, 4 * 16 * 1024, attr_set[0]);
    else if constexpr (EPI == OB_T16_GW) go(ob_t16_wr_kernel<EPI, TRL, SWAP, 8>, t8, ob_t16_wr_lds(8), attr_set[1]);
    else if (ob_wr_cost(t8, 8, cus) <= ob_wr_cost(t16, 16, cus)) go(ob_t16_wr_kernel<EPI, TRL, SWAP, 8>, t8, ob_t16_wr_lds(8), attr_set[1]);
    else go(ob_t16_wr_kernel<EPI, TRL, SWAP, 16>, t16, ob_t16_wr_lds(16), attr_set[2]);
}

// rows in registers where their width and alignment allow, else ob_train_ln_fwd_kernel
static void ob_t16_layernorm(const void *z, const void *g, const void *bias, void *y, float *stats, int64_t T, int64_t N, float eps, hipStream_t s)
{
#define OB_T16_LN(NV_) hipLaunchKernelGGL(ob_t16_ln_kernel<NV_>, dim3((unsigned)T), dim3(256), 0, s, (const _Float16 *)z, (const _Float16 *)g, \
                                          (const _Float16 *)bias, (_Float16 *)y, stats, (int)N, eps)
    if (N % 8 != 0 || N > 16384 || !ob_aligned(z, 16) || !ob_aligned(g, 16) || !ob_aligned(y, 16) || (bias && !ob_aligned(bias, 16)))
        hipLaunchKernelGGL((ob_train_ln_fwd_kernel<_Float16>), dim3((unsigned)T), dim3(256), 0, s, (const _Float16 *)z, (const _Float16 *)g,
                           (const _Float16 *)bias, (_Float16 *)y, stats, (int)N, eps);
    else if (N <= 2048) OB_T16_LN(1);
    else if (N <= 4096) OB_T16_LN(2);
    else if (N <= 8192) OB_T16_LN(4);
    else if (N <= 12288) OB_T16_LN(6);
    else OB_T16_LN(8);
#undef OB_T16_LN
}

// rows of x whose tiles the forward's scratch memory holds at once: all up to 512 MB of them, else equal portions
static int64_t ob_t16_portion(int64_t T, int64_t K)
{
    const int64_t fit = std::max<int64_t>(1, (int64_t)(((size_t)512 << 20) / ((size_t)ob_t16_up32(K) * 256))) * 128;
    if (T <= fit) return T;
    const int64_t n = (T + fit - 1) / fit;
    return ((T + n - 1) / n + 127) / 128 * 128;
}

static int ob_t16_forward(const void *x, const void *w, const void *h, const void *g, const void *bias, void *y, void *z, float *stats, char *ws, bool room,
                          int64_t T, int64_t K, int64_t N, float eps, hipStream_t s)
{
    char *sg = ws, *a = ws + ob_t16_bytes(N, K);
    ob_t16_tiles(true, w, nullptr, sg, N, K, s);
    const int kt = (int)(ob_t16_up32(K) / 32);
    const int64_t Tp = ob_t16_portion(T, K);
    const ObTrainPlan p = ob_train_plan(ONEBIT_F16, false, Tp, N, K, room);
    float *zp = (float *)(a + ob_t16_bytes(Tp, K));
    for (int64_t t0 = 0; t0 < T; t0 += Tp) {
        const int64_t n = std::min(Tp, T - t0);
        ob_t16_tiles(false, (const _Float16 *)x + t0 * K, h, a, n, K, s);
        ObT16Mm m = {sg, a, (int)((N + 15) / 16), (int)((n + 15) / 16), kt, kt, kt, (_Float16 *)z + t0 * N, (int)n, (int)N};
        m.vec4 = N % 4 == 0 && ob_aligned(z, 8);
        m.zp = zp; m.zld = ob_train_zld(n, N); m.ns = p.ns;
        ob_t16_mm<OB_T16_Z, false, false>(m, p, s);
        if (p.ns > 1) ob_train_zsum<_Float16>(zp, m.zld, p.ns, (_Float16 *)z + t0 * N, (size_t)n * N, s);
        if (const int rc = ob_launch_status("train_forward(product)")) return rc;
    }
    ob_t16_layernorm(z, g, bias, y, stats, T, N, eps, s);
    return ob_launch_status("train_forward(layernorm)");
}

static int ob_t16_backward(const void *gy, const void *x, const void *w, const void *h, const void *g, const void *z, const float *stats, void *gx, void *gw,
                           void *gh, void *gg, void *gbias, char *ws, bool room, int64_t T, int64_t K, int64_t N, hipStream_t s)
{
    // (the sign matrix and, once the input gradient is formed, x h in one place)
    char *sg = ws, *a = ws, *gz = ws + std::max(ob_t16_bytes(T, K), ob_t16_bytes(N, K));
    float *part = (float *)(gz + ob_t16_bytes(T, N)), *rowc = (float *)((char *)part + ob_t16_part_bytes(T, K, N));
    const int kt = (int)(ob_t16_up32(K) / 32), nt = (int)(ob_t16_up32(N) / 32), tt = (int)(ob_t16_up32(T) / 32), slices = ob_t16_slices(T);
    ObT16Gz q = {(const _Float16 *)gy, (const _Float16 *)z, (const _Float16 *)g, stats, rowc, part, gz, (int)T, (int)N, 2 * tt, nt, (2 * tt + slices - 1) / slices};
    int rc;
    hipLaunchKernelGGL(ob_t16_rowc_kernel, dim3((unsigned)T), dim3(256), 0, s, q);
    hipLaunchKernelGGL(ob_t16_gz_kernel, dim3((unsigned)((nt + 3) / 4), (unsigned)slices), dim3(256), 0, s, q);
    hipLaunchKernelGGL(ob_t16_cols_kernel<2>, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, (const float *)part, (_Float16 *)gg, (_Float16 *)gbias, (int)N, slices);
    ob_t16_tiles(true, w, nullptr, sg, N, K, s);
    if ((rc = ob_launch_status("train_backward(layernorm)"))) return rc;
    // gx [T, K] = fp16(gz S) h;  gh = sum_t fp16(gz S) x
    ObT16Mm m = {sg, gz, (int)((K + 15) / 16), (int)((T + 15) / 16), kt, nt, nt, (_Float16 *)gx, (int)T, (int)K, (const _Float16 *)h, (const _Float16 *)x, part};
    m.vec4 = K % 4 == 0 && ob_aligned(gx, 8) && ob_aligned(x, 8);
    const ObTrainPlan p = ob_train_plan(ONEBIT_F16, true, T, K, N, room);
    m.zp = (float *)((char *)rowc + ob_train_align((size_t)T * 8)); m.zld = ob_train_zld(T, K); m.ns = p.ns;
    ob_t16_mm<OB_T16_GX, true, false>(m, p, s);
    if (p.ns > 1) ob_train_gxsum<_Float16>(m.zp, p.ns, h, x, gx, part, T, K, s);
    hipLaunchKernelGGL(ob_t16_cols_kernel<1>, dim3((unsigned)((K + 255) / 256)), dim3(256), 0, s, (const float *)part, (_Float16 *)gh, (_Float16 *)nullptr, (int)K,
                       2 * (int)((T + 127) / 128));
    if ((rc = ob_launch_status("train_backward(grad input)"))) return rc;
    // gW [N, K] = (gz^T a) (1.001 - tanh(W)^2)
    ob_t16_turn(x, h, a, T, K, s);
    ObT16Mm v = {a, gz, (int)((K + 15) / 16), (int)((N + 15) / 16), tt, nt, tt, (_Float16 *)gw, (int)N, (int)K, (const _Float16 *)w};
    v.vec4 = K % 4 == 0 && ob_aligned(gw, 8) && ob_aligned(w, 8);
    ob_t16_mm<OB_T16_GW, false, true>(v, {1, false}, s);
    return ob_launch_status("train_backward(grad weight)");
}

// ---- float32 (ob_train32.h) ---------------------------------------------------------------------------------------------
static void ob_t32_tiles(bool sign, const void *p, const void *vec, char *out, int64_t rows, int64_t cols, hipStream_t s)
{
    ObT32Tiles a = {(const float *)p, (const float *)vec, out, ob_t16_bytes(rows, cols), (int)rows, (int)cols, (int)(ob_t16_up32(rows) / 16), (int)(ob_t16_up32(cols) / 32)};
    const unsigned grid = (unsigned)(((int64_t)a.bands * ((a.ct + 3) / 4) + 3) / 4);
    if (sign) hipLaunchKernelGGL(ob_t32_tiles_kernel<OB_T16_SIGN>, dim3(grid), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(ob_t32_tiles_kernel<OB_T16_SCALE>, dim3(grid), dim3(256), 0, s, a);
}

// the tiles of ob_t16_mm (which states both sides of each line); the weight gradient of up to 1280 rows with 128 of the other operand's, whose second workgroup
// multiplies while an epilogue reads W (whole backward, 256 / 128: 64 rows 4096 -> 11008 279 / 247 us, 300 428 / 389, 700 690 / 650, 1200 1087 / 1058, 2000 1490 / 1493)
template <int EPI, bool TRW, bool TRA>
static void ob_t32_mm(const ObT32Mm &a, const ObTrainPlan &p, hipStream_t s)
{
    constexpr bool SWAP = TRW, TRL = TRW || TRA;
    const int64_t cus = ob_cu_count(), narrow = (int64_t)((a.nw + 7) / 8) * ((a.na + 7) / 8), nd = ((SWAP ? a.na : a.nw) + 15) / 16, nl = SWAP ? a.nw : a.na;
    const auto go = [&](auto kern, int64_t grid, int lds, bool (&attr_set)[OB_MAX_DEVICES], int ns = 1) {
        ob_set_max_lds_once(kern, attr_set, lds);
        hipLaunchKernelGGL(kern, dim3((unsigned)grid, (unsigned)ns), dim3(256), lds, s, a);
    };
    static bool attr_set[5][OB_MAX_DEVICES] = {};
    const int64_t t8 = nd * ((nl + 7) / 8), t16 = nd * ((nl + 15) / 16);
    if constexpr (EPI != OB_T16_GW) if (p.ns > 1) {
        if (p.wide) go(ob_t32_wr_kernel<OB_T16_PART, TRL, SWAP, 8>, t8, ob_wr_steps(8) * 8 * 1024, attr_set[3], p.ns);
        else go(ob_t32_mm_kernel<OB_T16_PART, TRW, TRA>, narrow, 4 * 16 * 1024, attr_set[4], p.ns);
        return;
    }
    if (narrow <= cus) go(ob_t32_mm_kernel<EPI, TRW, TRA>, narrow, 4 * 16 * 1024, attr_set[0]);
    else if ((EPI == OB_T16_GW && a.nk[2] <= 40) || ob_wr_cost(t8, 8, cus) <= ob_wr_cost(t16, 16, cus)) go(ob_t32_wr_kernel<EPI, TRL, SWAP, 8>, t8, ob_wr_steps(8) * 8 * 1024, attr_set[1]);
    else go(ob_t32_wr_kernel<EPI, TRL, SWAP, 16>, t16, ob_wr_steps(16) * 16 * 1024, attr_set[2]);
}

static void ob_t32_layernorm(const void *z, const void *g, const void *bias, void *y, float *stats, int64_t T, int64_t N, float eps, hipStream_t s)
{
#define OB_T32_LN(NV_) hipLaunchKernelGGL(ob_t32_ln_kernel<NV_>, dim3((unsigned)T), dim3(256), 0, s, (const float *)z, (const float *)g, (const float *)bias, \
                                          (float *)y, stats, (int)N, eps)
    if (N % 4 != 0 || N > 16384 || !ob_aligned(z, 16) || !ob_aligned(g, 16) || !ob_aligned(y, 16) || (bias && !ob_aligned(bias, 16)))
        hipLaunchKernelGGL((ob_train_ln_fwd_kernel<float>), dim3((unsigned)T), dim3(256), 0, s, (const float *)z, (const float *)g, (const float *)bias,
                           (float *)y, stats, (int)N, eps);
    else if (N <= 1024) OB_T32_LN(1);
    else if (N <= 4096) OB_T32_LN(4);
    else if (N <= 8192) OB_T32_LN(8);
    else if (N <= 12288) OB_T32_LN(12);
    else OB_T32_LN(16);
#undef OB_T32_LN
}

static int64_t ob_t32_portion(int64_t T, int64_t K) { return ob_t16_portion(T, OB_T32_PARTS * K); }

static int ob_t32_forward(const void *x, const void *w, const void *h, const void *g, const void *bias, void *y, void *z, float *stats, char *ws, bool room,
                          int64_t T, int64_t K, int64_t N, float eps, hipStream_t s)
{
    char *sg = ws, *a = ws + ob_t16_bytes(N, K);
    ob_t32_tiles(true, w, nullptr, sg, N, K, s);
    const int kt = (int)(ob_t16_up32(K) / 32);
    const int64_t Tp = ob_t32_portion(T, K);
    const ObTrainPlan p = ob_train_plan(ONEBIT_F32, false, Tp, N, K, room);
    float *zp = (float *)(a + OB_T32_PARTS * ob_t16_bytes(Tp, K));
    for (int64_t t0 = 0; t0 < T; t0 += Tp) {
        const int64_t n = std::min(Tp, T - t0);
        ob_t32_tiles(false, (const float *)x + t0 * K, h, a, n, K, s);
        ObT32Mm m = {sg, a, (int)((N + 15) / 16), (int)((n + 15) / 16), kt, kt, {kt, kt, kt}, {}, {2 * ob_t16_bytes(n, K), ob_t16_bytes(n, K), 0},
                     (float *)z + t0 * N, (int)n, (int)N};
        m.vec4 = N % 4 == 0 && ob_aligned(z, 16);
        m.zp = zp; m.zld = ob_train_zld(n, N); m.ns = p.ns;
        ob_t32_mm<OB_T16_Z, false, false>(m, p, s);
        if (p.ns > 1) ob_train_zsum<float>(zp, m.zld, p.ns, (float *)z + t0 * N, (size_t)n * N, s);
        if (const int rc = ob_launch_status("train_forward(product)")) return rc;
    }
    ob_t32_layernorm(z, g, bias, y, stats, T, N, eps, s);
    return ob_launch_status("train_forward(layernorm)");
}

// (the sign matrix and, once the input gradient is formed, the parts of x h in one place)
static size_t ob_t32_operand_bytes(int64_t T, int64_t K, int64_t N) { return std::max(OB_T32_PARTS * ob_t16_bytes(T, K), ob_t16_bytes(N, K)); }

static int ob_t32_backward(const void *gy, const void *x, const void *w, const void *h, const void *g, const void *z, const float *stats, void *gx, void *gw,
                           void *gh, void *gg, void *gbias, char *ws, bool room, int64_t T, int64_t K, int64_t N, hipStream_t s)
{
    char *sg = ws, *a = ws, *gz = ws + ob_t32_operand_bytes(T, K, N);
    const size_t gzb = ob_t16_bytes(T, N);
    float *part = (float *)(gz + OB_T32_PARTS * gzb), *rowc = (float *)((char *)part + ob_t16_part_bytes(T, K, N));
    const int kt = (int)(ob_t16_up32(K) / 32), nt = (int)(ob_t16_up32(N) / 32), tt = (int)(ob_t16_up32(T) / 32), slices = ob_t16_slices(T);
    ObT32Gz q = {(const float *)gy, (const float *)z, (const float *)g, stats, rowc, part, gz, gzb, (int)T, (int)N, 2 * tt, nt, (2 * tt + slices - 1) / slices};
    int rc;
    hipLaunchKernelGGL(ob_t32_rowc_kernel, dim3((unsigned)T), dim3(256), 0, s, q);
    hipLaunchKernelGGL(ob_t32_gz_kernel, dim3((unsigned)((nt + 3) / 4), (unsigned)slices), dim3(256), 0, s, q);
    hipLaunchKernelGGL(ob_t32_cols_kernel<2>, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, (const float *)part, (float *)gg, (float *)gbias, (int)N, slices);
    ob_t32_tiles(true, w, nullptr, sg, N, K, s);
    if ((rc = ob_launch_status("train_backward(layernorm)"))) return rc;
    // gx [T, K] = (gz S) h;  gh = sum_t (gz S) x
    ObT32Mm m = {sg, gz, (int)((K + 15) / 16), (int)((T + 15) / 16), kt, nt, {nt, nt, nt}, {}, {2 * gzb, gzb, 0}, (float *)gx, (int)T, (int)K,
                 (const float *)h, (const float *)x, part};
    m.vec4 = K % 4 == 0 && ob_aligned(gx, 16) && ob_aligned(x, 16);
    const ObTrainPlan p = ob_train_plan(ONEBIT_F32, true, T, K, N, room);
    m.zp = (float *)((char *)rowc + ob_train_align((size_t)T * 8)); m.zld = ob_train_zld(T, K); m.ns = p.ns;
    ob_t32_mm<OB_T16_GX, true, false>(m, p, s);
    if (p.ns > 1) ob_train_gxsum<float>(m.zp, p.ns, h, x, gx, part, T, K, s);
    hipLaunchKernelGGL(ob_t32_cols_kernel<1>, dim3((unsigned)((K + 255) / 256)), dim3(256), 0, s, (const float *)part, (float *)gh, (float *)nullptr, (int)K,
                       2 * (int)((T + 127) / 128));
    if ((rc = ob_launch_status("train_backward(grad input)"))) return rc;
    // gW [N, K] = (gz^T a) (1.001 - tanh(W)^2): a's parts lie lowest first, gz's highest, so that a walk through both meets the pairs of one magnitude
    ObT32Turn tn = {(const float *)x, (const float *)h, a, (int)T, (int)K, tt, kt};
    hipLaunchKernelGGL(ob_t32_turn_kernel, dim3((unsigned)(((int64_t)tt * ((kt + 3) / 4) + 3) / 4)), dim3(256), 0, s, tn);
    ObT32Mm v = {a, gz, (int)((K + 15) / 16), (int)((N + 15) / 16), OB_T32_PARTS * tt, nt, {3 * tt, 2 * tt, tt}, {0, (size_t)tt * 1024, (size_t)tt * 2048}, {},
                 (float *)gw, (int)N, (int)K, (const float *)w};
    v.vec4 = K % 4 == 0 && ob_aligned(gw, 16) && ob_aligned(w, 16);
    ob_t32_mm<OB_T16_GW, false, true>(v, {1, false}, s);
    return ob_launch_status("train_backward(grad weight)");
}

// Workspace of the forward pass: a smaller or absent one takes the kernels that transform operands on their way into LDS, and so do small products, where two
// launches beat four (float16: 64 -> 64 up to 2048 rows 10.7 us against 16.3; 128 -> 128, 64 rows 12.9 / 16.1; 256 -> 128 18.0 / 16.4; 64 -> 128, 8192 rows 20.4 / 18.5;
// float32, below 64 M products: 64 rows 512 -> 512 in a trace 30 us / 25, but a call's host time has two launches more, 200 rows 31 / 26; 64 rows 1024 -> 1000, the
// first that takes it, 65 / 35).  One without room for slices' sums (ob_train_forward_least) takes products of one slice.
static size_t ob_train_forward_least(int64_t T, int64_t K, int64_t N, int dtype)
{
    if (T <= 0 || K <= 0 || N <= 0 || (dtype != ONEBIT_F16 && dtype != ONEBIT_F32)) return 0;
    if (K < 512 && (N < 128 || (K < 256 && T < 100000000 / (K * N)))) return 0;
    if (dtype == ONEBIT_F32) return T * K < 64000000 / N ? 0 : OB_T32_PARTS * ob_t16_bytes(ob_t32_portion(T, K), K) + ob_t16_bytes(N, K);
    return ob_t16_bytes(ob_t16_portion(T, K), K) + ob_t16_bytes(N, K);
}
extern "C" size_t onebit_train_forward_workspace_bytes(int64_t T, int64_t K, int64_t N, int dtype)
{
    const size_t n = ob_train_forward_least(T, K, N, dtype);
    if (n == 0) return 0;
    const int64_t Tp = dtype == ONEBIT_F32 ? ob_t32_portion(T, K) : ob_t16_portion(T, K);
    return n + ob_train_slice_bytes(ob_train_plan(dtype, false, Tp, N, K), Tp, N);
}

// the backward pass without room for slices' sums; float32 in products of parts (ob_train32.h)
static size_t ob_train_backward_bytes(int64_t T, int64_t K, int64_t N, int dtype)
{
    const size_t rest = ob_t16_part_bytes(T, K, N) + ob_train_align((size_t)T * 8);
    if (dtype == ONEBIT_F32) return ob_t32_operand_bytes(T, K, N) + OB_T32_PARTS * ob_t16_bytes(T, N) + rest;
    return std::max(ob_t16_bytes(T, K), ob_t16_bytes(N, K)) + ob_t16_bytes(T, N) + rest;
}
extern "C" size_t onebit_train_workspace_bytes(int64_t T, int64_t K, int64_t N, int dtype)
{
    if (T <= 0 || K <= 0 || N <= 0) return 0;
    return ob_train_backward_bytes(T, K, N, dtype) + ob_train_slice_bytes(ob_train_plan(dtype, true, T, K, N), T, K);
}
extern "C" size_t onebit_train_least_workspace_bytes(int64_t T, int64_t K, int64_t N, int dtype)
{
    if (T <= 0 || K <= 0 || N <= 0) return 0;
    const size_t n = ob_train_backward_bytes(T, K, N, dtype);
    if (dtype != ONEBIT_F32) return n;
    return std::min(n,                                                     // (gz, ga, the rows' means, the column sums' partials)
                    ob_train_align((size_t)T * N * 4) + ob_train_align((size_t)T * K * 4) + ob_train_align((size_t)T * 2 * sizeof(float)) +
                        ob_train_align((size_t)OB_TC_SLICES * std::max(2 * (size_t)N, (size_t)K) * sizeof(float)));
}

static int ob_train_check(const char *what, int64_t T, int64_t K, int64_t N, int dtype)
{
    if (T < 0 || K < 0 || N < 0) return ob_fail(ONEBIT_E_ARG, "%s: negative size", what);
    if (dtype != ONEBIT_F16 && dtype != ONEBIT_F32) return ob_fail(ONEBIT_E_DTYPE, "%s: dtype %d", what, dtype);
    if (T > 0x7fffffffLL || K > 0x7fffffffLL || N > 0x7fffffffLL) return ob_fail(ONEBIT_E_ARG, "%s: dimension too large", what);
    return 0;
}

template <typename TI>
static int ob_train_forward_t(const void *x, const void *w, const void *h, const void *g, const void *bias, void *y, void *z,
                              float *stats, int64_t T, int64_t K, int64_t N, float eps, hipStream_t s)
{
    ObTGemmArgs a = {};
    a.A = x; a.lda = K; a.va = h;            // A(t, k) = x[t, k] * h[k]
    a.B = w; a.ldb = K;                      // B(n, k) = sign(W[n, k])
    a.C = z; a.ldc = N; a.M = (int)T; a.N = (int)N; a.R = (int)K;
    if constexpr (std::is_same<TI, _Float16>::value) {
        static bool attr_set[OB_MAX_DEVICES] = {};
        ob_set_max_lds_once(ob_tgemm128_f16_kernel, attr_set, OB_TG2_LDS);
        hipLaunchKernelGGL(ob_tgemm128_f16_kernel, dim3((unsigned)((N + OB_TG2_B - 1) / OB_TG2_B), (unsigned)((T + OB_TG2_B - 1) / OB_TG2_B)), dim3(OB_TG_THREADS),
                           OB_TG2_LDS, s, a);
    } else ob_launch_tgemm<true, true, OB_TX_SCALE_R, OB_TX_SIGN, OB_TE_PLAIN>(a, s);
    int rc = ob_launch_status("train_forward(gemm)");
    if (rc) return rc;
    hipLaunchKernelGGL((ob_train_ln_fwd_kernel<TI>), dim3((unsigned)T), dim3(256), 0, s, (const TI *)z, (const TI *)g, (const TI *)bias,
                       (TI *)y, stats, (int)N, eps);
    return ob_launch_status("train_forward(layernorm)");
}

extern "C" int onebit_train_forward_ws(const void *x, const void *w_latent, const void *h, const void *g, const void *bias_or_null,
                                       void *y, void *z_save, float *ln_stats, void *workspace, size_t workspace_bytes, int64_t T, int64_t K, int64_t N,
                                       int dtype, float ln_eps, void *stream)
{
    int rc = ob_train_check("train_forward", T, K, N, dtype);
    if (rc) return rc;
    if (T == 0 || N == 0) return 0;
    if (K == 0) return ob_fail(ONEBIT_E_SHAPE, "train_forward: in_features = 0");
    if (!x || !w_latent || !h || !g || !y || !z_save || !ln_stats) return ob_fail(ONEBIT_E_ARG, "train_forward: null pointer");
    hipStream_t s = (hipStream_t)stream;
    const size_t least = ob_train_forward_least(T, K, N, dtype);
    if (least && workspace && ob_aligned(workspace, 16) && workspace_bytes >= least)
        return (dtype == ONEBIT_F16 ? ob_t16_forward : ob_t32_forward)(x, w_latent, h, g, bias_or_null, y, z_save, ln_stats, (char *)workspace,
                                                                       workspace_bytes >= onebit_train_forward_workspace_bytes(T, K, N, dtype), T, K, N, ln_eps, s);
    return dtype == ONEBIT_F16 ? ob_train_forward_t<_Float16>(x, w_latent, h, g, bias_or_null, y, z_save, ln_stats, T, K, N, ln_eps, s)
                               : ob_train_forward_t<float>(x, w_latent, h, g, bias_or_null, y, z_save, ln_stats, T, K, N, ln_eps, s);
}

extern "C" int onebit_train_forward(const void *x, const void *w_latent, const void *h, const void *g, const void *bias_or_null,
                                    void *y, void *z_save, float *ln_stats, int64_t T, int64_t K, int64_t N, int dtype,
                                    float ln_eps, void *stream)
{
    return onebit_train_forward_ws(x, w_latent, h, g, bias_or_null, y, z_save, ln_stats, nullptr, 0, T, K, N, dtype, ln_eps, stream);
}

// float32 with ob_train_least's workspace: the products on v_mfma_f32_16x16x4_f32, one float32 of gz and of ga each and no sign matrix
static int ob_train_backward_f32(const void *gy, const void *x, const void *w, const void *h, const void *g, const void *z,
                                 const float *stats, void *gx, void *gw, void *gh, void *gg, void *gbias, char *ws,
                                 int64_t T, int64_t K, int64_t N, hipStream_t s)
{
    float *gz = (float *)ws;
    float *ga = (float *)(ws + ob_train_align((size_t)T * N * sizeof(float)));
    float *rowc = (float *)(ws + ob_train_align((size_t)T * N * sizeof(float)) + ob_train_align((size_t)T * K * sizeof(float)));
    float *part = (float *)((char *)rowc + ob_train_align((size_t)T * 2 * sizeof(float)));     // [OB_TC_SLICES][2 N | K] column-sum partials
    int rc;
    // 1. through the LayerNorm and * g: gz [T, N]; column sums gg, gbias
    hipLaunchKernelGGL(ob_train_ln_bwd_kernel, dim3((unsigned)T), dim3(256), 0, s, (const float *)gy, (const float *)z, (const float *)g, stats, gz, rowc, (int)N);
    if ((rc = ob_launch_status("train_backward(layernorm)"))) return rc;
    hipLaunchKernelGGL(ob_train_cols_ln_kernel, dim3((unsigned)((N + 63) / 64), OB_TC_SLICES), dim3(256), 0, s, (const float *)gy, (const float *)z, (const float *)g, stats,
                       (const float *)rowc, part, (int)T, (int)N);
    hipLaunchKernelGGL(ob_train_cols_finish_kernel<2>, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s, (const float *)part, (float *)gg, (float *)gbias, (int)N);
    if ((rc = ob_launch_status("train_backward(gg)"))) return rc;
    // 2. ga [T, K] = gz . sign(W);  gx = ga * h;  gh = sum_t ga * x
    {
        ObTGemmArgs a = {};
        a.A = gz; a.lda = N;                 // A(t, n) = gz[t, n]            (n contiguous)
        a.B = w; a.ldb = K;                  // B(k, n) = sign(W[n, k])        (k = output index, contiguous)
        a.C = ga; a.C2 = gx; a.vc = h; a.ldc = K; a.M = (int)T; a.N = (int)K; a.R = (int)N;
        ob_launch_tgemm<true, false, OB_TX_NONE, OB_TX_SIGN, OB_TE_GX>(a, s);
        if ((rc = ob_launch_status("train_backward(grad input)"))) return rc;
        hipLaunchKernelGGL(ob_train_cols_gh_kernel, dim3((unsigned)((K + 63) / 64), OB_TC_SLICES), dim3(256), 0, s, (const float *)ga, (const float *)x, part, (int)T, (int)K);
        hipLaunchKernelGGL(ob_train_cols_finish_kernel<1>, dim3((unsigned)((K + 255) / 256)), dim3(256), 0, s, (const float *)part, (float *)gh, (float *)nullptr, (int)K);
        if ((rc = ob_launch_status("train_backward(gh)"))) return rc;
    }
    // 3. gW [N, K] = (gz^T . (x * h)) * (1.001 - tanh(W)^2)
    {
        ObTGemmArgs a = {};
        a.A = gz; a.lda = N;                 // A(n, t) = gz[t, n]            (n = output index, contiguous)
        a.B = x; a.ldb = K; a.vb = h;        // B(k, t) = x[t, k] * h[k]      (k = output index, contiguous)
        a.C = gw; a.vc = w; a.ldc = K; a.M = (int)N; a.N = (int)K; a.R = (int)T;
        ob_launch_tgemm<false, false, OB_TX_NONE, OB_TX_SCALE_I, OB_TE_STE>(a, s);
        if ((rc = ob_launch_status("train_backward(grad weight)"))) return rc;
    }
    return 0;
}

extern "C" int onebit_train_backward(const void *gy, const void *x, const void *w_latent, const void *h, const void *g,
                                     const void *z_save, const float *ln_stats, void *gx, void *gw, void *gh, void *gg,
                                     void *gbias_or_null, void *workspace, size_t workspace_bytes, int64_t T, int64_t K,
                                     int64_t N, int dtype, void *stream)
{
    int rc = ob_train_check("train_backward", T, K, N, dtype);
    if (rc) return rc;
    if (T == 0 || N == 0 || K == 0) return ob_fail(ONEBIT_E_SHAPE, "train_backward: empty problem");
    if (!gy || !x || !w_latent || !h || !g || !z_save || !ln_stats || !gx || !gw || !gh || !gg)
        return ob_fail(ONEBIT_E_ARG, "train_backward: null pointer");
    const size_t least = onebit_train_least_workspace_bytes(T, K, N, dtype);
    if (!workspace || workspace_bytes < least || !ob_aligned(workspace, 16))
        return ob_fail(ONEBIT_E_WSPACE, "train_backward: needs %zu bytes of 16-byte aligned workspace", least);
    hipStream_t s = (hipStream_t)stream;
    const bool room = workspace_bytes >= onebit_train_workspace_bytes(T, K, N, dtype);
    if (dtype == ONEBIT_F16) return ob_t16_backward(gy, x, w_latent, h, g, z_save, ln_stats, gx, gw, gh, gg, gbias_or_null, (char *)workspace, room, T, K, N, s);
    if (workspace_bytes >= ob_train_backward_bytes(T, K, N, dtype))
        return ob_t32_backward(gy, x, w_latent, h, g, z_save, ln_stats, gx, gw, gh, gg, gbias_or_null, (char *)workspace, room, T, K, N, s);
    return ob_train_backward_f32(gy, x, w_latent, h, g, z_save, ln_stats, gx, gw, gh, gg, gbias_or_null, (char *)workspace, T, K, N, s);
}
