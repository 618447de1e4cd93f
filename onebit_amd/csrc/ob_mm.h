// Inner loop of the LDS-staged 16-bit matrix products (ob_dense.h, ob_train16.h) and their numbering of output tiles.
//
// What bounds such a product here is the LDS (128 bytes a clock and CU) as soon as a wave's tile is small: 64 x 64 per wave asks for 12 KB of
// operands per 16 MFMA issue slots of its SIMD, 128 x 64 for 18 per 32.  A wave therefore keeps up to 128 x 64 sums, two workgroups share a CU,
// and
//   * a k step runs in two halves, rows 0 .. MN / 2 - 1 of the tile against all columns, then the others: every operand register is refilled for
//     the NEXT step as soon as its last MFMA is issued, half a step or more before it is needed again -- one operand set, no copies
//   * one barrier a step, between the halves: there every wave has read its last operand of tile k (lgkmcnt 0; the reads were issued half a step
//     ago) and tile k + 1 has landed (counted vmcnt), so tile k's buffer takes tile k + NST
//   * the MFMAs accumulate in place in AGPRs by inline assembly: with the builtin hipcc (ROCm 7.2) rotates accumulators between registers, 150
//     copies a step of 64 MFMAs, a quarter of the time
#pragma once
#include "ob_common.h"
#include <utility>

// Output tile of workgroup `orig` (of at least nnb * ntb; false: none).  Workgroup ids are dealt round-robin to the 8 XCDs, each with its own L2;
// every XCD takes a contiguous range of tiles numbered in bands of 8 token blocks, token block fastest: the 32-64 tiles in flight on it are about
// as many token blocks as weight blocks.  (Rows x k columns x columns, token blocks fastest over ALL token blocks -> in bands of 8, the same kernel: 6016 x
// 2048 x 9728 224 -> 208 us, 6016 x 2048 x 17920 418 -> 381, 16384 x 4096 x 11008 1229 -> 1202; bands of 4, 5, 6, 12 are within 2 % of 8.)
__device__ __forceinline__ bool ob_tile_of(int orig, int nnb, int ntb, int &nb, int &tb, int band_of = 8)
{
    const int nwg = nnb * ntb, xcd = orig & 7, j = orig >> 3, q8 = nwg >> 3, rem = nwg & 7;
    if (j >= q8 + (xcd < rem ? 1 : 0)) return false;
    const int id = (xcd < rem ? xcd * (q8 + 1) : rem * (q8 + 1) + (xcd - rem) * q8) + j;
    const int band = id / (band_of * nnb), r = id - band * band_of * nnb, w = min(band_of, ntb - band * band_of);
    nb = r / w;
    tb = band * band_of + r - nb * w;
    return true;
}

template <bool BF16> __device__ __forceinline__ void ob_mma_acc(ob_float4 &c, ob_u32x4 a, ob_u32x4 b)
{
    if constexpr (BF16) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// acc[i][j] = sum over nk k steps of w_i a_j.  rw(buf, i), ra(buf, j): operand fragments of the step in LDS buffer `buf`; dma(d, k, buf): transfer d
// of this wave's PER of step k into `buf` (steps beyond the last are requested too, nobody reads them: dma clamps k).  All waves of the workgroup.
// CONT: onto the sums that a loop before left in acc.
template <bool BF16, int MN, int MT, int PER, int NST, bool CONT = false, typename RW, typename RA, typename DMA>
__device__ __forceinline__ void ob_mm_loop(ob_float4 (&acc)[MN][MT], int nk, RW rw, RA ra, DMA dma)
{
    if constexpr (CONT) asm volatile("s_barrier" ::: "memory");         // (everyone is done with the buffers)
    constexpr int H = MN / 2, VM = (NST - 2) * PER, WAIT = (VM & 15) | 0x70 | (VM >> 4 << 14);        // vmcnt(VM), lgkmcnt(0)
    static_assert(MN % 2 == 0 && NST >= 3 && VM < 64, "steps in flight");
#pragma unroll
    for (int s = 0; s < NST; ++s)
#pragma unroll
        for (int d = 0; d < PER; ++d) dma(d, s, s);
    if constexpr (!CONT) {
#pragma unroll
        for (int i = 0; i < MN; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                acc[i][j] = (ob_float4){0.f, 0.f, 0.f, 0.f};
                asm volatile("" : "+a"(acc[i][j]));
            }
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"((NST - 1) * PER) : "memory");               // (the zeros above are long written)
    ob_u32x4 w[MN], a[MT];
#pragma unroll
    for (int j = 0; j < MT; ++j) a[j] = ra(0, j);
#pragma unroll
    for (int i = 0; i < H; ++i) w[i] = rw(0, i);
    int buf = 0;
    for (int k = 0; k < nk; ++k) {
#pragma unroll
        for (int j = 0; j < MT; ++j) {
#pragma unroll
            for (int i = j * H / MT; i < (j + 1) * H / MT; ++i) w[H + i] = rw(buf, H + i);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < H; ++i) ob_mma_acc<BF16>(acc[i][j], w[i], a[j]);
            __builtin_amdgcn_sched_barrier(0);
        }
        __builtin_amdgcn_s_waitcnt(WAIT);
        asm volatile("s_barrier" ::: "memory");
        const int nbuf = buf + 1 == NST ? 0 : buf + 1;
#pragma unroll
        for (int j = 0; j < MT; ++j) {
#pragma unroll
            for (int i = j * H / MT; i < (j + 1) * H / MT; ++i) w[i] = rw(nbuf, i);
#pragma unroll
            for (int d = j * PER / MT; d < (j + 1) * PER / MT; ++d) dma(d, k + NST, buf);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = H; i < MN; ++i) ob_mma_acc<BF16>(acc[i][j], w[i], a[j]);
            __builtin_amdgcn_sched_barrier(0);
            a[j] = ra(nbuf, j);
        }
        buf = nbuf;
    }
    // No transfer may land after the workgroup's LDS is released; the last sums leave the matrix pipe before anything reads them.
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < MN; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) asm volatile("" : "+a"(acc[i][j]));
}

// ---- one operand straight into registers --------------------------------------------------------------------------------------------------------
// Workgroup = 16 MT x 256 outputs: a wave has 64 of the "direct" operand's, whose tiles go from memory to its registers, times all 16 MT of the other's, which the
// four waves share through the LDS.  A direct tile belongs to one wave: with MT = 8 the LDS takes 8 KB and gives 32 for 128 MFMA, where both operands through it
// take 24 and 48 of the 64 KB that it moves meanwhile.  Up to MT = 8 two workgroups share a CU; above, one has it, all 512 registers, and asks for 32 instead
// of 48 bytes a clock (MT = 16), which is what bounds the smaller ones (8192^3 bf16: MFMA 77 % of the cycles with MT = 16, 70 % with 8, 64 % with both operands in
// the LDS).
//   * NST steps of the direct operand (16 registers each, refilled behind a step's last MFMA with them) and of the other (LDS) are on the way
//   * a step runs in two halves with its one barrier between them: there everyone has read all of tile k, and tile k + 1 has landed (counted vmcnt); the
//     first half's shared operands of step k + 1 are read in the second half of step k, the second half's in the first
//   * one load, transfer or LDS read behind an MFMA: an MFMA hides what issues in its 16 cycles
//   * whole turns of NST steps without a way out between them: where paths meet hipcc waits for every load
//   * the last steps, fewer than a turn, request nothing, and their waits count transfers alone: hipcc leaves out loads whose result nobody uses, and a count with
//     them in it would let the barrier pass before the tile has landed
// hipcc does not know that the assembly is an MFMA: an operand that it copies (a spill, a full register file) right in front of one is read too early, wrong by whole
// tiles.  No copy is left with these numbers of steps, and a test of the compiled code holds both, this and the waits; the sums are those of ob_mm_loop, bit for bit.
constexpr int ob_wr_steps(int mt) { return mt < 8 ? 5 : 4; }

// What a launch of t such workgroups costs by its rounds of them: a tile's time grows with its rows and a constant; half a round of two to a CU takes about as long
// as half their work (1.1 of it), more of one 1.5-2 tiles' time.  (Fitted to 152 products of the hybrid decoders, onebit_hybrid.hip.)
static inline double ob_wr_cost(int64_t t, int mt, int64_t cus)
{
    if (mt > 8) return 1.05 * (double)((t + cus - 1) / cus) * (mt + 5.6);
    if (t <= cus) return mt + 4.5;
    const int64_t full = t / (2 * cus), rem = t - full * 2 * cus;
    return 1.04 * (mt + 4.5) * (2.0 * (double)full + (rem == 0 ? 0.0 : rem <= cus ? (full ? 1.1 : 1.0) : 1.0 + 0.5 * (double)rem / (double)cus));
}

// acc[i][j] = sum over nk k steps of direct_i other_j (SWAP: the direct operand is the MFMA's second).  Direct tile i of step k: 16 bytes at wb[i] + 1024 k + wlane.
// ra(buf, j): operand j of the step in LDS buffer `buf`; dma(d, k, buf): transfer d of this wave's PER of step k < nk into `buf`; dma_next(d, u, buf): the
// same of step u + NST - 1 behind the turn's first one, in turns one behind the other from the first on.  All waves of the workgroup.  CONT: as above.
template <bool BF16, bool SWAP, int MT, int PER, int NST, bool CONT = false, typename RA, typename DMA, typename DMAN>
__device__ __forceinline__ void ob_wr_loop(ob_float4 (&acc)[4][MT], int nk, const char *const (&wb)[4], uint32_t wlane, RA ra, DMA dma, DMAN dma_next)
{
    if constexpr (CONT) asm volatile("s_barrier" ::: "memory");
    constexpr int MN = 4, H = MT / 2, G = MT - H, C = NST / 2, VM = (NST - 2) * (PER + MN), WAIT = (VM & 15) | 0x70 | (VM >> 4 << 14);
    static_assert(VM + 2 * MN < 64 && 2 * PER <= H * MN && 2 * G <= H * MN + 1 && 2 * H <= G * MN + 1, "vmcnt; places behind MFMAs");
    ob_u32x4 w[NST][MN], a[MT];
    // (past the end: the last step's again, nobody uses them)
    const auto wload = [&](int i, int k, int u) { w[u][i] = *reinterpret_cast<const ob_u32x4 *>(wb[i] + (size_t)((uint32_t)min(k, nk - 1) * 1024u + wlane)); };
    const auto mma = [&](ob_float4 &c, ob_u32x4 x, ob_u32x4 y) { if constexpr (SWAP) ob_mma_acc<BF16>(c, y, x); else ob_mma_acc<BF16>(c, x, y); };
#pragma unroll
    for (int s = 0; s < NST; ++s) {
#pragma unroll
        for (int d = 0; d < PER; ++d) if (s < NST - 1) dma(d, min(s, nk - 1), s);
#pragma unroll
        for (int i = 0; i < MN; ++i) wload(i, s, s);
    }
    if constexpr (!CONT) {
#pragma unroll
        for (int i = 0; i < MN; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
                acc[i][j] = (ob_float4){0.f, 0.f, 0.f, 0.f};
                asm volatile("" : "+a"(acc[i][j]));
            }
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" :: "n"(VM + 2 * MN) : "memory");                       // (the zeros above are long written)
#pragma unroll
    for (int j = 0; j < H; ++j) a[j] = ra(0, j);
    int k = 0;
    uint32_t woff = wlane + (NST + C) * 1024;                                        // (immediate offsets reach 4 KB either way)
    enum { MORE, TURN, REST };                                                       // another turn behind this one; the last whole turn; the steps behind it
    const auto step = [&]<int KIND, int u>() __attribute__((always_inline)) {
        constexpr int nu = (u + 1) % NST, pu = (u + NST - 1) % NST;
#pragma unroll
        for (int j = 0; j < H; ++j)
#pragma unroll
            for (int i = 0; i < MN; ++i) {
                const int m = j * MN + i;
                mma(acc[i][j], w[u][i], a[j]);
                __builtin_amdgcn_sched_barrier(0);
                if (m % 2 == 0 && m / 2 < G) a[H + m / 2] = ra(u, H + m / 2);
                if (m % 2 == 1 && m / 2 < PER) {
                    if constexpr (KIND == MORE) dma_next(m / 2, u, pu); else if constexpr (KIND == TURN) dma(m / 2, min(k + u + NST - 1, nk - 1), pu);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        // younger than tile k + 1's transfers: NST - 2 steps' loads of both (REST: the transfers of the tiles behind it, NST - 3 - u at most); lgkmcnt(0)
        constexpr int VR = u < NST - 3 ? (NST - 3 - u) * PER : 0;
        __builtin_amdgcn_s_waitcnt(KIND == REST ? (VR & 15) | 0x70 | (VR >> 4 << 14) : WAIT);
        asm volatile("s_barrier" ::: "memory");
#pragma unroll
        for (int i = 0; i < MN; ++i)
#pragma unroll
            for (int j = 0; j < G; ++j) {
                const int m = i * G + j;
                mma(acc[i][H + j], w[u][i], a[H + j]);
                __builtin_amdgcn_sched_barrier(0);
                if (m % 2 == 0 && m / 2 < H) a[m / 2] = ra(nu, m / 2);
                if (j == G - 1) {
                    if constexpr (KIND == MORE) w[u][i] = *reinterpret_cast<const ob_u32x4 *>(wb[i] + (size_t)woff + (u - C) * 1024);
                    else if constexpr (KIND == TURN) wload(i, k + u + NST, u);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
    };
    const auto turn = [&]<int KIND, int... U>(std::integer_sequence<int, U...>) __attribute__((always_inline)) { (step.template operator()<KIND, U>(), ...); };
    for (; k + 2 * NST <= nk; k += NST) {
        turn.template operator()<MORE>(std::make_integer_sequence<int, NST>{});
        woff += NST * 1024;
    }
    for (; k + NST <= nk; k += NST) turn.template operator()<TURN>(std::make_integer_sequence<int, NST>{});
    const auto rest = [&]<int... U>(std::integer_sequence<int, U...>) __attribute__((always_inline)) { ((k + U < nk ? step.template operator()<REST, U>() : (void)0), ...); };
    rest(std::make_integer_sequence<int, NST - 1>{});
    // No transfer may land after the workgroup's LDS is released; the last sums leave the matrix pipe before anything reads them.
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
#pragma unroll
    for (int i = 0; i < MN; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) asm volatile("" : "+a"(acc[i][j]));
}
