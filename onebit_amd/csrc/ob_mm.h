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
template <bool BF16, int MN, int MT, int PER, int NST, typename RW, typename RA, typename DMA>
__device__ __forceinline__ void ob_mm_loop(ob_float4 (&acc)[MN][MT], int nk, RW rw, RA ra, DMA dma)
{
    constexpr int H = MN / 2, VM = (NST - 2) * PER, WAIT = (VM & 15) | 0x70 | (VM >> 4 << 14);        // vmcnt(VM), lgkmcnt(0)
    static_assert(MN % 2 == 0 && NST >= 3 && VM < 64, "steps in flight");
#pragma unroll
    for (int s = 0; s < NST; ++s)
#pragma unroll
        for (int d = 0; d < PER; ++d) dma(d, s, s);
#pragma unroll
    for (int i = 0; i < MN; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) {
            acc[i][j] = (ob_float4){0.f, 0.f, 0.f, 0.f};
            asm volatile("" : "+a"(acc[i][j]));
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
