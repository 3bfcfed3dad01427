// bell_kernel.hpp -- SpMM C = A * B over a Blocked-ELL A on gfx950 matrix
// cores (fp16 / bf16 inputs, fp32 accumulation and output).
//
// Blocked-ELL is the format the reference hands to cusparseSpMM for its
// block baseline (src/spmm_cusparse.cu:201-342; layout in tca_host.h):
// every block is a dense BS x BS tile, so the format feeds the matrix cores
// with no condensing.  A workgroup owns one block row (BS rows) and 64 columns
// of C.  Its W wavefronts split the block row's list, each a contiguous range
// of it, and meet once at the end (reduce_store), so the loop has no barrier:
// a wavefront fills LDS of its own with global -> LDS transfers of the next
// unit as soon as it has read the last one into registers, and multiplies
// that meanwhile.  A unit is 64 columns of A (one block of 64 or two of 32),
// so every line of the row-major ELL values is used whole: lines from the L2
// to the CU bound the kernel (A 2 BS / 32 KiB, B 8 KiB a unit; 1.78M of them on
// the product below, one per 3.7 cycles and CU, the L1s active in 3.5 of these),
// and with one block of 32 at a time half of A's would be wasted.
//
// 4096 x 4096 fp16 with a quarter of its 32 x 32 blocks at N = 512: 15.6 us
// (31.9 with a workgroup per block row and 256 columns, B staged one block
// ahead through registers with a barrier per block).  128 columns per
// wavefront take 14.6 there with four wavefronts, but up to twice as long on
// small outputs.
//
// Sums run in list order within a wavefront's range, the ranges in order.  The
// missing half of an odd list's last unit, B rows past K and columns past N
// come from a zero piece; rows past M are not stored.  Padding blocks (colind
// -1) end the block row's list.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mfma_common.hpp"

namespace tca {

constexpr int kBellCols = 64;  // columns of C per workgroup

struct BellArgs {
    const int* colind;   // [block rows][ell_blocks] block column, -1 = padding
    const void* values;  // [block rows * BS][ell_blocks * BS] row-major
    const void* B;       // K x N row-major
    float* C;            // M x N row-major
    int M, N, K, ell_blocks;
    int row_groups, col_groups;  // block rows, column groups
};

// LDS of a wavefront: a unit's B tiles and A pieces.
template <int BS>
constexpr int bell_wave_bytes() {
    return 8192 + BS * 128;
}

template <bool kBf16, int BS, int W>
__global__ __launch_bounds__(64 * W) void bell_mfma_kernel(BellArgs a) {
    static_assert(BS == 32 || BS == 64, "block size");
    constexpr int RF = BS / 16;   // 16-row fragments per block row
    constexpr int kBlk = 64 / BS; // blocks of a unit
    constexpr int kLds = W * (bell_wave_bytes<BS>() > RF * 4096 ? bell_wave_bytes<BS>() : RF * 4096);
    __shared__ __attribute__((aligned(16))) char lds[kLds];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int brow, cg;
    xcd_tile(blockIdx.x, a.row_groups, a.col_groups, brow, cg);
    const int c0 = cg * kBellCols;
    const int* const cind = a.colind + static_cast<size_t>(brow) * a.ell_blocks;

    // number of blocks in this block row (the list is a prefix, -1 after it)
    int nblk = 0, first64 = -1;
    while (nblk < a.ell_blocks) {
        const int e = nblk + lane;
        const int c = cind[min(e, a.ell_blocks - 1)];
        const uint64_t ends = __ballot(e >= a.ell_blocks || c < 0);
        if (nblk == 0) first64 = c;
        nblk += ends ? __builtin_ctzll(ends) : 64;
        if (ends) break;
    }
    // First row of B of block e (the list's first 64 entries stay in registers;
    // a block column past K reads zeros).
    const int kblk = (a.K + BS - 1) / BS;
    auto block_row = [&](int e) {
        return min(nblk <= 64 ? __builtin_amdgcn_readlane(first64, e) : cind[e], kblk) * BS;
    };
    const int units = (nblk + kBlk - 1) / kBlk;
    const int u0 = static_cast<int>(static_cast<int64_t>(units) * wave / W);
    const int u1 = static_cast<int>(static_cast<int64_t>(units) * (wave + 1) / W);
    char* const mem = lds + wave * bell_wave_bytes<BS>();
    const uint32_t mem_at = lds_addr(mem);

    BTile<BS / 32> bt;
    bt.init(a.B, a.K, a.N, c0, lane);
    // A: transfer q holds rows 8 q + lane / 8 of the block row, 16-byte piece
    // (lane % 8) ^ row of the unit's 128 bytes.
    const int apiece = (lane & 7) ^ (lane >> 3);
    const size_t arow = static_cast<size_t>(a.ell_blocks) * BS * 2;  // bytes
    const char* const av = static_cast<const char*>(a.values) + (static_cast<size_t>(brow) * BS + (lane >> 3)) * arow +
                           16 * apiece;
    auto issue = [&](int u) {
        const bool half = kBlk == 2 && 2 * u + 1 >= nblk;
#pragma unroll
        for (int b = 0; b < kBlk; b++)
            bt.issue(b && half ? a.K : block_row(kBlk * u + b), mem_at + 4096 * b);
#pragma unroll
        for (int q = 0; q < BS / 8; q++) {
            const char* src = av + 8 * q * arow + static_cast<size_t>(u) * 128;
            if (half && apiece >= 4) src = reinterpret_cast<const char*>(&kZeroPiece);
            dma_x4(src, mem_at + 8192 + 1024 * q);
        }
    };

    f32x4 acc[RF][4];
#pragma unroll
    for (int rf = 0; rf < RF; rf++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[rf][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int r = lane & 15, g = lane >> 4;
    if (u0 < u1) issue(u0);
    for (int u = u0; u < u1; u++) {
        wait_vmcnt<0>();
        i32x4v bq[2][4], af[2][RF];
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
#pragma unroll
            for (int c = 0; c < 4; c++)
                bq[ks][c] = b_fragment(reinterpret_cast<const uint16_t*>(mem + 4096 * ks), c, lane);
#pragma unroll
            for (int rf = 0; rf < RF; rf++)
                af[ks][rf] =
                    *reinterpret_cast<const i32x4v*>(mem + 8192 + 2048 * rf + 128 * r + 16 * ((4 * ks + g) ^ (r & 7)));
        }
        wait_lds_reads();
        if (u + 1 < u1) issue(u + 1);
#pragma unroll
        for (int ks = 0; ks < 2; ks++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int rf = 0; rf < RF; rf++) {
                    if constexpr (kBf16)
                        acc[rf][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, af[ks][rf]),
                                                                             __builtin_bit_cast(bf16x8, bq[ks][c]),
                                                                             acc[rf][c], 0, 0, 0);
                    else
                        acc[rf][c] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, af[ks][rf]),
                                                                            __builtin_bit_cast(f16x8, bq[ks][c]),
                                                                            acc[rf][c], 0, 0, 0);
                }
    }
    reduce_store<RF, 4, W>(acc, lds, wave, lane, brow * BS, c0, a.M, a.N, a.C);
}

}  // namespace tca
