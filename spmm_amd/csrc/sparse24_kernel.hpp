// sparse24_kernel.hpp -- C = A * B with A in 2:4 structured sparsity on the
// gfx950 sparse matrix cores (v_smfmac_f32_16x16x64_{f16,bf16}), fp32
// accumulation and output.
//
// Replaces the reference's cuSPARSELt baseline
// (perform_cuSPARSELT_24sparsity, src/spmm_cusparse.cu:2-179).  A arrives
// compressed (tca_csr_to_24): vals [M][Kp/2], meta [M][Kp/16] uint16.
// Operand layout of v_smfmac_f32_16x16x64 (probed on the MI355X with one-hot
// inputs, 2048 cases):
//   * A: lane L holds row L % 16 and columns 16 (L / 16) .. + 15 as 4 groups
//     of 4; its 8 halves are the two kept values of each group (2 G, 2 G + 1);
//   * index: bits 4G .. 4G+1 and 4G+2 .. 4G+3 of the lane's word are the
//     positions of values 2 G and 2 G + 1 inside group G — exactly one meta
//     word of tca_csr_to_24 (placed in both 16-bit halves);
//   * B: lane n + 16 g holds column n, rows 8 g .. 8 g + 7 in halves 0..7 and
//     rows 32 + 8 g .. + 7 in halves 8..15: two fragments of the dense
//     v_mfma_f32_16x16x32 B operand, one per 32-row half of the 64-row step;
//   * D: as the dense 16x16 MFMA (lane l: column l % 16, rows 4 (l / 16) + r).
//
// A workgroup owns 16 RB rows and 64 columns of C.  Its W wavefronts split K,
// each a contiguous range of it, and meet once at the end (reduce_store), so
// the loop has no barrier: a wavefront fills LDS of its own with global -> LDS
// transfers of the next two 64-deep steps (128 rows of B, the compressed A
// pieces, every fourth time a window of index words) as soon as it has read
// the last two into registers, and multiplies those meanwhile.
//
// What bounds it is lines from the L2 to the CU, however much of a line is used:
// 2.36M of them on the product below, one per 4.6 cycles and CU, the L1s active
// in 3.3 of these.  Hence two steps at a time (a
// row of A is then one whole line; one step at a time reads half lines) and
// index words by windows of 64 bytes per row (one step's are 8 bytes): with
// one step and its index words at a time, rings up to three slots deep, a
// 4096 x 4096 bf16 product took 40 us at N = 512 whatever the depth, now 21.1
// (97.7 with 64 x 256 tiles of four wavefronts staging B through registers,
// one step ahead, on 128 of the 256 CUs).
//
// B rows past K, columns past N and A past Kp come from a zero piece; rows
// past M read row M - 1 and are not stored.  Index words lie at any 2-byte
// address: the window starts at the aligned dword at or before its first.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mfma_common.hpp"

namespace tca {

typedef _Float16 f16x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x16 __attribute__((ext_vector_type(16)));

constexpr int kS24Cols = 64;  // columns of C per workgroup

struct S24Args {
    const void* vals;       // [M][Kp / 2]
    const uint16_t* meta;   // [M][Kp / 16]
    const void* B;          // K x N row-major
    float* C;               // M x N row-major
    int M, N, K, Kp;
    int row_groups, col_groups;
};

// LDS of a wavefront: two steps' B tiles (16 KiB), A pieces (2 KiB per row
// block) and a window of index words (1 KiB per row block).
template <int RB>
constexpr int s24_wave_bytes() {
    return 16384 + RB * 3072;
}
template <int RB, int W>
constexpr int s24_lds_bytes() {
    return W * s24_wave_bytes<RB>() > W * RB * 4096 ? W * s24_wave_bytes<RB>() : W * RB * 4096;
}

template <bool kBf16, int RB, int W>
__global__ __launch_bounds__(64 * W) void sparse24_kernel(S24Args a) {
    __shared__ __attribute__((aligned(16))) char lds[s24_lds_bytes<RB, W>()];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int rg, cg;
    xcd_tile(blockIdx.x, a.row_groups, a.col_groups, rg, cg);
    const int row0 = rg * 16 * RB, c0 = cg * kS24Cols;
    const int steps = a.Kp / 64;
    const int pairs = (steps + 1) / 2;  // the second step of the last pair may be missing
    const int p0 = static_cast<int>(static_cast<int64_t>(pairs) * wave / W);
    const int p1 = static_cast<int>(static_cast<int64_t>(pairs) * (wave + 1) / W);
    char* const mem = lds + wave * s24_wave_bytes<RB>();
    const uint32_t mem_at = lds_addr(mem);

    BTile<4> bt;
    bt.init(a.B, a.K, a.N, c0, lane);
    // A: transfer q of row block rb holds its rows 8 q + lane / 8, 16-byte
    // piece (lane % 8) ^ row of the pair's 128 bytes.
    const char* const av = static_cast<const char*>(a.vals);
    const int apiece = (lane & 7) ^ (lane >> 3);
    // Index words: a window of `wsteps` steps from the aligned dword at or
    // before its first word (`odd`: the words start 2 bytes after it);
    // transfer q of row block rb holds its rows 4 q + lane / 16, dword
    // (lane % 16) ^ 4 q of the window.
    const char* const am = reinterpret_cast<const char*>(a.meta);
    const int odd = static_cast<int>(reinterpret_cast<uintptr_t>(am) & 2);
    const int wpairs = odd ? 3 : 4;
    const int row_dwords = (a.Kp / 8 + odd + 3) / 4;

    auto issue = [&](int p) {
        bt.issue(128 * p, mem_at);
        const bool half = 2 * p + 1 >= steps;  // the pair's second step lies past Kp
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const int row = min(row0 + 16 * rb + 8 * q + (lane >> 3), a.M - 1);
                const char* src = av + static_cast<size_t>(row) * a.Kp + static_cast<size_t>(p) * 128 + 16 * apiece;
                if (half && apiece >= 4) src = reinterpret_cast<const char*>(&kZeroPiece);
                dma_x4(src, mem_at + 16384 + 2048 * rb + 1024 * q);
            }
        if ((p - p0) % wpairs == 0) {
#pragma unroll
            for (int rb = 0; rb < RB; rb++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int row = min(row0 + 16 * rb + 4 * q + (lane >> 4), a.M - 1);
                    const int d = min(4 * p + ((lane & 15) ^ (4 * q)), row_dwords - 1);
                    const char* src = am - odd + static_cast<size_t>(row) * (a.Kp / 8) + static_cast<size_t>(d) * 4;
                    dma_x1(src, mem_at + 16384 + 2048 * RB + 1024 * rb + 256 * q);
                }
        }
    };

    f32x4 acc[RB][4];
#pragma unroll
    for (int rb = 0; rb < RB; rb++)
#pragma unroll
        for (int c = 0; c < 4; c++) acc[rb][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int r = lane & 15, g = lane >> 4;
    if (p0 < p1) issue(p0);
    for (int p = p0; p < p1; p++) {
        wait_vmcnt<0>();
        typedef int i32x8v __attribute__((ext_vector_type(8)));
        i32x8v bq[2][4];
        i32x4v af[2][RB];
        int ix[2][RB];
        const int w = (p - p0) % wpairs;
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const uint16_t* tile = reinterpret_cast<const uint16_t*>(mem + 8192 * t);
                const i32x4v b0 = b_fragment(tile, c, lane), b1 = b_fragment(tile + 2048, c, lane);
                bq[t][c] = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
            }
            const int word = 8 * (2 * w + t) + 2 * g + odd;  // byte of the lane's index word in its window
#pragma unroll
            for (int rb = 0; rb < RB; rb++) {
                af[t][rb] = *reinterpret_cast<const i32x4v*>(mem + 16384 + 2048 * rb + 128 * r +
                                                             16 * ((4 * t + g) ^ (r & 7)));
                const int m = *reinterpret_cast<const int*>(mem + 16384 + 2048 * RB + 1024 * rb + 64 * r +
                                                            4 * ((word >> 2) ^ (4 * (r >> 2))));
                const uint32_t x = (static_cast<uint32_t>(m) >> (8 * (word & 2))) & 0xffffu;
                ix[t][rb] = static_cast<int>(x | (x << 16));
            }
        }
        wait_lds_reads();
        if (p + 1 < p1) issue(p + 1);
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int rb = 0; rb < RB; rb++) {
                    if constexpr (kBf16)
                        acc[rb][c] = __builtin_amdgcn_smfmac_f32_16x16x64_bf16(__builtin_bit_cast(bf16x8, af[t][rb]),
                                                                               __builtin_bit_cast(bf16x16, bq[t][c]),
                                                                               acc[rb][c], ix[t][rb], 0, 0);
                    else
                        acc[rb][c] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(__builtin_bit_cast(f16x8, af[t][rb]),
                                                                              __builtin_bit_cast(f16x16, bq[t][c]),
                                                                              acc[rb][c], ix[t][rb], 0, 0);
                }
    }
    reduce_store<RB, 4, W>(acc, lds, wave, lane, row0, c0, a.M, a.N, a.C);
}

}  // namespace tca
