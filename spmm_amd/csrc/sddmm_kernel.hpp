// sddmm_kernel.hpp -- kernels of the PyTorch op's backward pass (gfx950).
//
// For C = A * B with A in CSR, the gradients are
//   dL/dB      = A^T * dL/dC         (an SpMM with the transposed plan), and
//   dL/dA[j]   = <dL/dC[row(j), :], B[col(j), :]>   for every nonzero j,
// the second being a sampled dense-dense product (SDDMM) over A's pattern.
// No counterpart in the reference, which has no backward pass.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "row_kernel.hpp"

namespace tca {

constexpr int kSddmmWaves = 4;          // wavefronts per workgroup (independent spans)
constexpr uint32_t kSddmmFill = 16384;  // wavefronts a launch is split into before spans grow
constexpr uint32_t kSddmmMaxBatches = 16;

struct SddmmArgs {
    const int* rowptr;
    const int* colidx;
    const float* G;
    const void* B;
    float* out;
    int M, N;
    uint32_t nnz;
    uint32_t batches;  // 64-nonzero batches per wavefront
    const int4* tasks;  // sddmm_tasks_kernel: the row kernel's task list
    const int* perm;
    const int4* longrows;
    int ntasks;
};

// Partner's value within 8 lanes: 7 - lane, lane ^ 2, lane ^ 1.
template <int kCtrl>
__device__ __forceinline__ float dpp_swap(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, x), kCtrl, 0xf, 0xf, true));
}

// The row of nonzero j: the last r in [lo, hi] with rowptr[r] <= j.
__device__ __forceinline__ int row_of(const int* __restrict__ rowptr, uint32_t j, int lo, int hi) {
    while (lo < hi) {
        const int mid = lo + (hi - lo + 1) / 2;
        if (static_cast<uint32_t>(rowptr[mid]) <= j) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// The same for one j per wavefront, 64 probes a step (M = 2^18: three dependent loads).
__device__ __forceinline__ int wave_row_of(const int* __restrict__ rowptr, uint32_t j, int M, int lane) {
    int lo = 0, n = M;  // the row is in [lo, lo + n)
    while (n > 1) {
        const int step = (n + 63) / 64;
        const int r = lo + lane * step;
        const bool le = lane * step < n && static_cast<uint32_t>(rowptr[r]) <= j;
        const int c = __popcll(__ballot(le));  // >= 1: rowptr[lo] <= j
        const int at = (c - 1) * step;
        n = min(step, n - at);
        lo += at;
    }
    return lo;
}

// out[j] = sum_n G[row(j), n] * B[colidx[j], n] for every nonzero j.
//
// Bound: gathering a row of B per nonzero (L2 -> CU).  The nonzeros are split
// evenly whatever their rows (a wavefront owns `batches` runs of 64; the rows
// at the ends of its span are searched in rowptr), so a power-law graph's
// longest row is spread over the chip.  A batch goes to 64 / L slots of L
// lanes, L nonzeros each; lane l of a slot reads 16-byte pieces l, l + L, ...
// of the L rows of B, L loads in flight per piece column, and the L partial
// sums per lane are exchanged and added in log2 L DPP steps (a reduce-scatter:
// L - 1 adds for L nonzeros) that leave lane i of the wavefront with nonzero
// i's sum, stored coalesced.  A slot whose nonzeros share a row reads that row
// of G once per piece (the wavefront takes this path when all its slots do),
// otherwise once per nonzero, mostly from the L1.  Sums run in a fixed order:
// a piece in fp32 (chains of four), a lane's pieces in fp64 (a lane adds up
// to N / 8 products, which in fp32 would round more often than the 64-lane
// tree that this replaced), the lanes of a slot in fp32.
//
// One wavefront per row with one nonzero at a time and a six-step shuffle sum
// per nonzero (the previous kernel): 25.2 ms on 11.4M nonzeros of an R-MAT
// graph of 131,072 nodes at N = 128 fp32, 650 us on a 2048 x 2048 layer of
// 10 % at N = 1024 bf16; gathered this way 0.60 ms and 63 us (9.7 and 13.6 TB/s of
// rows of B).  Few nonzeros take sddmm_wide_kernel (below).  Rows in panels take panel_sddmm_kernel (panel_kernel.hpp), and
// the others beside them sddmm_tasks_kernel (the spans above, skipping the
// panels' nonzeros, took 97 us for them: nearly every span holds a few).

// One batch: the sums of the wavefront's 64 nonzeros (lane i: row `row`, column
// `col`, a row's nonzeros side by side), lane i's own.
template <typename T, int E, int L>
__device__ __forceinline__ float sddmm_batch(const SddmmArgs& a, int row, int col, int lane) {
    const size_t N = static_cast<size_t>(a.N);
    const uint32_t rowbytes = static_cast<uint32_t>(a.N) * sizeof(T);
    const int l = lane & (L - 1), first = lane - l;
    const int V = (a.N + E - 1) / E;      // pieces of a row
    const int full = a.N / (E * L) * L;   // pieces of whole piece columns
    uint32_t brow[L];  // byte offsets of the rows of B (a plan's B is below 4 GiB)
    int grow[L];
#pragma unroll
    for (int u = 0; u < L; u++) {
        brow[u] = static_cast<uint32_t>(__shfl(col, first + u)) * rowbytes;
        grow[u] = __shfl(row, first + u);
    }
    const bool one_row = __ballot(grow[0] != grow[L - 1]) == 0;  // a row's nonzeros are side by side
    double acc[L];
#pragma unroll
    for (int u = 0; u < L; u++) acc[u] = 0.;
    auto add = [&](int u, const Pack<float, E>& g, const Pack<T, E>& b, int skip) {
        float t[(E + 3) / 4];
#pragma unroll
        for (int e = 0; e < E; e++) {
            float s = e % 4 == 0 ? g.v[e] * to_f32(b.v[e]) : __builtin_fmaf(g.v[e], to_f32(b.v[e]), t[e / 4]);
            if (skip > e) s = 0.f;
            t[e / 4] = s;
        }
        acc[u] += static_cast<double>(E == 8 ? t[0] + t[E / 8] : t[0]);
    };
    auto load_b = [&](int u, int at) {
        return load_unaligned<T, E>(reinterpret_cast<const T*>(static_cast<const char*>(a.B) +
                                                           (brow[u] + static_cast<uint32_t>(at) * sizeof(T))));
    };
    auto load_g = [&](int u, int at) { return load_unaligned<float, E>(a.G + static_cast<size_t>(grow[u]) * N + at); };
    auto piece = [&](int at, int skip) {  // columns [at, at + E), the first `skip` of them not counted
        Pack<T, E> b[L];
        const Pack<float, E> g = load_g(0, at);
#pragma unroll
        for (int u = 0; u < L; u++) b[u] = load_b(u, at);
#pragma unroll
        for (int u = 0; u < L; u++) add(u, g, b[u], skip);
    };
    auto piece_rows = [&](int at, int skip) {  // the same, every nonzero with its own row of G
        constexpr int H = L > 4 ? 4 : L;       // nonzeros loaded at a time (registers)
#pragma unroll
        for (int h = 0; h < L; h += H) {
            Pack<T, E> b[H];
            Pack<float, E> g[H];
#pragma unroll
            for (int u = 0; u < H; u++) {
                g[u] = load_g(h + u, at);
                b[u] = load_b(h + u, at);
            }
#pragma unroll
            for (int u = 0; u < H; u++) add(h + u, g[u], b[u], skip);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    const int tail = full + l;  // the last piece of a row that is no whole number of them ends at the row's end
    const int at = min(tail * E, a.N - E);
    if (one_row) {
        constexpr int kAhead = E == 8 ? 1 : 2;
#pragma unroll kAhead
        for (int p = 0; p < full; p += L) piece((p + l) * E, 0);
        if (tail < V) piece(at, tail * E - at);
    } else {
#pragma unroll 1
        for (int p = 0; p < full; p += L) piece_rows((p + l) * E, 0);
        if (tail < V) piece_rows(at, tail * E - at);
    }
    float sum[L];
#pragma unroll
    for (int u = 0; u < L; u++) sum[u] = static_cast<float>(acc[u]);
    if constexpr (L == 8) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const float give = l & 4 ? sum[u] : sum[u + 4], keep = l & 4 ? sum[u + 4] : sum[u];
            sum[u] = keep + dpp_swap<0x141>(give);  // row_half_mirror
        }
    }
    if constexpr (L >= 4) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const float give = l & 2 ? sum[u] : sum[u + 2], keep = l & 2 ? sum[u + 2] : sum[u];
            sum[u] = keep + dpp_swap<0x4e>(give);  // quad_perm [2, 3, 0, 1]
        }
    }
    if constexpr (L >= 2) {
        const float give = l & 1 ? sum[0] : sum[1], keep = l & 1 ? sum[1] : sum[0];
        sum[0] = keep + dpp_swap<0xb1>(give);  // quad_perm [1, 0, 3, 2]
    }
    return sum[0];
}

template <typename T, int E, int L>
__global__ __launch_bounds__(64 * kSddmmWaves, 4) void sddmm_kernel(SddmmArgs a) {
    const int lane = threadIdx.x & 63;
    const uint32_t wave = blockIdx.x * kSddmmWaves + (threadIdx.x >> 6);
    const uint32_t span = 64 * a.batches;
    const uint32_t j0 = wave * span;
    if (j0 >= a.nnz) return;
    const uint32_t j1 = min(j0 + span, a.nnz);
    const int r0 = wave_row_of(a.rowptr, j0, a.M, lane);
    const int r1 = wave_row_of(a.rowptr, j1 - 1, a.M, lane);
    int lo = r0;
    for (uint32_t jb = j0; jb < j1; jb += 64) {
        const uint32_t j = min(jb + lane, j1 - 1);
        const int col = a.colidx[j];
        const int row = row_of(a.rowptr, j, lo, r1);
        lo = __builtin_amdgcn_readlane(row, 63);
        const float sum = sddmm_batch<T, E, L>(a, row, col, lane);
        if (jb + lane < j1) a.out[j] = sum;
    }
}

// The same for few nonzeros and wide rows, where batches of 64 leave the chip
// idle: a wavefront per nonzero, lane l on pieces l, l + 64, ... of its rows.
// A piece's products in fp32 (chains of four), everything else in fp64.  us at
// N columns, batches / a wavefront each (one wavefront per row, before both, in
// brackets), fp32: 1200 nonzeros in 300 rows, N = 64 4.4 / 3.8 (4.0), N = 256 8.6 /
// 3.9 (5.1), N = 1024 24.8 / 4.5 (11.5), N = 4096 151 / 4.6 (42); 8000 in 1000, N = 64
// 3.8 / 4.8 (6.1), N = 256 5.6 / 4.8 (8.1), N = 1024 17.0 / 6.3 (24); 40,000 in 4000, N
// = 256 14.3 / 14.6 (13.2), N = 512 26.4 / 18.9 (31), N = 1024 48 / 28 (60); 80,000 in
// 2000, N = 512 14.8 / 32; bf16: 40,000, N = 512 11.8 / 17.2 (27), N = 1024 20.1 / 22.8
// (60).  A batch takes about 0.085 us a piece of its rows and a wavefront per
// nonzero 0.2 us per 1000 of them.
inline bool sddmm_wide(uint32_t nnz, int pieces) {
    return pieces >= 16 && nnz <= 65536u && nnz <= 256u * static_cast<uint32_t>(pieces);
}

template <typename T, int E>
__global__ __launch_bounds__(64 * kSddmmWaves) void sddmm_wide_kernel(SddmmArgs a) {
    const int lane = threadIdx.x & 63;
    const uint32_t j = blockIdx.x * kSddmmWaves + (threadIdx.x >> 6);
    if (j >= a.nnz) return;
    const float* const g = a.G + static_cast<size_t>(wave_row_of(a.rowptr, j, a.M, lane)) * a.N;
    const T* const b = static_cast<const T*>(a.B) + static_cast<size_t>(a.colidx[j]) * a.N;
    const int V = (a.N + E - 1) / E;
    double acc = 0.;
#pragma unroll 4
    for (int p = lane; p < V; p += 64) {
        const int at = min(p * E, a.N - E), skip = p * E - at;  // the last piece ends at the row's end
        const Pack<float, E> x = load_unaligned<float, E>(g + at);
        const Pack<T, E> y = load_unaligned<T, E>(b + at);
        float t[(E + 3) / 4];
#pragma unroll
        for (int e = 0; e < E; e++) {
            float s = e % 4 == 0 ? x.v[e] * to_f32(y.v[e]) : __builtin_fmaf(x.v[e], to_f32(y.v[e]), t[e / 4]);
            if (skip > e) s = 0.f;
            t[e / 4] = s;
        }
        acc += static_cast<double>(E == 8 ? t[0] + t[E / 8] : t[0]);
    }
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d);
    if (lane == 0) a.out[j] = static_cast<float>(acc);
}

// The same for the rows of the row kernel's task list (those outside the row
// panels, whose nonzeros lie scattered through the CSR): a wavefront per task;
// a group of short rows is walked nonzero by nonzero, 64 at a time.
template <typename T, int E, int L>
__global__ __launch_bounds__(64 * kSddmmWaves, 4) void sddmm_tasks_kernel(SddmmArgs a) {
    const int lane = threadIdx.x & 63;
    const int tid = blockIdx.x * kSddmmWaves + (threadIdx.x >> 6);
    if (tid >= a.ntasks) return;
    const int4 t = a.tasks[tid];
    if ((t.w & 3) != kTaskMulti) {  // a row, a quarter or a segment of one
        const int row = (t.w & 3) == kTaskSeg ? a.longrows[t.x].x : t.x;
        for (int jb = t.y; jb < t.z; jb += 64) {
            const int j = min(jb + lane, t.z - 1);
            const float sum = sddmm_batch<T, E, L>(a, row, a.colidx[j], lane);
            if (jb + lane < t.z) a.out[j] = sum;
        }
        return;
    }
    if (t.z == 0) return;  // empty rows
    int row = 0, beg = 0, len = 0;
    if (lane < t.y) {
        row = a.perm[t.x + lane];
        beg = a.rowptr[row];
        len = a.rowptr[row + 1] - beg;
    }
    int end = len;  // of the row among the group's nonzeros
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const int x = __shfl_up(end, d);
        if (lane >= d) end += x;
    }
    const int total = __builtin_amdgcn_readlane(end, 63);
    for (int qb = 0; qb < total; qb += 64) {
        const int q = min(qb + lane, total - 1);
        int i = 0;  // the row of nonzero q: the first that ends after it
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1)
            if (__shfl(end, i + d - 1) <= q) i += d;
        const int j = __shfl(beg + len - end, i) + q;
        const float sum = sddmm_batch<T, E, L>(a, __shfl(row, i), a.colidx[j], lane);
        if (qb + lane < total) a.out[j] = sum;
    }
}

// out[i] = value perm[i] of `val`, widened to fp32 (A's values in the order
// of the transpose).
template <typename T>
__global__ __launch_bounds__(256) void gather_values_kernel(const int* __restrict__ perm, int n,
                                                            const T* __restrict__ val, float* __restrict__ out) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = to_f32(val[perm[i]]);
}

}  // namespace tca
