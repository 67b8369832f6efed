// The matrix prefill's GEMM, C = X W^T on the matrix cores, with tiles loaded straight into LDS and
// an epilogue that does what follows the product.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

#include "device_common.hpp"

namespace tiles {

// What a block does with its tile of FP32 sums.
enum class GemmOut {
    kRows,      // c[m][n] = bf16(sum)
    kResidual,  // c[m][n] = bf16(bf16(sum) + residual[m][n])
    kSilu,      // w holds gate rows, w2 up rows: c[m][n] = bf16(bf16(silu(bf16(gate))) * bf16(up))
    kPartial,   // partial[split][m][n] = the sum over the split's part of K, for the next kernel to add
};

struct GemmArgs {
    const uint16_t* x;         // [m][k]
    const uint16_t* w;         // [n][k]
    const uint16_t* w2;        // kSilu: [n][k]
    const uint16_t* residual;  // kResidual: row stride ldc
    uint16_t* c;               // row stride ldc
    float* partial;            // kPartial: [splits][m][n]
    int m, n, k, ldc, splits;
    int m_tiles, n_tiles;
};

// m tiles a column walk covers before it goes to the next column: the blocks an XCD runs at a time
// (32 CUs) then read about 8 tiles of X rows and 4 of W rows between them.
constexpr int kGemmBand = 8;

// 16 bytes a lane from global memory straight into LDS, lane l's at lds + 16 l (lds wave-uniform).
__device__ inline void load_to_lds(const void* src, uint16_t* lds)
{
    __builtin_amdgcn_global_load_lds((const TILES_GLOBAL void*)(src), (__attribute__((address_space(3))) void*)(lds), 16, 0, 0);
}

// The row of W (or w2) whose values a tile keeps at its staged row `at`, from the tile's first column
// n0; past the last row, the last one (its sums are not stored).  The order makes a lane's sums 8
// adjacent columns, one 16-byte store, and four lanes' stores 64 adjacent bytes: lane group q holds
// rows 4 q .. 4 q + 3 of each 16-row MFMA tile, which in tiles 2 h and 2 h + 1 are columns
// 32 h + 8 q .. + 7.  kSilu: tiles 4 h .. 4 h + 3 are gate, up, gate, up rows of the same 32 columns.
// (Rows in plain order gave each lane 8-byte stores 32 bytes apart.)
template <GemmOut OUT>
__device__ inline int gemm_weight_row(const GemmArgs& g, int n0, int at)
{
    const int tile = at >> 4, r = at & 15, inner = 8 * (r >> 2) + (r & 3);
    const int n = OUT == GemmOut::kSilu ? n0 / 2 + 32 * (tile >> 2) + inner + 4 * ((tile >> 1) & 1)
                                        : n0 + 32 * (tile >> 1) + inner + 4 * (tile & 1);
    return min(n, g.n - 1);
}

__device__ inline uint32_t pair_bf16(float lo, float hi)
{
    return __builtin_bit_cast(uint32_t, bf16x2{static_cast<__bf16>(lo), static_cast<__bf16>(hi)});
}
__device__ inline u32x4 pack_bf16(const float (&v)[8])
{
    return u32x4{pair_bf16(v[0], v[1]), pair_bf16(v[2], v[3]), pair_bf16(v[4], v[5]), pair_bf16(v[6], v[7])};
}

// A wave's sums, tiles [WN / 16][WM / 16] from row m0 and (staged) column n0, to memory.
template <int WM, int WN, GemmOut OUT>
__device__ inline void gemm_store(const GemmArgs& g, int m0, int n0, int split, const f32x4 (&acc)[WN / 16][WM / 16])
{
    using Bf = Num<true>;
    constexpr int kTiles = OUT == GemmOut::kSilu ? 4 : 2;  // MFMA tiles of 8 adjacent columns
    static_assert(WN / 16 % kTiles == 0, "whole groups of columns");
    const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int j = 0; j < WM / 16; ++j) {
        const int m = m0 + j * 16 + r;
        if (m >= g.m)
            continue;
#pragma unroll
        for (int i = 0; i < WN / 16; i += kTiles) {
            const int n = (OUT == GemmOut::kSilu ? n0 / 2 + 8 * i : n0 + 16 * i) + 8 * q;
            if (n >= g.n)
                continue;
            if constexpr (OUT == GemmOut::kPartial) {
                f32x4* to = reinterpret_cast<f32x4*>(g.partial + (static_cast<size_t>(split) * g.m + m) * g.n + n);
                to[0] = acc[i][j];
                to[1] = acc[i + 1][j];
            } else {
                const size_t at = static_cast<size_t>(m) * g.ldc + n;
                u32x4 residual = {0u, 0u, 0u, 0u};
                if constexpr (OUT == GemmOut::kResidual)
                    residual = *reinterpret_cast<const u32x4*>(g.residual + at);
                float v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    if constexpr (OUT == GemmOut::kSilu) {
                        const float gate = Bf::round(acc[i + 2 * (e / 4)][j][e % 4]), up = Bf::round(acc[i + 2 * (e / 4) + 1][j][e % 4]);
                        v[e] = Bf::round(gate / (1.0f + expf(-gate))) * up;
                    } else if constexpr (OUT == GemmOut::kResidual) {
                        v[e] = Bf::round(acc[i + e / 4][j][e % 4]) + Bf::elem(residual, e);
                    } else {
                        v[e] = acc[i + e / 4][j][e % 4];
                    }
                }
                *reinterpret_cast<u32x4*>(g.c + at) = pack_bf16(v);
            }
        }
    }
}

// A tile of BM rows of X by BN rows of W (kSilu: BN / 2 of each matrix) per block, WM x WN of it per
// wave, K in steps of KS through STAGES LDS buffers.  Each load brings 16 bytes a lane from memory to
// LDS without passing registers, STAGES - 1 steps ahead of the products, so a step has one barrier
// and no LDS writes of its own.  The load fixes where in LDS each lane's bytes land, so the 16-byte
// chunks of a row are exchanged at the source: chunk c of staged row r lies at c ^ r mod 8 (KS 64), so
// that the 16 rows of an operand read fall on distinct banks (no bank conflicts counted).
// Rows past m and n are clamped on load and not stored.  k % KS == 0, n % 8 == 0, ldc % 8 == 0 and
// 16-byte aligned pointers (MatrixPrefill::supports
// holds widths to multiples of 16, so every row starts aligned).
template <int BM, int BN, int WM, int WN, int KS, int STAGES, GemmOut OUT>
__global__ void __launch_bounds__((BM / WM) * (BN / WN) * 64) gemm_tiles(GemmArgs g)
{
    constexpr int kWaves = (BM / WM) * (BN / WN);
    constexpr int kChunks = KS / 8;             // 16-byte chunks of a staged row
    constexpr int kRowsPerLoad = 64 / kChunks;  // rows one load of a wave covers
    constexpr int kLoads = (BM + BN) / kRowsPerLoad / kWaves;
    constexpr int kStage = (BM + BN) * KS;      // elements
    static_assert(KS == 32 || KS == 64, "swizzle of a row's chunks");
    static_assert((BM + BN) % (kRowsPerLoad * kWaves) == 0 && STAGES >= 2, "whole loads per wave");
    __shared__ __attribute__((aligned(16))) uint16_t lds[STAGES * kStage];
    auto swizzle = [](int row) { return kChunks == 8 ? row & 7 : (row >> 1) & 3; };
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int wm = (wave % (BM / WM)) * WM, wn = (wave / (BM / WM)) * WN;

    // Consecutive blocks go to the eight XCDs in turn; each XCD takes a contiguous range of tiles, so
    // that the rows its blocks share are read into its L2 once.
    const int per = gridDim.x / 8, rest = gridDim.x % 8, xcd = blockIdx.x % 8;
    const int id = xcd * per + min(xcd, rest) + blockIdx.x / 8;
    const int plane = g.m_tiles * g.n_tiles, split = id / plane, tile = id - split * plane;
    const int band = tile / (kGemmBand * g.n_tiles), in_band = tile - band * kGemmBand * g.n_tiles;
    const int band_rows = min(kGemmBand, g.m_tiles - band * kGemmBand);
    const int m0 = (band * kGemmBand + in_band % band_rows) * BM, n0 = in_band / band_rows * BN;
    const int all_steps = g.k / KS;
    const int first = OUT == GemmOut::kPartial ? split * all_steps / g.splits : 0;
    const int steps = (OUT == GemmOut::kPartial ? (split + 1) * all_steps / g.splits : all_steps) - first;

    const uint16_t* src[kLoads];  // of this lane's bytes of each of its wave's loads, at the first step
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int row = (wave * kLoads + i) * kRowsPerLoad + lane / kChunks;
        const uint16_t* line;
        if (row < BM)
            line = g.x + static_cast<size_t>(min(m0 + row, g.m - 1)) * g.k;
        else
            line = (OUT == GemmOut::kSilu && ((row - BM) / 16) % 2 ? g.w2 : g.w) +
                   static_cast<size_t>(gemm_weight_row<OUT>(g, n0, row - BM)) * g.k;
        src[i] = line + static_cast<size_t>(first) * KS + ((lane % kChunks) ^ swizzle(row)) * 8;
    }
    auto issue = [&](int step, int stage) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i)
            load_to_lds(src[i] + static_cast<size_t>(step) * KS, lds + stage * kStage + (wave * kLoads + i) * kRowsPerLoad * KS);
    };

    f32x4 acc[WN / 16][WM / 16];
#pragma unroll
    for (int i = 0; i < WN / 16; ++i)
#pragma unroll
        for (int j = 0; j < WM / 16; ++j)
            acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int s = 0; s < STAGES - 1; ++s)
        if (s < steps)
            issue(s, s);
    int stage = 0;
    for (int s = 0; s < steps; ++s) {
        // This step's tile is in LDS (loads arrive in order; those of later steps may be on their
        // way) for every wave, and every wave has read the tile whose buffer the next load takes.
        if (s + STAGES - 2 < steps)
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((STAGES - 2) * kLoads) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (s + STAGES - 1 < steps)
            issue(s + STAGES - 1, stage == 0 ? STAGES - 1 : stage - 1);
        const uint16_t* xs = lds + stage * kStage;
        const uint16_t* ws = xs + BM * KS;
#pragma unroll
        for (int kk = 0; kk < KS / 32; ++kk) {
            const int at = ((kk * 4 + q) ^ swizzle(r)) * 8;
            u32x4 fx[WM / 16], fw[WN / 16];
#pragma unroll
            for (int j = 0; j < WM / 16; ++j)
                fx[j] = *reinterpret_cast<const u32x4*>(xs + (wm + j * 16 + r) * KS + at);
#pragma unroll
            for (int i = 0; i < WN / 16; ++i)
                fw[i] = *reinterpret_cast<const u32x4*>(ws + (wn + i * 16 + r) * KS + at);
#pragma unroll
            for (int i = 0; i < WN / 16; ++i)
#pragma unroll
                for (int j = 0; j < WM / 16; ++j)
                    acc[i][j] = mfma_16x16x32_bf16(fw[i], fx[j], acc[i][j]);
        }
        stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
    gemm_store<WM, WN, OUT>(g, m0 + wm, n0 + wn, split, acc);
}

} // namespace tiles
