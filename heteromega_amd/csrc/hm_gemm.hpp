// Prefill GEMM: kernel arguments, tile shapes and launches shared by the planner (hm_gemm.hip) and the kernels
// (hm_gemm_kernel.hpp).
#pragma once

#include "hm_internal.hpp"

namespace hm {

struct GemmArgs {
    const uint4 *quant;
    const uint32_t *meta;
    const uint16_t *x;
    uint16_t *y;
    float *partial; // [splits][m][ncols] fp32 when the K range is split
    int64_t ldx, ldy;
    int kt_pitch;
    int kt_begin, kt_count, splits;
    int strip_begin;
    int m;
    int ncols; // 16 * strips of the call
    int tiles_m, tiles_n;
    int accumulate; // plain output: y = round(y + round(sum)) instead of y = round(sum)
    int group_m;    // tile order: bands of group_m row tiles, column-major inside a band (1: row-major)
    int xcds;       // XCDs of the device: the dispatcher places workgroup i on XCD i % xcds
};

// Tile shapes: 16 rbw rows x 32 wn columns, wk K groups of wn waves, depth LDS buffers, kpb K tiles per barrier (0: two
// barriers per K tile, the buffers hold half tiles). All but the last are eight waves, one workgroup per CU (LDS), and differ
// in how those waves are spread over columns and K.
struct GemmTile {
    int rbw, wn, wk, depth, kpb;
    constexpr int rows() const { return 16 * rbw; }
    constexpr int cols() const { return 32 * wn; }
};
constexpr GemmTile kGemmTiles[] = {
    // 64 columns, four K groups
    {2, 2, 4, 3, 1}, {3, 2, 4, 3, 1}, {4, 2, 4, 4, 0},
    // 128 columns, two K groups. From 112 rows LDS holds two whole tiles per group only, and requested one tile ahead the
    // activations came late (without them a timing copy ran 20-25% faster); as four half tiles they are requested 1.25 tiles
    // ahead: gate_ups of 128 rows 5-6% faster, of 100 rows 3%, downs of 200 rows 3%, runs of 5 K tiles 4% slower.
    {2, 4, 2, 4, 1}, {3, 4, 2, 4, 1}, {4, 4, 2, 4, 1}, {5, 4, 2, 3, 1}, {6, 4, 2, 3, 1}, {7, 4, 2, 4, 0}, {8, 4, 2, 4, 0},
    // 256 columns, 2 K tiles ahead in 4 buffers, one barrier per 2 K tiles (against one per K tile, the same bits:
    // Llama-3-8B M = 2048 gate_up 398.0 -> 392.9 us, down 193.9 -> 192.1)
    {5, 8, 1, 4, 2}, {6, 8, 1, 4, 2}, {7, 8, 1, 4, 2}, {8, 8, 1, 4, 2},
    // 128 x 128, four waves: two workgroups per CU (half tiles for the same reason: 2-7% faster at 640 rows)
    {8, 4, 1, 4, 0}};
constexpr int kGemmTileCount = sizeof(kGemmTiles) / sizeof(kGemmTiles[0]);
// The tile of bf16 matrices with scales from 2^117 on (Planes::large_scales): the only one that their dequantization is built for.
constexpr int kLargeScaleTile = kGemmTileCount - 1;
static_assert(kGemmTiles[kLargeScaleTile].cols() == 128 && kGemmTiles[kLargeScaleTile].wk == 1, "fits every call");

// The launches of one activation type (hm_gemm_f16.hip, hm_gemm_bf16.hip).
hipError_t launch_gemm_f16(const GemmArgs &a, int group, bool fused, int cfg, dim3 grid, hipStream_t s);
hipError_t launch_gemm_bf16(const GemmArgs &a, int group, bool fused, int cfg, dim3 grid, hipStream_t s);
hipError_t launch_gemm_bf16_large_scales(const GemmArgs &a, int group, bool fused, dim3 grid, hipStream_t s); // in kLargeScaleTile

} // namespace hm
