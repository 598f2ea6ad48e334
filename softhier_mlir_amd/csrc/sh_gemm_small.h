// Launch interface of the small-problem and any-alignment GEMM kernels (sh_gemm_small.hip). Not part of the C ABI.
#pragma once
#include "sh_gemm_dev.h"

// SMALL_RANGES_*: a tile's K ranges (a.kps k each, at most kSmallMaxRanges, kSmallMaxRanges64 for the 64-row tile) run in
// one workgroup, one wavefront each.
// SMALL_64x64 / SMALL_128x64: operands of any alignment, unsplit. SMALL_DMA*: the 64 x 64 direct-to-LDS tile (k_gemm5) with
// one or two K ranges (launched by sh_gemm.hip itself).
enum SmallTile { SMALL_RANGES_32 = 0, SMALL_RANGES_64 = 1, SMALL_64x64 = 2, SMALL_128x64 = 3, SMALL_ANY_TILES = 4,
                 SMALL_DMA = 4, SMALL_DMA2 = 5, SMALL_TILES = 6 };
constexpr uint32_t kSmallMaxRanges = 8, kSmallMaxRanges64 = 4;
struct SmallDims { uint32_t bm, bn; };
constexpr SmallDims kSmallDims[SMALL_TILES] = {{32, 32}, {64, 32}, {64, 64}, {128, 64}, {64, 64}, {64, 64}};

// Enqueue variant `v` (below SMALL_ANY_TILES) for a (tiles_m, tiles_n and kps set; `ranges` K ranges, 1 for the unsplit
// tiles). any: the ANY_ALIGN build (operands not 16-byte aligned, or K % 64 != 0). The caller checks the launch.
void sh_gemm_small_enqueue(const GemmArgs &a, SmallTile v, bool wt, bool any, uint32_t ranges, hipStream_t st);
