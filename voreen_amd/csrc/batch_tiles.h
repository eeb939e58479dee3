// batch_tiles.h -- the image tiles of batched launches (batch.hip,
// batch_learned.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace hipdvr {

// Tile shapes: regions of 64 pixels, 8x8, 16x4 or 32x2; a tile is 2x2 regions.
__host__ __device__ constexpr int wave_w(int tile) { return 8 << tile; }
__host__ __device__ constexpr int wave_h(int tile) { return 8 >> tile; }

// Job of a tile: the last j with tile_start[j] <= tile.
__device__ __forceinline__ uint32_t job_of_tile(const uint32_t* tile_start, uint32_t njobs, uint32_t tile) {
    uint32_t lo = 0, hi = njobs;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (tile_start[mid] <= tile) lo = mid;
        else hi = mid;
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// Tile (tx, ty) at position lt of a job of tiles_x x tiles_y tiles: blocks of
// BW x BH tiles row by row, tiles row by row inside a block, edge blocks
// smaller (a bijection of [0, tiles_x * tiles_y)).
template <int BW, int BH>
__device__ __forceinline__ void block_tile(uint32_t lt, uint32_t tiles_x, uint32_t tiles_y, uint32_t& tx,
                                           uint32_t& ty) {
    const uint32_t nby = (tiles_y + BH - 1) / BH, nbx = (tiles_x + BW - 1) / BW;
    uint32_t by = lt / (BH * tiles_x);
    if (by > nby - 1) by = nby - 1;
    const uint32_t r = lt - by * BH * tiles_x;
    const uint32_t bh = min((uint32_t)BH, tiles_y - by * BH);
    uint32_t bx = r / (BW * bh);
    if (bx > nbx - 1) bx = nbx - 1;
    const uint32_t r2 = r - bx * BW * bh;
    const uint32_t bw = min((uint32_t)BW, tiles_x - bx * BW);
    ty = by * BH + r2 / bw;
    tx = bx * BW + r2 % bw;
}

}  // namespace hipdvr
