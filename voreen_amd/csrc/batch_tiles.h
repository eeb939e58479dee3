// batch_tiles.h -- the image tiles of batched launches (batch.hip,
// batch_learned.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "march_common.h"

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

// The order of the tiles of a plain grid, whose workgroups each take a part of
// one.  The hardware hands consecutive workgroups to the 8 XCDs in turn (workgroup
// b to XCD b % 8), and each XCD has its own L2.  Tiles come in blocks of
// kTileBlockW x kTileBlockH tiles of one job (blocks row by row, tiles row by row
// inside a block; edge blocks smaller); consecutive runs of kTileRun tiles of the
// launch's tile range are dealt to the XCDs in turn, so the tiles an XCD marches
// at a time are a few compact blocks whose rays share that XCD's L2, and the eight
// march neighbouring ones.  Blocks of 2x2 tiles: 64 uneven volumes 709 us, 12
// views of 512^3 6.43 ms; 4x4 695 us, 6.51 ms; 8x4 824 us, 6.56 ms.
constexpr int kTileBlockW = 2, kTileBlockH = 2;
constexpr uint32_t kTileRun = kTileBlockW * kTileBlockH;

// The run that XCD x takes in round m: the round's eight runs in an order that
// changes from round to round without a pattern, so that no XCD meets the same
// column of an image whatever its width (dealt in a fixed order, 12 views of
// 1024^2 took 13.1 ms, the XCDs of the middle columns marching alone for half
// of it).
__host__ __device__ inline uint32_t xcd_run(uint32_t x, uint32_t m) {
    return kXcds * m + (x ^ ((m * 0x9E3779B1u) >> 29));
}

// Workgroups for `total` tiles in P parts each: whole rounds of runs (those
// past the last tile leave at once).
inline uint64_t batch_grid(uint32_t total, int parts) {
    const uint64_t chunks = ((uint64_t)total + kTileRun - 1) / kTileRun;
    return (chunks + kXcds - 1) / kXcds * kXcds * kTileRun * (uint64_t)parts;
}

}  // namespace hipdvr
