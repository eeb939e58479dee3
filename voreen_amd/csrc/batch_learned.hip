// batch_learned.hip -- the learned jobs of a batched launch
// (hipdvr_batch_launch_learned), in one of two forms (batch.hip,
// learned_batch_lanes, chooses by the launch's size).
//
// Large launches have rays enough to fill the chip and are bound by the
// instructions they issue.  A persistent launch marches every learned view's
// tiles with one lane per ray and two (Phong) or four samples in flight, which
// computes a pass's chain of positions once (learned_ray.h; 7.4 G vector
// instructions for 36 views, 9.7 G with two lanes); its grid stays resident and
// takes tiles from counters, so that a workgroup loads a job's tables once and
// starts no new wavefronts.  36 views of 512^3 at 1024^2 with Phong and a trained
// network, with the judges: 13.6 ms; as workgroups of their own with one lane
// 14.9 ms, with two 16.3, with four 22.5.
//
// The others are bound by the chain of a ray's samples, or by loads of records
// past 4 GiB: a plain grid marches the judges' rays, the plain jobs and the
// learned ones side by side with two or four lanes per ray.  One view of 512^3 at
// 1024^2 0.76 ms (in the persistent launch 0.90), 36 of 512^2 5.90 (7.44), 8 of
// 2048 x 2048 x 1024 at 3840 x 2160 66.9 (105).
#include <hip/hip_runtime.h>

#include "batch_tiles.h"
#include "errors.h"
#include "learned.h"
#include "learned_ray.h"
#include "march_cell.h"
#include "residency.h"

namespace hipdvr {

namespace {

// Tile queues.  The hardware hands the grid's workgroups to the 8 XCDs in turn
// (workgroup b to XCD b % 8), and each XCD has its own L2.  The tiles come in
// blocks of kBlockW x kBlockH tiles of one job; consecutive runs of kChunk
// tiles are dealt to the XCDs in turn, and each XCD takes its runs from a
// counter of its own, so the tiles an XCD marches at a time form a compact
// column of blocks whose rays share that XCD's L2.  An XCD whose runs are
// taken takes from the others' counters.  Blocks of 8x4 tiles 14.0 ms, 8x8
// 14.0, 4x4 14.5, 2x2 14.5.
constexpr int kBlockW = 8, kBlockH = 4;
constexpr uint32_t kChunk = kBlockW * kBlockH;
constexpr uint32_t kCounterStride = 32;   // counters 128 bytes apart
static_assert(kLearnedQueueBytes == kXcds * kCounterStride * 4, "a counter per XCD");

__global__ void reset_queue_kernel(uint32_t* counter) {
    if (threadIdx.x < kXcds) counter[threadIdx.x * kCounterStride] = 0;
}

// Tiles dealt to XCD x out of total.
__device__ __forceinline__ uint32_t xcd_tiles(uint32_t x, uint32_t total) {
    const uint32_t chunks = (total + kChunk - 1) / kChunk;
    if (x >= chunks) return 0;
    uint32_t n = ((chunks - 1 - x) / kXcds + 1) * kChunk;
    if ((chunks - 1) % kXcds == x) n -= chunks * kChunk - total;   // its last run is the short one
    return n;
}

// The next tile for a workgroup of XCD x (total: none is left, whatever the
// counters hold); drained: queues that this workgroup has seen empty.  (Taking
// it ahead, while the present tile is marched, gains nothing: 13.9 ms against
// 13.6.)
__device__ __forceinline__ uint32_t take_tile(uint32_t* counter, uint32_t x, uint32_t total, uint32_t& drained) {
    for (uint32_t k = 0; k < kXcds; ++k) {
        const uint32_t q = (x + k) % kXcds;
        if (drained & (1u << q)) continue;
        const uint32_t i = atomicAdd(counter + q * kCounterStride, 1u);
        if (i < xcd_tiles(q, total)) return (q + kXcds * (i / kChunk)) * kChunk + i % kChunk;
        drained |= 1u << q;
    }
    return total;
}

// A workgroup is a tile's 2x2 regions of 64 pixels, one per wavefront.
template <bool PHONG, bool COUNT>
__global__ __launch_bounds__(256) void learned_batch_kernel(const LearnedArgs* __restrict__ jobs,
                                                            const uint32_t* __restrict__ tile_start, uint32_t njobs,
                                                            uint32_t total_tiles, uint32_t tile_shape,
                                                            uint32_t* __restrict__ counter,
                                                            unsigned long long* __restrict__ counters) {
    __shared__ uint32_t s_tf[kMaxTfWidth];
    __shared__ float s_alpha[256];
    __shared__ uint32_t s_tile;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int WW = 8 << tile_shape, WH = 8 >> tile_shape;
    unsigned long long n_rays = 0, n_samples = 0, n_shaded = 0;
    uint32_t cur = 0xffffffffu, drained = 0;
    while (true) {
        if (tid == 0) s_tile = take_tile(counter, blockIdx.x % kXcds, total_tiles, drained);
        __syncthreads();   // also: every wave has finished the previous tile
        const uint32_t tile = __builtin_amdgcn_readfirstlane(s_tile);
        __syncthreads();   // s_tile is read before the next iteration writes it
        if (tile >= total_tiles) break;
        const uint32_t job = job_of_tile(tile_start, njobs, tile);
        const LearnedArgs& la = jobs[job];
        const MarchArgs& a = la.m;
        if (job != cur) {
            for (int i = tid; i < a.tf_width; i += 256) s_tf[i] = a.tf[i];
            s_alpha[tid] = la.alpha_m[tid];
            __syncthreads();
            cur = job;
        }
        uint32_t tx, ty;
        block_tile<kBlockW, kBlockH>(tile - tile_start[job], (uint32_t)(a.w + 2 * WW - 1) / (2 * WW),
                                     (uint32_t)(a.h + 2 * WH - 1) / (2 * WH), tx, ty);
        const int px = ((int)tx * 2 + (wave & 1)) * WW + lane % WW;
        const int py = ((int)ty * 2 + (wave >> 1)) * WH + lane / WW;
        if (px < a.w && py < a.h) {
            const size_t pix = (size_t)py * a.w + px;
            const float4 e = a.entry[pix], l = a.exit[pix];
            float4 res = make_float4(0.f, 0.f, 0.f, 0.f);
            if (!is_background(e, l)) {
                if (a.dtype == 0) {
                    const CellFetch<uint8_t, false> f = cell_fetch_of<uint8_t, false>(a);
                    res = learned_ray_single<uint8_t, false, PHONG>(la, f, s_tf, s_alpha, px, py, e, l, n_samples,
                                                                    n_shaded);
                } else {
                    const CellFetch<uint16_t, false> f = cell_fetch_of<uint16_t, false>(a);
                    res = learned_ray_single<uint16_t, false, PHONG>(la, f, s_tf, s_alpha, px, py, e, l, n_samples,
                                                                     n_shaded);
                }
                ++n_rays;
            }
            a.out[pix] = res;
        }
    }
    if (COUNT) {
        wave_add(counters + 0, n_rays);
        wave_add(counters + 1, n_samples);
        wave_add(counters + 2, n_samples);
        wave_add(counters + 3, n_shaded);
    }
}

// The plain jobs and the learned ones in one launch, the plain first (the judges'
// re-marches start while the chip fills), by workgroups of their own: one per
// P-th of a tile, P lanes per ray, as batch_kernel.
template <bool WIDE, bool PHONG, bool COUNT, int P>
__global__ __launch_bounds__(256, PHONG ? 5 : (COUNT ? 6 : 7)) void mixed_kernel(
    const MarchArgs* __restrict__ plain, const uint32_t* __restrict__ plain_start, uint32_t nplain, uint32_t plain_tiles,
    const LearnedArgs* __restrict__ jobs, const uint32_t* __restrict__ tile_start, uint32_t njobs, uint32_t total_tiles,
    uint32_t tile_shape, unsigned long long* __restrict__ counters) {
    const uint32_t block = linear_block(), slot = block / kXcds, part = slot % P, i = slot / P;
    uint32_t tile = xcd_run(block % kXcds, i / kTileRun) * kTileRun + i % kTileRun;
    if (tile >= plain_tiles + total_tiles) return;
    __shared__ uint32_t s_tf[kMaxTfWidth];
    __shared__ float s_alpha[256];
    const bool learned = tile >= plain_tiles;
    if (learned) tile -= plain_tiles;
    const uint32_t* start = learned ? tile_start : plain_start;
    const uint32_t job = job_of_tile(start, learned ? njobs : nplain, tile);
    const LearnedArgs& la = jobs[learned ? job : 0];
    const MarchArgs& a = learned ? la.m : plain[job];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ray = lane / P, sub = lane % P;
    const int WW = 8 << tile_shape, WH = 8 >> tile_shape;
    const int RH = ray_h<P>() < WH ? ray_h<P>() : WH, RW = 64 / P / RH, cols = WW / RW;
    uint32_t tx, ty;
    block_tile<kTileBlockW, kTileBlockH>(tile - start[job], (uint32_t)(a.grid_w + 2 * WW - 1) / (2 * WW),
                                         (uint32_t)(a.grid_h + 2 * WH - 1) / (2 * WH), tx, ty);
    const bool sparse = a.pix_block > 1;   // a judge's re-march (batch_kernel)
    const int q = (int)part * 4 + wave, region = q / P, rp = q % P;
    const int gx = ((int)tx * 2 + (region & 1)) * WW + (rp % cols) * RW + ray % RW;
    const int gy = ((int)ty * 2 + (region >> 1)) * WH + (rp / cols) * RH + ray / RW;
    const bool inside = gx < a.grid_w && gy < a.grid_h;
    const int px = sparse ? judge_pixel(gx, a.stride, a.pix_block, a.pix_offset) : gx;
    const int py = sparse ? judge_pixel(gy, a.stride, a.pix_block, a.pix_offset) : gy;
    float4 e = make_float4(0.f, 0.f, 0.f, 0.f), l = e, res = e;
    if (inside) {
        const size_t pix = (size_t)py * a.w + px;
        e = a.entry[pix];
        l = a.exit[pix];
    }
    const bool hit = !is_background(e, l);
    RayCounters n;
    if (__syncthreads_or(hit)) {
        for (int k = tid; k < a.tf_width; k += 256) s_tf[k] = a.tf[k];
        s_alpha[tid] = learned ? la.alpha_m[tid] : a.alpha_corr[tid];
        __syncthreads();
        if (hit) {
            if (learned) {
                unsigned long long ns = 0, nsh = 0;
                if (a.dtype == 0) {
                    const CellFetch<uint8_t, WIDE> f = cell_fetch_of<uint8_t, WIDE>(a);
                    res = learned_ray<uint8_t, WIDE, PHONG, P>(la, f, s_tf, s_alpha, px, py, sub, e, l, ns, nsh);
                } else {
                    const CellFetch<uint16_t, WIDE> f = cell_fetch_of<uint16_t, WIDE>(a);
                    res = learned_ray<uint16_t, WIDE, PHONG, P>(la, f, s_tf, s_alpha, px, py, sub, e, l, ns, nsh);
                }
                ++n.rays;
                n.fetched += sub == 0 ? (uint32_t)ns : 0;   // the ray's, counted by one lane
                n.shaded += sub == 0 ? (uint32_t)nsh : 0;
            } else if (a.dtype == 0) {
                const CellFetch<uint8_t, WIDE> f = cell_fetch_of<uint8_t, WIDE>(a);
                res = cell_ray<uint8_t, WIDE, PHONG ? 1 : 0, COUNT, P>(a, f, s_tf, s_alpha, px, py, sub, e, l, n);
            } else {
                const CellFetch<uint16_t, WIDE> f = cell_fetch_of<uint16_t, WIDE>(a);
                res = cell_ray<uint16_t, WIDE, PHONG ? 1 : 0, COUNT, P>(a, f, s_tf, s_alpha, px, py, sub, e, l, n);
            }
        }
    }
    if (inside && sub == 0) a.out[(size_t)gy * a.grid_w + gx] = res;
    if (sparse) n = RayCounters();
    if (COUNT) add_counters<P>(counters, n, sub == 0);
}

typedef void (*ResidentKernel)(const LearnedArgs*, const uint32_t*, uint32_t, uint32_t, uint32_t, uint32_t*,
                               unsigned long long*);
typedef void (*MixedKernel)(const MarchArgs*, const uint32_t*, uint32_t, uint32_t, const LearnedArgs*, const uint32_t*,
                            uint32_t, uint32_t, uint32_t, unsigned long long*);

ResidentKernel resident_kernel(bool phong, bool count) {
    if (phong) return count ? learned_batch_kernel<true, true> : learned_batch_kernel<true, false>;
    return count ? learned_batch_kernel<false, true> : learned_batch_kernel<false, false>;
}
template <bool WIDE, int P>
MixedKernel mixed_of(bool phong, bool count) {
    if (phong) return count ? mixed_kernel<WIDE, true, true, P> : mixed_kernel<WIDE, true, false, P>;
    return count ? mixed_kernel<WIDE, false, true, P> : mixed_kernel<WIDE, false, false, P>;
}
template <int P>
MixedKernel mixed_of(bool wide, bool phong, bool count) {
    return wide ? mixed_of<true, P>(phong, count) : mixed_of<false, P>(phong, count);
}

}  // namespace

void launch_learned_mixed(const MarchArgs* plain, const uint32_t* plain_start, uint32_t nplain, uint32_t plain_tiles,
                          const LearnedArgs* jobs, const uint32_t* tile_start, uint32_t njobs, uint32_t total_tiles,
                          int tile_shape, int lanes, bool phong, bool wide, int resident, unsigned long long* counters,
                          hipStream_t st) {
    const bool count = counters != nullptr;
    const MixedKernel k = lanes == 2 ? mixed_of<2>(wide, phong, count) : mixed_of<4>(wide, phong, count);
    size_t pad = 0;
    if (resident > 0) {
        hipFuncAttributes fa;
        hip_check(hipFuncGetAttributes(&fa, (const void*)k), "hipFuncGetAttributes");
        pad = residency_pad(fa.sharedSizeBytes, resident);
    }
    hipLaunchKernelGGL(k, linear_grid(batch_grid(plain_tiles + total_tiles, lanes)), dim3(256), pad, st, plain,
                       plain_start, nplain, plain_tiles, jobs, tile_start, njobs, total_tiles, (uint32_t)tile_shape,
                       counters);
    hip_check(hipGetLastError(), "learned batch launch");
}

void launch_learned_batch(const LearnedArgs* jobs, const uint32_t* tile_start, uint32_t njobs, uint32_t total_tiles,
                          int tile_shape, bool phong, int resident, uint32_t* queue, unsigned long long* counters,
                          hipStream_t st) {
    const bool count = counters != nullptr;
    const ResidentKernel k = resident_kernel(phong, count);
    int per_cu = 0, device = 0, cus = 0;
    hip_check(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k, 256, 0), "occupancy query");
    hip_check(hipGetDevice(&device), "hipGetDevice");
    hip_check(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device), "hipDeviceGetAttribute");
    if (per_cu < 1) per_cu = 1;
    if (resident > 0 && per_cu > resident) per_cu = resident;
    uint32_t grid = (uint32_t)(cus * per_cu);
    if (grid > total_tiles) grid = total_tiles ? total_tiles : 1;
    hipLaunchKernelGGL(reset_queue_kernel, dim3(1), dim3(64), 0, st, queue);
    hipLaunchKernelGGL(k, dim3(grid), dim3(256), 0, st, jobs, tile_start, njobs, total_tiles, (uint32_t)tile_shape,
                       queue, counters);
    hip_check(hipGetLastError(), "learned batch launch");
}

}  // namespace hipdvr
