// batch.hip -- many volumes in one launch (include/hipdvr_batch.h).
//
// Every job is the cell-record march of hipdvr_render_device (march_cell.h),
// so each job's image is bit-identical to its single-frame render.  The image
// tiles of all jobs form one list, jobs in decreasing order of estimated cost
// (pixels x longest volume axis: largest first), one workgroup per part of a
// tile, which finds its job in the list's prefix sums and loads that job's TF
// into LDS.  The hardware's dispatcher is the work queue: workgroups start in
// list order as others end.  (A persistent grid that took tiles from counters
// kept every job's arguments live across its loop, at two to four times the
// scalar registers that these kernels spill, and was slower: 12 views of 512^3
// with two lanes per ray 7.1 ms against 6.0.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <numeric>
#include <vector>

#include "../../include/hipdvr_batch.h"
#include "../../include/hipdvr_learned.h"
#include "batch_tiles.h"
#include "ctx.h"
#include "errors.h"
#include "kernels.h"
#include "learned.h"
#include "march_cell.h"
#include "objects.h"
#include "residency.h"
#include "volume.h"

namespace hipdvr {

namespace {

constexpr int kTileShapes = 3;
constexpr int kBrickSizes = 3;   // brick_log2 3, 4, 5

constexpr uint64_t kMaxTiles = 0x3fffff00;   // of a launch: four parts each below 2^32

// One workgroup per P-th of a tile, P lanes per ray (march_cell.h).  The
// tile's 2x2 regions of 64 pixels fall into parts of 64 / P rays; wavefront w
// marches part `part` of region w, or, where the parts of a region are
// narrower than it, its neighbours in the same part of the tile.  Wavefronts
// per SIMD, unshaded, 64 uneven volumes with two lanes, 6 / 7 / 8: 672 / 616 /
// 608 us.
template <bool WIDE, int SHADE, bool COUNT, int P>
__global__ __launch_bounds__(256, SHADE == 2 ? 4 : (SHADE == 1 ? (COUNT ? 5 : 6) : (COUNT ? 6 : 7))) void batch_kernel(
    const MarchArgs* __restrict__ jobs, const uint32_t* __restrict__ tile_start, uint32_t njobs,
    uint32_t total_tiles, unsigned long long* __restrict__ counters, uint32_t tile_shape) {
    const uint32_t block = linear_block(), slot = block / kXcds, part = slot % P, i = slot / P;
    const uint32_t tile = xcd_run(block % kXcds, i / kTileRun) * kTileRun + i % kTileRun;
    if (tile >= total_tiles) return;
    __shared__ uint32_t s_tf[kMaxTfWidth];
    __shared__ float s_alpha[256];
    const uint32_t job = job_of_tile(tile_start, njobs, tile);
    const MarchArgs& a = jobs[job];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ray = lane / P, sub = lane % P;
    // a region and its parts, all powers of two
    const int WW = 8 << tile_shape, WH = 8 >> tile_shape;
    const int RH = ray_h<P>() < WH ? ray_h<P>() : WH, RW = 64 / P / RH, cols = WW / RW;
    uint32_t tx, ty;
    block_tile<kTileBlockW, kTileBlockH>(tile - tile_start[job], (uint32_t)(a.grid_w + 2 * WW - 1) / (2 * WW),
                                 (uint32_t)(a.grid_h + 2 * WH - 1) / (2 * WH), tx, ty);
    // a job marches the pixels of its grid: the whole image, or (a judge's
    // re-march: pix_block > 1) the sparse pixels judge_pixel places, written
    // to out[gy * grid_w + gx]; their samples are not counted (the learned
    // frame's statistics leave the judge out)
    const bool sparse = a.pix_block > 1;
    // the workgroup's 4 waves take neighbouring parts
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
    if (__syncthreads_or(hit)) {   // a workgroup of background pixels needs no tables
        for (int k = tid; k < a.tf_width; k += 256) s_tf[k] = a.tf[k];
        s_alpha[tid] = a.alpha_corr[tid];
        __syncthreads();
        if (hit) {
            // WIDE: 64-bit record addressing for every job (a volume's
            // records exceed 4 GiB); else 32-bit buffer offsets
            if (a.dtype == 0) {
                const CellFetch<uint8_t, WIDE> f = cell_fetch_of<uint8_t, WIDE>(a);
                res = cell_ray<uint8_t, WIDE, SHADE, COUNT, P>(a, f, s_tf, s_alpha, px, py, sub, e, l, n);
            } else {
                const CellFetch<uint16_t, WIDE> f = cell_fetch_of<uint16_t, WIDE>(a);
                res = cell_ray<uint16_t, WIDE, SHADE, COUNT, P>(a, f, s_tf, s_alpha, px, py, sub, e, l, n);
            }
        }
    }
    if (inside && sub == 0) a.out[(size_t)gy * a.grid_w + gx] = res;
    if (sparse) n = RayCounters();
    if (COUNT) add_counters<P>(counters, n, sub == 0);
}

typedef void (*BatchKernel)(const MarchArgs*, const uint32_t*, uint32_t, uint32_t, unsigned long long*, uint32_t);

template <bool WIDE, int SHADE, bool COUNT>
BatchKernel pick_kernel(int lanes) {
    if (lanes == 2) return batch_kernel<WIDE, SHADE, COUNT, 2>;
    if (lanes == 4) return batch_kernel<WIDE, SHADE, COUNT, 4>;
    return batch_kernel<WIDE, SHADE, COUNT, 16>;
}

template <bool WIDE>
BatchKernel kernel_for_w(int shade, bool count, int lanes) {
    if (shade == 2) return count ? pick_kernel<WIDE, 2, true>(lanes) : pick_kernel<WIDE, 2, false>(lanes);
    if (shade == 1) return count ? pick_kernel<WIDE, 1, true>(lanes) : pick_kernel<WIDE, 1, false>(lanes);
    return count ? pick_kernel<WIDE, 0, true>(lanes) : pick_kernel<WIDE, 0, false>(lanes);
}

// Lanes per ray of a launch of `pixels` pixels whose finest step is `step`, for
// the configuration's batch.  `rays` are its pixels by the length of their
// rays, in those of the longest (BatchList): what a launch with few of them
// waits for is the chain of the longest rays, which more lanes shorten; a
// launch of many issues all the time, and more lanes issue more.  2 / 4 lanes,
// us: uneven volumes (64..384 an axis, unshaded) 8 of them (1.2 M rays) 349 /
// 239, 16 (2.4 M) 436 / 312, 32 (4.9 M) 480 / 463, 48 (7.3 M) 555 / 670, 64
// (9.8 M) 616 / 884; views of 512^3 at 1024^2 with Phong, 1 of them 1235 /
// 1193, 2 2025 / 2011, 4 3626 / 3790, 6 5209 / 5550, 12 9914 / 10841; unshaded
// 1 688 / 736, 4 1873 / 2244, 12 5032 / 6329.  So below the first line two
// lanes are never much better, above the second never worse; in between the
// configuration decides.
int batch_lanes(int batch, uint64_t pixels, double rays, float step) {
    if ((double)pixels * step <= 100.0) return 16;
    if (rays <= 1.5e6) return 4;
    return rays > 6.0e6 ? 2 : batch;
}

BatchKernel kernel_for(bool wide, int shade, bool count, int lanes) {
    return wide ? kernel_for_w<true>(shade, count, lanes) : kernel_for_w<false>(shade, count, lanes);
}

}  // namespace

}  // namespace hipdvr

using namespace hipdvr;

namespace {

// Jobs of one plain launch: their arguments per brick size, their tiles per
// tile shape.
struct BatchList {
    MarchArgs* d_args[kBrickSizes] = {};
    uint32_t* d_tile_start[kTileShapes] = {};
    uint32_t total_tiles[kTileShapes] = {};
    uint32_t n = 0;
    uint64_t pixels = 0;
    float step = 0.f;   // the finest
    double rays = 0.0;  // pixels, each counting as its step's share of the finest
};

}  // namespace

struct hipdvr_batch {
    hipdvr_ctx* ctx = nullptr;
    std::vector<hipdvr_batch_job> jobs;    // in launch order (largest first)
    std::vector<uint32_t> order;           // caller's index of each launch position
    int shade = 0;                         // 0 none, 1 Phong, 2 exact Phong
    bool wide = false;                     // some volume's cell records exceed 4 GiB
    // per brick size: device brick tables per job and the jobs' arguments
    std::vector<void*> allocations;
    std::vector<MarchArgs> h_args[kBrickSizes];
    BatchList plain;
    // learned jobs (hipdvr_batch_set_learned), per launch position: the judge's
    // grid, sparse image, sum and flag
    std::vector<hipdvr_learned*> learned;
    std::vector<char> plain_learned;   // given a learned state whose table cannot gain: marched plainly
    hipdvr_learned_opts lopts{};
    std::vector<hipdvr::JudgeGrid> grids;
    std::vector<float4*> d_sparse;
    std::vector<float*> d_sse;
    std::vector<int*> d_flag;
    // the learned launch's jobs (hipdvr_batch_launch_learned): those marched
    // plainly (first each learned view's judge re-march, its sparse grid into
    // its sparse image, then the plain jobs) and the learned ones
    BatchList with_learned;
    LearnedArgs* d_largs = nullptr;
    uint32_t n_learned = 0;
    uint64_t learned_pixels = 0;
    double learned_faces = 0.0;   // voxels of a face of each learned job's volume, if it were a cube
    uint32_t* d_ltile_start[kTileShapes] = {};
    uint32_t ltotal_tiles[kTileShapes] = {};
    uint32_t* d_queue = nullptr;
    hipStream_t queue_stream = nullptr;   // of the last learned launch
    hipdvr::JudgeJob* d_judge = nullptr;
    uint32_t n_judge = 0;
    hipdvr_batch_config cfg{0, 4, 4, 0};
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
};

namespace {

void drop_graph(hipdvr_batch* b) {
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
}

void free_batch(hipdvr_batch* b) {
    if (!b) return;
    drop_graph(b);
    for (void* p : b->allocations) (void)hipFree(p);
    delete b;
}

template <typename P>
P* dev_alloc(hipdvr_batch* b, size_t bytes) {
    void* p = nullptr;
    hip_check(hipMalloc(&p, bytes ? bytes : 4), "hipMalloc(batch)");
    b->allocations.push_back(p);
    return (P*)p;
}

void validate_config(const hipdvr_batch_config& c) {
    if (c.tile < HIPDVR_TILE_8x8 || c.tile > HIPDVR_TILE_32x2) fail(HIPDVR_ERR_INVALID, "unknown tile shape");
    if (c.brick_log2 < 3 || c.brick_log2 > 5) fail(HIPDVR_ERR_INVALID, "brick_log2 must be 3, 4 or 5");
    if (c.batch != 2 && c.batch != 4) fail(HIPDVR_ERR_INVALID, "batch must be 2 or 4");
    if (c.resident < 0 || c.resident > 8) fail(HIPDVR_ERR_INVALID, "resident must be 0 (default) or 1..8");
}

int list_lanes(const BatchList& l, int batch) { return batch_lanes(batch, l.pixels, l.rays, l.step); }

// Lanes per ray of the learned jobs: one, in a persistent launch of their own
// (launch_learned_batch), or 2 or 4 in one launch with the plain jobs
// (launch_learned_mixed).  One lane repeats no skipping among the lanes of a
// ray, so it is the better the more rays there are to fill the chip with; but a
// wavefront then holds 64 rays, which part ways where an image has few pixels
// for its volume's voxels, and the judges' few rays march alone before.  One /
// two lanes, ms (blobs in 512^3): 1024^2 with Phong 4 views 2.10 / 1.93, 12 5.11
// / 5.32, 24 9.56 / 10.68, unshaded 4 1.27 / 1.23, 12 3.03 / 3.29, 24 5.62 /
// 6.48; 1080p 4 views 2.38 / 2.10, 8 3.98 / 4.02, unshaded 1.40 / 1.35, 2.32 /
// 2.53; 768^2 (2.25 pixels to a voxel) 36 views 10.6 / 10.3, 5.71 / 5.91; 512^2
// (one pixel) 96 views 18.6 / 14.8, 8.67 / 7.86.  Turbulence in 512^3 and blobs
// in 256^3 have their lines within a factor of 1.5 of these.  Records past 4 GiB,
// whose loads take longer, never take one lane: 8 views of 2048 x 2048 x 1024 at
// 3840 x 2160 105 / 66.6 ms.
int learned_batch_lanes(const hipdvr_batch* b) {
    if (!b->wide && b->learned_pixels > (b->shade ? 12000000u : 9000000u) &&
        (double)b->learned_pixels >= 2.5 * b->learned_faces)
        return 1;
    const uint64_t pixels = b->learned_pixels + b->with_learned.pixels;
    if (pixels <= 1500000) return 4;
    return pixels > 6000000 ? 2 : b->cfg.batch;
}

void launch_list(hipdvr_batch* b, const BatchList& list, bool count, hipStream_t st) {
    if (list.n == 0) return;
    const int t = b->cfg.tile, bs = b->cfg.brick_log2 - 3;
    const int lanes = list_lanes(list, b->cfg.batch);
    BatchKernel k = kernel_for(b->wide, b->shade, count, lanes);
    size_t pad = 0;
    if (b->cfg.resident > 0) {
        hipFuncAttributes fa;
        hip_check(hipFuncGetAttributes(&fa, (const void*)k), "hipFuncGetAttributes");
        pad = residency_pad(fa.sharedSizeBytes, b->cfg.resident);
    }
    hipLaunchKernelGGL(k, linear_grid(batch_grid(list.total_tiles[t], lanes)), dim3(256), pad, st,
                       (const MarchArgs*)list.d_args[bs], (const uint32_t*)list.d_tile_start[t], list.n,
                       list.total_tiles[t], b->ctx->d_counters, (uint32_t)t);
    hip_check(hipGetLastError(), "batch launch");
}

void launch_batch(hipdvr_batch* b, bool count) { launch_list(b, b->plain, count, ctx_stream(b->ctx)); }

// Tiles of the jobs' grids: start[k] of job k, start[n] in all.
template <typename Job>
std::vector<uint32_t> tile_starts(const std::vector<Job>& jobs, int t, const MarchArgs& (*args)(const Job&)) {
    std::vector<uint32_t> start(jobs.size() + 1, 0);
    const uint32_t tw = 2 * wave_w(t), th = 2 * wave_h(t);
    for (size_t k = 0; k < jobs.size(); ++k) {
        const MarchArgs& m = args(jobs[k]);
        const uint64_t tiles = (uint64_t)((m.grid_w + tw - 1) / tw) * ((m.grid_h + th - 1) / th);
        if (start[k] + tiles > kMaxTiles) fail(HIPDVR_ERR_UNSUPPORTED, "batch too large");
        start[k + 1] = start[k] + (uint32_t)tiles;
    }
    return start;
}
const MarchArgs& plain_args(const MarchArgs& a) { return a; }
const MarchArgs& learned_args(const LearnedArgs& a) { return a.m; }

template <typename T>
void upload(T* dst, const std::vector<T>& src, hipStream_t st) {
    if (!src.empty())
        hip_check(hipMemcpyAsync(dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice, st), "upload");
}

// A list's host side: what upload_list takes over.
struct HostList {
    std::vector<MarchArgs> args[kBrickSizes];
    std::vector<uint32_t> start[kTileShapes];
    void tiles() {
        for (int t = 0; t < kTileShapes; ++t) start[t] = tile_starts(args[0], t, plain_args);
    }
};

// Uploads a list into buffers of at least `capacity` jobs (asynchronous: the
// caller waits before `h` goes).
void upload_list(hipdvr_batch* b, BatchList& list, const HostList& h, size_t capacity, hipStream_t st) {
    for (int bs = 0; bs < kBrickSizes; ++bs) {
        if (!list.d_args[bs]) list.d_args[bs] = dev_alloc<MarchArgs>(b, capacity * sizeof(MarchArgs));
        upload(list.d_args[bs], h.args[bs], st);
    }
    for (int t = 0; t < kTileShapes; ++t) {
        if (!list.d_tile_start[t]) list.d_tile_start[t] = dev_alloc<uint32_t>(b, (capacity + 1) * 4);
        upload(list.d_tile_start[t], h.start[t], st);
        list.total_tiles[t] = h.start[t].back();
    }
    list.n = (uint32_t)h.args[0].size();
    list.pixels = 0;
    list.step = INFINITY;
    for (const MarchArgs& m : h.args[0]) {
        list.pixels += (uint64_t)m.grid_w * m.grid_h;
        list.step = std::min(list.step, m.step);
    }
    list.rays = 0.0;
    for (const MarchArgs& m : h.args[0]) list.rays += (double)m.grid_w * m.grid_h * (list.step / m.step);
}

}  // namespace

extern "C" {

int hipdvr_batch_create(hipdvr_ctx* ctx, const hipdvr_batch_job* jobs, uint32_t n, hipdvr_batch** out) {
    if (!ctx) return HIPDVR_ERR_INVALID;
    return ctx_guarded(ctx, [&] {
        if (!out || !jobs || n == 0) fail(HIPDVR_ERR_INVALID, "a batch needs at least one job");
        int shade = -1;
        for (uint32_t i = 0; i < n; ++i) {
            const hipdvr_batch_job& j = jobs[i];
            if (!j.volume || !j.tf || !j.d_entry || !j.d_exit || !j.d_out || !j.w || !j.h)
                fail(HIPDVR_ERR_INVALID, "job " + std::to_string(i) + ": NULL argument or empty image");
            if (j.volume->ctx != ctx || j.tf->ctx != ctx) fail(HIPDVR_ERR_INVALID, "handle from another context");
            validate_params(&j.params, j.tf);
            if (j.params.filter != HIPDVR_FILTER_LINEAR || j.params.classification != HIPDVR_CLASS_TF ||
                j.params.compositing != HIPDVR_COMPOSITE_DVR)
                fail(HIPDVR_ERR_UNSUPPORTED, "batched jobs use the linear filter, TF classification and DVR");
            if (j.params.shading != HIPDVR_SHADE_NONE && j.params.gradient != HIPDVR_GRADIENT_CENTRAL)
                fail(HIPDVR_ERR_UNSUPPORTED, "batched jobs shade with central-difference gradients");
            const int ph = j.params.shading == HIPDVR_SHADE_NONE ? 0
                         : (j.params.shading == HIPDVR_SHADE_PHONG && !j.params.exact_shading) ? 1 : 2;
            if (shade >= 0 && ph != shade) fail(HIPDVR_ERR_UNSUPPORTED, "all jobs of a batch share the shading path");
            shade = ph;
        }
        ctx_set_device(ctx);
        hipStream_t st = ctx_stream(ctx);
        hipdvr_batch* b = new hipdvr_batch();
        b->ctx = ctx;
        b->shade = shade;
        try {
            // largest estimated cost first
            std::vector<uint32_t> order(n);
            std::iota(order.begin(), order.end(), 0u);
            auto cost = [&](uint32_t i) {
                const hipdvr_volume* v = jobs[i].volume;
                const uint32_t m = std::max(v->desc.dims[0], std::max(v->desc.dims[1], v->desc.dims[2]));
                return (double)jobs[i].w * jobs[i].h * m;
            };
            std::stable_sort(order.begin(), order.end(), [&](uint32_t x, uint32_t y) { return cost(x) > cost(y); });
            for (uint32_t i : order) b->jobs.push_back(jobs[i]);
            b->order = order;
            // cell records, then per brick size the brick tables of every job
            for (const hipdvr_batch_job& j : b->jobs) {
                ensure_cells(const_cast<hipdvr_volume*>(j.volume), st);
                b->wide = b->wide || j.volume->cells_wide;
            }
            for (int bs = 0; bs < kBrickSizes; ++bs) {
                std::vector<MarchArgs>& args = b->h_args[bs];
                args.assign(n, MarchArgs{});
                const uint32_t bl = (uint32_t)bs + 3;
                for (uint32_t i = 0; i < n; ++i) {
                    const hipdvr_batch_job& j = b->jobs[i];
                    const hipdvr_volume* v = j.volume;
                    uint32_t nb[3];
                    uint64_t count = 1;
                    for (int k = 0; k < 3; ++k) {
                        nb[k] = (v->desc.dims[k] + (1u << bl) - 1) >> bl;
                        count *= nb[k];
                    }
                    // ranges, skip grid and its scratch
                    uint2* mm = dev_alloc<uint2>(b, count * (sizeof(uint2) + 2));
                    uint8_t* skip = (uint8_t*)(mm + count);
                    launch_brick_minmax(v, bl, nb, mm, st);
                    launch_skip_grid(occupancy_args(v, j.tf, mm, count), nb, skip, skip + count, st);
                    MarchArgs& a = args[i];
                    fill_march_args(a, v, j.tf, &j.params, j.d_entry, j.d_exit, j.d_out, j.w, j.h, nullptr);
                    a.cells = v->d_cells;
                    a.skip = skip;
                    a.skip_log2 = bl;
                    for (int k = 0; k < 3; ++k) a.nskip[k] = nb[k];
                }
            }
            HostList list;
            for (int bs = 0; bs < kBrickSizes; ++bs) list.args[bs] = b->h_args[bs];
            list.tiles();
            upload_list(b, b->plain, list, n, st);
            if (list_lanes(b->plain, b->cfg.batch) == 2) b->cfg.batch = 2;
            hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
            b->learned.assign(n, nullptr);
            b->plain_learned.assign(n, 0);
            hip_check(hipGetLastError(), "batch setup");
            hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
        } catch (...) {
            free_batch(b);
            throw;
        }
        *out = b;
    });
}

int hipdvr_batch_destroy(hipdvr_batch* b) {
    if (!b) return HIPDVR_OK;
    (void)hipStreamSynchronize(ctx_stream(b->ctx));
    free_batch(b);
    return HIPDVR_OK;
}

int hipdvr_batch_set_config(hipdvr_batch* b, const hipdvr_batch_config* cfg) {
    if (!b) return HIPDVR_ERR_INVALID;
    return ctx_guarded(b->ctx, [&] {
        if (!cfg) fail(HIPDVR_ERR_INVALID, "NULL argument");
        validate_config(*cfg);
        b->cfg = *cfg;
        drop_graph(b);
    });
}

int hipdvr_batch_get_config(const hipdvr_batch* b, hipdvr_batch_config* cfg) {
    if (!b || !cfg) return HIPDVR_ERR_INVALID;
    *cfg = b->cfg;
    return HIPDVR_OK;
}

int hipdvr_batch_capture(hipdvr_batch* b) {
    if (!b) return HIPDVR_ERR_INVALID;
    return ctx_guarded(b->ctx, [&] {
        ctx_set_device(b->ctx);
        hipStream_t st = ctx_stream(b->ctx);
        drop_graph(b);
        hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
        hip_check(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal), "hipStreamBeginCapture");
        try {
            launch_batch(b, false);
        } catch (...) {
            hipGraph_t g = nullptr;
            (void)hipStreamEndCapture(st, &g);
            if (g) (void)hipGraphDestroy(g);
            throw;
        }
        hip_check(hipStreamEndCapture(st, &b->graph), "hipStreamEndCapture");
        hip_check(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0), "hipGraphInstantiate");
    });
}

int hipdvr_batch_launch(hipdvr_batch* b, hipdvr_stats* stats) {
    if (!b) return HIPDVR_ERR_INVALID;
    return ctx_guarded(b->ctx, [&] {
        ctx_set_device(b->ctx);
        hipStream_t st = ctx_stream(b->ctx);
        if (stats) {
            launch_zero_u64(b->ctx->d_counters, kNumCounters, st);
            hip_check(hipEventRecord(b->ctx->ev0, st), "hipEventRecord");
            launch_batch(b, true);
            hip_check(hipEventRecord(b->ctx->ev1, st), "hipEventRecord");
            unsigned long long c[kNumCounters];
            hip_check(hipMemcpyAsync(c, b->ctx->d_counters, sizeof c, hipMemcpyDeviceToHost, st), "download");
            hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
            float ms = 0.f;
            hip_check(hipEventElapsedTime(&ms, b->ctx->ev0, b->ctx->ev1), "hipEventElapsedTime");
            stats->rays = c[0];
            stats->samples = c[1];
            stats->fetched = c[2];
            stats->shaded = c[3];
            stats->lane_slots = c[4];
            stats->shade_slots = c[5];
            stats->kernel_ms = ms;
            return;
        }
        const bool timed = ctx_timing_start(b->ctx);
        if (b->exec) hip_check(hipGraphLaunch(b->exec, st), "hipGraphLaunch");
        else launch_batch(b, false);
        if (timed) ctx_timing_stop(b->ctx);
    });
}

int hipdvr_batch_autotune(hipdvr_batch* b, uint32_t reps, hipdvr_batch_config* best, float* best_ms) {
    if (!b) return HIPDVR_ERR_INVALID;
    return ctx_guarded(b->ctx, [&] {
        if (reps == 0) fail(HIPDVR_ERR_INVALID, "reps must be > 0");
        ctx_set_device(b->ctx);
        hipStream_t st = ctx_stream(b->ctx);
        drop_graph(b);
        hipEvent_t e0 = nullptr, e1 = nullptr;
        hip_check(hipEventCreate(&e0), "hipEventCreate");
        hip_check(hipEventCreate(&e1), "hipEventCreate");
        hipdvr_batch_config win = b->cfg;
        float win_ms = 1e30f;
        // mean launch time of configuration c over reps launches after a warm-up
        auto time_config = [&](const hipdvr_batch_config& c) {
            b->cfg = c;
            launch_batch(b, false);
            hip_check(hipEventRecord(e0, st), "hipEventRecord");
            for (uint32_t r = 0; r < reps; ++r) launch_batch(b, false);
            hip_check(hipEventRecord(e1, st), "hipEventRecord");
            hip_check(hipEventSynchronize(e1), "hipEventSynchronize");
            float ms = 0.f;
            hip_check(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
            return ms / (float)reps;
        };
        try {
            for (int t = 0; t < 3; ++t)
                for (int bl = 3; bl <= 5; ++bl)
                    for (int k : {2, 4}) {
                        // (where the size decides, both are the same launch)
                        const int lanes = list_lanes(b->plain, k);
                        if (list_lanes(b->plain, 6 - k) == lanes && k != (lanes == 2 ? 2 : 4)) continue;
                        const float ms = time_config(hipdvr_batch_config{t, bl, k, 0});
                        if (ms < win_ms) {
                            win_ms = ms;
                            win = b->cfg;
                        }
                    }
            const hipdvr_batch_config shape = win;
            for (int r : {3, 4, 5}) {
                const float ms = time_config(hipdvr_batch_config{shape.tile, shape.brick_log2, shape.batch, r});
                if (ms < win_ms) {
                    win_ms = ms;
                    win = b->cfg;
                }
            }
        } catch (...) {
            (void)hipEventDestroy(e0);
            (void)hipEventDestroy(e1);
            throw;
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        b->cfg = win;
        if (best) *best = win;
        if (best_ms) *best_ms = win_ms;
    });
}

int hipdvr_batch_set_learned(hipdvr_batch* b, hipdvr_learned* const* learned, uint32_t n,
                             const hipdvr_learned_opts* o) {
    if (!b) return HIPDVR_ERR_INVALID;
    return ctx_guarded(b->ctx, [&] {
        if (!learned || n != b->jobs.size()) fail(HIPDVR_ERR_INVALID, "one learned state (or NULL) per job");
        ctx_set_device(b->ctx);
        hipStream_t st = ctx_stream(b->ctx);
        const hipdvr_learned_opts lopts = learned_options(o);
        const size_t nj = b->jobs.size();
        // built aside and taken over only when every job is accepted
        std::vector<hipdvr_learned*> lv(nj, nullptr);
        std::vector<char> plain_lv(nj, 0);
        std::vector<const hipdvr_learned*> given(nj, nullptr);   // the state given for each job
        std::vector<JudgeGrid> grids(nj, JudgeGrid{});
        std::vector<float4*> sparse(nj, nullptr);
        std::vector<float*> sse(nj, nullptr);
        std::vector<int*> flag(nj, nullptr);
        std::vector<LearnedArgs> largs;
        for (size_t i = 0; i < nj; ++i) {
            hipdvr_learned* l = learned[b->order[i]];
            const hipdvr_batch_job& j = b->jobs[i];
            if (!l) continue;
            const std::string job = "job " + std::to_string(b->order[i]);
            if (learned_volume(l) != j.volume) fail(HIPDVR_ERR_INVALID, job + ": the learned state of another volume");
            if (learned_prepared_tf(l) != j.tf)
                fail(HIPDVR_ERR_INVALID, job + ": the learned state was not prepared for the job's TF");
            if (b->shade == 2) fail(HIPDVR_ERR_UNSUPPORTED, "learned jobs shade with the approximate Phong path");
            // a learned state holds the opacity tables of one step
            for (size_t k = 0; k < i; ++k)
                if (given[k] == l && b->jobs[k].params.step != j.params.step)
                    fail(HIPDVR_ERR_INVALID, "jobs sharing a learned state must share the step");
            given[i] = l;
            if (!learned_gains(l)) {
                // every occupied brick at the base step: the plain march
                // gives the exact frame at a lower cost
                plain_lv[i] = 1;
                continue;
            }
            largs.push_back(LearnedArgs{});
            largs.back().m = b->h_args[0][i];
            learned_stepping_args(l, &j.params, largs.back());
            lv[i] = l;
            grids[i] = learned_judge_grid(j.w, j.h, lopts);
        }
        for (size_t i = 0; i < nj; ++i) {
            if (!lv[i]) continue;
            if (i < b->d_sparse.size() && b->d_sparse[i] && b->grids[i].w == grids[i].w &&
                b->grids[i].h == grids[i].h) {   // same grid as before: keep its buffers
                sparse[i] = b->d_sparse[i];
                sse[i] = b->d_sse[i];
                flag[i] = b->d_flag[i];
                continue;
            }
            const size_t px = (size_t)grids[i].w * grids[i].h;
            sparse[i] = dev_alloc<float4>(b, px * sizeof(float4));
            sse[i] = dev_alloc<float>(b, 64);
            flag[i] = dev_alloc<int>(b, 64);
        }
        // the learned launch's jobs: each learned view's judge re-march
        // (plain, into its sparse image), the plain jobs, the learned ones; and
        // the judges
        HostList list;
        std::vector<JudgeJob> judges;
        const float mse_max = powf(10.f, -lopts.psnr_floor / 10.f);
        for (size_t i = 0; i < nj; ++i) {
            if (!lv[i]) continue;
            const JudgeGrid& g = grids[i];
            const hipdvr_batch_job& j = b->jobs[i];
            for (int bs = 0; bs < kBrickSizes; ++bs) {
                MarchArgs sj = b->h_args[bs][i];
                sj.out = sparse[i];
                sj.grid_w = g.w;
                sj.grid_h = g.h;
                sj.stride = (int32_t)g.stride;
                sj.pix_block = (int32_t)g.block;
                sj.pix_offset = (int32_t)g.offs;
                list.args[bs].push_back(sj);
            }
            JudgeJob jj;
            jj.learned = (const float4*)j.d_out;
            jj.sparse = sparse[i];
            jj.sse = sse[i];
            jj.flag = flag[i];
            jj.w = (int32_t)j.w;
            jj.h = (int32_t)j.h;
            jj.sw = g.w;
            jj.sh = g.h;
            jj.stride = (int32_t)g.stride;
            jj.block = (int32_t)g.block;
            jj.offs = (int32_t)g.offs;
            jj.denom = (float)(g.w * g.h * 4);
            jj.mse_max = mse_max;
            judges.push_back(jj);
        }
        for (int bs = 0; bs < kBrickSizes; ++bs)
            for (size_t i = 0; i < nj; ++i)
                if (!lv[i]) list.args[bs].push_back(b->h_args[bs][i]);
        list.tiles();
        std::vector<uint32_t> lstart[kTileShapes];
        for (int t = 0; t < kTileShapes; ++t) {
            lstart[t] = tile_starts(largs, t, learned_args);
            if ((uint64_t)lstart[t].back() + list.start[t].back() > kMaxTiles)
                fail(HIPDVR_ERR_UNSUPPORTED, "batch too large");
        }
        if (!b->d_largs) b->d_largs = dev_alloc<LearnedArgs>(b, nj * sizeof(LearnedArgs));
        for (int t = 0; t < kTileShapes; ++t)
            if (!b->d_ltile_start[t]) b->d_ltile_start[t] = dev_alloc<uint32_t>(b, (nj + 1) * 4);
        if (!b->d_queue) b->d_queue = dev_alloc<uint32_t>(b, kLearnedQueueBytes);
        if (!b->d_judge) b->d_judge = dev_alloc<JudgeJob>(b, nj * sizeof(JudgeJob));
        // every learned view gives a judge's job, the others themselves
        upload_list(b, b->with_learned, list, nj, st);
        upload(b->d_largs, largs, st);
        for (int t = 0; t < kTileShapes; ++t) upload(b->d_ltile_start[t], lstart[t], st);
        upload(b->d_judge, judges, st);
        hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
        b->n_learned = (uint32_t)largs.size();
        b->learned_pixels = 0;
        b->learned_faces = 0.0;
        for (size_t i = 0; i < nj; ++i) {
            if (!lv[i]) continue;
            const hipdvr_batch_job& j = b->jobs[i];
            b->learned_pixels += (uint64_t)j.w * j.h;
            const uint32_t* d = j.volume->desc.dims;
            b->learned_faces += std::pow((double)d[0] * d[1] * d[2], 2.0 / 3.0);
        }
        for (int t = 0; t < kTileShapes; ++t) b->ltotal_tiles[t] = lstart[t].back();
        b->n_judge = (uint32_t)judges.size();
        b->lopts = lopts;
        b->learned.swap(lv);
        b->plain_learned.swap(plain_lv);
        b->grids.swap(grids);
        b->d_sparse.swap(sparse);
        b->d_sse.swap(sse);
        b->d_flag.swap(flag);
    });
}

int hipdvr_batch_launch_learned(hipdvr_batch* b, hipdvr_learned_stats* stats) {
    if (!b) return HIPDVR_ERR_INVALID;
    return ctx_guarded(b->ctx, [&] {
        ctx_set_device(b->ctx);
        hipStream_t st = ctx_stream(b->ctx);
        const size_t nj = b->jobs.size();
        const int bs = b->cfg.brick_log2 - 3;
        const int shade = b->shade;
        bool any = false;
        for (size_t i = 0; i < nj; ++i) {
            if (!b->learned[i]) continue;
            any = true;
            // the state's opacity tables follow the last step it rendered with
            learned_ensure_step(b->learned[i], b->jobs[i].params.step);
        }
        const bool count = stats != nullptr;
        if (count) launch_zero_u64(b->ctx->d_counters, kNumCounters, st);
        const bool timed = ctx_timing_start(b->ctx);
        if (!b->d_largs) fail(HIPDVR_ERR_INVALID, "hipdvr_batch_set_learned has not been called");
        // 1. the judges' plain re-marches of the learned views' sparse pixels,
        //    the plain jobs and the learned ones
        const BatchList& plain = b->with_learned;
        const int t = b->cfg.tile;
        const int lanes = any ? learned_batch_lanes(b) : 0;
        if (lanes < 2) launch_list(b, plain, count, st);
        if (lanes == 1) {
            // the queue's counters serve one launch at a time
            if (b->queue_stream && b->queue_stream != st) ctx_wait_left(b->ctx, b->queue_stream, ctx_capturing(b->ctx));
            b->queue_stream = st;
            launch_learned_batch(b->d_largs, b->d_ltile_start[t], b->n_learned, b->ltotal_tiles[t], t, shade != 0,
                                 b->cfg.resident, b->d_queue, count ? b->ctx->d_counters : nullptr, st);
        }
        if (lanes > 1)
            launch_learned_mixed(plain.d_args[bs], plain.d_tile_start[t], plain.n, plain.n ? plain.total_tiles[t] : 0,
                                 b->d_largs, b->d_ltile_start[t], b->n_learned, b->ltotal_tiles[t], t, lanes,
                                 shade != 0, b->wide, b->cfg.resident, count ? b->ctx->d_counters : nullptr, st);
        if (any) {
            // 2. the judges of all learned views in one launch, then per
            //    learned view the plain frame, launched always, which runs
            //    only when its view was flagged
            launch_judge_multi(b->d_judge, b->n_judge, st);
            for (size_t i = 0; i < nj; ++i) {
                if (!b->learned[i]) continue;
                const hipdvr_batch_job& j = b->jobs[i];
                MarchArgs fb = b->h_args[bs][i];
                fb.counters = nullptr;
                fb.cond_flag = b->d_flag[i];
                launch_march_cell(fb, fb.dtype, shade, false, j.volume->cells_wide, 0, st);
            }
        }
        hip_check(hipGetLastError(), "batched learned launch");
        if (timed) ctx_timing_stop(b->ctx);
        if (count) {
            unsigned long long c[kNumCounters];
            std::vector<float> sse(nj, 0.f);
            std::vector<int> flag(nj, 0);
            hip_check(hipMemcpyAsync(c, b->ctx->d_counters, sizeof c, hipMemcpyDeviceToHost, st), "download");
            for (size_t i = 0; i < nj; ++i) {
                if (!b->learned[i]) continue;
                hip_check(hipMemcpyAsync(&sse[i], b->d_sse[i], 4, hipMemcpyDeviceToHost, st), "download");
                hip_check(hipMemcpyAsync(&flag[i], b->d_flag[i], 4, hipMemcpyDeviceToHost, st), "download");
            }
            hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
            for (size_t i = 0; i < nj; ++i) {
                hipdvr_learned_stats& s = stats[b->order[i]];
                s.samples = c[1];
                s.shaded = c[3];
                if (b->learned[i]) {
                    const JudgeGrid& g = b->grids[i];
                    const double mse = (double)sse[i] / ((double)g.w * g.h * 4);
                    s.sparse_psnr = mse > 0 ? (float)(10.0 * std::log10(1.0 / mse)) : 999.f;
                    s.fell_back = flag[i];
                } else {
                    s.sparse_psnr = b->plain_learned[i] ? 999.f : 0.f;
                    s.fell_back = 0;
                }
            }
        }
    });
}

}  // extern "C"
