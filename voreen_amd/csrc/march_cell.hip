// march_cell.hip -- per-frame launches of the cell-record ray march (the
// device code and its parity argument are in march_cell.h): one workgroup per
// 16x16 pixel tile, tiles in XCD-compact order.
#include "kernels.h"
#include "march_cell.h"
#include "march_common.h"

namespace hipdvr {

// A workgroup is 2x2 waves of ray_w<P>() x ray_h<P>() rays, P lanes per ray: a
// P-th of a 16x16 pixel tile.
template <typename T, bool WIDE, int SHADE, bool COUNT, int P>
__global__ __launch_bounds__(256, SHADE == 2 ? 4 : 6) void march_cell_kernel(const MarchArgs a, const uint32_t tiles_x,
                                                         const uint32_t tiles_y) {
    // XCD-compact tile order (xcd_tile): each XCD marches one compact region
    // of tiles, the chip one compact image area; the P workgroups of a tile
    // follow each other on its XCD
    const uint32_t block = linear_block(), slot = block / kXcds, part = slot % P;
    uint32_t tile_x, tile_y;
    if (!xcd_tile((slot / P) * kXcds + block % kXcds, tiles_x, tiles_y, tile_x, tile_y))
        return;   // whole workgroup leaves together
    if (a.cond_flag && *a.cond_flag == 0) return;
    __shared__ uint32_t s_tf[kMaxTfWidth];
    __shared__ float s_alpha[256];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6, ray = lane / P, sub = lane % P;
    constexpr int RW = ray_w<P>(), RH = ray_h<P>(), PX = 16 / (2 * RW);   // parts of the tile per row
    const int gx = (int)tile_x * 16 + ((int)(part % PX) * 2 + (wave & 1)) * RW + ray % RW;
    const int gy = (int)tile_y * 16 + ((int)(part / PX) * 2 + (wave >> 1)) * RH + ray / RW;
    const int px = judge_pixel(gx, a.stride, a.pix_block, a.pix_offset);
    const int py = judge_pixel(gy, a.stride, a.pix_block, a.pix_offset);
    const bool inside = (gx < a.grid_w) && (gy < a.grid_h) && (px < a.w) && (py < a.h);
    float4 e = make_float4(0.f, 0.f, 0.f, 0.f), l = e;
    if (inside) {
        const size_t pix = (size_t)py * a.w + px;
        e = a.entry[pix];
        l = a.exit[pix];
    }
    const bool hit = !is_background(e, l);
    float4 res = make_float4(0.f, 0.f, 0.f, 0.f);
    RayCounters n;
    if (__syncthreads_or(hit)) {   // a workgroup of background pixels needs no tables
        for (int i = tid; i < a.tf_width; i += 256) s_tf[i] = a.tf[i];
        s_alpha[tid] = a.alpha_corr[tid];
        __syncthreads();
        const CellFetch<T, WIDE> f = cell_fetch_of<T, WIDE>(a);
        if (hit) res = cell_ray<T, WIDE, SHADE, COUNT, P>(a, f, s_tf, s_alpha, px, py, sub, e, l, n);
    }
    if (inside && sub == 0) a.out[(size_t)gy * a.grid_w + gx] = res;
    if (COUNT) add_counters<P>(a.counters, n, sub == 0);
}

template <typename T, bool WIDE, int SHADE, int P>
static void launch_k(const MarchArgs& a, bool count, hipStream_t st) {
    const uint32_t tx = (a.grid_w + 15) / 16, ty = (a.grid_h + 15) / 16;
    const dim3 grid = linear_grid((uint64_t)xcd_tile_grid(tx, ty) * P);
    if (count)
        hipLaunchKernelGGL((march_cell_kernel<T, WIDE, SHADE, true, P>), grid, dim3(256), 0, st, a, tx, ty);
    else
        hipLaunchKernelGGL((march_cell_kernel<T, WIDE, SHADE, false, P>), grid, dim3(256), 0, st, a, tx, ty);
}

template <typename T, bool WIDE, int SHADE>
static void launch_ks(const MarchArgs& a, bool count, int lanes, hipStream_t st) {
    if (lanes == 2) launch_k<T, WIDE, SHADE, 2>(a, count, st);
    else if (lanes == 4) launch_k<T, WIDE, SHADE, 4>(a, count, st);
    else launch_k<T, WIDE, SHADE, 16>(a, count, st);
}

template <typename T, bool WIDE>
static void launch_cw(const MarchArgs& a, int shade, bool count, int lanes, hipStream_t st) {
    if (shade == 2) launch_ks<T, WIDE, 2>(a, count, lanes, st);
    else if (shade == 1) launch_ks<T, WIDE, 1>(a, count, lanes, st);
    else launch_ks<T, WIDE, 0>(a, count, lanes, st);
}

int frame_lanes(int batch, uint64_t pixels, float step) {
    if (batch) return batch <= 2 ? 2 : (batch == 4 ? 4 : 16);
    if ((double)pixels * step <= 100.0) return 16;
    return pixels <= 1500000 ? 4 : 2;
}

void launch_march_cell(const MarchArgs& a, int dtype, int shade, bool count, bool wide, int batch,
                       hipStream_t st) {
    const int lanes = frame_lanes(batch, (uint64_t)a.grid_w * a.grid_h, a.step);
    if (dtype == 0) {
        if (wide) launch_cw<uint8_t, true>(a, shade, count, lanes, st);
        else launch_cw<uint8_t, false>(a, shade, count, lanes, st);
    } else {
        if (wide) launch_cw<uint16_t, true>(a, shade, count, lanes, st);
        else launch_cw<uint16_t, false>(a, shade, count, lanes, st);
    }
}

}  // namespace hipdvr
