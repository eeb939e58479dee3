// kernels.h -- launchers of the HIP kernels (internal to libhipdvr.so).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "march_common.h"

namespace hipdvr {

// Ray-generation constants of the unit-cube proxy, texture space.
struct RayGen {
    float o[3];     // camera position
    float f[3];     // view direction
    float r[3];     // right * tan(fovy/2) * aspect
    float u[3];     // up * tan(fovy/2)
    float near_t;   // near-plane ray parameter
    int32_t w, h;
    int32_t quantize;
};

void launch_march_ref(const MarchArgs& a, int dtype, int filter, int classif, bool phong,
                      bool count, hipStream_t st);
// compositing modes other than DVR (TF classification), reference layout
void launch_march_modes(const MarchArgs& a, int dtype, int filter, bool phong, hipStream_t st);
void launch_march_fast(const MarchArgs& a, int dtype, int filter, bool phong, bool count, bool wide,
                       hipStream_t st);
// shade: 0 none, 1 Phong (interior gradient, approximate lighting), 2 Phong
// bit-identical to the reference kernel; batch: hipdvr_params::batch.  The
// grid's pixels are placed by judge_pixel (a.pix_block; 1 for a whole frame).
void launch_march_cell(const MarchArgs& a, int dtype, int shade, bool count, bool wide, int batch,
                       hipStream_t st);
// The other compositing modes (preint false) or the pre-integrated
// classification on the cell records, linear filter and central differences:
// the reference-layout kernels' results bit for bit.  Without a.skip nothing
// is skipped.
void launch_march_cell_modes(const MarchArgs& a, int dtype, bool wide, bool preint, bool shaded, bool count, int batch,
                             hipStream_t st);
// Lanes per ray of a frame (march_cell.h) for hipdvr_params::batch: 1 and 2
// two, 4 four, 8 sixteen; 0 by the grid's size.  A frame of few rays waits
// for their chains, a frame of many for issue slots, of which more lanes per
// ray use more.  Measured on square frames of 128^3 u8, 256^3 and 512^3 u16
// shells, unshaded and Phong, in microseconds for 2 / 4 / 16 lanes:
//   512^3 Phong 128^2 604 / 339 / 170, 256^2 600 / 355 / 237, 512^2 656 / 396
//   / 443, 1024^2 714 / 674 / 1344, 1536^2 1139 / 1254 / 2864;
//   256^3 unshaded 128^2 222 / 138 / 87, 512^2 252 / 192 / 252, 1024^2 274 /
//   296 / 743; 128^3 unshaded 128^2 109 / 68 / 45, 512^2 117 / 95 / 135.
// The line between 16 and 4 follows the samples of the longest ray (1/step):
// a 256^2 frame of 28 samples per ray takes 12 us with four, 17 with 16.
// (Eight lanes lie behind both neighbours: 512^3 Phong 128^2 300, 512^2 458.)
int frame_lanes(int batch, uint64_t pixels, float step);
// The slab-staged march (march_slab.h): linear filter, TF classification,
// DVR; shade as for the cell kernel.  Reads the linear volume.
void launch_march_slab(const MarchArgs& a, int dtype, int shade, bool count, hipStream_t st);
// Zero n 64-bit counters with a kernel (graph-capture safe, unlike a memset node).
void launch_zero_u64(unsigned long long* p, int n, hipStream_t st);
// Streaming copy of n 16-byte vectors (bandwidth calibration).
void launch_copy16(void* dst, const void* src, size_t n, hipStream_t st);
void launch_entry_exit(const RayGen& g, float4* entry, float4* exit, hipStream_t st);

}  // namespace hipdvr
