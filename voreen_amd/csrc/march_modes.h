// march_modes.h -- the compositing modes other than DVR, one sample at a time:
// shared by the reference-layout kernel (march_ref.hip) and the cell-record
// kernel (march_cell_modes.hip).
#pragma once

#include "march_common.h"

namespace hipdvr {

// compositeMIDAhelper, mod_compositing.frag:112-129.
__device__ __forceinline__ void mida_step(float res[4], float voxel, const float c[3], float alpha, float max_int,
                                          float gamma) {
    float delta = 0.0f;
    if (voxel > max_int) delta = voxel - max_int;
    const float beta = 1.0f - delta * (1.0f + gamma);
    const float k = (1.0f - beta * res[3]) * alpha;
#pragma unroll
    for (int i = 0; i < 3; ++i) res[i] = beta * res[i] + k * c[i];
    res[3] = beta * res[3] + (1.0f - beta * res[3]) * alpha;
}

// One sample of alpha > 0 taken into the ray's result
// (mod_compositing.frag:85-213): its real-world intensity rw, what the mode
// shows of it in c (colour; FHP the position, FHN the normal) and the alpha it
// is composited with (MIDA: the corrected one).  ISO: the caller has found the
// alpha in the band.
__device__ __forceinline__ void mode_composite(const MarchArgs& a, int mode, float rw, const float c[3], float alpha,
                                               float out[4], float& max_int) {
    if (mode == kCompMIP) {
        if (rw > max_int) {
            out[0] = c[0];
            out[1] = c[1];
            out[2] = c[2];
            out[3] = alpha;
            max_int = rw;
        }
    } else if (mode == kCompMOP) {
        if (alpha > out[3]) {
            out[0] = c[0];
            out[1] = c[1];
            out[2] = c[2];
            out[3] = alpha;
        }
    } else if (mode == kCompMIDA) {
        if (a.gamma <= 0.0f) {
            mida_step(out, rw, c, alpha, max_int, a.gamma);
        } else {
            float mip[4], mida[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) mip[i] = mida[i] = out[i];
            if (rw > max_int) {
                mip[0] = c[0];
                mip[1] = c[1];
                mip[2] = c[2];
                mip[3] = alpha;
                max_int = rw;
            }
            mida_step(mida, rw, c, alpha, max_int, 0.0f);
#pragma unroll
            for (int i = 0; i < 4; ++i) out[i] = a.gamma * mip[i] + (1.0f - a.gamma) * mida[i];
        }
    } else if (mode == kCompISO) {
        out[0] = c[0];
        out[1] = c[1];
        out[2] = c[2];
        out[3] = 1.0f;
    } else {   // FHP, FHN: the first hit
        if (out[0] == 0.f && out[1] == 0.f && out[2] == 0.f) {
            out[0] = c[0];
            out[1] = c[1];
            out[2] = c[2];
            out[3] = 1.0f;
        }
    }
}

}  // namespace hipdvr
