// march_cell.h -- device code of the cell-record ray march, shared by the
// per-frame kernel (march_cell.hip) and the batched kernel
// (batch.hip).
//
// The record of cell (x, y, z) holds the eight voxels of its trilinear
// footprint, (x..x+1, y..y+1, z..z+1) clamped to the volume, in the order the
// trilinear sum visits them (llB, lrB, urB, ulB, llF, lrF, urF, ulF of
// VolumeRAM::getVoxelNormalizedLinear, volumeram.cpp:78-97).  One sample is
// one 16-byte (uint16) or 8-byte (uint8) load instead of eight 2- or 1-byte
// gathers: the march is bound by the vector-memory issue rate per load
// instruction, not by bytes, so one wide load per sample is the MI355X trade
// of HBM capacity (8x the voxel bytes) for load instructions.
//
// Sample positions, corners, weights, the 8-term sum, TF classification,
// opacity correction, Phong's six central-difference lookups
// (mod_gradients.frag:202-214) and the lighting are the same expressions as
// the reference-layout kernel (march_ref.hip, restating
// CPURaycaster::directRendering, cpuraycaster.cpp:210-326), so the image is
// bit-identical to it, shaded or not.  Empty-space skipping is the exact
// fast-forward of the bricked kernel over the skip grid (volume.h); P lanes
// march a ray together, one sample each, and composite in order; a sample
// fetched past early termination is dropped.
#pragma once

#include <type_traits>

#include "cell_layout.h"
#include "march_common.h"
#include "step_run.h"

namespace hipdvr {

template <typename T>
struct CellRecord;
template <>
struct CellRecord<uint16_t> {
    typedef uint4 type;
    // stored values as floats (no normalization)
    static __device__ __forceinline__ void raw(const uint4& r, float v[8]) {
        v[0] = (float)(r.x & 0xffffu);
        v[1] = (float)(r.x >> 16);
        v[2] = (float)(r.y & 0xffffu);
        v[3] = (float)(r.y >> 16);
        v[4] = (float)(r.z & 0xffffu);
        v[5] = (float)(r.z >> 16);
        v[6] = (float)(r.w & 0xffffu);
        v[7] = (float)(r.w >> 16);
    }
    static __device__ __forceinline__ void unpack(const uint4& r, float v[8]) {
        v[0] = VoxNorm<uint16_t>::apply(r.x & 0xffffu);
        v[1] = VoxNorm<uint16_t>::apply(r.x >> 16);
        v[2] = VoxNorm<uint16_t>::apply(r.y & 0xffffu);
        v[3] = VoxNorm<uint16_t>::apply(r.y >> 16);
        v[4] = VoxNorm<uint16_t>::apply(r.z & 0xffffu);
        v[5] = VoxNorm<uint16_t>::apply(r.z >> 16);
        v[6] = VoxNorm<uint16_t>::apply(r.w & 0xffffu);
        v[7] = VoxNorm<uint16_t>::apply(r.w >> 16);
    }
};
template <>
struct CellRecord<uint8_t> {
    typedef uint2 type;
    // stored values as floats (no normalization)
    static __device__ __forceinline__ void raw(const uint2& r, float v[8]) {
        v[0] = (float)(r.x & 0xffu);
        v[1] = (float)((r.x >> 8) & 0xffu);
        v[2] = (float)((r.x >> 16) & 0xffu);
        v[3] = (float)(r.x >> 24);
        v[4] = (float)(r.y & 0xffu);
        v[5] = (float)((r.y >> 8) & 0xffu);
        v[6] = (float)((r.y >> 16) & 0xffu);
        v[7] = (float)(r.y >> 24);
    }
    static __device__ __forceinline__ void unpack(const uint2& r, float v[8]) {
        v[0] = VoxNorm<uint8_t>::apply(r.x & 0xffu);
        v[1] = VoxNorm<uint8_t>::apply((r.x >> 8) & 0xffu);
        v[2] = VoxNorm<uint8_t>::apply((r.x >> 16) & 0xffu);
        v[3] = VoxNorm<uint8_t>::apply(r.x >> 24);
        v[4] = VoxNorm<uint8_t>::apply(r.y & 0xffu);
        v[5] = VoxNorm<uint8_t>::apply((r.y >> 8) & 0xffu);
        v[6] = VoxNorm<uint8_t>::apply((r.y >> 16) & 0xffu);
        v[7] = VoxNorm<uint8_t>::apply(r.y >> 24);
    }
};

// Record addressing (cell_layout.h): 2x2x2 cells per group (one 128-byte
// line for uint16), groups x-fastest inside bricks of kCellBrick^3 groups,
// bricks x-fastest.
template <typename T, bool WIDE>
struct CellFetch {
    typedef typename CellRecord<T>::type rec_t;
    typedef typename std::conditional<WIDE, uint64_t, uint32_t>::type off_t;
    const rec_t* p;
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t nbx, nby;   // bricks along x and y

    __device__ __forceinline__ off_t index(const uint32_t lo[3]) const { return cell_index<off_t>(lo, nbx, nby); }
    // brick stride of axis i, in records
    __device__ __forceinline__ off_t brick_stride(int i) const {
        const off_t one = (off_t)1 << kCellBrickRecLog2;
        return i == 0 ? one : (i == 1 ? one * nbx : one * nbx * nby);
    }
    __device__ __forceinline__ rec_t load(off_t i) const {
        if constexpr (WIDE) {
            return p[i];
        } else if constexpr (sizeof(T) == 2) {
            const auto v = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (uint32_t)i * 16u, 0, 0);
            return rec_t{v[0], v[1], v[2], v[3]};
        } else {
            const auto v = __builtin_amdgcn_raw_buffer_load_b64(rsrc, (uint32_t)i * 8u, 0, 0);
            rec_t r;
            r.x = v[0];
            r.y = v[1];
            return r;
        }
    }
};

// Voxel position, corners and record index of the texture-space point s.
template <typename T, bool WIDE>
__device__ __forceinline__ typename CellFetch<T, WIDE>::off_t cell_of(const CellFetch<T, WIDE>& f,
                                                                      const MarchArgs& a, const float s[3],
                                                                      float p[3]) {
    // corners() of volumeram.cpp:79-86 on a clamped position (vp >= 0, so
    // max(vp, 0) == vp): the record holds the clamped upper corners, so only
    // the lower corner and the fraction are needed
    uint32_t lo[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float vp = tex_to_voxel(s[i], a.fdims[i], a.fdm1[i]);
        p[i] = vp - floorf(vp);
        const uint32_t l = (uint32_t)vp, m = a.dims[i] - 1;
        lo[i] = l < m ? l : m;
    }
    return f.index(lo);
}

// Central differences of six trilinear lookups at s +- one voxel per axis,
// as march_ref.hip computes them; the six loads are issued together.  RAW
// (kernels whose shading is checked by tolerance): the lookups interpolate
// the stored values and the difference is scaled once by grad_raw, equal up
// to float rounding.
template <typename T, bool WIDE, bool RAW = false>
__device__ __forceinline__ void cell_gradient(const CellFetch<T, WIDE>& f, const MarchArgs& a,
                                              const float s[3], float gr[3]) {
    typename CellFetch<T, WIDE>::rec_t rec[6];
    float p[6][3];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const int axis = k % 3;
        const float off = (k < 3) ? a.grad_off[axis] : -a.grad_off[axis];
        float q[3] = {s[0], s[1], s[2]};
        q[axis] = s[axis] + off;
        q[(axis + 1) % 3] = s[(axis + 1) % 3] + 0.0f;
        q[(axis + 2) % 3] = s[(axis + 2) % 3] + 0.0f;
        rec[k] = f.load(cell_of<T, WIDE>(f, a, q, p[k]));
    }
    float vals[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        float v[8];
        if (RAW) CellRecord<T>::raw(rec[k], v);
        else CellRecord<T>::unpack(rec[k], v);
        vals[k] = trilerp(v, p[k]);
    }
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        if (RAW) gr[i] = (vals[3 + i] - vals[i]) * a.grad_raw[i];
        else gr[i] = ((vals[3 + i] - vals[i]) * a.grad_scale[i]) * a.rwm_scale;
    }
}

// Interior central differences from the cell records at unclamped voxel
// position u: when every axis has u_i in [1, dim_i - 3) and a proper fraction, the six lookups at +-1 voxel
// have the sample's own weights p, and their footprints are the sample's
// corner planes plus the outer planes lo-1 and lo+2 (records of the cells
// lo -+ e_i).  Equal to the six-lookup form up to float rounding (for the
// kernels whose shading is checked by tolerance): the differences are taken
// in stored units and scaled once by grad_raw = grad_scale * rwm_scale /
// range, the four-term sums use fused multiply-adds, and the neighbour
// records are found from the sample's own record index `own` (its low three
// bits are the parities of lo; a step to the neighbouring group moves by the
// group stride inside a brick, else to the neighbouring brick's facing group;
// cell_layout.h).  Returns false (and leaves gr) outside the interior.
template <typename T, bool WIDE>
__device__ __forceinline__ bool cell_gradient_interior(const CellFetch<T, WIDE>& f, const MarchArgs& a,
                                                       const float u[3],
                                                       const typename CellFetch<T, WIDE>::rec_t& rec,
                                                       typename CellFetch<T, WIDE>::off_t own, const float p[3],
                                                       float gr[3]) {
    typedef typename CellFetch<T, WIDE>::off_t off_t;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        if (!(u[i] >= 1.0f) || !(u[i] + 3.0f < a.fdims[i]) || !(p[i] > 0.0f)) return false;
    }
    off_t nb[6];
#pragma unroll
    for (int i = 0; i < 3; ++i) cell_neighbours<off_t>(own, i, f.brick_stride(i), nb[i], nb[3 + i]);
    typename CellFetch<T, WIDE>::rec_t nr[6];
#pragma unroll
    for (int k = 0; k < 6; ++k) nr[k] = f.load(nb[k]);
    float v[8], m[3][8], q[3][8];
    CellRecord<T>::raw(rec, v);
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        CellRecord<T>::raw(nr[i], m[i]);
        CellRecord<T>::raw(nr[3 + i], q[i]);
    }
    const float px = p[0], py = p[1], pz = p[2];
    const float qx = 1.f - px, qy = 1.f - py, qz = 1.f - pz;
    auto dot4 = [](float a0, float a1, float a2, float a3, const float w[4]) {
        return __builtin_fmaf(a3, w[3], __builtin_fmaf(a2, w[2], __builtin_fmaf(a1, w[1], a0 * w[0])));
    };
    // (qa*bm + pa*b0) - (qa*b1 + pa*bp): the lookup at -1 voxel minus the one at +1
    auto diff = [](float qa, float pa, float bm, float b0, float b1, float bp) {
        return __builtin_fmaf(-pa, bp, __builtin_fmaf(-qa, b1, __builtin_fmaf(pa, b0, qa * bm)));
    };
    // corner order: 0 x0y0z0, 1 x1y0z0, 2 x1y1z0, 3 x0y1z0, 4 x0y0z1, 5 x1y0z1, 6 x1y1z1, 7 x0y1z1
    {
        const float w[4] = {qy * qz, py * qz, qy * pz, py * pz};
        const float bm = dot4(m[0][0], m[0][3], m[0][4], m[0][7], w);
        const float b0 = dot4(v[0], v[3], v[4], v[7], w);
        const float b1 = dot4(v[1], v[2], v[5], v[6], w);
        const float bp = dot4(q[0][1], q[0][2], q[0][5], q[0][6], w);
        gr[0] = diff(qx, px, bm, b0, b1, bp) * a.grad_raw[0];
    }
    {
        const float w[4] = {qx * qz, px * qz, qx * pz, px * pz};
        const float bm = dot4(m[1][0], m[1][1], m[1][4], m[1][5], w);
        const float b0 = dot4(v[0], v[1], v[4], v[5], w);
        const float b1 = dot4(v[3], v[2], v[7], v[6], w);
        const float bp = dot4(q[1][3], q[1][2], q[1][7], q[1][6], w);
        gr[1] = diff(qy, py, bm, b0, b1, bp) * a.grad_raw[1];
    }
    {
        const float w[4] = {qx * qy, px * qy, qx * py, px * py};
        const float bm = dot4(m[2][0], m[2][1], m[2][3], m[2][2], w);
        const float b0 = dot4(v[0], v[1], v[3], v[2], w);
        const float b1 = dot4(v[4], v[5], v[7], v[6], w);
        const float bp = dot4(q[2][4], q[2][5], q[2][7], q[2][6], w);
        gr[2] = diff(qz, pz, bm, b0, b1, bp) * a.grad_raw[2];
    }
    return true;
}

// Counters of a lane (COUNT builds); a lane marches at most 2^31 samples (the
// loop cap), sums have 64 bits.  rays, skipped and the passes are the
// ray's, alike in its P lanes; fetched and shaded are the lane's own samples.
struct RayCounters {
    uint32_t rays = 0, skipped = 0, fetched = 0, shaded = 0, passes = 0, shade_passes = 0;
};

// Adds the lanes' counters to the launch's, the wavefronts marching 64 / P rays
// with P lanes each.  Slots: samples a wavefront's rays could have taken, a
// skipped sample counting as one.  Every thread of a workgroup of 256 calls it:
// the counters lie in one line, so a workgroup adds them with one instruction.
// Counted 256^3 Phong frame, 512^2 with four lanes per ray: 559 us with an
// atomic per wavefront and counter and samples counted by every lane of a ray,
// 326 so (270 without counters).
template <int P>
__device__ __forceinline__ void add_counters(unsigned long long* c, const RayCounters& n, bool own) {
    typedef unsigned long long count_t;
    __shared__ count_t s_count[4][kNumCounters];
    count_t v[kNumCounters] = {own ? n.rays : 0, (count_t)(own ? n.skipped : 0) + n.fetched, n.fetched, n.shaded,
                               (count_t)n.passes * P + n.skipped, (count_t)n.shade_passes * P};
#pragma unroll
    for (int off = 32; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < kNumCounters; ++k) {
            const count_t o = __shfl_xor(v[k], off, 64);
            v[k] = k < 4 ? v[k] + o : (o > v[k] ? o : v[k]);
        }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < kNumCounters; ++k) s_count[threadIdx.x >> 6][k] = k < 4 ? v[k] : v[k] * (64 / P);
    }
    __syncthreads();
    if (threadIdx.x < kNumCounters) {
        count_t sum = 0;
#pragma unroll
        for (int w = 0; w < 4; ++w) sum += s_count[w][threadIdx.x];
        if (sum) atomicAdd(c + threadIdx.x, sum);
    }
}

// Lanes per ray.  P neighbouring lanes of a wavefront (2, 4 or 16)
// march one ray together: in every pass lane `sub` of the ray fetches,
// classifies and shades sample `sub` of the next P, and all P lanes then
// composite the P results in order, so each lane holds the ray's state and
// every branch of the ray is taken by its P lanes alike.  The results equal
// the one-lane march bit for bit.  A ray is one dependent chain of memory
// round trips and several hundred instructions per pass; P lanes cut it P
// times, and neighbouring lanes read neighbouring samples, mostly of one
// record group, in one load.  sub_value reads lane j's value (a move within
// the VALU, no LDS).  What that gives is in kernels.h (frame_lanes).  One
// sample per lane fits six wavefronts per SIMD but for 1 to 7 of the shaded
// kernels' registers (10 in batches): 512^3 / 1024^2 with Phong went from 1.04
// ms (two samples in flight in one lane, four wavefronts) to 0.68.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}
// value of lane j of the row of 16
__device__ __forceinline__ float row_value(float v, int j) {
    switch (j) {
        case 0: return dpp_move<0x150>(v);
        case 1: return dpp_move<0x151>(v);
        case 2: return dpp_move<0x152>(v);
        case 3: return dpp_move<0x153>(v);
        case 4: return dpp_move<0x154>(v);
        case 5: return dpp_move<0x155>(v);
        case 6: return dpp_move<0x156>(v);
        case 7: return dpp_move<0x157>(v);
        case 8: return dpp_move<0x158>(v);
        case 9: return dpp_move<0x159>(v);
        case 10: return dpp_move<0x15a>(v);
        case 11: return dpp_move<0x15b>(v);
        case 12: return dpp_move<0x15c>(v);
        case 13: return dpp_move<0x15d>(v);
        case 14: return dpp_move<0x15e>(v);
        default: return dpp_move<0x15f>(v);
    }
}
template <int P>
__device__ __forceinline__ float sub_value(float v, int j) {
    static_assert(P == 2 || P == 4 || P == 16, "lanes per ray");
    if (P == 2) return j == 0 ? dpp_move<0xA0>(v) : dpp_move<0xF5>(v);   // quad permutations
    if (P == 4) return j == 0 ? dpp_move<0x00>(v) : j == 1 ? dpp_move<0x55>(v) : j == 2 ? dpp_move<0xAA>(v)
                                                                                       : dpp_move<0xFF>(v);
    return row_value(v, j);
}
template <int P>
__device__ __forceinline__ uint32_t sub_value(uint32_t v, int j) {
    return __float_as_uint(sub_value<P>(__uint_as_float(v), j));
}

// Counts this lane's sample of a pass (COUNT builds): ca its opacity (-1: past
// the ray's end); A0 and A the ray's opacity before and after the pass.  Where
// the ray ended in the pass, the samples up to the one that ended it count.
template <int SHADE, int P>
__device__ __forceinline__ void count_pass(RayCounters& n, float ca, float A0, float A, int sub) {
    bool on = ca >= 0.0f;
    if (A >= kErtOpacity) {
        const float cz = fmaxf(ca, 0.0f);
        float before = A0;
#pragma unroll
        for (int j = 0; j < P - 1; ++j) {
            const float next = before + (1.0f - before) * sub_value<P>(cz, j);
            before = j < sub ? next : before;
        }
        on = on && before < kErtOpacity;
    }
    n.fetched += on ? 1 : 0;
    if (SHADE) n.shaded += on && ca > 0.0f ? 1 : 0;
}

// The place of a wavefront's rays in the image: 64 / P rays, ray_w<P>() wide.
template <int P>
__host__ __device__ constexpr int ray_w() { return P <= 2 ? 8 : (P == 4 ? 4 : 2); }
template <int P>
__host__ __device__ constexpr int ray_h() { return 64 / P / ray_w<P>(); }

// Takes the run of samples that starts at (t, loop) and lies before t_lim, the
// ray's end and the cap: (t, loop) becomes its last sample, the next sample's
// t is returned.  bound = fminf(t_lim, tend).
__device__ __forceinline__ float skip_run(float step, float bound, float t_lim, float tend, int cap, float& t,
                                          int& loop) {
    // most of the run in closed form; the last steps below take the
    // reference's float sequence step by step
    float d = 0.0f;
    const int j = closed_form_steps(t, step, bound, cap - loop, d);
    if (j > 0) {
        t = t + (float)j * d;
        loop += j;
    }
    float tn = t + step;
    while (tn < t_lim && !(tn > tend) && loop + 1 < cap) {
        t = tn;
        ++loop;
        tn = t + step;
    }
    return tn;
}

// The sample loop of one ray from state (t, loop, r, g, bb, A) up to sample
// index cap (exclusive) or the ray's end.  SHADE: 0 none, 1 Phong with the
// interior gradient and the hardware-approximate lighting terms (within the
// oracle's tolerance), 2 Phong bit-identical to the reference-layout kernel.
// s_tf / s_alpha are the TF and the opacity-correction table in LDS; a may
// live in kernel arguments or in global memory (batched launches).  `sub` is
// this lane's place among the ray's P lanes.
//
// The skip grid is asked only after a pass that composited nothing: inside
// visible matter there is nothing to skip, and the grid's byte is a memory
// round trip ahead of the sample's own.
template <typename T, bool WIDE, int SHADE, bool COUNT, int P>
__device__ __forceinline__ void cell_march(const MarchArgs& a, const CellFetch<T, WIDE>& f, const uint32_t* s_tf,
                                           const float* s_alpha, int px, int py, int sub, const float first[3],
                                           const float dir[3], float tend, int cap, float& t, int& loop, float& r,
                                           float& g, float& bb, float& A, RayCounters& n) {
    typedef typename CellFetch<T, WIDE>::rec_t rec_t;
    const uint32_t bl = a.skip_log2;
    uint32_t cur_brick = 0xffffffffu;
    uint32_t empty = 0;   // the skip grid's entry of the current brick
    float t_lim = 0.0f;
    // reciprocals for the empty-brick bound (a bound with a 0.05-voxel
    // margin needs no correctly rounded quotient); an axis with |dir| below
    // 1e-30 cannot move 0.05 voxel within a ray and bounds nothing
    float rdir[3], rfd[3];
    // a degenerate ray (its direction or start is not a number): the clamps
    // below map its positions into the volume, its intensities are NaN
    bool nan_ray = false;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        rdir[i] = fabsf(dir[i]) < 1e-30f ? 0.0f : __builtin_amdgcn_rcpf(dir[i]);
        rfd[i] = __builtin_amdgcn_rcpf(a.fdims[i]);
        nan_ray = nan_ray || !(fabsf(dir[i]) < INFINITY) || first[i] != first[i];
    }
    bool probe = true, finished = false;
    while (!finished && loop < cap) {
        // this lane's sample and the next pass's first
        float tm = t, t_next = t;
#pragma unroll
        for (int j = 1; j < P; ++j) {
            t_next = t_next + a.step;
            tm = sub == j ? t_next : tm;
        }
        t_next = t_next + a.step;
        float s[3], u[3], vp[3];
        uint32_t lo[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            s[i] = first[i] + tm * dir[i];
            u[i] = (a.fdims[i] * s[i]) + (-0.5f);
            vp[i] = __builtin_amdgcn_fmed3f(u[i], 0.0f, a.fdm1[i]);   // tex_to_voxel of a number
            lo[i] = (uint32_t)vp[i];                                  // <= dims - 1
        }
        if (probe) {
            uint32_t b[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) b[i] = sub_value<P>(lo[i], 0) >> bl;   // the pass's first sample
            const uint32_t brick = cell_mul24(cell_mul24(b[2], a.nskip[1]) + b[1], a.nskip[0]) + b[0];
            if (brick != cur_brick) {
                cur_brick = brick;
                empty = nan_ray ? a.nan_empty : a.skip[brick];
                if (empty) t_lim = empty_box_limit_rcp(a.nskip, first, rdir, rfd, b, bl, empty);
            }
            if (empty) {
                // every sample at t' < t_lim lies in empty bricks: only the
                // count and the float sequence t += step remain
                const int loop0 = loop;
                const float tn = skip_run(a.step, fminf(t_lim, tend), t_lim, tend, cap, t, loop);
                ++loop;
                t = tn;
                finished = t > tend;
                if (COUNT) n.skipped += (uint32_t)(loop - loop0);
                continue;
            }
        }
        // ca: the sample's corrected opacity; -1 past the ray's end or the cap
        float ca = -1.0f, col[3] = {0.f, 0.f, 0.f};
        if (sub == 0 || (!(tm > tend) && loop + sub < cap)) {
            float p[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) p[i] = vp[i] - floorf(vp[i]);
            const typename CellFetch<T, WIDE>::off_t own = f.index(lo);
            const rec_t rec = f.load(own);
            float v[8];
            CellRecord<T>::unpack(rec, v);
            const float inten = nan_ray ? NAN : trilerp(v, p);
            const uint32_t c8 = s_tf[tf_index(inten, a)];
            ca = s_alpha[c8 >> 24];
            if (ca > 0.0f) {
                col[0] = byte_norm(c8 & 0xffu);
                col[1] = byte_norm((c8 >> 8) & 0xffu);
                col[2] = byte_norm((c8 >> 16) & 0xffu);
                if (SHADE) {
                    float gr[3], pos[3];
                    if (tm == 0.0f) clip_border_gradient(a, px, py, s, dir, gr);
                    else if (SHADE == 2 || nan_ray) cell_gradient<T, WIDE>(f, a, s, gr);
                    else if (!cell_gradient_interior<T, WIDE>(f, a, u, rec, own, p, gr))
                        cell_gradient<T, WIDE, true>(f, a, s, gr);
                    if (SHADE == 2) {
#pragma unroll
                        for (int i = 0; i < 3; ++i)
                            pos[i] = (((s[i] * a.fdims[i]) - 0.5f) * a.spacing[i]) + a.offset[i];
                        shade_model(a, gr, pos, col);
                    } else {
#pragma unroll
                        for (int i = 0; i < 3; ++i) pos[i] = __builtin_fmaf(u[i], a.spacing[i], a.offset[i]);
                        phong_fast(a, gr, pos, col);
                    }
                }
            }
        }
        if (COUNT) {
            ++n.passes;
            if (SHADE) n.shade_passes += (__ballot(ca > 0.0f) != 0ull) ? 1 : 0;
        }
        // the ray's lanes composite the pass's samples in order.  A terminated
        // ray has A = 1, so later samples weigh zero and a sample of alpha 0
        // changes nothing: no branches, unless a colour is not a finite
        // number (degenerate lighting), which a zero weight would not keep out
        const float A0 = A;
        if (SHADE && __any(!(fabsf((col[0] + col[1]) + col[2]) < INFINITY))) {
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const float cj = sub_value<P>(ca, j);
                const float c0 = sub_value<P>(col[0], j), c1 = sub_value<P>(col[1], j), c2 = sub_value<P>(col[2], j);
                if (cj > 0.0f && A < kErtOpacity) {
                    const float wgt = (1.0f - A) * cj;
                    r = r + wgt * c0;
                    g = g + wgt * c1;
                    bb = bb + wgt * c2;
                    A = A + wgt;
                    A = A >= kErtOpacity ? 1.0f : A;
                }
            }
        } else {
            const float cz = fmaxf(ca, 0.0f);
#pragma unroll
            for (int j = 0; j < P; ++j) {
                const float wgt = (1.0f - A) * sub_value<P>(cz, j);
                r = r + wgt * sub_value<P>(col[0], j);
                g = g + wgt * sub_value<P>(col[1], j);
                bb = bb + wgt * sub_value<P>(col[2], j);
                A = A + wgt;
                A = A >= kErtOpacity ? 1.0f : A;
            }
        }
        if (COUNT) count_pass<SHADE, P>(n, ca, A0, A, sub);
        probe = A == A0;
        loop += P;
        t = t_next;
        finished = A >= kErtOpacity || t > tend;
    }
}

// One ray of the cell march from entry point e to exit point l (neither the
// background): returns the composited RGBA (in each of the ray's P lanes).
template <typename T, bool WIDE, int SHADE, bool COUNT, int P>
__device__ __forceinline__ float4 cell_ray(const MarchArgs& a, const CellFetch<T, WIDE>& f, const uint32_t* s_tf,
                                           const float* s_alpha, int px, int py, int sub, float4 e, float4 l,
                                           RayCounters& n) {
    ++n.rays;
    const float first[3] = {e.x, e.y, e.z};
    const float last[3] = {l.x, l.y, l.z};
    float dir[3];
    const float tend = ray_setup(first, last, a.step, dir);
    float t = 0.0f, r = 0.f, g = 0.f, bb = 0.f, A = 0.f;
    int loop = 0;   // samples taken (the reference loop counter)
    cell_march<T, WIDE, SHADE, COUNT, P>(a, f, s_tf, s_alpha, px, py, sub, first, dir, tend, a.loop_cap, t, loop, r, g,
                                         bb, A, n);
    return make_float4(r, g, bb, A);
}

// Cell-record addressing of the volume in a (buffer descriptor when narrow).
template <typename T, bool WIDE>
__device__ __forceinline__ CellFetch<T, WIDE> cell_fetch_of(const MarchArgs& a) {
    typedef typename CellFetch<T, WIDE>::rec_t rec_t;
    CellFetch<T, WIDE> f;
    f.p = (const rec_t*)a.cells;
    f.nbx = cell_bricks(a.dims[0]);
    f.nby = cell_bricks(a.dims[1]);
    if (!WIDE) {
        const uint32_t dims[3] = {a.dims[0], a.dims[1], a.dims[2]};
        const uint32_t bytes = (uint32_t)(cell_record_count(dims) * sizeof(rec_t));
        f.rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a.cells, (short)0, (int)bytes, 0x00020000);
    }
    return f;
}

}  // namespace hipdvr
