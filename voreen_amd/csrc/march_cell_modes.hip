// march_cell_modes.hip -- the compositing modes other than DVR and the
// pre-integrated classification on the cell records, several lanes per ray
// (march_cell.h): linear filter, central differences.
//
// The reference-layout kernels (march_ref.hip) read eight voxels per sample
// and reconstruct every sample of every ray; their results are these kernels'
// to the bit, since positions, sums, lookups and the order of compositing are
// the same.  What is left out contributes nothing:
//   modes   samples of alpha 0 composite nothing in any mode: the exact skip
//           grid of the DVR march serves them all.  MIP also passes bricks
//           whose largest value does not exceed the ray's maximum so far, and
//           lights only samples above it; ISO lights only samples in its band.
//   preint  the table pairs a sample with the one before it; a brick is
//           skipped when every entry that pairs an index of its own range with
//           one of its 3^3 neighbourhood's range has alpha 0.
//           The run's last sample is reconstructed again, for its index.
// What bounds them is what bounds the DVR march: record loads and the chain of
// the longest rays.  Whole frames, reference-layout kernel / this one, us:
// 512x512x361 u16 MIP 1024^2 5222 / 831; 301x257x199 u8 isosurface with Phong
// 811x613 3825 / 291; 381x255x317 u16 pre-integrated (256) 1019x763 1635 / 372.
#include <cmath>

#include "kernels.h"
#include "march_cell.h"
#include "march_common.h"

namespace hipdvr {

namespace {

// What one lane's sample gives the compositing of its ray.
struct ModeSample {
    float alpha;    // alpha composited; -1: nothing to composite, -2: past the ray's end
    float rw;       // real-world intensity
    float c[3];     // colour, position (FHP) or normal (FHN)
};

// Classifies (and lights) this lane's sample: mod_compositing.frag's inputs.
template <typename T, bool WIDE, bool GRAD>
__device__ __forceinline__ void mode_sample(const MarchArgs& a, const CellFetch<T, WIDE>& f, const uint32_t* s_tf,
                                            const float* s_alpha, int mode, int px, int py, const float s[3],
                                            const float dir[3], float tm, float inten, float max_int, float max_alpha,
                                            ModeSample& m, bool& shaded) {
    const uint32_t c8 = s_tf[tf_index(inten, a)];
    const float al = byte_norm(c8 >> 24);
    m.alpha = -1.0f;
    m.rw = (inten * a.rwm_scale) + a.rwm_offset;
    if (!(al > 0.0f)) return;
    shaded = GRAD && a.shade_model != kShadeNone;
    // a sample that the ray's state before the pass already rules out is not lit
    if (mode == kCompMIP && !(m.rw > max_int)) return;
    if (mode == kCompMOP && !(al > max_alpha)) return;
    if (mode == kCompISO && !(al >= a.iso_value - 0.02f && al <= a.iso_value + 0.02f)) return;
    m.alpha = mode == kCompMIDA ? s_alpha[c8 >> 24] : al;
    if (mode == kCompFHP) {
#pragma unroll
        for (int i = 0; i < 3; ++i) m.c[i] = s[i];
        return;
    }
    m.c[0] = byte_norm(c8 & 0xffu);
    m.c[1] = byte_norm((c8 >> 8) & 0xffu);
    m.c[2] = byte_norm((c8 >> 16) & 0xffu);
    if (GRAD) {
        float gr[3];
        if (tm == 0.0f) clip_border_gradient(a, px, py, s, dir, gr);
        else cell_gradient<T, WIDE>(f, a, s, gr);
        if (mode == kCompFHN) {
            const float l2 = gr[0] * gr[0] + gr[1] * gr[1] + gr[2] * gr[2];
            const float rl = l2 > 0.f ? 1.0f / sqrtf(l2) : 0.f;
#pragma unroll
            for (int i = 0; i < 3; ++i) m.c[i] = ((gr[i] * rl) / 2.0f) + 0.5f;
        } else if (a.shade_model != kShadeNone) {
            float pos[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) pos[i] = (((s[i] * a.fdims[i]) - 0.5f) * a.spacing[i]) + a.offset[i];
            shade_model(a, gr, pos, m.c);
        }
    }
}

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

// One sample taken into the ray's result (mod_compositing.frag:85-213).  (The
// reference-layout kernel has these steps written out in its loop: through a
// shared function it ran 2 to 5% slower.)
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

// Brick of voxel lo on a grid of nb bricks of 2^bl voxels.
__device__ __forceinline__ uint32_t brick_of(const uint32_t lo[3], const uint32_t nb[3], uint32_t bl, uint32_t b[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) b[i] = lo[i] >> bl;
    return cell_mul24(cell_mul24(b[2], nb[1]) + b[1], nb[0]) + b[0];
}

// The index of the sample before lane sub's: the lane below, or `carry`.
template <int P>
__device__ __forceinline__ int previous_index(int idx, int carry, int sub) {
    const float v = __int_as_float(idx);
    const int below = __float_as_int(P == 4 ? dpp_move<0x90>(v) : dpp_move<0x111>(v));   // quad 0,0,1,2; row shift 1
    return sub == 0 ? carry : below;
}

// GRAD: a gradient may be needed (lighting or FHN); its registers leave four
// wavefronts per SIMD, without it six.
template <typename T, bool WIDE, bool PREINT, bool GRAD, bool COUNT, int P>
__global__ __launch_bounds__(256, GRAD ? 4 : 6) void march_modes_cell_kernel(const MarchArgs a, const uint32_t tiles_x,
                                                                             const uint32_t tiles_y) {
    const uint32_t block = linear_block(), slot = block / kXcds, part = slot % P;
    uint32_t tile_x, tile_y;
    if (!xcd_tile((slot / P) * kXcds + block % kXcds, tiles_x, tiles_y, tile_x, tile_y)) return;
    __shared__ uint32_t s_tf[PREINT ? 1 : kMaxTfWidth];
    __shared__ float s_alpha[PREINT ? 1 : 256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, ray = lane / P, sub = lane % P;
    constexpr int RW = ray_w<P>(), RH = ray_h<P>(), PX = 16 / (2 * RW);
    const int px = (int)tile_x * 16 + ((int)(part % PX) * 2 + (wave & 1)) * RW + ray % RW;
    const int py = (int)tile_y * 16 + ((int)(part / PX) * 2 + (wave >> 1)) * RH + ray / RW;
    const bool inside = px < a.w && py < a.h;
    const size_t pix = (size_t)py * a.w + px;
    float4 e = make_float4(0.f, 0.f, 0.f, 0.f), l = e;
    if (inside) {
        e = a.entry[pix];
        l = a.exit[pix];
    }
    const bool hit = !is_background(e, l);
    float out[4] = {0.f, 0.f, 0.f, 0.f};
    RayCounters n;
    if (__syncthreads_or(hit)) {
        if (!PREINT) {
            for (int i = tid; i < a.tf_width; i += 256) s_tf[i] = a.tf[i];
            s_alpha[tid] = a.alpha_corr[tid];
        }
        __syncthreads();
        if (hit) {
            n.rays = 1;
            const CellFetch<T, WIDE> f = cell_fetch_of<T, WIDE>(a);
            const int mode = a.compositing;
            const bool ert = PREINT || mode == kCompISO || mode == kCompFHP || mode == kCompFHN;
            // (the counters hold every sample that a light would have reached)
            const bool mip = !PREINT && mode == kCompMIP && !(COUNT && GRAD);
            const float first[3] = {e.x, e.y, e.z}, last[3] = {l.x, l.y, l.z};
            float dir[3];
            const float tend = ray_setup(first, last, a.step, dir);
            const int cap = a.loop_cap;
            float rdir[3], rfd[3];
            bool nan_ray = false;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                rdir[i] = fabsf(dir[i]) < 1e-30f ? 0.0f : __builtin_amdgcn_rcpf(dir[i]);
                rfd[i] = __builtin_amdgcn_rcpf(a.fdims[i]);
                nan_ray = nan_ray || !(fabsf(dir[i]) < INFINITY) || first[i] != first[i];
            }
            float t = 0.0f, max_int = 0.0f;
            int loop = 0, carry = 0;   // carry: table index of the sample before the pass (last_x = 0 at first)
            uint32_t cur = 0xffffffffu, empty = 0;
            float t_lim = 0.0f;
            // PREINT: the first sample pairs with index 0, in no brick's range
            // a degenerate ray's positions say nothing about its samples
            const bool skips = a.skip && !nan_ray;
            bool probe = skips && !PREINT, ghost = false, finished = false;
            float top = INFINITY;   // MIP: no sample of the current brick lies above
            while (!finished && loop < cap) {
                float tm = t, t_next = t;
#pragma unroll
                for (int j = 1; j < P; ++j) {
                    t_next = t_next + a.step;
                    tm = sub == j ? t_next : tm;
                }
                t_next = t_next + a.step;
                float s[3], vp[3];
                uint32_t lo[3];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    s[i] = first[i] + tm * dir[i];
                    vp[i] = __builtin_amdgcn_fmed3f((a.fdims[i] * s[i]) + (-0.5f), 0.0f, a.fdm1[i]);
                    lo[i] = (uint32_t)vp[i];
                }
                if (probe) {
                    uint32_t l0[3], b[3];
#pragma unroll
                    for (int i = 0; i < 3; ++i) l0[i] = sub_value<P>(lo[i], 0);   // the pass's first sample
                    const uint32_t brick = brick_of(l0, a.nskip, a.skip_log2, b);
                    if (brick != cur) {
                        cur = brick;
                        empty = a.skip[brick];
                        if (mip) {   // the brick's range, widened as the skip grid's
                            const uint2 mm = a.skip_minmax[brick];
                            const float lo_n = VoxNorm<T>::apply(mm.x) - 1e-5f, hi_n = VoxNorm<T>::apply(mm.y) + 1e-5f;
                            top = fmaxf((lo_n * a.rwm_scale) + a.rwm_offset, (hi_n * a.rwm_scale) + a.rwm_offset);
                        }
                        if (empty || mip)
                            t_lim = empty_box_limit_rcp(a.nskip, first, rdir, rfd, b, a.skip_log2, empty ? empty : 1);
                    }
                    const bool skip = empty != 0 || (mip && top <= max_int);
                    if (skip) {
                        const int loop0 = loop;
                        const float tn = skip_run(a.step, fminf(t_lim, tend), t_lim, tend, cap, t, loop);
                        finished = tn > tend;
                        if (PREINT && !finished && loop + 1 < cap) {
                            ghost = true;   // march on from the run's last sample, for its index
                            probe = false;
                        } else {
                            ++loop;
                            t = tn;
                        }
                        if (COUNT) n.skipped += (uint32_t)(loop - loop0);
                        continue;
                    }
                }
                ModeSample m;
                m.alpha = -2.0f;
                m.rw = 0.0f;
                m.c[0] = m.c[1] = m.c[2] = 0.0f;
                bool shaded = false;
                const bool mine = sub == 0 || (!(tm > tend) && loop + sub < cap);
                float inten = 0.0f;
                int idx = 0;
                if (mine) {
                    float p[3], v[8];
#pragma unroll
                    for (int i = 0; i < 3; ++i) p[i] = vp[i] - floorf(vp[i]);
                    CellRecord<T>::unpack(f.load(f.index(lo)), v);
                    inten = nan_ray ? NAN : trilerp(v, p);
                    if (PREINT) idx = preint_index(norm_rw(inten, a), a.preint_n);
                }
                if (PREINT) {
                    const int before = previous_index<P>(idx, carry, sub);
                    if (mine) {
                        const float4 c = a.preint[(size_t)idx * a.preint_n + before];
                        m.alpha = (ghost && sub == 0) || !(c.w > 0.0f) ? -1.0f : c.w;
                        m.c[0] = c.x;
                        m.c[1] = c.y;
                        m.c[2] = c.z;
                        if (GRAD && m.alpha >= 0.0f) {
                            float gr[3], pos[3];
                            if (tm == 0.0f) clip_border_gradient(a, px, py, s, dir, gr);
                            else cell_gradient<T, WIDE>(f, a, s, gr);
#pragma unroll
                            for (int i = 0; i < 3; ++i)
                                pos[i] = (((s[i] * a.fdims[i]) - 0.5f) * a.spacing[i]) + a.offset[i];
                            shade_model(a, gr, pos, m.c);
                            shaded = true;
                        }
                    }
                    carry = (int)sub_value<P>((uint32_t)idx, P - 1);
                } else if (mine) {
                    mode_sample<T, WIDE, GRAD>(a, f, s_tf, s_alpha, mode, px, py, s, dir, tm, inten, max_int, out[3], m,
                                               shaded);
                }
                ghost = false;
                // the ray's lanes composite the pass's samples in order
                probe = skips;
                if (COUNT || __any(m.alpha >= 0.0f)) {
#pragma unroll
                    for (int j = 0; j < P; ++j) {
                        const float aj = sub_value<P>(m.alpha, j);
                        const float c[3] = {sub_value<P>(m.c[0], j), sub_value<P>(m.c[1], j), sub_value<P>(m.c[2], j)};
                        const float rj = PREINT ? 0.0f : sub_value<P>(m.rw, j);
                        if (!(aj >= -1.0f) || finished) continue;
                        if (COUNT && sub == j) {
                            ++n.fetched;
                            n.shaded += shaded ? 1 : 0;
                        }
                        if (!(aj >= 0.0f)) continue;
                        probe = mip && skips;   // MIP: the bricks ahead may lie below the new maximum
                        if (PREINT) {
                            const float wgt = (1.0f - out[3]) * aj;
                            out[0] = out[0] + wgt * c[0];
                            out[1] = out[1] + wgt * c[1];
                            out[2] = out[2] + wgt * c[2];
                            out[3] = out[3] + (1.0f - out[3]) * aj;
                        } else {
                            mode_composite(a, mode, rj, c, aj, out, max_int);
                        }
                        if (ert && out[3] >= kErtOpacity) {
                            out[3] = 1.0f;
                            finished = true;
                        }
                    }
                }
                if (COUNT) ++n.passes;
                loop += P;
                t = t_next;
                finished = finished || (t > tend);
            }
        }
    }
    if (inside && sub == 0) a.out[pix] = make_float4(out[0], out[1], out[2], out[3]);
    if (COUNT) add_counters<P>(a.counters, n, sub == 0);
}

template <typename T, bool WIDE, bool PREINT, bool GRAD, bool COUNT>
void launch_p(const MarchArgs& a, int lanes, hipStream_t st) {
    const uint32_t tx = (a.w + 15) / 16, ty = (a.h + 15) / 16;
    const uint64_t blocks = xcd_tile_grid(tx, ty);
    if (lanes == 16)
        hipLaunchKernelGGL((march_modes_cell_kernel<T, WIDE, PREINT, GRAD, COUNT, 16>), linear_grid(blocks * 16),
                           dim3(256), 0, st, a, tx, ty);
    else
        hipLaunchKernelGGL((march_modes_cell_kernel<T, WIDE, PREINT, GRAD, COUNT, 4>), linear_grid(blocks * 4),
                           dim3(256), 0, st, a, tx, ty);
}

template <typename T, bool WIDE, bool PREINT>
void launch_g(const MarchArgs& a, bool grad, bool count, int lanes, hipStream_t st) {
    if (grad) {
        if (count) launch_p<T, WIDE, PREINT, true, true>(a, lanes, st);
        else launch_p<T, WIDE, PREINT, true, false>(a, lanes, st);
    } else {
        if (count) launch_p<T, WIDE, PREINT, false, true>(a, lanes, st);
        else launch_p<T, WIDE, PREINT, false, false>(a, lanes, st);
    }
}

template <bool PREINT>
void launch_m(const MarchArgs& a, int dtype, bool wide, bool grad, bool count, int lanes, hipStream_t st) {
    if (dtype == 0) {
        if (wide) launch_g<uint8_t, true, PREINT>(a, grad, count, lanes, st);
        else launch_g<uint8_t, false, PREINT>(a, grad, count, lanes, st);
    } else {
        if (wide) launch_g<uint16_t, true, PREINT>(a, grad, count, lanes, st);
        else launch_g<uint16_t, false, PREINT>(a, grad, count, lanes, st);
    }
}

}  // namespace

void launch_march_cell_modes(const MarchArgs& a, int dtype, bool wide, bool preint, bool shaded, bool count, int batch,
                             hipStream_t st) {
    const int lanes = frame_lanes(batch, (uint64_t)a.w * a.h, a.step) == 16 ? 16 : 4;
    if (preint) launch_m<true>(a, dtype, wide, shaded, count, lanes, st);
    else launch_m<false>(a, dtype, wide, shaded || a.compositing == kCompFHN, count, lanes, st);
}

}  // namespace hipdvr
