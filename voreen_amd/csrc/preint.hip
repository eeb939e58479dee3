// preint.hip -- pre-integration tables built on the device.
//
// PreIntegrationTable::computeTable (src/core/datastructures/transfunc/1d/
// preintegrationtable.cpp:67-204), both variants: the exact variant composites the TF from sf to sb with the opacity
// correction exponent step*200/(|sb-sf|+1) and early termination at 0.95,
// then un-premultiplies; the integral variant differences prefix sums
// (alpha = 1 - exp(-dA*step*200/ds)).  The TF colours per table index and the
// integral prefix sums are made on the host in the reference's float order
// (hipdvr_preint_build, tf.cpp); the device evaluates pow/exp with its own
// library functions (within an ulp of the host's).
#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "../../include/hipdvr.h"
#include "ctx.h"
#include "errors.h"
#include "objects.h"

namespace hipdvr {

namespace {

__device__ __forceinline__ float dmaxf(float a, float b) { return (a < b) ? b : a; }
__device__ __forceinline__ float dminf(float a, float b) { return (b < a) ? b : a; }
__device__ __forceinline__ float clamp01(float v) { return dminf(dmaxf(v, 0.f), 1.f); }

// Entries of one lane: the diagonals' entries at kRun neighbouring sf.
constexpr int kRun = 4;

// Place of TF entry s in LDS: lanes kRun entries apart read different banks
// (16-byte entries, sixteen to a row of 64 banks).
__device__ __forceinline__ int lds_slot(int s) { return (s & ~3) | ((s + (s >> 4)) & 3); }

// One entry's compositing step: nothing once its alpha has passed 0.95.  The
// reference compares the float alpha with the double 0.95
// (preintegrationtable.cpp:115); 0.95f < 0.95 < the next float up, so that
// test is a <= 0.95f, without double arithmetic.  A zero weight keeps every
// finite sum as it is.  The colour sums are fused; alpha, which decides where
// an entry ends, takes the reference's roundings.
__device__ __forceinline__ void entry_step(float e[4], const float4 c) {
    const float w = e[3] <= 0.95f ? (1.0f - e[3]) * c.w : 0.0f;
    e[0] = __builtin_fmaf(w, c.x, e[0]);
    e[1] = __builtin_fmaf(w, c.y, e[1]);
    e[2] = __builtin_fmaf(w, c.z, e[2]);
    e[3] = e[3] + w;
}

// The d + 1 steps of the entries sf0 .. sf0 + kRun - 1 (DIR 1: to sb = sf + d,
// -1: to sf - d).  A sample read for one entry is the next step's of its
// neighbour, so each step reads one; the samples of the next four steps are on
// their way while four are taken.  Reads past either end stay in the table
// (any entry of it) and belong to entries that are not stored.
template <int DIR>
__device__ __forceinline__ void diagonal_run(const float4* s_tf, int n, int sf0, int d, float e[kRun][4]) {
    static_assert(kRun == 4, "the ring below");
    const uint32_t last = (((uint32_t)n + 3) & ~3u) - 1;
    auto at = [&](int s) { return s_tf[min((uint32_t)lds_slot(s), last)]; };
    // the run's first sample in marching direction comes first; entry j's
    // sample of step k is the (k + j)-th of the run
    const int s0 = DIR > 0 ? sf0 : sf0 + kRun - 1;
#pragma unroll
    for (int j = 0; j < kRun; ++j)
#pragma unroll
        for (int c = 0; c < 4; ++c) e[j][c] = 0.f;
    int k = 0;
    if (d + 1 >= 12) {
        float4 ring[12];   // sample q in ring[q % 12]
#pragma unroll
        for (int q = 0; q < 7; ++q) ring[q] = at(s0 + DIR * q);
        for (; k + 12 <= d + 1; k += 12) {
#pragma unroll
            for (int g = 0; g < 12; g += 4) {
#pragma unroll
                for (int q = g + 7; q < g + 11; ++q) ring[q % 12] = at(s0 + DIR * (k + q));
#pragma unroll
                for (int u = g; u < g + 4; ++u)
#pragma unroll
                    for (int j = 0; j < kRun; ++j) entry_step(e[j], ring[(u + j) % 12]);
            }
            bool done = true;
#pragma unroll
            for (int j = 0; j < kRun; ++j) done = done && !(e[j][3] <= 0.95f);
            if (done) return;
        }
    }
    for (; k <= d; ++k)
#pragma unroll
        for (int j = 0; j < kRun; ++j) entry_step(e[j], at(s0 + DIR * (k + j)));
}

// Exact variant, one workgroup per diagonal d = |sb - sf|.  The corrected
// opacity of a TF entry depends on the entry and on d alone, so a diagonal
// needs n powers instead of one per entry and step, and the entries of a lane
// share their samples: n^3/3 steps of eight operations and a quarter of an LDS
// read remain (1024^2: 184 us; one power per entry and step took 772, this
// split without the reads ahead and fused sums 294).
// Longest chains first; four neighbouring diagonals, whose entries share
// 64-byte pieces of the table, go to the same XCD one after another.
__global__ __launch_bounds__(256) void preint_exact_kernel(const float4* __restrict__ tfb, int n, float step,
                                                           float4* __restrict__ table) {
    extern __shared__ float4 s_tf[];
    const int slot = blockIdx.x / 8;
    const int r = ((slot / 4) * 8 + blockIdx.x % 8) * 4 + slot % 4;
    if (r >= n) return;
    const int d = n - 1 - r;
    if (d == 0) {
        for (int sf = threadIdx.x; sf < n; sf += 256) {
            const float4 cc = tfb[sf];
            table[(size_t)sf * n + sf] = make_float4(clamp01(cc.x), clamp01(cc.y), clamp01(cc.z),
                                                     1.f - powf(1.f - clamp01(cc.w), step * 200.0f));
        }
        return;
    }
    const float scale = 1.0f / ((float)d + 1);
    const float ex = step * 200.0f * scale;
    for (int s = threadIdx.x; s < n; s += 256) {
        float4 cc = tfb[s];
        cc.w = cc.w > 0.0f ? 1.f - powf(1.f - cc.w, ex) : 0.0f;
        s_tf[lds_slot(s)] = cc;
    }
    __syncthreads();
    const int runs = (n - d + kRun - 1) / kRun;
    for (int i = threadIdx.x; i < 2 * runs; i += 256) {
        const bool down = i >= runs;   // entries with sb < sf
        const int sf0 = (down ? i - runs : i) * kRun + (down ? d : 0);
        float e[kRun][4];
        if (down) diagonal_run<-1>(s_tf, n, sf0, d, e);
        else diagonal_run<1>(s_tf, n, sf0, d, e);
#pragma unroll
        for (int j = 0; j < kRun; ++j) {
            const int sf = down ? sf0 + kRun - 1 - j : sf0 + j;
            const int sb = down ? sf - d : sf + d;
            if (sf >= n || sb >= n) continue;
            const float den = dmaxf(e[j][3], 0.001f);
            table[(size_t)sb * n + sf] =
                make_float4(clamp01(e[j][0] / den), clamp01(e[j][1] / den), clamp01(e[j][2] / den), clamp01(e[j][3]));
        }
    }
}

__global__ __launch_bounds__(256) void preint_integral_kernel(const float4* __restrict__ tfb,
                                                              const float4* __restrict__ intf, int n, float step,
                                                              float4* __restrict__ table) {
    const int sf = blockIdx.x * blockDim.x + threadIdx.x;
    const int sb = blockIdx.y;
    if (sf >= n) return;
    const int smin = sb < sf ? sb : sf;
    const int smax = sb < sf ? sf : sb;
    float col[4];
    if (smax != smin) {
        const float factor = step * 200.f / (float)(smax - smin);
        const float4 hi = intf[smax], lo = intf[smin];
        col[0] = (hi.x - lo.x) * factor;
        col[1] = (hi.y - lo.y) * factor;
        col[2] = (hi.z - lo.z) * factor;
        col[3] = 1.f - expf(-(hi.w - lo.w) * factor);
        const float den = dmaxf(col[3], 0.001f);
        for (int c = 0; c < 3; ++c) col[c] /= den;
    } else {
        const float4 cc = tfb[smin];
        col[0] = cc.x;
        col[1] = cc.y;
        col[2] = cc.z;
        col[3] = 1.f - powf(1.f - cc.w, step * 200.0f);
    }
    table[(size_t)sb * n + sf] = make_float4(clamp01(col[0]), clamp01(col[1]), clamp01(col[2]), clamp01(col[3]));
}

}  // namespace

}  // namespace hipdvr

using namespace hipdvr;

extern "C" int hipdvr_tf_preint_device(hipdvr_tf* tf, const hipdvr_tf_key* keys, int32_t nkeys, float gamma,
                                       float thr_lo, float thr_hi, int32_t alpha_mode, uint32_t n, float step,
                                       int32_t use_integral) {
    if (!tf) return HIPDVR_ERR_INVALID;
    return ctx_guarded(tf->ctx, [&] {
        if (n < 2 || n > 4096 || !(step > 0.f) || nkeys < 0 || (nkeys > 0 && !keys))
            fail(HIPDVR_ERR_INVALID, "bad pre-integration arguments");
        // TF colours per table index: the host builder's first stage
        std::vector<float> tfb((size_t)n * 4);
        if (!preint_index_colors(keys, nkeys, gamma, thr_lo, thr_hi, alpha_mode, n, tfb.data()))
            fail(HIPDVR_ERR_INVALID, "invalid transfer-function keys");
        std::vector<float> intf;
        if (use_integral) {
            intf.assign((size_t)n * 4, 0.f);
            float acc[4] = {0.f, 0.f, 0.f, 0.f};
            for (uint32_t i = 0; i < n; ++i) {
                const float* cc = &tfb[4 * (size_t)i];
                if (cc[3] > 0.0f) {
                    acc[0] += cc[0] * cc[3];
                    acc[1] += cc[1] * cc[3];
                    acc[2] += cc[2] * cc[3];
                    acc[3] += cc[3];
                }
                for (int c = 0; c < 4; ++c) intf[4 * (size_t)i + c] = acc[c];
            }
        }
        ctx_set_device(tf->ctx);
        hipStream_t st = ctx_stream(tf->ctx);
        hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
        // the table, with the colours (and prefix sums) behind it
        float4* d_tab = nullptr;
        try {
            hip_check(hipMalloc((void**)&d_tab, ((size_t)n * n + (use_integral ? 2 : 1) * (size_t)n) * sizeof(float4)),
                      "hipMalloc(preint)");
            float4* d_tfb = d_tab + (size_t)n * n;
            hip_check(hipMemcpyAsync(d_tfb, tfb.data(), (size_t)n * sizeof(float4), hipMemcpyHostToDevice, st),
                      "upload");
            const dim3 grid((n + 255) / 256, n);
            if (use_integral) {
                float4* d_int = d_tfb + n;
                hip_check(hipMemcpyAsync(d_int, intf.data(), (size_t)n * sizeof(float4), hipMemcpyHostToDevice, st),
                          "upload");
                hipLaunchKernelGGL(preint_integral_kernel, grid, dim3(256), 0, st, d_tfb, d_int, (int)n, step, d_tab);
            } else {
                const unsigned groups = (n + 31) / 32;   // of eight times four diagonals
                const size_t lds = (((size_t)n + 3) & ~(size_t)3) * sizeof(float4);   // lds_slot stays within four
                hipLaunchKernelGGL(preint_exact_kernel, dim3(groups * 32), dim3(256), lds, st, d_tfb, (int)n, step,
                                   d_tab);
            }
            hip_check(hipGetLastError(), "pre-integration kernel launch");
            hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
        } catch (...) {
            if (d_tab) (void)hipFree(d_tab);
            throw;
        }
        if (tf->d_preint) (void)hipFree(tf->d_preint);
        tf->d_preint = d_tab;
        tf->preint_n = n;
        tf->preint_serial = next_serial();
    });
}
