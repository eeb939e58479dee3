// mlp.hip -- the per-brick stepping network: 16 -> 64 -> 64 -> 2, GELU,
// BF16 weights, FP32 accumulation on MFMA (v_mfma_f32_16x16x16_bf16).
//
// One wavefront handles tiles of 16 rows.  For a 16x16x16 MFMA the operand
// layout is: A[m][k] lives in lane m + 16*(k/4), element k%4; B[k][n] in lane
// n + 16*(k/4), element k%4; the accumulator D[m][n] in lane n + 16*(m/4),
// element m%4.  Activations go through LDS between layers to move from the
// accumulator layout to the A layout.
//
// Parameters (FP32 master copy, flat): W1[16][64] b1[64] W2[64][64] b2[64]
// W3[64][2] b3[2]; the kernels read BF16 copies of W1, W2, W3 (W3 padded to
// 64x16 with zero columns) that every update writes with the master (pack_param).
//
// Loss per row (targets t0 in {0,1}, t1 in [0,3], weight t2):
//   BCE-with-logits(y0, t0) + t2 * (y1 - t1)^2, averaged over the batch.
#include <hip/hip_runtime.h>

#include "mlp.h"

namespace hipdvr {

typedef __attribute__((ext_vector_type(4))) float f4;
typedef __attribute__((ext_vector_type(4))) short s4;

__device__ __forceinline__ short f2bf(float x) {
    const uint32_t u = __float_as_uint(x);
    const uint32_t r = ((u >> 16) & 1u) + 0x7fffu;   // round to nearest even
    return (short)((u + r) >> 16);
}
__device__ __forceinline__ float bf2f(short b) { return __uint_as_float(((uint32_t)(uint16_t)b) << 16); }

// GELU (erf form).
__device__ __forceinline__ float gelu(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }
__device__ __forceinline__ f4 mfma(s4 a, s4 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, c, 0, 0, 0);
}

// Shared weights of one workgroup (BF16) and biases.
struct MlpShared {
    short w1[kMlpIn * kMlpHidden];        // [16][64]
    short w2[kMlpHidden * kMlpHidden];    // [64][64]
    short w3[kMlpHidden * 16];            // [64][16] (columns >= 2 are zero)
    float b1[kMlpHidden], b2[kMlpHidden], b3[16];
};

// Per-wave scratch: activations of the 16-row tile.
struct WaveTile {
    short x[16 * kMlpIn];       // input rows (bf16)
    short h1[16 * kMlpHidden];  // GELU(z1) (bf16)
    short h2[16 * kMlpHidden];  // GELU(z2) (bf16)
};

__device__ void load_shared(MlpShared& sh, const MlpDevParams& p) {
    for (int i = threadIdx.x; i < kMlpIn * kMlpHidden; i += blockDim.x) sh.w1[i] = p.w1[i];
    for (int i = threadIdx.x; i < kMlpHidden * kMlpHidden; i += blockDim.x) sh.w2[i] = p.w2[i];
    for (int i = threadIdx.x; i < kMlpHidden * 16; i += blockDim.x) sh.w3[i] = p.w3[i];
    for (int i = threadIdx.x; i < kMlpHidden; i += blockDim.x) {
        sh.b1[i] = p.b[i];
        sh.b2[i] = p.b[kMlpHidden + i];
    }
    for (int i = threadIdx.x; i < 16; i += blockDim.x) sh.b3[i] = i < kMlpOut ? p.b[2 * kMlpHidden + i] : 0.f;
}

// Forward pass of one 16-row tile whose inputs are already in t.x.
// Returns y0/y1 of the lane's rows in y (lanes with n = lane%16 < 2 hold
// output column n for rows 4*(lane/16) .. +3).
__device__ void tile_forward(const MlpShared& sh, WaveTile& t, f4& y) {
    const int lane = threadIdx.x & 63;
    const int n0 = lane & 15, kq = (lane >> 4) * 4;
    // layer 1: [16x16] x [16x64]
    s4 a;
    for (int i = 0; i < 4; ++i) a[i] = t.x[n0 * kMlpIn + kq + i];
    for (int nt = 0; nt < 4; ++nt) {
        s4 b;
        for (int i = 0; i < 4; ++i) b[i] = sh.w1[(kq + i) * kMlpHidden + nt * 16 + n0];
        f4 acc = {0.f, 0.f, 0.f, 0.f};
        acc = mfma(a, b, acc);
        for (int i = 0; i < 4; ++i) {
            const int row = kq + i, col = nt * 16 + n0;
            const float z = acc[i] + sh.b1[col];
            t.h1[row * kMlpHidden + col] = f2bf(gelu(z));
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    // layer 2: [16x64] x [64x64]
    for (int nt = 0; nt < 4; ++nt) {
        f4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int kc = 0; kc < 4; ++kc) {
            s4 aa, b;
            for (int i = 0; i < 4; ++i) {
                aa[i] = t.h1[n0 * kMlpHidden + kc * 16 + kq + i];
                b[i] = sh.w2[(kc * 16 + kq + i) * kMlpHidden + nt * 16 + n0];
            }
            acc = mfma(aa, b, acc);
        }
        for (int i = 0; i < 4; ++i) {
            const int row = kq + i, col = nt * 16 + n0;
            const float z = acc[i] + sh.b2[col];
            t.h2[row * kMlpHidden + col] = f2bf(gelu(z));
        }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
    // layer 3: [16x64] x [64x16]
    f4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int kc = 0; kc < 4; ++kc) {
        s4 aa, b;
        for (int i = 0; i < 4; ++i) {
            aa[i] = t.h2[n0 * kMlpHidden + kc * 16 + kq + i];
            b[i] = sh.w3[(kc * 16 + kq + i) * 16 + n0];
        }
        acc = mfma(aa, b, acc);
    }
    for (int i = 0; i < 4; ++i) y[i] = acc[i] + sh.b3[n0];
}

// Load 16 input rows (zero rows past `rows`) into the tile as BF16.
__device__ void tile_load_x(WaveTile& t, const float* x, uint32_t row0, uint32_t rows) {
    const int lane = threadIdx.x & 63;
    for (int e = lane; e < 16 * kMlpIn; e += 64) {
        const uint32_t r = row0 + e / kMlpIn;
        t.x[e] = f2bf(r < rows ? x[(size_t)r * kMlpIn + e % kMlpIn] : 0.f);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_wave_barrier();
}

__global__ __launch_bounds__(256) void mlp_forward_kernel(MlpDevParams p, const float* __restrict__ x,
                                                          uint32_t rows, float* __restrict__ y) {
    __shared__ MlpShared sh;
    __shared__ WaveTile tiles[4];
    load_shared(sh, p);
    __syncthreads();
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    WaveTile& t = tiles[wave];
    const uint32_t ntiles = (rows + 15) / 16;
    for (uint32_t tile = blockIdx.x * 4 + wave; tile < ntiles; tile += gridDim.x * 4) {
        tile_load_x(t, x, tile * 16, rows);
        f4 out;
        tile_forward(sh, t, out);
        const int n0 = lane & 15, kq = (lane >> 4) * 4;
        if (n0 < kMlpOut)
            for (int i = 0; i < 4; ++i) {
                const uint32_t r = tile * 16 + kq + i;
                if (r < rows) y[(size_t)r * kMlpOut + n0] = out[i];
            }
        __builtin_amdgcn_wave_barrier();
    }
}

// Value of lane j of the lane's row of 16.
template <int J>
__device__ __forceinline__ float row_lane(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + J, 0xf, 0xf, true));
}

// GELU of z rounded to BF16, and its derivative (one erf for both).
__device__ __forceinline__ short gelu_both(float z, float& grad) {
    const float e = 1.0f + erff(z * 0.70710678118654752f);
    const float pdf = 0.39894228040143268f * expf(-0.5f * z * z);
    grad = 0.5f * e + z * pdf;
    return f2bf(0.5f * z * e);
}

// Forward + backward over the batch: the workgroup's sums of dL/dparam and of
// the loss.
//
// A tile of 16 rows is a chain of small products and GELUs (a batch has only a
// few tiles per compute unit), so its length bounds the kernel: the four
// wavefronts share each tile, wavefront w the hidden units 16w .. 16w+15.
// In the accumulator layout a lane holds four rows of one unit, which is also
// the operand layout of the products over rows (dW1, dW2): those operands, the
// weights (packed in operand order), z's derivatives and the sums stay in
// registers, and only h1, h2 and dZ2 pass through LDS.  The sums are stored
// per workgroup and added by the update kernel.  8192 rows: 14 us; with one
// atomic addition per wavefront and parameter and a tile per wavefront 51.
constexpr int kRowPad = kMlpHidden + 8;   // shorts: 8-byte reads down the rows meet no bank twice

__global__ __launch_bounds__(256) void mlp_grad_kernel(const MlpDevParams p, const float* __restrict__ x,
                                                       const float* __restrict__ tgt, uint32_t rows, float inv_batch,
                                                       float* __restrict__ partial) {
    __shared__ __align__(8) short s_h1[16 * kRowPad], s_h2[16 * kRowPad], s_dz[16 * kRowPad];
    __shared__ s4 s_dzf[4][64];   // dZ2 as the operand of dW2
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int n0 = lane & 15, kg = lane >> 4, kq = kg * 4, col = wave * 16 + n0;
    const s4* frag = (const s4*)p.frag;
    const s4 w1 = frag[wave * 64 + lane];
    s4 w2[4], w2t[4], w3[4];
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) {
        w2[kc] = frag[256 + (wave * 4 + kc) * 64 + lane];
        w2t[kc] = frag[256 + 1024 + (wave * 4 + kc) * 64 + lane];
        w3[kc] = s4{0, 0, 0, 0};
        if (n0 < kMlpOut) w3[kc] = frag[256 + 2048 + (kc * 4 + kg) * kMlpOut + n0];
    }
    const float b1 = p.b[col], b2 = p.b[kMlpHidden + col], b3 = n0 < kMlpOut ? p.b[2 * kMlpHidden + n0] : 0.f;
    const float w30 = bf2f(p.w3[col * 16]), w31 = bf2f(p.w3[col * 16 + 1]);
    const f4 zero = {0.f, 0.f, 0.f, 0.f};
    f4 gw1 = zero, gw2[4] = {zero, zero, zero, zero};
    float gb1 = 0.f, gb2 = 0.f, gb3 = 0.f, gw3[2] = {0.f, 0.f}, lsum = 0.f;
    const uint32_t ntiles = (rows + 15) / 16;
    for (uint32_t tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        s4 xa, xt;   // rows as the operand of layer 1, and of dW1
        float t0[4], t2[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t ra = tile * 16 + n0, rt = tile * 16 + kq + i;
            xa[i] = f2bf(ra < rows ? x[(size_t)ra * kMlpIn + kq + i] : 0.f);
            xt[i] = f2bf(rt < rows ? x[(size_t)rt * kMlpIn + n0] : 0.f);
            t0[i] = t2[i] = 0.f;
            if (n0 < kMlpOut && rt < rows) {
                t0[i] = tgt[(size_t)rt * kMlpTargets + n0];
                t2[i] = tgt[(size_t)rt * kMlpTargets + 2];
            }
        }
        s4 h1, h2;
        float g1[4], g2[4];
        f4 acc = mfma(xa, w1, zero);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h1[i] = gelu_both(acc[i] + b1, g1[i]);
            s_h1[(kq + i) * kRowPad + col] = h1[i];
        }
        __syncthreads();
        acc = zero;
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) acc = mfma(*(const s4*)&s_h1[n0 * kRowPad + kc * 16 + kq], w2[kc], acc);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h2[i] = gelu_both(acc[i] + b2, g2[i]);
            s_h2[(kq + i) * kRowPad + col] = h2[i];
        }
        __syncthreads();
        acc = zero;   // every wavefront takes the two outputs
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) acc = mfma(*(const s4*)&s_h2[n0 * kRowPad + kc * 16 + kq], w3[kc], acc);
        float d[4] = {0.f, 0.f, 0.f, 0.f};   // dL/dy: lanes 0 and 1 of a row of 16
        if (n0 < kMlpOut)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float y = acc[i] + b3;
                if (tile * 16 + kq + i >= rows) continue;
                if (n0 == 0) {
                    const float s = 1.f / (1.f + expf(-y));
                    d[i] = s - t0[i];
                    lsum += fmaxf(y, 0.f) - y * t0[i] + log1pf(expf(-fabsf(y)));
                } else {
                    const float e = y - t0[i];
                    d[i] = 2.f * t2[i] * e;
                    lsum += t2[i] * e * e;
                }
                d[i] = d[i] * inv_batch;
                gb3 += d[i];
            }
        s4 dz2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float d0 = row_lane<0>(d[i]), d1 = row_lane<1>(d[i]);
            const float h = bf2f(h2[i]);
            gw3[0] += h * d0;
            gw3[1] += h * d1;
            const float dz = (d0 * w30 + d1 * w31) * g2[i];
            gb2 += dz;
            dz2[i] = f2bf(dz);
            s_dz[(kq + i) * kRowPad + col] = dz2[i];
        }
        s_dzf[wave][lane] = dz2;
        __syncthreads();
        // dW2[k][j] += sum_r h1[r][k] dz2[r][j]   (M = k, N = j, K = r)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) gw2[nt] = mfma(h1, s_dzf[nt][lane], gw2[nt]);
        // dH1[r][k] = sum_j dz2[r][j] W2[k][j]   (M = r, N = k, K = j)
        acc = zero;
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) acc = mfma(*(const s4*)&s_dz[n0 * kRowPad + kc * 16 + kq], w2t[kc], acc);
        s4 dz1;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float dz = acc[i] * g1[i];
            gb1 += dz;
            dz1[i] = f2bf(dz);
        }
        // dW1[f][k] += sum_r x[r][f] dz1[r][k]   (M = f, N = k, K = r)
        gw1 = mfma(xt, dz1, gw1);
        // the next tile writes s_h1, s_h2 and s_dz one barrier or more after
        // this tile's last read of each
    }
    // sums over the four groups of rows
    auto over_groups = [](float v) {
        v += __shfl_xor(v, 16, 64);
        return v + __shfl_xor(v, 32, 64);
    };
    gb1 = over_groups(gb1);
    gb2 = over_groups(gb2);
    gb3 = over_groups(gb3);
    gw3[0] = over_groups(gw3[0]);
    gw3[1] = over_groups(gw3[1]);
    for (int off = 32; off > 0; off >>= 1) lsum += __shfl_xor(lsum, off, 64);
    float* gW1 = partial + (size_t)blockIdx.x * kMlpPartial;
    float* gB1 = gW1 + kMlpIn * kMlpHidden;
    float* gW2 = gB1 + kMlpHidden;
    float* gB2 = gW2 + kMlpHidden * kMlpHidden;
    float* gW3 = gB2 + kMlpHidden;
    float* gB3 = gW3 + kMlpHidden * kMlpOut;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        gW1[(kq + i) * kMlpHidden + col] = gw1[i];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) gW2[(wave * 16 + kq + i) * kMlpHidden + nt * 16 + n0] = gw2[nt][i];
    }
    if (kg == 0) {
        gB1[col] = gb1;
        gB2[col] = gb2;
        gW3[col * kMlpOut] = gw3[0];
        gW3[col * kMlpOut + 1] = gw3[1];
        if (wave == 0 && n0 < kMlpOut) gB3[n0] = gb3;
        if (wave == 0 && n0 == 0) gB3[kMlpOut] = lsum * inv_batch;
    }
}

// Writes parameter i's packed copies: FP32 biases, BF16 weights row by row
// (W3 padded to 16 columns) and in operand order: of the K x N matrix a
// product multiplies by, tile (nt, kc) of 16 x 16 holds for lane n + 16*(k/4)
// elements k%4 (W1; W2; W2 transposed, for dH1; W3's two columns).
__device__ __forceinline__ void pack_param(int i, float w, const MlpDevParams& p) {
    constexpr int H = kMlpHidden;
    auto tile = [](int k, int n) { return (((n >> 4) * 4 + (k >> 4)) * 64 + ((k >> 2) & 3) * 16 + (n & 15)) * 4 + (k & 3); };
    if (i < kMlpIn * H) {
        const int k = i / H, n = i % H;
        p.w1[i] = f2bf(w);
        p.frag[((n >> 4) * 64 + (k >> 2) * 16 + (n & 15)) * 4 + (k & 3)] = f2bf(w);
        return;
    }
    i -= kMlpIn * H;
    if (i < H) {
        p.b[i] = w;
        return;
    }
    i -= H;
    if (i < H * H) {
        const int k = i / H, n = i % H;
        p.w2[i] = f2bf(w);
        p.frag[kMlpIn * H + tile(k, n)] = f2bf(w);
        p.frag[kMlpIn * H + H * H + tile(n, k)] = f2bf(w);
        return;
    }
    i -= H * H;
    if (i < H) {
        p.b[H + i] = w;
        return;
    }
    i -= H;
    if (i < H * kMlpOut) {
        const int k = i / kMlpOut, n = i % kMlpOut;
        p.w3[k * 16 + n] = f2bf(w);
        p.frag[kMlpIn * H + 2 * H * H + ((k >> 2) * kMlpOut + n) * 4 + (k & 3)] = f2bf(w);
        return;
    }
    p.b[2 * H + i - H * kMlpOut] = w;
}

// Sums the workgroups' gradients, 32 parameters per workgroup, eight lanes to
// a parameter; ADAM: the step on the FP32 master parameters and the packed
// copies with it.  One launch (4.7 us) for what were two fills, the step and the
// packing (18 us); it reads the partial sums once (5.5 MB at 256 workgroups).
template <bool ADAM>
__global__ __launch_bounds__(256) void mlp_update_kernel(const float* __restrict__ partial, uint32_t blocks,
                                                         float* __restrict__ grad, float* __restrict__ loss,
                                                         float* __restrict__ w, float* __restrict__ m,
                                                         float* __restrict__ v, const MlpDevParams p, float lr,
                                                         float b1, float b2, float eps, float c1, float c2) {
    __shared__ float s_sum[8][32];
    const int c = threadIdx.x & 31, part = threadIdx.x >> 5, i = blockIdx.x * 32 + c;
    float sum = 0.f;
    if (i <= kMlpParams)
#pragma unroll 8
        for (uint32_t b = part; b < blocks; b += 8) sum += partial[(size_t)b * kMlpPartial + i];
    s_sum[part][c] = sum;
    __syncthreads();
    if (part != 0 || i > kMlpParams) return;
    float gi = s_sum[0][c];
#pragma unroll
    for (int k = 1; k < 8; ++k) gi += s_sum[k][c];
    if (i == kMlpParams) {
        *loss = gi;
        return;
    }
    grad[i] = gi;
    if (!ADAM) return;
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    w[i] = wi;
    pack_param(i, wi, p);
}

__global__ void mlp_pack_kernel(const float* __restrict__ w, MlpDevParams p) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < kMlpHidden * 16 && i % 16 >= kMlpOut) p.w3[i] = 0;
    if (i < kMlpParams) pack_param(i, w[i], p);
}

void launch_mlp_pack(const float* master, const MlpDevParams& p, hipStream_t st) {
    hipLaunchKernelGGL(mlp_pack_kernel, dim3((kMlpParams + 255) / 256), dim3(256), 0, st, master, p);
}

void launch_mlp_forward(const MlpDevParams& p, const float* x, uint32_t rows, float* y, hipStream_t st) {
    const uint32_t ntiles = (rows + 15) / 16;
    uint32_t blocks = (ntiles + 3) / 4;
    if (blocks > 2048) blocks = 2048;
    if (blocks == 0) return;
    hipLaunchKernelGGL(mlp_forward_kernel, dim3(blocks), dim3(256), 0, st, p, x, rows, y);
}

uint32_t launch_mlp_grad(const MlpDevParams& p, const float* x, const float* tgt, uint32_t rows, float* partial,
                         hipStream_t st) {
    const uint32_t ntiles = (rows + 15) / 16;
    const uint32_t blocks = ntiles < kMlpGradBlocks ? ntiles : kMlpGradBlocks;
    if (blocks)
        hipLaunchKernelGGL(mlp_grad_kernel, dim3(blocks), dim3(256), 0, st, p, x, tgt, rows, 1.0f / (float)rows, partial);
    return blocks;
}

void launch_mlp_sum(const float* partial, uint32_t blocks, float* grad, float* loss, hipStream_t st) {
    hipLaunchKernelGGL(mlp_update_kernel<false>, dim3((kMlpParams + 1 + 31) / 32), dim3(256), 0, st, partial, blocks, grad,
                       loss, nullptr, nullptr, nullptr, MlpDevParams{}, 0.f, 0.f, 0.f, 0.f, 1.f, 1.f);
}

void launch_mlp_update(const float* partial, uint32_t blocks, float* grad, float* loss, float* w, float* m, float* v,
                       const MlpDevParams& p, float lr, int step, hipStream_t st) {
    const float b1 = 0.9f, b2 = 0.999f;
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(mlp_update_kernel<true>, dim3((kMlpParams + 1 + 31) / 32), dim3(256), 0, st, partial, blocks, grad,
                       loss, w, m, v, p, lr, b1, b2, 1e-8f, c1, c2);
}

}  // namespace hipdvr
