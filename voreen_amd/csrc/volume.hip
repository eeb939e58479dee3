// volume.hip -- volume upload: linear copy, 4^3-block tiled copy, brick
// min/max, and the per-TF brick occupancy used for exact empty-space skipping.
#include <hip/hip_runtime.h>

#include <string>

#include "cell_layout.h"
#include "errors.h"
#include "march_common.h"
#include "volume.h"

namespace hipdvr {

namespace {

// One lane per tiled element: gather from the linear copy (clamped), write
// the tiled copy contiguously.
// (Grid-stride: the element count of an 8 GiB volume reaches 2^32, beyond
// what one dispatch addresses.)
template <typename T>
__global__ __launch_bounds__(256) void tile_kernel(const T* __restrict__ src, T* __restrict__ dst,
                                                   uint32_t X, uint32_t Y, uint32_t Z, uint32_t nbx,
                                                   uint32_t nby, uint64_t total) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        const uint32_t in = (uint32_t)(i & 63);
        const uint64_t blk = i >> 6;
        const uint32_t bx = (uint32_t)(blk % nbx);
        const uint64_t r = blk / nbx;
        const uint32_t by = (uint32_t)(r % nby);
        const uint32_t bz = (uint32_t)(r / nby);
        uint32_t x = bx * 4 + (in & 3), y = by * 4 + ((in >> 2) & 3), z = bz * 4 + (in >> 4);
        x = x < X ? x : X - 1;
        y = y < Y ? y : Y - 1;
        z = z < Z ? z : Z - 1;
        dst[i] = src[((uint64_t)z * Y + y) * X + x];
    }
}

// Workgroups of a grid-stride launch: one per per_block items, at most 2^20.
inline unsigned stride_grid(uint64_t items, uint64_t per_block = 256) {
    const uint64_t want = (items + per_block - 1) / per_block;
    const uint64_t cap = 1ull << 20;
    return (unsigned)(want < 1 ? 1 : (want < cap ? want : cap));
}

// One workgroup per brick (grid-stride over the bricks): min/max over
// [b*B, b*B + B] per axis, clamped.
template <typename T>
__global__ __launch_bounds__(256) void minmax_kernel(const T* __restrict__ src, uint2* __restrict__ mm,
                                                     uint32_t X, uint32_t Y, uint32_t Z, uint32_t bl,
                                                     uint32_t nbx, uint32_t nby, uint64_t nbricks) {
    for (uint64_t b64 = blockIdx.x; b64 < nbricks; b64 += gridDim.x) {
        const uint32_t b = (uint32_t)b64;
        const uint32_t bx = b % nbx, by = (b / nbx) % nby, bz = b / (nbx * nby);
        const uint32_t B1 = (1u << bl) + 1;
        const uint32_t n = B1 * B1 * B1;
        uint32_t lo = 0xffffffffu, hi = 0;
        for (uint32_t k = threadIdx.x; k < n; k += blockDim.x) {
            uint32_t x = (bx << bl) + k % B1;
            uint32_t y = (by << bl) + (k / B1) % B1;
            uint32_t z = (bz << bl) + k / (B1 * B1);
            x = x < X ? x : X - 1;
            y = y < Y ? y : Y - 1;
            z = z < Z ? z : Z - 1;
            const uint32_t v = src[((uint64_t)z * Y + y) * X + x];
            lo = v < lo ? v : lo;
            hi = v > hi ? v : hi;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const uint32_t l2 = __shfl_xor(lo, off, 64), h2 = __shfl_xor(hi, off, 64);
            lo = l2 < lo ? l2 : lo;
            hi = h2 > hi ? h2 : hi;
        }
        __shared__ uint32_t s_lo[4], s_hi[4];
        const int w = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 0) {
            s_lo[w] = lo;
            s_hi[w] = hi;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int i = 1; i < (int)(blockDim.x >> 6); ++i) {
                lo = s_lo[i] < lo ? s_lo[i] : lo;
                hi = s_hi[i] > hi ? s_hi[i] : hi;
            }
            mm[b] = make_uint2(lo, hi);
        }
        __syncthreads();   // s_lo / s_hi are rewritten for the next brick
    }
}

// Ranges of 8^3 bricks (plus the upper one-voxel apron): a workgroup takes 32
// bricks of a brick row, lane i the voxels of column 256*bx + i over the 9 x 9
// rows (coalesced; the last column of the apron by one more load of lane 0's
// wave), then one lane per brick folds its 9 columns from LDS.  Each voxel is
// read 1.27 times.
template <typename T>
__global__ __launch_bounds__(256) void minmax8_kernel(const T* __restrict__ src, uint2* __restrict__ mm, uint32_t X,
                                                      uint32_t Y, uint32_t Z, uint32_t nbx, uint32_t nby,
                                                      uint32_t groups_x, uint64_t groups) {
    __shared__ uint32_t s_lo[257], s_hi[257];
    for (uint64_t gr = blockIdx.x; gr < groups; gr += gridDim.x) {
        const uint32_t gx = (uint32_t)(gr % groups_x);
        const uint64_t row = gr / groups_x;
        const uint32_t by = (uint32_t)(row % nby), bz = (uint32_t)(row / nby);
        for (uint32_t c = threadIdx.x; c < 257; c += 256) {
            const uint32_t xc = gx * 256 + c, x = xc < X ? xc : X - 1;
            uint32_t lo = 0xffffffffu, hi = 0;
            for (uint32_t dz = 0; dz < 9; ++dz) {
                const uint32_t zc = bz * 8 + dz, z = zc < Z ? zc : Z - 1;
#pragma unroll
                for (uint32_t dy = 0; dy < 9; ++dy) {
                    const uint32_t yc = by * 8 + dy, y = yc < Y ? yc : Y - 1;
                    const uint32_t v = src[((uint64_t)z * Y + y) * X + x];
                    lo = v < lo ? v : lo;
                    hi = v > hi ? v : hi;
                }
            }
            s_lo[c] = lo;
            s_hi[c] = hi;
        }
        __syncthreads();
        const uint32_t bx = gx * 32 + threadIdx.x;
        if (threadIdx.x < 32 && bx < nbx) {
            uint32_t lo = 0xffffffffu, hi = 0;
            for (uint32_t k = 0; k < 9; ++k) {
                const uint32_t l2 = s_lo[threadIdx.x * 8 + k], h2 = s_hi[threadIdx.x * 8 + k];
                lo = l2 < lo ? l2 : lo;
                hi = h2 > hi ? h2 : hi;
            }
            mm[((uint64_t)bz * nby + by) * nbx + bx] = make_uint2(lo, hi);
        }
        __syncthreads();   // the columns are rewritten for the next group
    }
}

// Ranges of bricks of 8 * 2^s voxels per edge from those of the 8^3 bricks
// (the apron of the last child is the brick's).
__global__ __launch_bounds__(256) void minmax_fold_kernel(const uint2* __restrict__ mm8, uint2* __restrict__ mm,
                                                          uint32_t n8x, uint32_t n8y, uint32_t n8z, uint32_t s,
                                                          uint32_t nbx, uint32_t nby, uint64_t count) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; b < count; b += stride) {
        const uint32_t bx = (uint32_t)(b % nbx), by = (uint32_t)((b / nbx) % nby), bz = (uint32_t)(b / nbx / nby);
        uint32_t lo = 0xffffffffu, hi = 0;
        for (uint32_t z = bz << s; z < ((bz + 1) << s) && z < n8z; ++z)
            for (uint32_t y = by << s; y < ((by + 1) << s) && y < n8y; ++y)
                for (uint32_t x = bx << s; x < ((bx + 1) << s) && x < n8x; ++x) {
                    const uint2 v = mm8[((uint64_t)z * n8y + y) * n8x + x];
                    lo = v.x < lo ? v.x : lo;
                    hi = v.y > hi ? v.y : hi;
                }
        mm[b] = make_uint2(lo, hi);
    }
}

// One lane per record: the 8 footprint voxels of cell (x, y, z), clamped.
// Records in the order of cell_layout.h; cells of the padding hold zeros.
template <typename T>
__global__ __launch_bounds__(256) void cells_kernel(const T* __restrict__ src, void* __restrict__ dst, uint32_t X,
                                                    uint32_t Y, uint32_t Z, uint64_t total) {
    const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
    const uint32_t dims[3] = {X, Y, Z};
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += stride) {
        uint32_t c[3];
        cell_of_record(i, dims, c);
        const uint32_t x = c[0], y = c[1], z = c[2];
        uint32_t v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        if (x < X && y < Y && z < Z) {
            const uint32_t x1 = x + 1 < X ? x + 1 : X - 1;
            const uint32_t y1 = y + 1 < Y ? y + 1 : Y - 1;
            const uint32_t z1 = z + 1 < Z ? z + 1 : Z - 1;
            const uint64_t XY = (uint64_t)X * Y;
            const uint64_t b0 = (uint64_t)z * XY, b1 = (uint64_t)z1 * XY;
            // trilinear order: llB lrB urB ulB llF lrF urF ulF
            v[0] = src[b0 + (uint64_t)y * X + x];
            v[1] = src[b0 + (uint64_t)y * X + x1];
            v[2] = src[b0 + (uint64_t)y1 * X + x1];
            v[3] = src[b0 + (uint64_t)y1 * X + x];
            v[4] = src[b1 + (uint64_t)y * X + x];
            v[5] = src[b1 + (uint64_t)y * X + x1];
            v[6] = src[b1 + (uint64_t)y1 * X + x1];
            v[7] = src[b1 + (uint64_t)y1 * X + x];
        }
        if (sizeof(T) == 2) {
            ((uint4*)dst)[i] = make_uint4(v[0] | (v[1] << 16), v[2] | (v[3] << 16), v[4] | (v[5] << 16),
                                          v[6] | (v[7] << 16));
        } else {
            ((uint2*)dst)[i] = make_uint2(v[0] | (v[1] << 8) | (v[2] << 16) | (v[3] << 24),
                                          v[4] | (v[5] << 8) | (v[6] << 16) | (v[7] << 24));
        }
    }
}

template <typename T>
void build_layouts(hipdvr_volume* v, hipStream_t st) {
    const uint32_t X = v->desc.dims[0], Y = v->desc.dims[1], Z = v->desc.dims[2];
    const uint64_t total = v->tiled_elems;
    hipLaunchKernelGGL(tile_kernel<T>, dim3(stride_grid(total)), dim3(256), 0, st,
                       (const T*)v->d_linear, (T*)v->d_tiled, X, Y, Z, v->nblocks[0], v->nblocks[1],
                       total);
    hip_check(hipGetLastError(), "tile kernel launch");
    const uint32_t gx = (v->nskip[0] + 31) / 32;
    const uint64_t groups = (uint64_t)gx * v->nskip[1] * v->nskip[2];
    hipLaunchKernelGGL(minmax8_kernel<T>, dim3(stride_grid(groups, 1)), dim3(256), 0, st, (const T*)v->d_linear,
                       v->d_minmax8, X, Y, Z, v->nskip[0], v->nskip[1], gx, groups);
    hip_check(hipGetLastError(), "min/max kernel launch");
    launch_brick_minmax(v, v->desc.brick_log2, v->nbricks, v->d_minmax, st);
    hip_check(hipGetLastError(), "min/max kernel launch");
}

__device__ __forceinline__ float norm_raw(uint32_t v, int dtype) {
    return dtype == 0 ? VoxNorm<uint8_t>::apply(v) : VoxNorm<uint16_t>::apply(v);
}

__device__ __forceinline__ int map_index(float n, const OccArgs& a) {
    const float rw = (n * a.rwm_scale) + a.rwm_offset;
    const float x = rw_to_norm(rw, a.dom_lo, a.dom_hi);
    const int w1 = a.tf_width - 1;
    const int idx = iround_tgt(x * (float)w1);
    return idx < 0 ? 0 : (idx > w1 ? w1 : idx);
}

// Table indices that samples of raw range mm may take, one more to each side.
__device__ __forceinline__ void index_range(const OccArgs& a, uint2 mm, int& i0, int& i1) {
    const float n0 = norm_raw(mm.x, a.dtype) - 1e-5f;
    const float n1 = norm_raw(mm.y, a.dtype) + 1e-5f;
    i0 = map_index(n0, a);
    i1 = map_index(n1, a);
    if (i0 > i1) {
        const int t = i0;
        i0 = i1;
        i1 = t;
    }
    i0 = i0 > 0 ? i0 - 1 : 0;
    i1 = i1 < a.tf_width - 1 ? i1 + 1 : a.tf_width - 1;
}

// Whether a brick of raw range mm may hold alpha > 0.
__device__ __forceinline__ bool brick_occupied(const OccArgs& a, uint2 mm) {
    int i0, i1;
    index_range(a, mm, i0, i1);
    return (a.alpha_prefix[i1 + 1] - a.alpha_prefix[i0]) != 0u;
}

__global__ __launch_bounds__(256) void occupancy_kernel(const OccArgs a) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.count) a.occ[i] = brick_occupied(a, a.minmax[i]) ? 1 : 0;
}

// The same for the pairs of a pre-integration table: brick (x, y, z) of the
// grid nb.
__device__ __forceinline__ bool brick_pairs_occupied(const OccArgs& a, const uint32_t nb[3], uint32_t x, uint32_t y,
                                                     uint32_t z) {
    uint32_t lo = 0xffffffffu, hi = 0;
    for (uint32_t k = z > 0 ? z - 1 : 0; k <= z + 1 && k < nb[2]; ++k)
        for (uint32_t j = y > 0 ? y - 1 : 0; j <= y + 1 && j < nb[1]; ++j)
            for (uint32_t i = x > 0 ? x - 1 : 0; i <= x + 1 && i < nb[0]; ++i) {
                const uint2 v = a.minmax[((uint64_t)k * nb[1] + j) * nb[0] + i];
                lo = v.x < lo ? v.x : lo;
                hi = v.y > hi ? v.y : hi;
            }
    int i0, i1;
    index_range(a, make_uint2(lo, hi), i0, i1);
    return a.pair_reach[i0] <= (uint32_t)i1;
}

// The skip grid in three passes, one per axis: the Chebyshev distance to the
// nearest occupied brick is the minimum over k of max(|k|, distance within
// the row k bricks away), taken axis after axis.  Pass 1 classifies 256
// bricks of an x row and their neighbours into LDS and writes the distance
// within the row.
template <bool PAIRS>
__global__ __launch_bounds__(256) void skip_x_kernel(const OccArgs a, uint8_t* __restrict__ out, uint32_t nbx,
                                                     uint32_t nby, uint32_t nbz, uint32_t parts, uint64_t groups) {
    constexpr int R = (int)kSkipReach;
    const uint32_t nb[3] = {nbx, nby, nbz};
    __shared__ uint8_t s_occ[256 + 2 * R];
    for (uint64_t gr = blockIdx.x; gr < groups; gr += gridDim.x) {
        const uint64_t row = gr / parts;
        const int x0 = (int)(gr % parts) * 256;
        const uint2* mm = a.minmax + row * nbx;
        for (int i = (int)threadIdx.x; i < 256 + 2 * R; i += 256) {
            const int x = x0 + i - R;
            bool occ = x >= 0 && x < (int)nbx;
            if (occ) {
                if constexpr (PAIRS) occ = brick_pairs_occupied(a, nb, x, (uint32_t)(row % nby), (uint32_t)(row / nby));
                else occ = brick_occupied(a, mm[x]);
            }
            s_occ[i] = occ ? 1 : 0;
        }
        __syncthreads();
        const int x = x0 + (int)threadIdx.x;
        if (x < (int)nbx) {
            int d = 0;
            while (d < R && !s_occ[threadIdx.x + R - d] && !s_occ[threadIdx.x + R + d]) ++d;
            out[row * nbx + x] = (uint8_t)d;
        }
        __syncthreads();   // the classes are rewritten for the next group
    }
}

// Passes 2 and 3: n bricks along the axis, `stride` bytes apart.
__global__ __launch_bounds__(256) void skip_axis_kernel(const uint8_t* __restrict__ in, uint8_t* __restrict__ out,
                                                        uint64_t stride, uint32_t n, uint64_t count) {
    const uint64_t step = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += step) {
        const int c = (int)((i / stride) % n);
        int d = in[i];
        for (int k = 1; k < d; ++k) {
            if (c - k >= 0) d = min(d, max(k, (int)in[i - (uint64_t)k * stride]));
            if (c + k < (int)n) d = min(d, max(k, (int)in[i + (uint64_t)k * stride]));
        }
        out[i] = (uint8_t)d;
    }
}

// One workgroup: inclusive scan of v over its 1024 lanes (s: 1024 words).
template <bool MIN>
__device__ __forceinline__ uint32_t block_scan(uint32_t v, uint32_t* s) {
    const int tid = threadIdx.x;
    s[tid] = v;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        const uint32_t o = tid >= off ? s[tid - off] : (MIN ? 0xffffffffu : 0u);
        __syncthreads();
        v = MIN ? (o < v ? o : v) : v + o;
        s[tid] = v;
        __syncthreads();
    }
    return v;
}

// One workgroup, four entries per lane: width <= 4096.
__global__ __launch_bounds__(1024) void iso_prefix_kernel(const uint32_t* __restrict__ rgba, uint32_t width, float iso,
                                                          uint32_t* __restrict__ prefix) {
    __shared__ uint32_t s[1024];
    uint32_t c[4], sum = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t i = threadIdx.x * 4 + k;
        const float al = i < width ? VoxNorm<uint8_t>::apply(rgba[i] >> 24) : 0.0f;
        sum += al > 0.0f && al >= iso - 0.02f && al <= iso + 0.02f ? 1 : 0;
        c[k] = sum;
    }
    const uint32_t before = block_scan<false>(sum, s) - sum;
    if (threadIdx.x == 0) prefix[0] = 0;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k)
        if (threadIdx.x * 4 + k < width) prefix[threadIdx.x * 4 + k + 1] = before + c[k];
}

// Block i: the smallest j >= i whose entry (i, j) or (j, i) has alpha > 0 (n:
// none), from i upward, so a table that is mostly visible is hardly read.
__global__ __launch_bounds__(256) void pair_first_kernel(const float4* __restrict__ table, uint32_t n,
                                                         uint32_t* __restrict__ first) {
    __shared__ uint32_t s_min[4];
    const uint32_t i = blockIdx.x;
    uint32_t found = n;
    for (uint32_t j0 = i; j0 < n; j0 += 256) {
        const uint32_t j = j0 + threadIdx.x;
        bool hit = false;
        if (j < n) hit = !(table[(size_t)i * n + j].w <= 0.0f) || !(table[(size_t)j * n + i].w <= 0.0f);
        const unsigned long long b = __ballot(hit);
        if ((threadIdx.x & 63) == 0) s_min[threadIdx.x >> 6] = b ? j + (uint32_t)__builtin_ctzll(b) : n;
        __syncthreads();
        for (int w = 3; w >= 0; --w) found = s_min[w] < found ? s_min[w] : found;
        __syncthreads();
        if (found < n) break;
    }
    if (threadIdx.x == 0) first[i] = found;
}

// One workgroup: reach[i] = minimum of first over [i, n), in place, n <= 4096
// (entries beyond i's square have a first beyond it as well).
__global__ __launch_bounds__(1024) void pair_reach_kernel(uint32_t* __restrict__ first, uint32_t n) {
    __shared__ uint32_t s[1024];
    uint32_t c[4], m = 0xffffffffu;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {   // from the table's end
        const uint32_t r = threadIdx.x * 4 + k;
        const uint32_t v = r < n ? first[n - 1 - r] : 0xffffffffu;
        m = v < m ? v : m;
        c[k] = m;
    }
    block_scan<true>(m, s);
    const uint32_t before = threadIdx.x > 0 ? s[threadIdx.x - 1] : 0xffffffffu;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
        const uint32_t r = threadIdx.x * 4 + k;
        if (r < n) first[n - 1 - r] = before < c[k] ? before : c[k];
    }
}

__global__ __launch_bounds__(256) void occupancy_bits_kernel(const uint8_t* __restrict__ occ,
                                                             uint32_t* __restrict__ bits, uint64_t count) {
    const uint64_t w = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (w * 32 >= count) return;
    uint32_t word = 0;
    for (uint32_t k = 0; k < 32 && w * 32 + k < count; ++k) word |= (occ[w * 32 + k] != 0 ? 1u : 0u) << k;
    bits[w] = word;
}

}  // namespace

void launch_occupancy(const OccArgs& a, hipStream_t st) {
    hipLaunchKernelGGL(occupancy_kernel, dim3((unsigned)((a.count + 255) / 256)), dim3(256), 0, st, a);
    const uint64_t words = (a.count + 31) / 32;
    hipLaunchKernelGGL(occupancy_bits_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st, a.occ, a.bits,
                       a.count);
}

void launch_skip_grid(const OccArgs& a, const uint32_t nb[3], uint8_t* skip, uint8_t* scratch, hipStream_t st) {
    const uint64_t count = (uint64_t)nb[0] * nb[1] * nb[2];
    const uint32_t parts = (nb[0] + 255) / 256;
    const uint64_t groups = (uint64_t)parts * nb[1] * nb[2];
    if (a.pair_reach)
        hipLaunchKernelGGL(skip_x_kernel<true>, dim3(stride_grid(groups, 1)), dim3(256), 0, st, a, skip, nb[0], nb[1],
                           nb[2], parts, groups);
    else
        hipLaunchKernelGGL(skip_x_kernel<false>, dim3(stride_grid(groups, 1)), dim3(256), 0, st, a, skip, nb[0], nb[1],
                           nb[2], parts, groups);
    hipLaunchKernelGGL(skip_axis_kernel, dim3(stride_grid(count)), dim3(256), 0, st, (const uint8_t*)skip, scratch,
                       (uint64_t)nb[0], nb[1], count);
    hipLaunchKernelGGL(skip_axis_kernel, dim3(stride_grid(count)), dim3(256), 0, st, (const uint8_t*)scratch, skip,
                       (uint64_t)nb[0] * nb[1], nb[2], count);
}

void launch_iso_prefix(const uint32_t* rgba, uint32_t width, float iso, uint32_t* prefix, hipStream_t st) {
    hipLaunchKernelGGL(iso_prefix_kernel, dim3(1), dim3(1024), 0, st, rgba, width, iso, prefix);
}

void launch_pair_reach(const float4* table, uint32_t n, uint32_t* reach, hipStream_t st) {
    hipLaunchKernelGGL(pair_first_kernel, dim3(n), dim3(256), 0, st, table, n, reach);
    hipLaunchKernelGGL(pair_reach_kernel, dim3(1), dim3(1024), 0, st, reach, n);
}

SkipGrid& add_skip_grid(hipdvr_volume* v, SkipRule rule) {
    SkipGrid g;
    g.rule = rule;
    // an allocation is no part of a graph, and disturbs none
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    hip_check(hipThreadExchangeStreamCaptureMode(&mode), "hipThreadExchangeStreamCaptureMode");
    const hipError_t e = hipMalloc((void**)&g.d_band, kBandWords * 4 + 2 * v->skip_count);
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    hip_check(e, "hipMalloc(skip grid)");
    g.d = (uint8_t*)(g.d_band + kBandWords);
    v->skips.push_back(g);
    return v->skips.back();
}

hipdvr_volume* volume_create(hipdvr_ctx* ctx, hipStream_t st, const hipdvr_volume_desc* d,
                             const void* voxels, bool on_device) {
    for (int i = 0; i < 3; ++i)
        if (d->dims[i] < 1 || d->dims[i] > (1u << 20))
            fail(HIPDVR_ERR_INVALID, "volume dimensions must be in [1, 2^20]");
    if (d->dtype != HIPDVR_U8 && d->dtype != HIPDVR_U16)
        fail(HIPDVR_ERR_INVALID, "dtype must be HIPDVR_U8 or HIPDVR_U16");
    uint32_t bl = d->brick_log2 ? d->brick_log2 : 3;
    if (bl < 2 || bl > 5) fail(HIPDVR_ERR_INVALID, "brick_log2 must be in [2, 5]");
    hipdvr_volume* v = new hipdvr_volume();
    v->ctx = ctx;
    v->tiled_elems = 64;
    v->brick_count = 1;
    for (int i = 0; i < 3; ++i) {
        v->desc.dims[i] = d->dims[i];
        v->desc.spacing[i] = d->spacing[i];
        v->desc.offset[i] = d->offset[i];
        v->nblocks[i] = (d->dims[i] + 3) / 4;
        v->nbricks[i] = (d->dims[i] + (1u << bl) - 1) >> bl;
        v->tiled_elems *= v->nblocks[i];
        v->brick_count *= v->nbricks[i];
        v->nskip[i] = (d->dims[i] + (1u << kSkipLog2) - 1) >> kSkipLog2;
    }
    v->skip_count = (uint64_t)v->nskip[0] * v->nskip[1] * v->nskip[2];
    v->desc.dtype = d->dtype;
    v->desc.rwm_scale = d->rwm_scale;
    v->desc.rwm_offset = d->rwm_offset;
    v->desc.brick_log2 = bl;
    const size_t vsz = d->dtype == HIPDVR_U8 ? 1 : 2;
    const size_t bytes = (size_t)d->dims[0] * d->dims[1] * d->dims[2] * vsz;
    try {
        hip_check(hipMalloc(&v->d_linear, bytes), "hipMalloc(volume)");
        hip_check(hipMalloc(&v->d_tiled, v->tiled_elems * vsz), "hipMalloc(tiled volume)");
        // the brick tables in one allocation: ranges of the volume's bricks and
        // of the 8^3 bricks, occupancy bits, the tables and grids (with scratch)
        // of the skip rules, occupancy bytes
        v->occ_words = (uint32_t)((v->brick_count + 31) / 32);
        const size_t mm = v->brick_count * sizeof(uint2), mm8 = v->skip_count * sizeof(uint2);
        const size_t words = ((size_t)v->occ_words * 4 + 7) & ~(size_t)7;
        char* p = nullptr;
        hip_check(hipMalloc((void**)&p, mm + mm8 + words + kSkipRules * (kBandWords * 4 + 2 * v->skip_count) +
                                              v->brick_count),
                  "hipMalloc(bricks)");
        v->d_minmax = (uint2*)p;
        v->d_minmax8 = (uint2*)(p + mm);
        v->d_occ_bits = (uint32_t*)(p + mm + mm8);
        uint32_t* band = (uint32_t*)(p + mm + mm8 + words);
        uint8_t* bytes_at = (uint8_t*)(band + kSkipRules * kBandWords);
        v->skips.resize(kSkipRules);
        for (int r = 0; r < kSkipRules; ++r) {
            v->skips[r].rule = (SkipRule)r;
            v->skips[r].d_band = band + r * kBandWords;
            v->skips[r].d = bytes_at;
            bytes_at += 2 * v->skip_count;
        }
        v->d_occ = bytes_at;
        hip_check(hipMemcpyAsync(v->d_linear, voxels, bytes,
                                 on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, st),
                  "volume upload");
        if (d->dtype == HIPDVR_U8) build_layouts<uint8_t>(v, st);
        else build_layouts<uint16_t>(v, st);
        hip_check(hipStreamSynchronize(st), "hipStreamSynchronize");
    } catch (...) {
        volume_destroy(v);
        throw;
    }
    return v;
}

namespace {
// One workgroup: minimum and maximum over the brick table (every voxel lies
// in some brick's range).
__global__ __launch_bounds__(1024) void minmax_reduce_kernel(const uint2* __restrict__ mm, uint64_t n,
                                                            uint32_t* __restrict__ out) {
    uint32_t lo = 0xffffffffu, hi = 0;
    for (uint64_t i = threadIdx.x; i < n; i += blockDim.x) {
        const uint2 v = mm[i];
        lo = v.x < lo ? v.x : lo;
        hi = v.y > hi ? v.y : hi;
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const uint32_t l2 = __shfl_xor(lo, off, 64), h2 = __shfl_xor(hi, off, 64);
        lo = l2 < lo ? l2 : lo;
        hi = h2 > hi ? h2 : hi;
    }
    __shared__ uint32_t s_lo[16], s_hi[16];
    if ((threadIdx.x & 63) == 0) {
        s_lo[threadIdx.x >> 6] = lo;
        s_hi[threadIdx.x >> 6] = hi;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) {
            lo = s_lo[w] < lo ? s_lo[w] : lo;
            hi = s_hi[w] > hi ? s_hi[w] : hi;
        }
        out[0] = lo;
        out[1] = hi;
    }
}
}  // namespace

void volume_raw_minmax(const hipdvr_volume* v, hipStream_t st, uint32_t out[2]) {
    uint32_t* d = nullptr;
    hip_check(hipMalloc((void**)&d, 8), "hipMalloc(minmax)");
    hipLaunchKernelGGL(minmax_reduce_kernel, dim3(1), dim3(1024), 0, st, v->d_minmax, v->brick_count, d);
    const hipError_t e1 = hipGetLastError();
    const hipError_t e2 = e1 == hipSuccess ? hipMemcpyAsync(out, d, 8, hipMemcpyDeviceToHost, st) : e1;
    const hipError_t e3 = e2 == hipSuccess ? hipStreamSynchronize(st) : e2;
    (void)hipFree(d);
    hip_check(e3, "volume min/max");
}

void launch_brick_minmax(const hipdvr_volume* v, uint32_t bl, const uint32_t nb[3], uint2* out, hipStream_t st) {
    const uint32_t X = v->desc.dims[0], Y = v->desc.dims[1], Z = v->desc.dims[2];
    const uint64_t count = (uint64_t)nb[0] * nb[1] * nb[2];
    if (bl >= kSkipLog2) {
        hipLaunchKernelGGL(minmax_fold_kernel, dim3(stride_grid(count)), dim3(256), 0, st, (const uint2*)v->d_minmax8,
                           out, v->nskip[0], v->nskip[1], v->nskip[2], bl - kSkipLog2, nb[0], nb[1], count);
        return;
    }
    const dim3 grid(stride_grid(count, 1));
    if (v->desc.dtype == HIPDVR_U8)
        hipLaunchKernelGGL(minmax_kernel<uint8_t>, grid, dim3(256), 0, st, (const uint8_t*)v->d_linear, out, X, Y,
                           Z, bl, nb[0], nb[1], count);
    else
        hipLaunchKernelGGL(minmax_kernel<uint16_t>, grid, dim3(256), 0, st, (const uint16_t*)v->d_linear, out, X,
                           Y, Z, bl, nb[0], nb[1], count);
}

uint64_t cell_record_bytes(const hipdvr_volume* v) {
    return cell_record_count(v->desc.dims) * (v->desc.dtype == HIPDVR_U8 ? 8 : 16);
}

bool cells_allowed(const hipdvr_volume* v) { return cell_record_bytes(v) <= kMaxCellBytes; }

namespace {

// Builds the records; false, and nothing done, where the memory for them is
// not there.
bool build_cells(hipdvr_volume* v, hipStream_t st) {
    const uint64_t bytes = cell_record_bytes(v);
    const uint64_t total = bytes / (v->desc.dtype == HIPDVR_U8 ? 8 : 16);
    void* p = nullptr;
    const hipError_t e0 = hipMalloc(&p, bytes);
    if (e0 == hipErrorOutOfMemory) {
        (void)hipGetLastError();   // not left for the next call
        return false;
    }
    hip_check(e0, "hipMalloc(cell records)");
    const dim3 grid(stride_grid(total));
    if (v->desc.dtype == HIPDVR_U8)
        hipLaunchKernelGGL(cells_kernel<uint8_t>, grid, dim3(256), 0, st, (const uint8_t*)v->d_linear, p,
                           v->desc.dims[0], v->desc.dims[1], v->desc.dims[2], total);
    else
        hipLaunchKernelGGL(cells_kernel<uint16_t>, grid, dim3(256), 0, st, (const uint16_t*)v->d_linear, p,
                           v->desc.dims[0], v->desc.dims[1], v->desc.dims[2], total);
    const hipError_t e1 = hipGetLastError();
    const hipError_t e2 = hipStreamSynchronize(st);
    if (e1 != hipSuccess || e2 != hipSuccess) {
        (void)hipFree(p);
        hip_check(e1 != hipSuccess ? e1 : e2, "cell record build");
    }
    v->d_cells = p;
    v->cell_bytes = bytes;
    v->cells_wide = bytes > 0xffffff00ull;
    return true;
}

}  // namespace

bool try_cells(hipdvr_volume* v, hipStream_t st) {
    if (v->d_cells) return true;
    size_t free_bytes = 0, all = 0;
    hip_check(hipMemGetInfo(&free_bytes, &all), "hipMemGetInfo");
    return cells_allowed(v) && cell_record_bytes(v) <= free_bytes / 2 && build_cells(v, st);
}

void ensure_cells(hipdvr_volume* v, hipStream_t st) {
    if (v->d_cells) return;
    if (!cells_allowed(v)) fail(HIPDVR_ERR_UNSUPPORTED, "cell records of this volume exceed the size limit");
    if (!build_cells(v, st)) hip_check(hipErrorOutOfMemory, "hipMalloc(cell records)");
}

void volume_destroy(hipdvr_volume* v) {
    if (!v) return;
    if (v->d_cells) (void)hipFree(v->d_cells);
    if (v->d_linear) (void)hipFree(v->d_linear);
    if (v->d_tiled) (void)hipFree(v->d_tiled);
    if (v->d_minmax) (void)hipFree(v->d_minmax);   // and the tables behind it
    for (size_t i = kSkipRules; i < v->skips.size(); ++i) (void)hipFree(v->skips[i].d_band);
    if (v->d_grad) (void)hipFree(v->d_grad);
    delete v;
}

}  // namespace hipdvr
