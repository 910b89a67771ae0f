// Quantile binning on the device: the reference's quantile_bin / apply_bins (data.py:44-111).
//
//  * edges: for each column, the interior quantiles np.quantile(x, q, method="linear") of the
//    column's values, cast to float32. NumPy's arithmetic (numpy lib/_function_base_impl.py,
//    _quantile / _get_indexes / _lerp) is restated exactly, in double without contraction:
//        v = (n - 1) * q;  i = floor(v);  j = i + 1;  (both n - 1 when v >= n - 1)
//        g = v - i;  a = x(i), b = x(j) (float32, sorted ascending);  d = b - a (float32)
//        e = g >= 0.5 ? b - d * (1 - g) : a + d * g          (double), then float32
//    A column holding a NaN gets NaN edges (NumPy sorts NaN last and propagates it).
//  * bins: searchsorted(edges, x, side="left") clipped to [0, max_bins - 1], with NumPy's
//    NaN-last order (NaN > every number), written column-major for the histogram kernel,
//    optionally gathering rows through a permutation (era-major order).
#include <algorithm>

#include "pb_internal.h"

namespace pb {
namespace {

__global__ void quantile_edges_kernel(const float* __restrict__ sorted, int64_t n, int64_t ld,
                                      int32_t F, const double* __restrict__ q, int32_t nq,
                                      float* __restrict__ edges, int32_t edge_stride) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)F * nq) return;
    const int f = (int)(t / nq);
    const int k = (int)(t - (int64_t)f * nq);
    const float* col = sorted + (int64_t)f * ld;
    float out;
    if (n <= 0) {
        out = __int_as_float(0x7fc00000);
    } else if (isnan(col[n - 1])) {
        out = __int_as_float(0x7fc00000);
    } else {
        const double v = (double)(n - 1) * q[k];
        double prev = floor(v);
        double next = prev + 1.0;
        if (v >= (double)(n - 1)) {
            prev = (double)(n - 1);
            next = (double)(n - 1);
        }
        if (v < 0.0) {
            prev = 0.0;
            next = 0.0;
        }
        const double g = v - floor(v);
        const float a = col[(int64_t)prev];
        const float b = col[(int64_t)next];
        const float d = b - a;
        const double e = (g >= 0.5) ? ((double)b - (double)d * (1.0 - g))
                                    : ((double)a + (double)d * g);
        out = (float)e;
    }
    edges[(int64_t)k * edge_stride + f] = out;
}

// NumPy's float order for searchsorted: a < b, with NaN after every number
__device__ __forceinline__ bool np_less(float a, float b) {
    return a < b || (isnan(b) && !isnan(a));
}

__global__ __launch_bounds__(kBlock) void apply_bins_kernel(
    const float* __restrict__ xt, int64_t n, int64_t ld_x, const float* __restrict__ edges,
    int32_t ne, int32_t edge_stride, int32_t max_bins, const int64_t* __restrict__ perm,
    uint8_t* __restrict__ bins, int64_t ld_out, int32_t rows_per_block) {
    __shared__ float s_edges[256];
    const int f = blockIdx.y;
    for (int i = threadIdx.x; i < ne; i += kBlock) s_edges[i] = edges[(int64_t)i * edge_stride + f];
    __syncthreads();
    const float* col = xt + (int64_t)f * ld_x;
    const int64_t r0 = (int64_t)blockIdx.x * rows_per_block;
    const int64_t r1 = min(n, r0 + rows_per_block);
    for (int64_t r = r0 + threadIdx.x; r < r1; r += kBlock) {
        const float x = col[perm ? perm[r] : r];
        int lo = 0, hi = ne;
        while (lo < hi) {
            const int mid = lo + ((hi - lo) >> 1);
            if (np_less(s_edges[mid], x))
                lo = mid + 1;
            else
                hi = mid;
        }
        bins[(int64_t)f * ld_out + r] = (uint8_t)min(lo, max_bins - 1);
    }
}

// NumPy's float order for searchsorted as an unsigned order: -0.0 equals +0.0, NaN after all.
__device__ __forceinline__ uint32_t order_key(float x) {
    const uint32_t b = __float_as_uint(x);
    const uint32_t k = b == 0x80000000u ? 0x80000000u : b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
    return isnan(x) ? 0xffffffffu : k;
}

// apply_bins from row-major values [n][F] (row stride in elements) straight to the column-major
// bins, optionally gathering rows through a permutation; rows n .. n_out-1 become 0. A workgroup
// keeps the sorted edges of 32 features in LDS as order keys (2^STEPS - 1 per feature, padded with
// the last key) and walks tiles of 128 rows: a thread reads 4 features of 4 rows (8 lanes cover 128
// contiguous bytes of a row) and runs its 16 searches side by side, STEPS branchless LDS probes
// each, so the probes' latencies overlap; the bins leave through LDS as 128-byte runs per column.
// An odd stride between the features' edges keeps the first probes (the same index in every
// feature) on distinct banks; the later ones are random. The LDS probes bound it (8.7 clocks each, three
// quarters of them bank conflicts; the LDS is active 78% of the time): 1M x 500 values through 254 edges
// take 1.13 to 1.17 ms (430 G values/s; 0.65 ms through 15 edges), where transposed copies and one search
// per lane took 9.0 ms. The 32 features are searched however few there are: long tables of up to 7 are
// binned column by column instead.
// Edges that do not ascend (a column with infinities between its quantiles has NaN edges below
// finite ones) take searchsorted's own probe order instead, which decides what it finds there.
// All feature groups of a row range run on one XCD, where its rows' split cache lines are shared.
typedef __attribute__((address_space(3))) uint32_t lds_word;
constexpr int kBrRows = 128;
constexpr int kBrFeats = 32;

template <int STEPS>
__global__ __launch_bounds__(kBlock) void bin_rows_kernel(const float* __restrict__ x, int64_t n, int64_t stride,
                                                      int32_t F, const float* __restrict__ edges, int32_t ne,
                                                      int32_t edge_stride, int32_t max_bins,
                                                      const int64_t* __restrict__ perm, uint8_t* __restrict__ out,
                                                      int64_t n_out, int64_t ld, int32_t groups,
                                                      int32_t tiles_per_block) {
    constexpr int kCap = (1 << STEPS) - 1, kStride = kCap + (STEPS == 1 ? 0 : 2);
    __shared__ uint32_t s_edge[kBrFeats * kStride];
    __shared__ uint32_t s_tile[kBrFeats][kBrRows / 4 + 1];
    __shared__ uint32_t s_mixed;  // some feature's edges do not ascend
    const int64_t item = blockIdx.x >> 3;
    const int64_t chunk = item / groups * 8 + (blockIdx.x & 7);
    const int f0 = (int)(item % groups) * kBrFeats;
    const int64_t row_lo = chunk * tiles_per_block * kBrRows;
    if (row_lo >= n_out) return;  // uniform
    for (int i = threadIdx.x; i < kBrFeats * kCap; i += kBlock) {
        const int fl = i & (kBrFeats - 1), e = i / kBrFeats;
        const bool in = e < ne && f0 + fl < F;
        s_edge[fl * kStride + e] = in ? order_key(edges[(int64_t)e * edge_stride + f0 + fl]) : 0xffffffffu;
    }
    if (threadIdx.x == 0) s_mixed = 0u;
    __syncthreads();
    for (int i = threadIdx.x; i < kBrFeats * (kCap - 1); i += kBlock) {
        const int fl = i & (kBrFeats - 1), e = i / kBrFeats;
        if (s_edge[fl * kStride + e] > s_edge[fl * kStride + e + 1]) s_mixed = 1u;
    }
    const int fq = threadIdx.x & 7, rq = threadIdx.x >> 3;
    const int f = f0 + 4 * fq;
    struct __attribute__((packed, aligned(4))) Floats4 {
        float v[4];
    };
    // the searches hold LDS byte addresses, so that a probe is one read at an immediate offset, a
    // compare, a select and an add
    const uint32_t edge0 = (uint32_t)(size_t)(lds_word*)s_edge + (uint32_t)(4 * fq * kStride * 4);
    const uint32_t last = (uint32_t)(max_bins - 1);
    for (int t = 0; t < tiles_per_block; ++t) {
        const int64_t r0 = row_lo + (int64_t)t * kBrRows;
        if (r0 >= n_out) break;  // uniform
        Floats4 v[4];
        if (r0 + kBrRows <= n && f0 + kBrFeats <= F) {  // uniform
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t r = r0 + 4 * rq + i;
                v[i] = *reinterpret_cast<const Floats4*>(x + (perm ? perm[r] : r) * stride + f);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t r = r0 + 4 * rq + i;
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    v[i].v[k] = r < n && f + k < F ? x[(perm ? perm[r] : r) * stride + f + k] : 0.0f;
            }
        }
        __syncthreads();  // the edges are staged; the last tile is stored
        uint32_t key[4][4], at[4][4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                key[i][k] = order_key(v[i].v[k]);
                at[i][k] = edge0;
            }
        if (s_mixed) {  // uniform
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t* edge = s_edge + (4 * fq + k) * kStride;
                    int lo = 0, hi = ne;
                    while (lo < hi) {
                        const int mid = lo + ((hi - lo) >> 1);
                        if (edge[mid] < key[i][k])
                            lo = mid + 1;
                        else
                            hi = mid;
                    }
                    at[i][k] = edge0 + 4u * (uint32_t)lo;
                }
        } else
#pragma unroll
        for (int s = STEPS - 1; s >= 0; --s)
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t probe = *((const lds_word*)(size_t)at[i][k] + k * kStride + (1 << s) - 1);
                    at[i][k] += probe < key[i][k] ? 4u << s : 0u;
                }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            uint32_t w = 0u;
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w |= (r0 + 4 * rq + i < n ? min((at[i][k] - edge0) >> 2, last) : 0u) << (8 * i);
            s_tile[4 * fq + k][rq] = w;
        }
        __syncthreads();
        const int c = threadIdx.x >> 3, q = threadIdx.x & 7;  // column, 16 rows of it
        const int64_t row = r0 + 16 * q;
        if (f0 + c < F && row < n_out) {
            const uint32_t* w = &s_tile[c][4 * q];
            *reinterpret_cast<uint4*>(out + (int64_t)(f0 + c) * ld + row) = make_uint4(w[0], w[1], w[2], w[3]);
        }
    }
}

template <int STEPS>
void launch_bin_rows_steps(const float* x, int64_t n, int64_t stride, int32_t F, const float* edges, int32_t ne,
                           int32_t edge_stride, int32_t max_bins, const int64_t* perm, uint8_t* out, int64_t n_out,
                           int64_t ld, int32_t groups, int32_t tiles_per_block, int64_t grid, hipStream_t s) {
    hipLaunchKernelGGL(bin_rows_kernel<STEPS>, dim3((unsigned)grid), dim3(kBlock), 0, s, x, n, stride, F, edges, ne,
                       edge_stride, max_bins, perm, out, n_out, ld, groups, tiles_per_block);
}

// Nibble layout for nb <= 16: every 8 rows of a uint8 column (bytes b0..b7) become one dword
// whose byte j is b_j | b_{j+4} << 4. One thread converts 16 rows (one 16-byte load, one
// 8-byte store); bins above 15 lose their high bits (callers guarantee bins < nb <= 16).
// Rows n .. ld-1 (padding) are written as bin 0: the histogram reads them unmasked.
__global__ __launch_bounds__(kBlock) void pack_bins4_kernel(const uint8_t* __restrict__ bins,
                                                         int64_t ld, int64_t n,
                                                         int64_t units_per_col, int64_t units,
                                                         uint8_t* __restrict__ out) {
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t t = (int64_t)blockIdx.x * kBlock + threadIdx.x; t < units; t += stride) {
        const int64_t f = t / units_per_col;
        const int64_t u = t - f * units_per_col;
        uint4 v = *reinterpret_cast<const uint4*>(bins + f * ld + u * 16);
        const int64_t r0 = u * 16;  // first row of this unit
        if (r0 + 16 > n) {
            uint32_t wv[4] = {v.x, v.y, v.z, v.w};
    #pragma unroll
            for (int q = 0; q < 4; ++q)
    #pragma unroll
                for (int b = 0; b < 4; ++b)
                    if (r0 + 4 * q + b >= n) wv[q] &= ~(0xffu << (8 * b));
            v = make_uint4(wv[0], wv[1], wv[2], wv[3]);
        }
        uint2 o;
        o.x = (v.x & 0x0f0f0f0fu) | ((v.y & 0x0f0f0f0fu) << 4);
        o.y = (v.z & 0x0f0f0f0fu) | ((v.w & 0x0f0f0f0fu) << 4);
        *reinterpret_cast<uint2*>(out + f * (ld / 2) + u * 8) = o;
    }
}

// Row-major bin codes [n][F] (row stride `stride` bytes, any alignment) to the histogram's
// column-major [F][ld], optionally gathering rows through a permutation; rows n .. n_out-1 become 0.
// Bound by HBM (every byte read and written once). A workgroup moves a tile of 256 rows x 128
// features: each thread reads 16 features of 4 consecutive rows (8 lanes cover 128 contiguous
// bytes of a row), transposes them as 4x4 bytes in registers and puts one dword (4 rows) per
// feature into LDS, whose odd row stride spreads the 8 lanes of a row over the banks; the tile then
// leaves as 16-byte stores, 256 contiguous bytes per column. Feature tiles are the fastest grid
// dimension, so the workgroups in flight read whole rows. 2.4M x 2376 codes take 2.34 ms (4.9 TB/s,
// this card's copy rate; 4.65 ms with the loads behind per-row guards, 28 ms as torch's strided
// copy), 2.72 ms through a random row permutation.
// limit > 0: *over is set when some code is >= limit (codes compared four at a time).
constexpr int kTrRows = 256;
constexpr int kTrFeats = 128;

struct __attribute__((packed)) Bytes16 {
    uint32_t w[4];
};

__device__ __forceinline__ void transpose4x4_bytes(const uint32_t (&r)[4], uint32_t (&c)[4]) {
    const uint32_t ab0 = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);  // a0 b0 a1 b1
    const uint32_t ab1 = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);  // a2 b2 a3 b3
    const uint32_t cd0 = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
    const uint32_t cd1 = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
    c[0] = __builtin_amdgcn_perm(cd0, ab0, 0x05040100u);
    c[1] = __builtin_amdgcn_perm(cd0, ab0, 0x07060302u);
    c[2] = __builtin_amdgcn_perm(cd1, ab1, 0x05040100u);
    c[3] = __builtin_amdgcn_perm(cd1, ab1, 0x07060302u);
}

__global__ __launch_bounds__(kBlock) void transpose_bins_kernel(const uint8_t* __restrict__ src, int64_t n,
                                                            int64_t stride, int32_t F,
                                                            const int64_t* __restrict__ perm,
                                                            uint8_t* __restrict__ out, int64_t n_out, int64_t ld,
                                                            int32_t ftiles, uint32_t limit,
                                                            int32_t* __restrict__ over) {
    __shared__ uint32_t tile[kTrFeats][kTrRows / 4 + 1];
    const int64_t r0 = (int64_t)(blockIdx.x / (uint32_t)ftiles) * kTrRows;
    const int f0 = (int)(blockIdx.x % (uint32_t)ftiles) * kTrFeats;
    const int fg = threadIdx.x & 7;  // 16-feature group
    const int f = f0 + fg * 16;
    constexpr int kIt = kTrRows / 128;  // row quads per thread: rows r0 + 4 rq .. for rq = tid / 8 + 32 it
    Bytes16 v[kIt][4];
    if (r0 + kTrRows <= n && f0 + kTrFeats <= F) {  // uniform: no guard, every load in flight at once
        const int64_t rb = r0 + 4 * (int)(threadIdx.x >> 3);
#pragma unroll
        for (int it = 0; it < kIt; ++it)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t r = rb + 128 * it + i;
                v[it][i] = *reinterpret_cast<const Bytes16*>(src + (perm ? perm[r] : r) * stride + f);
            }
    } else {
#pragma unroll
        for (int it = 0; it < kIt; ++it)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int64_t r = r0 + 4 * ((int)(threadIdx.x >> 3) + 32 * it) + i;
                v[it][i] = Bytes16{{0u, 0u, 0u, 0u}};
                if (r >= n || f >= F) continue;
                const uint8_t* p = src + (perm ? perm[r] : r) * stride + f;
                if (f + 16 <= F) {
                    v[it][i] = *reinterpret_cast<const Bytes16*>(p);
                } else {  // the last features of a row: no byte past the row is read
#pragma unroll
                    for (int b = 0; b < 16; ++b)
                        if (b < F - f) v[it][i].w[b >> 2] |= (uint32_t)p[b] << (8 * (b & 3));
                }
            }
    }
    uint32_t hit = 0u;
#pragma unroll
    for (int it = 0; it < kIt; ++it) {
        const int rq = (int)(threadIdx.x >> 3) + it * 32;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t rows4[4] = {v[it][0].w[q], v[it][1].w[q], v[it][2].w[q], v[it][3].w[q]};
            uint32_t cols4[4];
            transpose4x4_bytes(rows4, cols4);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (limit) hit |= bytes_at_least(cols4[k], limit);
                tile[fg * 16 + q * 4 + k][rq] = cols4[k];
            }
        }
    }
    if (limit && hit) atomicOr(over, 1);
    __syncthreads();
    // 16 lanes per column, 16 bytes (16 rows) each
    const int q = threadIdx.x & 15;
    const int64_t row = r0 + 16 * q;
    if (row >= n_out) return;
#pragma unroll
    for (int it = 0; it < kTrFeats / 16; ++it) {
        const int k = (int)(threadIdx.x >> 4) + it * 16;
        if (f0 + k >= F) break;
        const uint4 w = make_uint4(tile[k][4 * q], tile[k][4 * q + 1], tile[k][4 * q + 2], tile[k][4 * q + 3]);
        *reinterpret_cast<uint4*>(out + (int64_t)(f0 + k) * ld + row) = w;
    }
}

}  // namespace

hipError_t launch_transpose_bins(const uint8_t* src, int64_t n, int64_t stride, int32_t F, const int64_t* perm,
                                 uint8_t* out, int64_t n_out, int64_t ld, int32_t limit, int32_t* over,
                                 hipStream_t s) {
    const int64_t ftiles = (F + kTrFeats - 1) / kTrFeats;
    const int64_t grid = (n_out + kTrRows - 1) / kTrRows * ftiles;
    if (grid > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(transpose_bins_kernel, dim3((unsigned)grid), dim3(kBlock), 0, s, src, n, stride, F, perm,
                       out, n_out, ld, (int32_t)ftiles, (uint32_t)limit, over);
    return hipGetLastError();
}

hipError_t launch_bin_rows(const float* x, int64_t n, int64_t stride, int32_t F, const float* edges, int32_t ne,
                           int32_t edge_stride, int32_t max_bins, const int64_t* perm, uint8_t* out,
                           int64_t n_out, int64_t ld, hipStream_t s) {
    if (ne < 1 || ne > 254) return hipErrorInvalidValue;
    const int64_t groups = (F + kBrFeats - 1) / kBrFeats;
    const int64_t tiles = (n_out + kBrRows - 1) / kBrRows;
    // a workgroup loads its features' edges once (as many bytes as two tiles of rows at 254 edges)
    // and walks up to 16 tiles, fewer while that would leave less than about 2048 workgroups
    const int64_t per = std::max<int64_t>(1, std::min<int64_t>(16, tiles * groups / 2048));
    const int64_t chunks = (tiles + per - 1) / per;
    const int64_t grid = (chunks + 7) / 8 * 8 * groups;
    if (grid > INT32_MAX) return hipErrorInvalidValue;
    int steps = 1;
    while ((1 << steps) - 1 < ne) ++steps;
    auto go = [&](auto launch) {
        launch(x, n, stride, F, edges, ne, edge_stride, max_bins, perm, out, n_out, ld, (int32_t)groups, (int32_t)per,
               grid, s);
    };
    switch (steps) {
        case 1: go(launch_bin_rows_steps<1>); break;
        case 2: go(launch_bin_rows_steps<2>); break;
        case 3: go(launch_bin_rows_steps<3>); break;
        case 4: go(launch_bin_rows_steps<4>); break;
        case 5: go(launch_bin_rows_steps<5>); break;
        case 6: go(launch_bin_rows_steps<6>); break;
        case 7: go(launch_bin_rows_steps<7>); break;
        default: go(launch_bin_rows_steps<8>); break;
    }
    return hipGetLastError();
}

hipError_t launch_pack_bins4(const uint8_t* bins, int64_t n, int64_t ld, int32_t F, uint8_t* out,
                             hipStream_t s) {
    const int64_t per_col = ld / 16;
    const int64_t units = per_col * F;
    const int grid = (int)std::min<int64_t>((units + kBlock - 1) / kBlock, 65536);
    hipLaunchKernelGGL(pack_bins4_kernel, dim3(std::max(grid, 1)), dim3(kBlock), 0, s, bins, ld, n,
                       per_col, units, out);
    return hipGetLastError();
}

hipError_t launch_quantile_edges(const float* sorted, int64_t n, int64_t ld, int32_t F,
                                 const double* q, int32_t nq, float* edges, int32_t edge_stride,
                                 hipStream_t s) {
    const int64_t work = (int64_t)F * nq;
    const int grid = (int)((work + kBlock - 1) / kBlock);
    hipLaunchKernelGGL(quantile_edges_kernel, dim3(grid), dim3(kBlock), 0, s, sorted, n, ld, F, q,
                       nq, edges, edge_stride);
    return hipGetLastError();
}

hipError_t launch_apply_bins(const float* xt, int64_t n, int64_t ld_x, int32_t F,
                             const float* edges, int32_t ne, int32_t edge_stride, int32_t max_bins,
                             const int64_t* perm, uint8_t* bins, int64_t ld_out, hipStream_t s) {
    const int rows_per_block = 8192;
    const int64_t gx = (n + rows_per_block - 1) / rows_per_block;
    hipLaunchKernelGGL(apply_bins_kernel, dim3((unsigned)gx, (unsigned)F), dim3(kBlock), 0, s, xt,
                       n, ld_x, edges, ne, edge_stride, max_bins, perm, bins, ld_out,
                       rows_per_block);
    return hipGetLastError();
}

}  // namespace pb
