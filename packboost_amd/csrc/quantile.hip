// Quantile edges by selection: np.quantile(x, q, method="linear") of every column of a float table
// (the reference's quantile_bin, data.py:44-56), without sorting the columns.
//
// A quantile needs two neighbouring order statistics of its column; num_q of them pin at most
// 2 num_q elements, so a sort (a library segmented sort took 110 ms for 1M x 500, and held the
// sorted values and 64-bit indices) orders far more than is asked. Here, per column:
//   keys     the values as unsigned order keys, column-major (-0.0 before +0.0, NaN as the last key);
//            row-major input is transposed through LDS, 256 contiguous bytes each way
//   sample   a sorted sample's every fourth key gives the splitters (2^STEPS - 1 of them)
//   count    every key's class by a branchless search in LDS: 2i = strictly between splitters
//            i - 1 and i, 2i + 1 = equal to splitter i (so a heavy tie fills a class that needs no
//            look inside); the classes are counted and kept, 2 bytes a key
//   ranks    prefix sums place each wanted rank in a class; intervals that hold one get space
//   gather   the keys of those intervals are moved together
//   select   a workgroup per quantile picks its ranks from its interval by radix selection, at any
//            interval size, and interpolates in NumPy's order of operations
// Columns of at most kSmall rows are sorted in LDS instead. Every step is exact; only speed depends
// on the sample. 1M x 500 values and 254 quantiles take 6.6 ms (keys 0.9, count 2.5, gather 1.8,
// select 1.2), where transposed copies, a segmented sort and its reading took 127 ms;
// 200k x 100 and 127 quantiles 0.4 ms for 4.8.
#include <algorithm>

#include "pb_internal.h"

namespace pb {
namespace {

typedef __attribute__((address_space(3))) uint32_t lds_word;

constexpr int kSmall = 16384;      // rows a column may have to be sorted in LDS
constexpr int kTile = 64;          // rows and features of a transposed tile
constexpr int kChunkKeys = 32768;  // keys per workgroup of the count pass
constexpr uint32_t kNanKey = 0xffffffffu;

// A total order that keeps every bit of a number: a zero edge has the sign that its ranks' zeros give
// it. (Where a column holds zeros of both signs, which tie in NumPy's sort, -0.0 comes first.)
__device__ __forceinline__ uint32_t key_of(float x) {
    const uint32_t b = __float_as_uint(x);
    return isnan(x) ? kNanKey : b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
}

__device__ __forceinline__ float value_of(uint32_t k) {
    return __uint_as_float((k >> 31) ? k ^ 0x80000000u : ~k);
}

// the ranks a quantile interpolates between, and its edge from the values there (NumPy's
// _get_indexes and _lerp, in double without contraction)
__device__ __forceinline__ void quantile_ranks(int64_t n, double q, int64_t& lo, int64_t& hi, double& g) {
    const double v = (double)(n - 1) * q;
    double prev = floor(v), next = prev + 1.0;
    if (v >= (double)(n - 1)) prev = next = (double)(n - 1);
    if (v < 0.0) prev = next = 0.0;
    g = v - floor(v);
    lo = (int64_t)prev;
    hi = (int64_t)next;
}

__device__ __forceinline__ float quantile_edge(float a, float b, double g) {
    const float d = b - a;
    return (float)(g >= 0.5 ? (double)b - (double)d * (1.0 - g) : (double)a + (double)d * g);
}

// keys[f][r] = key of x[r * stride + f]: 64 x 64 tiles through LDS (odd row stride: no conflicts)
__global__ __launch_bounds__(kBlock) void keys_from_rows_kernel(const float* __restrict__ x, int64_t n, int64_t stride,
                                                            int32_t F, uint32_t* __restrict__ keys, int64_t ld,
                                                            int32_t ftiles) {
    __shared__ uint32_t tile[kTile][kTile + 1];
    struct __attribute__((packed, aligned(4))) Floats4 {
        float v[4];
    };
    const int64_t r0 = (int64_t)(blockIdx.x / (uint32_t)ftiles) * kTile;
    const int f0 = (int)(blockIdx.x % (uint32_t)ftiles) * kTile;
    const int fq = threadIdx.x & 15, rr = threadIdx.x >> 4;
    Floats4 v[4];
    if (r0 + kTile <= n && f0 + kTile <= F) {  // uniform
#pragma unroll
        for (int i = 0; i < 4; ++i)
            v[i] = *reinterpret_cast<const Floats4*>(x + (r0 + rr + 16 * i) * stride + f0 + 4 * fq);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int64_t r = r0 + rr + 16 * i;
                const int f = f0 + 4 * fq + k;
                v[i].v[k] = r < n && f < F ? x[r * stride + f] : 0.0f;
            }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int k = 0; k < 4; ++k) tile[4 * fq + k][rr + 16 * i] = key_of(v[i].v[k]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int f = rr + 16 * i;
        const int64_t r = r0 + 4 * fq;
        if (f0 + f < F && r < ld) {
            const uint32_t* t = &tile[f][4 * fq];
            *reinterpret_cast<uint4*>(keys + (int64_t)(f0 + f) * ld + r) = make_uint4(t[0], t[1], t[2], t[3]);
        }
    }
}

// keys[f][r] = key of x[f * xld + r] (feature-major values)
__global__ __launch_bounds__(kBlock) void keys_from_columns_kernel(const float* __restrict__ x, int64_t n, int64_t xld,
                                                               uint32_t* __restrict__ keys, int64_t ld) {
    const float* col = x + (int64_t)blockIdx.y * xld;
    uint32_t* out = keys + (int64_t)blockIdx.y * ld;
    const int64_t stride = (int64_t)gridDim.x * kBlock;
    for (int64_t r = (int64_t)blockIdx.x * kBlock + threadIdx.x; r < n; r += stride) out[r] = key_of(col[r]);
}

// ascending bitonic sort of the P (a power of two) keys in LDS
template <int NT>
__device__ void sort_lds(uint32_t* s, int P) {
    for (int k = 2; k <= P; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            __syncthreads();
            for (int t = threadIdx.x; t < P / 2; t += NT) {
                const int i = 2 * t - (t & (j - 1));
                const uint32_t a = s[i], b = s[i + j];
                const bool up = (i & k) == 0;
                if ((a > b) == up) {
                    s[i] = b;
                    s[i + j] = a;
                }
            }
        }
    __syncthreads();
}

constexpr int kSortBlock = 1024;

// A whole column in LDS: sorted, and its edges read off.
__global__ __launch_bounds__(kSortBlock) void small_columns_kernel(const uint32_t* __restrict__ keys, int32_t n,
                                                               int64_t ld, int32_t P, const double* __restrict__ q,
                                                               int32_t nq, float* __restrict__ edges,
                                                               int32_t edge_stride) {
    extern __shared__ uint32_t s_key[];
    const uint32_t* col = keys + (int64_t)blockIdx.x * ld;
    for (int i = threadIdx.x; i < P; i += kSortBlock) s_key[i] = i < n ? col[i] : kNanKey;
    sort_lds<kSortBlock>(s_key, P);
    const bool nan = s_key[n - 1] == kNanKey;
    for (int k = threadIdx.x; k < nq; k += kSortBlock) {
        int64_t lo, hi;
        double g;
        quantile_ranks(n, q[k], lo, hi, g);
        edges[(int64_t)k * edge_stride + blockIdx.x] =
            nan ? __uint_as_float(0x7fc00000u) : quantile_edge(value_of(s_key[lo]), value_of(s_key[hi]), g);
    }
}

// per-column state of the selection, in the caller's workspace
struct Select {
    uint32_t* keys;    // [F][ld]
    uint32_t* packed;  // [F][ld] keys of the intervals that hold a wanted rank
    uint16_t* cls;     // [F][ld] class of every key
    uint32_t* split;   // [F][1 << STEPS] splitters (the last entry unused)
    uint32_t* count;   // [F][2 << STEPS] keys per class
    uint2* seg;        // [F][1 << STEPS] first packed key of an interval (~0: not needed), its keys
    uint32_t* cursor;  // [F][1 << STEPS]
    uint4* want;       // [F][nq] class and rank in it, of the lower and the upper rank
    uint32_t* nan;     // [F] 1 if the column holds a NaN
    int64_t n, ld;
};

// Splitters from a sorted sample of 4 << STEPS keys (one from each of as many equal stretches, at a
// hashed place), and the column's counters cleared.
template <int STEPS>
__global__ __launch_bounds__(kSortBlock) void sample_kernel(Select st) {
    constexpr int kSample = 4 << STEPS, kClasses = 2 << STEPS;
    __shared__ uint32_t s_key[kSample];
    const uint32_t* col = st.keys + (int64_t)blockIdx.x * st.ld;
    for (int i = threadIdx.x; i < kSample; i += kSortBlock) {
        const int64_t a = st.n * i / kSample, b = st.n * (i + 1) / kSample;  // n > kSmall >= kSample: not empty
        const uint64_t h = (uint64_t)((uint32_t)i * 2654435761u ^ 0x9e3779b9u);
        s_key[i] = col[a + (int64_t)((h * (uint64_t)(b - a)) >> 32)];
    }
    sort_lds<kSortBlock>(s_key, kSample);
    for (int i = threadIdx.x; i < (1 << STEPS); i += kSortBlock)
        st.split[((int64_t)blockIdx.x << STEPS) + i] = s_key[min(4 * i + 3, kSample - 1)];
    for (int i = threadIdx.x; i < kClasses; i += kSortBlock) st.count[(int64_t)blockIdx.x * kClasses + i] = 0u;
    if (threadIdx.x == 0) st.nan[blockIdx.x] = 0u;
}

// Bound by the LDS probes (STEPS + 1 per key, mostly random: 16 clocks each at STEPS 10, the LDS active
// 95% of the time); 8 searches per thread run side by side.
template <int STEPS>
__global__ __launch_bounds__(kBlock) void count_kernel(Select st) {
    constexpr int kSplits = (1 << STEPS) - 1, kClasses = 2 << STEPS, kPer = 8;
    __shared__ uint32_t s_split[kSplits + 1];
    __shared__ uint32_t s_count[kClasses];
    __shared__ uint32_t s_nan;
    const int64_t f = blockIdx.y;
    for (int i = threadIdx.x; i <= kSplits; i += kBlock) s_split[i] = st.split[(f << STEPS) + i];
    for (int i = threadIdx.x; i < kClasses; i += kBlock) s_count[i] = 0u;
    if (threadIdx.x == 0) s_nan = 0u;
    __syncthreads();
    const uint32_t base = (uint32_t)(size_t)(lds_word*)s_split;
    const int64_t r1 = min(st.n, (int64_t)(blockIdx.x + 1) * kChunkKeys);
    const uint32_t* col = st.keys + f * st.ld;
    uint16_t* out = st.cls + f * st.ld;
    bool nan = false;
    for (int64_t r = (int64_t)blockIdx.x * kChunkKeys + (int64_t)threadIdx.x * kPer; r < r1; r += kBlock * kPer) {
        // ld is a multiple of 16: the vector accesses stay inside the column's stride
        const uint4 a = *reinterpret_cast<const uint4*>(col + r), b = *reinterpret_cast<const uint4*>(col + r + 4);
        const uint32_t key[kPer] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
        uint32_t at[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) at[k] = base;
#pragma unroll
        for (int s = STEPS - 1; s >= 0; --s)
#pragma unroll
            for (int k = 0; k < kPer; ++k)
                at[k] += *((const lds_word*)(size_t)at[k] + (1 << s) - 1) < key[k] ? 4u << s : 0u;
        uint32_t c[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const uint32_t i = (at[k] - base) >> 2;
            c[k] = 2u * i + (i < (uint32_t)kSplits && *(const lds_word*)(size_t)at[k] == key[k] ? 1u : 0u);
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            if (r + k < r1) {
                atomicAdd(&s_count[c[k]], 1u);
                nan |= key[k] == kNanKey;
            }
        *reinterpret_cast<uint4*>(out + r) =
            make_uint4(c[0] | c[1] << 16, c[2] | c[3] << 16, c[4] | c[5] << 16, c[6] | c[7] << 16);
    }
    if (nan) s_nan = 1u;
    __syncthreads();
    for (int i = threadIdx.x; i < kClasses; i += kBlock)
        if (s_count[i]) atomicAdd(&st.count[f * kClasses + i], s_count[i]);
    if (threadIdx.x == 0 && s_nan) atomicOr(&st.nan[f], 1u);
}

// exclusive prefix over the workgroup's threads of one value each; ends with a barrier
__device__ __forceinline__ uint32_t scan_excl(uint32_t v, uint32_t* s_w) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    uint32_t incl = v;
#pragma unroll
    for (int m = 1; m < kWave; m <<= 1) {
        const uint32_t o = __shfl_up(incl, m);
        if (lane >= m) incl += o;
    }
    if (lane == kWave - 1) s_w[wave] = incl;
    __syncthreads();
    uint32_t before = 0u;
#pragma unroll
    for (int w = 0; w < kBlock / kWave; ++w) before += w < wave ? s_w[w] : 0u;
    __syncthreads();
    return before + incl - v;
}

template <int STEPS>
__global__ __launch_bounds__(kBlock) void ranks_kernel(Select st, const double* __restrict__ q, int32_t nq) {
    constexpr int kClasses = 2 << STEPS, kIntervals = 1 << STEPS;
    constexpr int kPer = (kClasses + kBlock - 1) / kBlock, kPerI = (kIntervals + kBlock - 1) / kBlock;
    __shared__ uint32_t s_cum[kClasses + 1];  // keys before a class
    __shared__ uint32_t s_need[kIntervals];
    __shared__ uint32_t s_w[kBlock / kWave];
    const int64_t f = blockIdx.x;
    uint32_t v[kPer], sum = 0u;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int c = (int)threadIdx.x * kPer + i;
        v[i] = c < kClasses ? st.count[f * kClasses + c] : 0u;
        sum += v[i];
    }
    uint32_t run = scan_excl(sum, s_w);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const int c = (int)threadIdx.x * kPer + i;
        if (c < kClasses) s_cum[c] = run;
        run += v[i];
    }
    if (threadIdx.x == kBlock - 1) s_cum[kClasses] = run;
    for (int i = threadIdx.x; i < kIntervals; i += kBlock) s_need[i] = 0u;
    __syncthreads();
    for (int k = threadIdx.x; k < nq; k += kBlock) {
        int64_t rank[2];
        double g;
        quantile_ranks(st.n, q[k], rank[0], rank[1], g);
        uint32_t out[4];
        for (int j = 0; j < 2; ++j) {
            int lo = 0, hi = kClasses - 1;  // the class with cum[c] <= rank < cum[c + 1]
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (s_cum[mid + 1] > (uint32_t)rank[j])
                    hi = mid;
                else
                    lo = mid + 1;
            }
            if (!(lo & 1)) s_need[lo >> 1] = 1u;
            out[2 * j] = (uint32_t)lo;
            out[2 * j + 1] = (uint32_t)rank[j] - s_cum[lo];
        }
        st.want[f * nq + k] = make_uint4(out[0], out[1], out[2], out[3]);
    }
    __syncthreads();
    uint32_t m[kPerI];
    sum = 0u;
#pragma unroll
    for (int i = 0; i < kPerI; ++i) {
        const int x = (int)threadIdx.x * kPerI + i;
        m[i] = x < kIntervals && s_need[x] ? s_cum[2 * x + 1] - s_cum[2 * x] : 0u;
        sum += m[i];
    }
    run = scan_excl(sum, s_w);
#pragma unroll
    for (int i = 0; i < kPerI; ++i) {
        const int x = (int)threadIdx.x * kPerI + i;
        if (x < kIntervals) {
            st.seg[(f << STEPS) + x] = make_uint2(s_need[x] ? run : ~0u, m[i]);
            st.cursor[(f << STEPS) + x] = 0u;
        }
        run += m[i];
    }
}

// The keys of the needed intervals to their places: per 2048 keys, ranks within the workgroup by
// LDS atomics and one global reservation per interval. The order within an interval is free (the
// selection does not depend on it).
template <int STEPS>
__global__ __launch_bounds__(kBlock) void gather_kernel(Select st) {
    constexpr int kIntervals = 1 << STEPS, kPer = 8;
    __shared__ uint32_t s_off[kIntervals];
    __shared__ uint32_t s_cnt[kIntervals];
    const int64_t f = blockIdx.y;
    for (int i = threadIdx.x; i < kIntervals; i += kBlock) s_off[i] = st.seg[(f << STEPS) + i].x;
    const int64_t r1 = min(st.n, (int64_t)(blockIdx.x + 1) * kChunkKeys);
    const uint32_t* col = st.keys + f * st.ld;
    const uint16_t* cls = st.cls + f * st.ld;
    uint32_t* out = st.packed + f * st.ld;
    for (int64_t rb = (int64_t)blockIdx.x * kChunkKeys; rb < r1; rb += kBlock * kPer) {
        for (int i = threadIdx.x; i < kIntervals; i += kBlock) s_cnt[i] = 0u;
        __syncthreads();
        const int64_t r = rb + (int64_t)threadIdx.x * kPer;
        uint32_t at[kPer], rank[kPer];
        uint4 w = make_uint4(0u, 0u, 0u, 0u), k0 = w, k1 = w;
        if (r < r1) {
            w = *reinterpret_cast<const uint4*>(cls + r);
            k0 = *reinterpret_cast<const uint4*>(col + r);
            k1 = *reinterpret_cast<const uint4*>(col + r + 4);
        }
        const uint32_t cw[4] = {w.x, w.y, w.z, w.w};
        const uint32_t key[kPer] = {k0.x, k0.y, k0.z, k0.w, k1.x, k1.y, k1.z, k1.w};
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const uint32_t c = (cw[k >> 1] >> (16 * (k & 1))) & 0xffffu;
            const bool take = r + k < r1 && !(c & 1u) && s_off[c >> 1] != ~0u;
            at[k] = take ? c >> 1 : ~0u;
            rank[k] = take ? atomicAdd(&s_cnt[c >> 1], 1u) : 0u;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < kIntervals; i += kBlock)
            if (s_cnt[i]) s_cnt[i] = s_off[i] + atomicAdd(&st.cursor[(f << STEPS) + i], s_cnt[i]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < kPer; ++k)
            if (at[k] != ~0u) out[s_cnt[at[k]] + rank[k]] = key[k];
        __syncthreads();
    }
}

// One workgroup per (quantile, column). Its lower rank by radix selection over its interval, eight
// bits a pass (an interval of up to 8 keys per thread stays in registers); the upper rank is the
// next key: the same one while copies are left, else the least greater key of the interval, or the
// least key of the upper rank's own class.
template <int STEPS>
__global__ __launch_bounds__(kBlock) void select_kernel(Select st, const double* __restrict__ q, int32_t nq,
                                                    float* __restrict__ edges, int32_t edge_stride) {
    constexpr int kRegs = 8;
    __shared__ uint32_t s_hist[256];
    __shared__ uint32_t s_w[kBlock / kWave];
    __shared__ uint32_t s_pick[3];  // digit, keys below it, keys in it
    __shared__ uint32_t s_min;
    const int k = blockIdx.x;
    const int64_t f = blockIdx.y;
    float* edge = edges + (int64_t)k * edge_stride + f;
    if (st.nan[f]) {  // uniform
        if (threadIdx.x == 0) *edge = __uint_as_float(0x7fc00000u);
        return;
    }
    const uint4 want = st.want[f * nq + k];
    const uint32_t* split = st.split + (f << STEPS);
    // f(key) over an interval's keys, from registers or memory
    const uint2 seg = want.x & 1u ? make_uint2(0u, 0u) : st.seg[(f << STEPS) + (want.x >> 1)];
    const uint32_t* src = st.packed + f * st.ld + seg.x;
    uint32_t reg[kRegs];
    const bool in_regs = seg.y <= kRegs * kBlock;
#pragma unroll
    for (int i = 0; i < kRegs; ++i) {
        const uint32_t x = threadIdx.x + i * kBlock;
        reg[i] = in_regs && x < seg.y ? src[x] : 0u;
    }
    auto each = [&](auto fn) {
        if (in_regs) {
#pragma unroll
            for (int i = 0; i < kRegs; ++i)
                if (threadIdx.x + i * kBlock < seg.y) fn(reg[i]);
        } else {
            for (uint32_t x = threadIdx.x; x < seg.y; x += kBlock) fn(src[x]);
        }
    };
    uint32_t lower, copies = 0u, rank = want.y;  // copies: keys equal to `lower` in its class
    if (want.x & 1u) {
        lower = split[want.x >> 1];
    } else {
        uint32_t prefix = 0u, mask = 0u;
        for (int shift = 24; shift >= 0; shift -= 8) {
            s_hist[threadIdx.x] = 0u;
            __syncthreads();
            each([&](uint32_t x) {
                if ((x & mask) == prefix) atomicAdd(&s_hist[(x >> shift) & 255u], 1u);
            });
            __syncthreads();
            const uint32_t h = s_hist[threadIdx.x];
            const uint32_t before = scan_excl(h, s_w);
            if (rank >= before && rank - before < h) {
                s_pick[0] = threadIdx.x;
                s_pick[1] = before;
                s_pick[2] = h;
            }
            __syncthreads();
            prefix |= s_pick[0] << shift;
            mask |= 255u << shift;
            rank -= s_pick[1];
            copies = s_pick[2];
            __syncthreads();
        }
        lower = prefix;
    }
    uint32_t upper = lower;
    if (want.z != want.x) {  // the first key of a later class
        if (want.z & 1u) {
            upper = split[want.z >> 1];
        } else {
            const uint2 next = st.seg[(f << STEPS) + (want.z >> 1)];
            if (threadIdx.x == 0) s_min = kNanKey;
            __syncthreads();
            uint32_t m = kNanKey;
            for (uint32_t x = threadIdx.x; x < next.y; x += kBlock) m = min(m, st.packed[f * st.ld + next.x + x]);
            atomicMin(&s_min, m);
            __syncthreads();
            upper = s_min;
        }
    } else if (!(want.x & 1u) && rank + (want.w - want.y) >= copies) {  // past the copies of `lower`
        if (threadIdx.x == 0) s_min = kNanKey;
        __syncthreads();
        uint32_t m = kNanKey;
        each([&](uint32_t x) { m = x > lower ? min(m, x) : m; });
        atomicMin(&s_min, m);
        __syncthreads();
        upper = s_min;
    }
    if (threadIdx.x == 0) {
        int64_t lo, hi;
        double g;
        quantile_ranks(st.n, q[k], lo, hi, g);
        *edge = quantile_edge(value_of(lower), value_of(upper), g);
    }
}

int64_t key_ld(int64_t n) { return (n + 15) / 16 * 16; }

// 1023 splitters keep an interval of 1M rows near 1000 keys; below half a million rows 255 do, and
// a search is two probes shorter
int steps_for(int64_t n) { return n > (1 << 19) ? 10 : 8; }

// carves the workspace (256-byte pieces); returns its size
int64_t carve(Select& st, char* work, int64_t n, int32_t F, int32_t nq) {
    const int64_t ld = key_ld(n), I = int64_t(1) << steps_for(n);
    int64_t at = 0;
    auto take = [&](auto** p, int64_t count) {
        *p = reinterpret_cast<std::remove_reference_t<decltype(**p)>*>(work + at);
        at += (count * (int64_t)sizeof(**p) + 255) / 256 * 256;
    };
    take(&st.keys, F * ld);
    if (n > kSmall) {
        take(&st.packed, F * ld);
        take(&st.cls, F * ld);
        take(&st.split, F * I);
        take(&st.count, F * 2 * I);
        take(&st.seg, F * I);
        take(&st.cursor, F * I);
        take(&st.want, (int64_t)F * nq);
        take(&st.nan, F);
    }
    st.n = n;
    st.ld = ld;
    return at;
}

template <int STEPS>
hipError_t select_columns(const Select& st, int32_t F, const double* q, int32_t nq, float* edges, int32_t edge_stride,
                          hipStream_t s) {
    const unsigned chunks = (unsigned)((st.n + kChunkKeys - 1) / kChunkKeys);
    hipLaunchKernelGGL(sample_kernel<STEPS>, dim3(F), dim3(kSortBlock), 0, s, st);
    hipLaunchKernelGGL(count_kernel<STEPS>, dim3(chunks, F), dim3(kBlock), 0, s, st);
    hipLaunchKernelGGL(ranks_kernel<STEPS>, dim3(F), dim3(kBlock), 0, s, st, q, nq);
    hipLaunchKernelGGL(gather_kernel<STEPS>, dim3(chunks, F), dim3(kBlock), 0, s, st);
    hipLaunchKernelGGL(select_kernel<STEPS>, dim3(nq, F), dim3(kBlock), 0, s, st, q, nq, edges, edge_stride);
    return hipGetLastError();
}

}  // namespace

int64_t quantile_work_bytes(int64_t n, int32_t F, int32_t nq) {
    Select st{};
    return carve(st, nullptr, n, F, nq);
}

hipError_t launch_column_quantiles(const float* x, int64_t n, int64_t row_stride, int64_t col_stride, int32_t F,
                                   const double* q, int32_t nq, float* edges, int32_t edge_stride, void* work,
                                   hipStream_t s) {
    if (n < 1 || n > kMaxQuantileRows || F < 1 || F > 65535 || nq < 1 || nq > 254 ||
        (row_stride != 1 && col_stride != 1))
        return hipErrorInvalidValue;
    Select st{};
    carve(st, static_cast<char*>(work), n, F, nq);
    if (col_stride == 1) {
        const int64_t ftiles = (F + kTile - 1) / kTile;
        const int64_t grid = (n + kTile - 1) / kTile * ftiles;
        if (grid > INT32_MAX) return hipErrorInvalidValue;
        hipLaunchKernelGGL(keys_from_rows_kernel, dim3((unsigned)grid), dim3(kBlock), 0, s, x, n, row_stride, F,
                           st.keys, st.ld, (int32_t)ftiles);
    } else {
        const unsigned gx = (unsigned)std::min<int64_t>((n + kBlock * 8 - 1) / (kBlock * 8), 4096);
        hipLaunchKernelGGL(keys_from_columns_kernel, dim3(gx, F), dim3(kBlock), 0, s, x, n, col_stride, st.keys,
                           st.ld);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (n <= kSmall) {
        int P = 2;
        while (P < n) P *= 2;
        hipLaunchKernelGGL(small_columns_kernel, dim3(F), dim3(kSortBlock), (size_t)P * 4, s, st.keys, (int32_t)n,
                           st.ld, P, q, nq, edges, edge_stride);
        return hipGetLastError();
    }
    return steps_for(n) == 10 ? select_columns<10>(st, F, q, nq, edges, edge_stride, s)
                              : select_columns<8>(st, F, q, nq, edges, edge_stride, s);
}

}  // namespace pb
