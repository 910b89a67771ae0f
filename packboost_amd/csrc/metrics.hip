// Round metrics on the device: mean over eras of the Pearson correlation of target and
// predictions (PackBoost._era_correlation_np, booster.py:909-929). Rows are era-major, so era
// e is the row range [era_off[e], era_off[e+1]).
//
// One workgroup per era (or, for long eras, per window of rows), two passes in double (means, then
// centred sums), each reduced in a fixed order (per-thread strided sums, then a fixed tree), so
// results are identical run to run. An era counts when it has >= 2 rows, both population standard
// deviations exceed 1e-12 and the correlation is finite, as in the reference (the mean is NaN when
// none counts).
#include "pb_internal.h"

namespace pb {
namespace {

__device__ double block_sum(double v, double* sh) {
    // fixed-order tree: lanes of a wave, then the waves in order
#pragma unroll
    for (int m = kWave / 2; m >= 1; m >>= 1) v += __shfl_down(v, m);
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = threadIdx.x / kWave;
    __syncthreads();
    if (lane == 0) sh[wave] = v;
    __syncthreads();
    double t = 0.0;
    for (int w = 0; w < kBlock / kWave; ++w) t += sh[w];
    return t;  // every thread holds the total
}

// The correlation of an era of n rows from its centred sums, NaN where the era does not count.
__device__ __forceinline__ double corr_of(double n, double syy, double spp, double syp) {
    const double nan = __longlong_as_double(0x7ff8000000000000ll);
    if (!(n >= 2.0)) return nan;
    const double sdy = sqrt(syy / n), sdp = sqrt(spp / n);
    if (!(sdy > 1e-12 && sdp > 1e-12)) return nan;
    const double v = (syp / n) / (sdy * sdp);
    return isfinite(v) ? v : nan;
}

__global__ __launch_bounds__(kBlock) void era_corr_kernel(const float* __restrict__ y,
                                                      const float* __restrict__ p,
                                                      const int32_t* __restrict__ era_off,
                                                      double* __restrict__ era_corr) {
    __shared__ double sh[kBlock / kWave];
    const int e = blockIdx.x;
    const int r0 = era_off[e], r1 = era_off[e + 1];
    const int n = r1 - r0;
    double sy = 0.0, sp = 0.0;
    for (int64_t r = (int64_t)r0 + threadIdx.x; r < r1; r += kBlock) {  // past 2^31 at the last rows
        sy += (double)y[r];
        sp += (double)p[r];
    }
    sy = block_sum(sy, sh);
    sp = block_sum(sp, sh);
    const double my = n > 0 ? sy / n : 0.0, mp = n > 0 ? sp / n : 0.0;
    double syy = 0.0, spp = 0.0, syp = 0.0;
    for (int64_t r = (int64_t)r0 + threadIdx.x; r < r1; r += kBlock) {
        const double dy = (double)y[r] - my, dp = (double)p[r] - mp;
        syy += dy * dy;
        spp += dp * dp;
        syp += dy * dp;
    }
    syy = block_sum(syy, sh);
    spp = block_sum(spp, sh);
    syp = block_sum(syp, sh);
    if (threadIdx.x == 0) era_corr[e] = corr_of(n, syy, spp, syp);
}

// Mean over the counted eras by one workgroup in a fixed order (strided sums, then a tree): a single
// thread walking them waited on a load per era (40 us for 574).
__global__ __launch_bounds__(kBlock) void era_corr_mean_kernel(const double* __restrict__ era_corr, int32_t E,
                                                           double* __restrict__ out) {
    __shared__ double sh[kBlock / kWave];
    double s = 0.0, k = 0.0;
    for (int e = threadIdx.x; e < E; e += kBlock) {
        const double c = era_corr[e];
        if (!isnan(c)) {
            s += c;
            k += 1.0;
        }
    }
    s = block_sum(s, sh);
    k = block_sum(k, sh);
    if (threadIdx.x == 0) out[0] = k > 0.0 ? s / k : __longlong_as_double(0x7ff8000000000000ll);
}

// Eras of any length over many workgroups: one per window of kCorrWin consecutive rows, which keeps
// its rows in registers and takes, for each era that overlaps it, the two passes of era_corr_kernel
// over the overlap (means, then centred sums, in double). The pair (window w, era e) has slot w + e:
// going up through the rows either w or e steps. era_corr_merge_kernel joins an era's windows.
// One workgroup per era left a fit without eras (one era of 200k rows) 188 us per call; 12 + 4 us so.
constexpr int kCorrRows = 16;  // rows per thread
constexpr int kCorrWin = kBlock * kCorrRows;

// One past the last row of the window that starts at w0 (a multiple of kCorrWin below n): w0 +
// kCorrWin passes 2^31 - 1 in the last window of the longest tables. Every row of the window, of the
// last one's lanes too, is then at most w0 + kCorrWin - 1 <= 2^31 - 1.
__host__ __device__ constexpr int window_end(int w0, int n) { return n - w0 < kCorrWin ? n : w0 + kCorrWin; }
constexpr int kLastWin = INT32_MAX - (kCorrWin - 1);
static_assert(kLastWin % kCorrWin == 0 && window_end(kLastWin, INT32_MAX) == INT32_MAX &&
                  window_end(kLastWin, kLastWin + 1) == kLastWin + 1 &&
                  window_end(kLastWin - kCorrWin, INT32_MAX) == kLastWin && window_end(0, 1) == 1 &&
                  window_end(0, kCorrWin) == kCorrWin,
              "a window ends within the rows, up to 2^31 - 1 of them");

struct Moments {  // of one era's rows in one window
    double n, my, mp, syy, spp, syp;
};

template <int K>
__device__ __forceinline__ void block_sums(double (&v)[K], double (*sh)[4]) {
    static_assert(K <= 4, "four sums at a time");
#pragma unroll
    for (int m = kWave / 2; m >= 1; m >>= 1)
#pragma unroll
        for (int k = 0; k < K; ++k) v[k] += __shfl_down(v[k], m);
    __syncthreads();
    if ((threadIdx.x & (kWave - 1)) == 0)
#pragma unroll
        for (int k = 0; k < K; ++k) sh[threadIdx.x / kWave][k] = v[k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < K; ++k) {
        v[k] = 0.0;
        for (int w = 0; w < kBlock / kWave; ++w) v[k] += sh[w][k];
    }
}

__global__ __launch_bounds__(kBlock) void era_corr_windows_kernel(const float* __restrict__ y, const float* __restrict__ p,
                                                              int32_t n, const int32_t* __restrict__ era_off, int32_t E,
                                                              Moments* __restrict__ slots) {
    __shared__ double sh[kBlock / kWave][4];
    const int w0 = blockIdx.x * kCorrWin;
    const int w1 = window_end(w0, n);
    float yv[kCorrRows], pv[kCorrRows];
#pragma unroll
    for (int i = 0; i < kCorrRows; ++i) {
        const int r = w0 + i * kBlock + (int)threadIdx.x;
        yv[i] = r < w1 ? y[r] : 0.0f;
        pv[i] = r < w1 ? p[r] : 0.0f;
    }
    int lo = 0, hi = E - 1;  // the last era that starts at or before the window
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (era_off[mid] <= w0)
            lo = mid;
        else
            hi = mid - 1;
    }
    for (int e = lo; e < E; ++e) {
        const int r0 = max(era_off[e], w0), r1 = min(era_off[e + 1], w1);
        if (era_off[e] >= w1) break;
        if (r1 <= r0) continue;
        double m[2] = {0.0, 0.0};
#pragma unroll
        for (int i = 0; i < kCorrRows; ++i) {
            const int r = w0 + i * kBlock + (int)threadIdx.x;
            if (r >= r0 && r < r1) {
                m[0] += (double)yv[i];
                m[1] += (double)pv[i];
            }
        }
        block_sums(m, sh);
        const double cnt = (double)(r1 - r0), my = m[0] / cnt, mp = m[1] / cnt;
        double c[3] = {0.0, 0.0, 0.0};
#pragma unroll
        for (int i = 0; i < kCorrRows; ++i) {
            const int r = w0 + i * kBlock + (int)threadIdx.x;
            if (r >= r0 && r < r1) {
                const double dy = (double)yv[i] - my, dp = (double)pv[i] - mp;
                c[0] += dy * dy;
                c[1] += dp * dp;
                c[2] += dy * dp;
            }
        }
        block_sums(c, sh);
        if (threadIdx.x == 0) slots[(int64_t)blockIdx.x + e] = Moments{cnt, my, mp, c[0], c[1], c[2]};
    }
}

// a joined with b (Chan, Golub and LeVeque's pairwise update)
__device__ __forceinline__ void join(Moments& a, const Moments& b) {
    const double n = a.n + b.n;
    if (!(b.n > 0.0)) return;
    const double dy = b.my - a.my, dp = b.mp - a.mp, f = b.n / n, g = a.n * f;
    a.syy += b.syy + dy * dy * g;
    a.spp += b.spp + dp * dp * g;
    a.syp += b.syp + dy * dp * g;
    a.my += dy * f;
    a.mp += dp * f;
    a.n = n;
}

// `lanes` (a power of two) lanes per era: each joins every lanes-th window of the era, then the lanes
// are joined pairwise.
__global__ __launch_bounds__(kBlock) void era_corr_merge_kernel(const Moments* __restrict__ slots,
                                                            const int32_t* __restrict__ era_off, int32_t E,
                                                            int32_t lanes, double* __restrict__ era_corr) {
    const int t = blockIdx.x * kBlock + (int)threadIdx.x;
    const int e = t / lanes, l = t & (lanes - 1);
    Moments a{0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (e < E) {
        const int r0 = era_off[e], r1 = era_off[e + 1];
        if (r1 > r0)
            for (int w = r0 / kCorrWin + l; w <= (r1 - 1) / kCorrWin; w += lanes) join(a, slots[(int64_t)w + e]);
    }
    for (int m = 1; m < lanes; m <<= 1) {
        const Moments b{__shfl_xor(a.n, m),   __shfl_xor(a.my, m),  __shfl_xor(a.mp, m),
                        __shfl_xor(a.syy, m), __shfl_xor(a.spp, m), __shfl_xor(a.syp, m)};
        join(a, b);
    }
    if (e < E && l == 0) era_corr[e] = corr_of(a.n, a.syy, a.spp, a.syp);
}

}  // namespace

hipError_t launch_era_corr(const float* y, const float* p, const int32_t* era_off, int32_t E,
                           double* era_corr, double* out, hipStream_t s) {
    hipLaunchKernelGGL(era_corr_kernel, dim3(E), dim3(kBlock), 0, s, y, p, era_off, era_corr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(era_corr_mean_kernel, dim3(1), dim3(kBlock), 0, s, era_corr, E, out);
    return hipGetLastError();
}

int64_t era_corr_slots(int64_t n, int32_t E) { return (n + kCorrWin - 1) / kCorrWin + E; }

hipError_t launch_era_corr_rows(const float* y, const float* p, int64_t n, const int32_t* era_off, int32_t E,
                                double* era_corr, double* work, double* out, hipStream_t s) {
    const int64_t wins = (n + kCorrWin - 1) / kCorrWin;
    // up to two windows per era on average, a workgroup per era is as wide and skips the join (574
    // eras of 4180 rows beside a running histogram: 32 us against 49 + 5). The average does not see one
    // long era among many short ones: 3M rows beside 400 eras of 3 are one workgroup's, 6 ms.
    if (n < (int64_t)E * (kCorrWin * 2)) return launch_era_corr(y, p, era_off, E, era_corr, out, s);
    int32_t lanes = 1;
    while (lanes < kWave && (int64_t)lanes * E < wins) lanes *= 2;
    Moments* slots = reinterpret_cast<Moments*>(work);
    hipLaunchKernelGGL(era_corr_windows_kernel, dim3((unsigned)wins), dim3(kBlock), 0, s, y, p, (int32_t)n, era_off, E,
                       slots);
    const int64_t threads = (int64_t)E * lanes;
    hipLaunchKernelGGL(era_corr_merge_kernel, dim3((unsigned)((threads + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                       slots, era_off, E, lanes, era_corr);
    hipLaunchKernelGGL(era_corr_mean_kernel, dim3(1), dim3(kBlock), 0, s, era_corr, E, out);
    return hipGetLastError();
}

}  // namespace pb
