// Row-list entry points: the reference's CUDA backend hands its split finder and partition
// per-node, per-era row lists (rows_index with node_row_splits / node_era_splits,
// frontier_cuda.cu:576-716, 719-851). This file serves that interface on the device:
//
//  * partition (frontier_cuda.cu:719-851, frontier_cpu.cpp:446-497): every (node, era)
//    segment of the lists splits stably into its left rows (bin <= threshold) and right rows.
//    Left counts per segment (one wavefront per segment), an exclusive scan over the segments
//    in node-major order, then a stable scatter per segment (a ballot gives each row its rank
//    among the rows of its side that precede it).
//  * gather: the listed rows of a range of nodes, reordered era-major (era, then node, then
//    list order: the layout the histogram kernel reads), with their K sampled bins, values and
//    node slots, placed by a scan over the segment sizes in era-major order.
//  * best thresholds: per (node, feature) the CUDA split finder's sequential choice over
//    thresholds (frontier_cuda.cu:537-560) from the scorer's candidate records.
//
// Every read and write is bounds-checked: a segment outside the row list, a row id outside
// [0, N), a feature outside [0, F) or an output past its capacity sets a status word (the
// first entries of the workspace) instead of touching memory out of range.
#include <algorithm>

#include <mutex>

#include "pb_internal.h"

// Workspace of pb_rowlist_partition_noalloc: a fixed device array instead of caller or
// library allocations (for callers that cannot allocate device memory, e.g. under HIP graph
// capture). Every device the library runs on holds one copy until the process ends. Host code
// never passes `scratch` itself to a kernel (on the host it names a shadow variable, not
// device memory): pb::noalloc_scratch looks up each device's address once, with that device
// current, and launches take that address.
static __device__ __align__(256) int32_t scratch[pb::kNoAllocScratchInts];

namespace pb {

// Device address of `scratch` on the current device, looked up on the first call per device
// (hipGetSymbolAddress with that device current) and kept.
hipError_t noalloc_scratch(int32_t** out) {
    static std::mutex mu;
    static int32_t* addr[kNoAllocMaxDevices] = {};
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kNoAllocMaxDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void* p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        addr[dev] = static_cast<int32_t*>(p);
    }
    *out = addr[dev];
    return hipSuccess;
}

namespace {

constexpr int kRlBlock = 256;
constexpr int kRlWaves = kRlBlock / kWave;
constexpr int kScanItems = 8;
constexpr int kScanTile = kRlBlock * kScanItems;  // pairs per scan tile

// Status words (the first kRlStatus entries of the workspace).
constexpr int kRlStatus = 4;
enum : int { kBadSegment = 0, kBadRow = 1, kBadFeature = 2, kOverflow = 3 };

__device__ __forceinline__ void raise_status(int32_t* status, int which) { status[which] = 1; }

// Segment (s, e) of the row lists: positions [lo, hi) of rows_index. An inconsistent segment
// (outside [0, R) or reversed) counts as empty and reports false.
__device__ __forceinline__ bool seg_range(const int32_t* nrs, const int32_t* nes, int32_t E, int64_t R,
                                          int32_t s, int32_t e, int64_t& lo, int64_t& hi) {
    const int64_t base = nrs[s];
    lo = base + nes[(int64_t)s * (E + 1) + e];
    hi = base + nes[(int64_t)s * (E + 1) + e + 1];
    if (lo < 0 || hi < lo || hi > R) {
        lo = hi = 0;
        return false;
    }
    return true;
}

__device__ __forceinline__ uint64_t lanes_below(int lane) {
    return lane == 0 ? 0ull : (~0ull >> (kWave - lane));
}

__global__ void rl_clear_kernel(int32_t* status) {
    if (threadIdx.x < kRlStatus) status[threadIdx.x] = 0;
}

// vals[2 seg] = left rows of segment seg = s * E + e, vals[2 seg + 1] = right rows.
__global__ __launch_bounds__(kRlBlock) void rl_count_kernel(
    const uint8_t* __restrict__ bins, int64_t N, int64_t ld, int32_t F, const int32_t* __restrict__ rows,
    int64_t R, const int32_t* nrs, const int32_t* nes, int32_t S, int32_t E, const int32_t* feat,
    const int32_t* thr, int32_t* vals, int32_t* status) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t n = (int64_t)S * E;
    for (int64_t seg = (int64_t)blockIdx.x * kRlWaves + threadIdx.x / kWave; seg < n;
         seg += (int64_t)gridDim.x * kRlWaves) {
        const int32_t s = (int32_t)(seg / E), e = (int32_t)(seg - (int64_t)s * E);
        int64_t lo, hi;
        if (!seg_range(nrs, nes, E, R, s, e, lo, hi) && lane == 0) raise_status(status, kBadSegment);
        const int32_t f = feat[s], t = thr[s];
        const bool fok = f >= 0 && f < F;
        if (!fok && lane == 0 && hi > lo) raise_status(status, kBadFeature);
        const uint8_t* col = bins + (fok ? (int64_t)f * ld : 0);
        int left = 0;
        bool bad = false;
        for (int64_t i = lo + lane; i < hi; i += kWave) {
            const int32_t r = rows[i];
            if (r < 0 || r >= N) {
                bad = true;
                continue;
            }
            left += fok && (int32_t)col[r] <= t;
        }
        if (bad) raise_status(status, kBadRow);
        for (int m = kWave / 2; m > 0; m >>= 1) left += __shfl_xor(left, m);
        if (lane == 0) {
            vals[2 * seg] = left;
            vals[2 * seg + 1] = (int32_t)(hi - lo) - left;
        }
    }
}

// Block-wide inclusive scan of pairs (kRlBlock threads). Returns this thread's inclusive value
// and the block total.
__device__ __forceinline__ int2 block_scan_pairs(int2 v, int2& total, int2* s_w) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
    for (int m = 1; m < kWave; m <<= 1) {
        const int32_t y0 = __shfl_up(v.x, m), y1 = __shfl_up(v.y, m);
        if (lane >= m) {
            v.x += y0;
            v.y += y1;
        }
    }
    __syncthreads();
    if (lane == kWave - 1) s_w[wave] = v;
    __syncthreads();
    int2 before = make_int2(0, 0);
    total = make_int2(0, 0);
    for (int w = 0; w < kRlWaves; ++w) {
        if (w < wave) {
            before.x += s_w[w].x;
            before.y += s_w[w].y;
        }
        total.x += s_w[w].x;
        total.y += s_w[w].y;
    }
    return make_int2(v.x + before.x, v.y + before.y);
}

// Tile sums of the n pairs: tiles[2 t + c] = sum of vals[2 j + c] over tile t's pairs.
__global__ __launch_bounds__(kRlBlock) void rl_tile_sums_kernel(const int32_t* vals, int64_t n,
                                                             int32_t* tiles) {
    __shared__ int2 s_w[kRlWaves];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    int2 acc = make_int2(0, 0);
    for (int k = 0; k < kScanItems; ++k) {
        const int64_t j = base + k;
        if (j < n) {
            acc.x += vals[2 * j];
            acc.y += vals[2 * j + 1];
        }
    }
    int2 total;
    block_scan_pairs(acc, total, s_w);
    if (threadIdx.x == 0) {
        tiles[2 * blockIdx.x] = total.x;
        tiles[2 * blockIdx.x + 1] = total.y;
    }
}

// Exclusive scan of the nt tile sums in place, in one workgroup; tiles[2 nt + c] = the totals.
__global__ __launch_bounds__(kRlBlock) void rl_scan_tiles_kernel(int32_t* tiles, int64_t nt) {
    __shared__ int2 s_w[kRlWaves];
    int2 carry = make_int2(0, 0);
    for (int64_t b = 0; b < nt; b += kRlBlock) {
        const int64_t j = b + threadIdx.x;
        const int2 v = j < nt ? make_int2(tiles[2 * j], tiles[2 * j + 1]) : make_int2(0, 0);
        int2 total;
        const int2 inc = block_scan_pairs(v, total, s_w);
        if (j < nt) {
            tiles[2 * j] = carry.x + inc.x - v.x;
            tiles[2 * j + 1] = carry.y + inc.y - v.y;
        }
        carry.x += total.x;
        carry.y += total.y;
    }
    if (threadIdx.x == 0) {
        tiles[2 * nt] = carry.x;
        tiles[2 * nt + 1] = carry.y;
    }
}

// Exclusive scan of the pairs: scan[2 j + c] = sum_{i < j} vals[2 i + c]; scan[2 n + c] = the
// totals (copied from the scanned tiles by block 0).
__global__ __launch_bounds__(kRlBlock) void rl_tile_scan_kernel(const int32_t* vals, int64_t n,
                                                             const int32_t* tiles, int64_t nt,
                                                             int32_t* scan) {
    __shared__ int2 s_w[kRlWaves];
    const int64_t base = (int64_t)blockIdx.x * kScanTile + (int64_t)threadIdx.x * kScanItems;
    int2 v[kScanItems];
    int2 acc = make_int2(0, 0);
    for (int k = 0; k < kScanItems; ++k) {
        const int64_t j = base + k;
        v[k] = j < n ? make_int2(vals[2 * j], vals[2 * j + 1]) : make_int2(0, 0);
        acc.x += v[k].x;
        acc.y += v[k].y;
    }
    int2 total;
    const int2 inc = block_scan_pairs(acc, total, s_w);
    if (blockIdx.x < nt) {
        int2 run = make_int2(tiles[2 * blockIdx.x] + inc.x - acc.x, tiles[2 * blockIdx.x + 1] + inc.y - acc.y);
        for (int k = 0; k < kScanItems; ++k) {
            const int64_t j = base + k;
            if (j < n) {
                scan[2 * j] = run.x;
                scan[2 * j + 1] = run.y;
            }
            run.x += v[k].x;
            run.y += v[k].y;
        }
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        scan[2 * n] = tiles[2 * nt];
        scan[2 * n + 1] = tiles[2 * nt + 1];
    }
}

// [S][E+1] split offsets from the scan (node s's entries are scan pairs s*E .. s*E + E); totals [2]:
// the left and right rows of all segments.
__global__ void rl_splits_kernel(const int32_t* scan, int32_t S, int32_t E, int32_t* left_splits,
                                 int32_t* right_splits, int32_t* totals) {
    if (blockIdx.x == 0 && threadIdx.x < 2) totals[threadIdx.x] = scan[2 * (int64_t)S * E + threadIdx.x];
    const int64_t n = (int64_t)S * (E + 1);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t s = i / (E + 1), e = i - s * (E + 1);
        const int64_t j = s * E + e;
        left_splits[i] = scan[2 * j];
        right_splits[i] = scan[2 * j + 1];
    }
}

// Stable scatter of every segment's rows to its side, in list order (one wavefront per
// segment; the same left test as rl_count_kernel).
__global__ __launch_bounds__(kRlBlock) void rl_scatter_kernel(
    const uint8_t* __restrict__ bins, int64_t N, int64_t ld, int32_t F, const int32_t* __restrict__ rows,
    int64_t R, const int32_t* nrs, const int32_t* nes, int32_t S, int32_t E, const int32_t* feat,
    const int32_t* thr, const int32_t* scan, int32_t* left_out, int32_t* right_out, int64_t cap,
    int32_t* status) {
    const int lane = threadIdx.x & (kWave - 1);
    const uint64_t below = lanes_below(lane);
    const int64_t n = (int64_t)S * E;
    for (int64_t seg = (int64_t)blockIdx.x * kRlWaves + threadIdx.x / kWave; seg < n;
         seg += (int64_t)gridDim.x * kRlWaves) {
        const int32_t s = (int32_t)(seg / E), e = (int32_t)(seg - (int64_t)s * E);
        int64_t lo, hi;
        seg_range(nrs, nes, E, R, s, e, lo, hi);
        const int32_t f = feat[s], t = thr[s];
        const bool fok = f >= 0 && f < F;
        const uint8_t* col = bins + (fok ? (int64_t)f * ld : 0);
        int64_t lpos = scan[2 * seg], rpos = scan[2 * seg + 1];
        bool over = false;
        for (int64_t c = lo; c < hi; c += kWave) {
            const int64_t i = c + lane;
            const bool in = i < hi;
            const int32_t r = in ? rows[i] : -1;
            const bool left = in && fok && r >= 0 && r < N && (int32_t)col[r] <= t;
            const uint64_t bl = __ballot(left);
            const int lrank = __popcll(bl & below);
            const int n_in = (int)min<int64_t>(kWave, hi - c);
            if (in) {
                const int64_t p = left ? lpos + lrank : rpos + (lane - lrank);
                if (p >= 0 && p < cap)
                    (left ? left_out : right_out)[p] = r;
                else
                    over = true;
            }
            const int nl = __popcll(bl);
            lpos += nl;
            rpos += n_in - nl;
        }
        if (over) raise_status(status, kOverflow);
    }
}

// Era-major sizes of the segments of nodes [m0, m1): vals[2 j] = size of segment (m0 + sl, e)
// with j = e * (m1 - m0) + sl; vals[2 j + 1] = 0.
__global__ void rl_sizes_kernel(const int32_t* nrs, const int32_t* nes, int64_t R, int32_t m0, int32_t m1,
                                int32_t E, int32_t* vals, int32_t* status) {
    const int32_t Mc = m1 - m0;
    const int64_t n = (int64_t)Mc * E;
    for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
        const int32_t e = (int32_t)(j / Mc), sl = (int32_t)(j - (int64_t)e * Mc);
        int64_t lo, hi;
        if (!seg_range(nrs, nes, E, R, m0 + sl, e, lo, hi)) raise_status(status, kBadSegment);
        vals[2 * j] = (int32_t)(hi - lo);
        vals[2 * j + 1] = 0;
    }
}

// One wavefront per (segment, block of kGatherFeats features): the segment's rows to their era-major
// positions, with those features' bins (the first block also moves values and slots). The block's
// loads of a row are in flight together; a wavefront per segment left 800 segments of 250 rows and
// 100 features to 3 waves a CU, each waiting on one byte load after another: 416 us for those, 50 us so.
constexpr int kGatherFeats = 8;

__global__ __launch_bounds__(kRlBlock) void rl_gather_kernel(
    const uint8_t* __restrict__ bins, int64_t N, int64_t ld, int32_t F, const int32_t* __restrict__ feats, int32_t K,
    const float* __restrict__ values, const int32_t* __restrict__ rows, int64_t R, const int32_t* nrs,
    const int32_t* nes, int32_t m0, int32_t m1, int32_t E, const int32_t* scan, uint8_t* __restrict__ out_bins,
    int64_t out_ld, float* __restrict__ out_values, uint16_t* __restrict__ out_slot, int32_t* status) {
    const int lane = threadIdx.x & (kWave - 1);
    const int32_t Mc = m1 - m0;
    const int64_t blocks = (K + kGatherFeats - 1) / kGatherFeats > 0 ? (K + kGatherFeats - 1) / kGatherFeats : 1;
    const int64_t n = (int64_t)Mc * E * blocks;
    bool bad_row = false, bad_feat = false, over = false;
    for (int64_t x = (int64_t)blockIdx.x * kRlWaves + threadIdx.x / kWave; x < n;
         x += (int64_t)gridDim.x * kRlWaves) {
        // an era's segments are next to one another for one feature block: its column lines are shared
        const int64_t fb = x / ((int64_t)Mc * E), j = x - fb * ((int64_t)Mc * E);
        const int32_t e = (int32_t)(j / Mc), sl = (int32_t)(j - (int64_t)e * Mc);
        const int k0 = (int)fb * kGatherFeats;
        int64_t lo, hi;
        seg_range(nrs, nes, E, R, m0 + sl, e, lo, hi);
        const int64_t dst = scan[2 * j];
        const uint8_t* col[kGatherFeats];
        bool ok[kGatherFeats];
#pragma unroll
        for (int q = 0; q < kGatherFeats; ++q) {
            const int32_t f = k0 + q < K ? feats[k0 + q] : 0;
            ok[q] = k0 + q < K && f >= 0 && f < F;
            bad_feat |= k0 + q < K && !ok[q] && hi > lo;
            col[q] = bins + (ok[q] ? (int64_t)f * ld : 0);
        }
        for (int64_t i = lo + lane; i < hi; i += kWave) {
            const int64_t d = dst + (i - lo);
            if (d < 0 || d >= out_ld) {
                over = true;
                continue;
            }
            const int32_t r = rows[i];
            const bool rok = r >= 0 && r < N;
            bad_row |= !rok;
            if (fb == 0) {
                out_values[d] = values[i];
                out_slot[d] = (uint16_t)sl;
            }
            uint8_t b[kGatherFeats];
#pragma unroll
            for (int q = 0; q < kGatherFeats; ++q) b[q] = rok && ok[q] ? col[q][r] : (uint8_t)0;
#pragma unroll
            for (int q = 0; q < kGatherFeats; ++q)
                if (k0 + q < K) out_bins[(int64_t)(k0 + q) * out_ld + d] = b[q];
        }
    }
    if (bad_row) raise_status(status, kBadRow);
    if (bad_feat) raise_status(status, kBadFeature);
    if (over) raise_status(status, kOverflow);
}

// era_off[e] = first era-major position of era e; era_off[E] = the row total.
__global__ void rl_era_off_kernel(const int32_t* scan, int32_t Mc, int32_t E, int32_t* era_off) {
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e <= E) era_off[e] = scan[2 * e * Mc];
}

// Per (node, feature): frontier_cuda.cu:537-560's pick over the thresholds in their order
// (score within 1e-12 of the best: the larger left count, then the larger threshold wins; a
// non-finite best leaves threshold -1 and zero sums). One wavefront each: 64 candidate records are
// loaded together and the pick runs over them in order on values every lane reads from the lane
// that holds them (the rule is not transitive, so the order is kept). 16 x 100 picks of 127 records:
// 16 us, where rl_best_lane_kernel waits on each record in turn, 40 us.
__global__ __launch_bounds__(kRlBlock) void rl_best_kernel(const pb_candidate* __restrict__ cand, int64_t MK, int32_t T,
                                                        float* __restrict__ score, int32_t* __restrict__ thr,
                                                        float* __restrict__ left_grad, float* __restrict__ left_hess,
                                                        int64_t* __restrict__ left_count) {
    const int lane = threadIdx.x & (kWave - 1);
    const int64_t i = (int64_t)blockIdx.x * kRlWaves + threadIdx.x / kWave;
    if (i >= MK) return;  // whole wavefronts
    float bs = -__builtin_inff(), blg = 0.0f;
    int32_t bt = -1, bl = 0;
    for (int t0 = 0; t0 < T; t0 += kWave) {
        pb_candidate c;
        c.valid = 0;
        c.score = c.left_grad = 0.0f;
        c.threshold = -1;
        c.left_total = 0;
        if (t0 + lane < T) c = cand[i * T + t0 + lane];
        uint64_t todo = __ballot(c.valid != 0);
        while (todo) {
            const int l = __builtin_ctzll(todo);
            todo &= todo - 1;
            const float sc = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.score), l));
            const int32_t lc = __builtin_amdgcn_readlane(c.left_total, l);
            const int32_t th = __builtin_amdgcn_readlane(c.threshold, l);
            bool better = sc > bs;
            if (!better && fabsf(sc - bs) <= 1e-12f) better = lc > bl || (lc == bl && th > bt);
            if (better) {
                bs = sc;
                bt = th;
                blg = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c.left_grad), l));
                bl = lc;
            }
        }
    }
    if (!(bs == bs) || isinf(bs)) {
        bt = -1;
        blg = 0.0f;
        bl = 0;
    }
    if (lane) return;
    score[i] = bs;
    thr[i] = bt;
    left_grad[i] = blg;
    left_hess[i] = (float)(int64_t)bl;  // squared loss: hess == 1 per row
    left_count[i] = bl;
}

// The same pick by one lane, 64 picks to a wavefront.
__global__ __launch_bounds__(kRlBlock) void rl_best_lane_kernel(const pb_candidate* __restrict__ cand, int64_t MK,
                                                             int32_t T, float* __restrict__ score,
                                                             int32_t* __restrict__ thr, float* __restrict__ left_grad,
                                                             float* __restrict__ left_hess,
                                                             int64_t* __restrict__ left_count) {
    const int64_t i = (int64_t)blockIdx.x * kRlBlock + threadIdx.x;
    if (i >= MK) return;
    float bs = -__builtin_inff(), blg = 0.0f;
    int32_t bt = -1;
    int64_t bl = 0;
    for (int t = 0; t < T; ++t) {
        const pb_candidate c = cand[i * T + t];
        if (!c.valid) continue;
        const float sc = c.score;
        const int64_t lc = c.left_total;
        bool better = sc > bs;
        if (!better && fabsf(sc - bs) <= 1e-12f) better = lc > bl || (lc == bl && c.threshold > bt);
        if (better) {
            bs = sc;
            bt = c.threshold;
            blg = c.left_grad;
            bl = lc;
        }
    }
    if (!(bs == bs) || isinf(bs)) {
        bt = -1;
        blg = 0.0f;
        bl = 0;
    }
    score[i] = bs;
    thr[i] = bt;
    left_grad[i] = blg;
    left_hess[i] = (float)bl;  // squared loss: hess == 1 per row
    left_count[i] = bl;
}

// A lane a pick where that leaves no wait uncovered: few records each, or enough picks to fill the chip,
// where a wavefront each would leave most of its lanes idle. T = 4: equal up to 32768 picks, 262144 in
// 11 us by lanes against 46 by wavefronts; T = 31: 8192 in 11.4 against 8.7, 16384 in 11.4 against
// 14.2; T = 62: 16384 in 31 against 25, 65536 in 36 against 84; T = 127: 32768 in 82 against 88. Records
// past the caches go to wavefronts, which read them side by side: 587776 x 15 in 220 against 256,
// 262144 x 127 in 646 against 1529.
bool pick_by_lane(int64_t MK, int32_t T) {
    const int64_t records = MK * T;
    return T < 48 ? (T <= 16 || MK >= 12288) && records <= 1 << 23 : MK >= 24576 && records <= 1 << 24;
}

// What a call's inputs must satisfy, looked up in one launch (RowlistFacts, cleared by the caller):
// the first `wblocks` workgroups cover the weights and row counts, one (node, era) pair a thread up
// to 512 workgroups (a single workgroup waited on its loads pair after pair: split search over
// 1024 x 574 lists and 8 features 2.25 ms, 1.10 so), the others hess and the drawn columns' bins.
// The least and greatest weight - rows are joined as the bit patterns of non-negative doubles, whose
// order is the numbers'; the least as its complement, so that a cleared record is the neutral one
// of both.
__global__ __launch_bounds__(kRlBlock) void rl_facts_kernel(
    const uint8_t* __restrict__ bins, int64_t N, int64_t ld, int32_t F, const int32_t* __restrict__ feats, int32_t K,
    const float* __restrict__ hess, int64_t n_hess, const float* __restrict__ weights, const int32_t* __restrict__ nes,
    int32_t M, int32_t E, uint32_t limit, int32_t wblocks, pb_rowlist_facts* out) {
    const int lane = threadIdx.x & (kWave - 1);
    if ((int)blockIdx.x < wblocks) {
        unsigned long long least = 0ull, most = 0ull, total = 0ull;
        bool stray = false, counted = false, unit = true;
        for (int64_t x = (int64_t)blockIdx.x * kRlBlock + threadIdx.x; x < (int64_t)M * E;
             x += (int64_t)wblocks * kRlBlock) {
            const int64_t s = x / E, e = x - s * E;
            const int32_t c = nes[s * (E + 1) + e + 1] - nes[s * (E + 1) + e];
            const float w = weights[x];
            if (c > 0) {
                const double d = (double)w - (double)c;
                const unsigned long long key = d > 0.0 ? (unsigned long long)__double_as_longlong(d) : 0ull;  // 0: NaN too
                counted = true;
                unit &= w == 1.0f;
                least = max(least, ~key);
                most = max(most, key);
            } else {
                stray |= !(w == 0.0f);
            }
            if (e == 0) {
                const int64_t rows = (int64_t)nes[s * (E + 1) + E] - nes[s * (E + 1)];
                total += rows > 0 ? (unsigned long long)rows : 0ull;
            }
        }
        if (blockIdx.x == 0)
            for (int32_t k = threadIdx.x; k < K; k += kRlBlock)
                if (feats[k] < 0 || feats[k] >= F) out->bad_feature = 1;
        if (stray) out->stray_weight = 1;
        if (counted) out->counted = 1;
        if (!unit) out->not_unit = 1;
#pragma unroll
        for (int m = 1; m < kWave; m <<= 1) {
            least = max(least, (unsigned long long)__shfl_xor(least, m));
            most = max(most, (unsigned long long)__shfl_xor(most, m));
            total += __shfl_xor(total, m);
        }
        if (lane == 0) {
            if (least) atomicMax(reinterpret_cast<unsigned long long*>(&out->alpha_least), least);
            if (most) atomicMax(reinterpret_cast<unsigned long long*>(&out->alpha_most), most);
            if (total) atomicAdd(reinterpret_cast<unsigned long long*>(&out->rows), total);
        }
        return;
    }
    const int64_t t = (int64_t)((int)blockIdx.x - wblocks) * kRlBlock + threadIdx.x;
    const int64_t stride = (int64_t)((int)gridDim.x - wblocks) * kRlBlock;
    bool bad = false;
    for (int64_t i = t; i < n_hess; i += stride) bad |= !(hess[i] == 1.0f);
    if (bad) out->bad_hess = 1;
    // 16 bytes of a drawn column at a time (byte by byte at its end): any alignment
    struct __attribute__((packed)) Bytes16 {
        uint32_t w[4];
    };
    const int64_t per_col = (N + 15) / 16;
    bool over = false;
    for (int64_t x = t; x < per_col * K; x += stride) {
        const int64_t k = x / per_col, r = (x - k * per_col) * 16;
        const int32_t f = feats[k];
        if (f < 0 || f >= F) continue;
        const uint8_t* p = bins + (int64_t)f * ld + r;
        if (r + 16 <= N) {
            const Bytes16 v = *reinterpret_cast<const Bytes16*>(p);
#pragma unroll
            for (int q = 0; q < 4; ++q) over |= bytes_at_least(v.w[q], limit) != 0u;
        } else {
            for (int64_t b = r; b < N; ++b) over |= p[b - r] >= limit;
        }
    }
    if (over) out->bin_over = 1;
}

int grid_of(int64_t work, int64_t per_block, int64_t cap) {
    return (int)std::max<int64_t>(1, std::min<int64_t>((work + per_block - 1) / per_block, cap));
}

int64_t tiles_of(int64_t n) { return (n + kScanTile - 1) / kScanTile; }

// Exclusive scan of n pairs into scan[2n + 2]; tiles: [2 nt + 2] scratch.
void scan_pairs(const int32_t* vals, int64_t n, int32_t* tiles, int32_t* scan, hipStream_t s) {
    const int64_t nt = tiles_of(n);
    if (nt > 0)
        hipLaunchKernelGGL(rl_tile_sums_kernel, dim3((unsigned)nt), dim3(kRlBlock), 0, s, vals, n, tiles);
    hipLaunchKernelGGL(rl_scan_tiles_kernel, dim3(1), dim3(kRlBlock), 0, s, tiles, nt);
    hipLaunchKernelGGL(rl_tile_scan_kernel, dim3((unsigned)std::max<int64_t>(1, nt)), dim3(kRlBlock), 0, s,
                       vals, n, tiles, nt, scan);
}

}  // namespace

int64_t rowlist_work_elems(int64_t segments) {
    return kRlStatus + 2 * segments + (2 * segments + 2) + (2 * tiles_of(segments) + 2);
}

namespace {

void rowlist_partition_stages(const uint8_t* bins, int64_t N, int64_t ld, int32_t F, const int32_t* rows,
                              int64_t R, const int32_t* nrs, const int32_t* nes, int32_t S, int32_t E,
                              const int32_t* feat, const int32_t* thr, int32_t* left_out,
                              int32_t* right_out, int64_t cap, int32_t* left_splits,
                              int32_t* right_splits, int32_t* status, int32_t* rest, hipStream_t s) {
    const int64_t n = (int64_t)S * E;
    int32_t* vals = rest;               // [2n]
    int32_t* scan = vals + 2 * n;       // [2n + 2]
    int32_t* tiles = scan + 2 * n + 2;  // [2 nt + 2]
    const int g = grid_of(n, kRlWaves, 1 << 16);
    hipLaunchKernelGGL(rl_clear_kernel, dim3(1), dim3(kWave), 0, s, status);
    hipLaunchKernelGGL(rl_count_kernel, dim3(g), dim3(kRlBlock), 0, s, bins, N, ld, F, rows, R, nrs, nes,
                       S, E, feat, thr, vals, status);
    scan_pairs(vals, n, tiles, scan, s);
    hipLaunchKernelGGL(rl_splits_kernel, dim3(grid_of((int64_t)S * (E + 1), 256, 1 << 14)), dim3(256), 0, s,
                       scan, S, E, left_splits, right_splits, vals);  // the scan is done with the counts
    hipLaunchKernelGGL(rl_scatter_kernel, dim3(g), dim3(kRlBlock), 0, s, bins, N, ld, F, rows, R, nrs, nes,
                       S, E, feat, thr, scan, left_out, right_out, cap, status);
}

}  // namespace

hipError_t launch_rowlist_partition(const uint8_t* bins, int64_t N, int64_t ld, int32_t F,
                                    const int32_t* rows, int64_t R, const int32_t* nrs,
                                    const int32_t* nes, int32_t S, int32_t E, const int32_t* feat,
                                    const int32_t* thr, int32_t* left_out, int32_t* right_out,
                                    int64_t cap, int32_t* left_splits, int32_t* right_splits,
                                    int32_t* work, hipStream_t s) {
    rowlist_partition_stages(bins, N, ld, F, rows, R, nrs, nes, S, E, feat, thr, left_out, right_out,
                             cap, left_splits, right_splits, work, work + kRlStatus, s);
    return hipGetLastError();
}

int64_t rowlist_noalloc_max_segments() {
    // largest n with rowlist_work_elems(n) - kRlStatus <= kNoAllocScratchInts
    int64_t lo = 0, hi = kNoAllocScratchInts;
    while (lo < hi) {
        const int64_t mid = (lo + hi + 1) / 2;
        if (rowlist_work_elems(mid) - kRlStatus <= kNoAllocScratchInts) lo = mid; else hi = mid - 1;
    }
    return lo;
}

hipError_t launch_rowlist_partition_noalloc(const uint8_t* bins, int64_t N, int64_t ld, int32_t F,
                                            const int32_t* rows, int64_t R, const int32_t* nrs,
                                            const int32_t* nes, int32_t S, int32_t E,
                                            const int32_t* feat, const int32_t* thr, int32_t* left_out,
                                            int32_t* right_out, int64_t cap, int32_t* left_splits,
                                            int32_t* right_splits, int32_t* status, hipStream_t s) {
    int32_t* rest = nullptr;
    hipError_t e = noalloc_scratch(&rest);
    if (e != hipSuccess) return e;
    rowlist_partition_stages(bins, N, ld, F, rows, R, nrs, nes, S, E, feat, thr, left_out, right_out,
                             cap, left_splits, right_splits, status, rest, s);
    return hipGetLastError();
}

hipError_t launch_rowlist_gather(const uint8_t* bins, int64_t N, int64_t ld, int32_t F,
                                 const int32_t* feats, int32_t K, const float* values,
                                 const int32_t* rows, int64_t R, const int32_t* nrs,
                                 const int32_t* nes, int32_t m0, int32_t m1, int32_t E,
                                 uint8_t* out_bins, int64_t out_ld, float* out_values,
                                 uint16_t* out_slot, int32_t* era_off, int32_t* work, hipStream_t s) {
    const int32_t Mc = m1 - m0;
    const int64_t n = (int64_t)Mc * E;
    int32_t* status = work;
    int32_t* vals = status + kRlStatus;
    int32_t* scan = vals + 2 * n;
    int32_t* tiles = scan + 2 * n + 2;
    hipLaunchKernelGGL(rl_clear_kernel, dim3(1), dim3(kWave), 0, s, status);
    hipLaunchKernelGGL(rl_sizes_kernel, dim3(grid_of(n, 256, 1 << 14)), dim3(256), 0, s, nrs, nes, R, m0, m1,
                       E, vals, status);
    scan_pairs(vals, n, tiles, scan, s);
    const int64_t units = n * std::max<int64_t>(1, (K + kGatherFeats - 1) / kGatherFeats);
    hipLaunchKernelGGL(rl_gather_kernel, dim3(grid_of(units, kRlWaves, 1 << 16)), dim3(kRlBlock), 0, s, bins, N,
                       ld, F, feats, K, values, rows, R, nrs, nes, m0, m1, E, scan, out_bins, out_ld,
                       out_values, out_slot, status);
    hipLaunchKernelGGL(rl_era_off_kernel, dim3(grid_of((int64_t)E + 1, 256, 1 << 14)), dim3(256), 0, s, scan,
                       Mc, E, era_off);
    return hipGetLastError();
}

hipError_t launch_best_thresholds(const pb_candidate* cand, int32_t M, int32_t K, int32_t T,
                                  float* score, int32_t* thr, float* left_grad, float* left_hess,
                                  int64_t* left_count, hipStream_t s) {
    const int64_t n = (int64_t)M * K;
    const bool lanes = pick_by_lane(n, T);
    const int64_t grid = std::max<int64_t>(1, (n + (lanes ? kRlBlock : kRlWaves) - 1) / (lanes ? kRlBlock : kRlWaves));
    if (grid > INT32_MAX) return hipErrorInvalidValue;
    hipLaunchKernelGGL(lanes ? rl_best_lane_kernel : rl_best_kernel, dim3((unsigned)grid), dim3(kRlBlock), 0, s, cand, n, T,
                       score, thr, left_grad, left_hess, left_count);
    return hipGetLastError();
}

hipError_t launch_rowlist_facts(const uint8_t* bins, int64_t N, int64_t ld, int32_t F, const int32_t* feats, int32_t K,
                                const float* hess, int64_t n_hess, const float* weights, const int32_t* nes, int32_t M,
                                int32_t E, int32_t limit, pb_rowlist_facts* out, hipStream_t s) {
    const int64_t work = std::max<int64_t>(n_hess, (N + 15) / 16 * K);
    const int32_t wblocks = grid_of((int64_t)M * E, kRlBlock, 512);
    hipLaunchKernelGGL(rl_facts_kernel, dim3(wblocks + grid_of(work, kRlBlock, 2048)), dim3(kRlBlock), 0, s, bins, N, ld,
                       F, feats, K, hess, n_hess, weights, nes, M, E, (uint32_t)limit, wblocks, out);
    return hipGetLastError();
}

}  // namespace pb
