// Descending sort along the middle of a contiguous f32 [outer, n, inner] of a Device::Hip tensor
// (GpuBackend::sort_desc, src/tensor/gpu/mod.rs:186-191): the values and their I32 source
// positions, in CpuRef's order (src/tensor/kernels.rs:374-413, `sort_order`): every NaN above
// +inf and equal to every other NaN, otherwise total_cmp (+0 above -0), stable (ties keep
// ascending source position). The CUDA backend sorts lanes of up to 4096 on the device and sends
// longer ones through the host (cuda/backend.rs:919-937); here every lane length stays on the
// device.
//
// Each element becomes one 64-bit key, (order key << 32) | ~position, so that a plain descending
// comparison of keys is CpuRef's order with ties broken by position, and no two keys are equal.
// A lane of up to kSortCap elements is sorted by one workgroup (four counting passes over the order
// key in LDS). A longer lane is cut into runs of kSortCap, or of a quarter of it where few lanes
// leave CUs idle, each sorted that way into a scratch buffer, and the runs are merged pairwise
// (merge path: each workgroup stages the two input windows that feed its tile of outputs into LDS
// and merges them there) until one run remains. The last step writes each position's value,
// decoded from its key (a NaN is read back from its source to keep the payload), and its index.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <string>

#include "../../include/noetic_hip.h"
#include "../../include/noetic_ops.h"
#include "nt_internal.hpp"

namespace nt {
namespace {

constexpr int kSortCap = 16384;  // elements one workgroup sorts in LDS (the longest run)
constexpr int kMergeThreads = 256;
constexpr int kMergeItems = 8;   // outputs per thread of a merge pass
constexpr int kMergeTile = kMergeThreads * kMergeItems;  // outputs per workgroup (divides twice a run)
constexpr int kWaveSize = 64;

// CpuRef's order as an unsigned key: every NaN, whatever its sign and payload, above +inf, then
// total_cmp's order.
__device__ __forceinline__ uint32_t order_key(float v) {
    if (v != v) return 0xffffffffu;
    const uint32_t b = __float_as_uint(v);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

__device__ __forceinline__ uint32_t key_pos(uint64_t c) { return ~uint32_t(c); }

// The element a key came from: the order key is a bijection of the value's bits except for NaN
// (every NaN has one key), so only a NaN is read back from x to keep its payload.
__device__ __forceinline__ float key_value(uint64_t c, const float *x, int64_t at_src) {
    const uint32_t k = uint32_t(c >> 32);
    if (k == 0xffffffffu) return x[at_src];
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

struct SortP {
    const float *x;
    float *vals;
    int32_t *idx;
    uint64_t *runs;   // [lanes][n] sorted runs (multi-run lanes)
    int64_t outer, n, inner;
    int32_t chunks;   // runs per lane
    int32_t run;      // elements per run
    int32_t wide;     // merges find their co-ranks with a wave each
};

// Sort run `chunk` of lane `lane` (at most THREADS x E elements) by four stable counting passes over
// the key's bytes, lowest first; a lane of one run is written out directly. Wave w holds elements
// 64 E w .. in E registers per lane, element 64 E w + 64 e + lane in register e, so (w, e, lane) is
// their order. In a pass each wave counts its elements per digit in its own LDS row, E steps of 64
// elements: the lanes of one digit find each other by a ballot per bit, an element's rank is the
// count before its step plus the peers before its lane, and the last peer adds the step's peers to
// the count (a wave's LDS operations run in order). The workgroup then sums the counts over digits
// and waves, and each element moves to its place in LDS. Keys are stored inverted, so that the
// ascending passes give the descending order and equal keys keep their positions; padding takes the
// largest inverted key, above every real one. Bound by VALU issue (about 70 instructions per step and
// pass): [64, 128256] in runs of 16384 takes 116 us; the bitonic network of 91 stages before it took
// 254 us for runs of 8192.
template <int THREADS, int E>
__global__ __launch_bounds__(THREADS) void k_sort_runs(SortP p) {
    constexpr int W = THREADS / kWaveSize, CAP = THREADS * E, D = 256;
    __shared__ uint32_t skey[CAP];
    __shared__ uint16_t spos[CAP];
    __shared__ uint32_t cnt[W][D];  // a wave's counts; then each digit's exclusive sum over the waves
    __shared__ uint32_t first[D];   // each digit's first place
    __shared__ uint32_t wsum[D / kWaveSize];
    const int64_t lane_id = blockIdx.x / p.chunks;
    const int chunk = int(blockIdx.x - lane_id * p.chunks);
    const int64_t o = lane_id / p.inner, i = lane_id - o * p.inner;
    const int64_t beg = int64_t(chunk) * p.run;
    const int len = int(std::min<int64_t>(CAP, p.n - beg));
    const int tid = threadIdx.x, lane = tid % kWaveSize, w = tid / kWaveSize;
    const int t0 = w * kWaveSize * E + lane;  // element of register 0
    uint32_t key[E], pos[E], rank[E];
#pragma unroll
    for (int e = 0; e < E; e++) {
        const int t = t0 + e * kWaveSize;
        key[e] = t < len ? ~order_key(p.x[(o * p.n + beg + t) * p.inner + i]) : 0xffffffffu;
        pos[e] = uint32_t(t);
    }
#pragma unroll 1
    for (int shift = 0; shift < 32; shift += 8) {
        for (int d = lane; d < D; d += kWaveSize) cnt[w][d] = 0;
#pragma unroll
        for (int e = 0; e < E; e++) {
            const uint32_t d = (key[e] >> shift) & 255u;
            uint32_t lo = ~0u, hi = ~0u;  // the lanes of this lane's digit
#pragma unroll
            for (int b = 0; b < 8; b++) {
                const uint32_t bit = uint32_t(int32_t(key[e] << (31 - shift - b)) >> 31);  // all ones or none
                const uint64_t bal = __builtin_amdgcn_ballot_w64(bit != 0);
                lo &= ~(uint32_t(bal) ^ bit);
                hi &= ~(uint32_t(bal >> 32) ^ bit);
            }
            const uint32_t before = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0u));
            const uint32_t total = uint32_t(__popc(lo) + __popc(hi));
            asm volatile("" ::: "memory");
            const uint32_t old = cnt[w][d];
            asm volatile("" ::: "memory");
            if (before + 1 == total) cnt[w][d] = old + total;
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            rank[e] = old + before;
        }
        __syncthreads();
        uint32_t sum = 0, incl = 0;
        if (tid < D) {
#pragma unroll
            for (int v = 0; v < W; v++) {
                const uint32_t c = cnt[v][tid];
                cnt[v][tid] = sum;
                sum += c;
            }
            incl = sum;
#pragma unroll
            for (int s = 1; s < kWaveSize; s <<= 1) {
                const uint32_t up = uint32_t(__shfl_up(int(incl), s, kWaveSize));
                if (lane >= s) incl += up;
            }
            if (lane == kWaveSize - 1) wsum[w] = incl;
        }
        __syncthreads();
        if (tid < D) {
            uint32_t base = 0;
            for (int v = 0; v < w; v++) base += wsum[v];
            first[tid] = base + incl - sum;
        }
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; e++) {
            const uint32_t d = (key[e] >> shift) & 255u;
            const uint32_t at = first[d] + cnt[w][d] + rank[e];
            skey[at] = key[e];
            spos[at] = uint16_t(pos[e]);
        }
        __syncthreads();
        if (shift < 24) {
#pragma unroll
            for (int e = 0; e < E; e++) {
                key[e] = skey[t0 + e * kWaveSize];
                pos[e] = spos[t0 + e * kWaveSize];
            }
        }
    }
    for (int t = tid; t < len; t += THREADS) {
        const uint32_t src = uint32_t(beg) + spos[t];
        const uint64_t c = (uint64_t(~skey[t]) << 32) | uint64_t(~src);
        if (p.chunks == 1) {
            const int64_t at = (o * p.n + t) * p.inner + i;
            p.vals[at] = key_value(c, p.x, (o * p.n + src) * p.inner + i);
            p.idx[at] = int32_t(src);
        } else {
            p.runs[lane_id * p.n + beg + t] = c;
        }
    }
}

// Elements per run. A lane that one workgroup can hold is one run. Longer lanes whose runs of kSortCap
// would leave most CUs idle are cut four times finer: the runs are bound by one workgroup's time, and two
// more merge passes (8.5 us each) cost less than it saves. Measured (us, runs of 16384 and halving co-ranks /
// this rule): 1 row of 32000 57.1 / 40.9, 1 of 128256 80.9 / 59.0, 8 of 50257 70.4 / 56.1, 8 of 128256 (64
// runs) 95.0 / 85.8; from there on the two meet (16 of 128256 keep runs of 16384, 102.5).
int32_t sort_run(int64_t lanes, int64_t n) {
    if (n <= kSortCap) return kSortCap;
    return lanes * ((n + kSortCap - 1) / kSortCap) <= 64 ? kSortCap / 4 : kSortCap;
}

// Up to this many workgroups a merge pass waits for its co-ranks' dependent loads, past it for the loads'
// number: a pass over [1, 128256] takes 8.5 us with a wave's co-ranks and 12 by halving, over
// [64, 128256] (4032 workgroups) 44.6 and 35.9.
constexpr int64_t kWideMerges = 512;

// Threads and elements per thread for runs of up to `longest` elements: the smallest that hold them.
void launch_runs(const SortP &p, int64_t longest, int64_t blocks, hipStream_t s) {
    const dim3 grid{unsigned(blocks)};
    if (longest <= 256) hipLaunchKernelGGL((k_sort_runs<256, 1>), grid, dim3(256), 0, s, p);
    else if (longest <= 1024) hipLaunchKernelGGL((k_sort_runs<256, 4>), grid, dim3(256), 0, s, p);
    else if (longest <= 4096 && p.chunks == 1) hipLaunchKernelGGL((k_sort_runs<256, 16>), grid, dim3(256), 0, s, p);
    else if (longest <= 4096) hipLaunchKernelGGL((k_sort_runs<1024, 4>), grid, dim3(1024), 0, s, p);
    else if (longest <= 8192) hipLaunchKernelGGL((k_sort_runs<1024, 8>), grid, dim3(1024), 0, s, p);
    else hipLaunchKernelGGL((k_sort_runs<1024, 16>), grid, dim3(1024), 0, s, p);
}

// How many of the first d outputs of merging descending runs A (la keys) and B (lb keys) come
// from A (the merge path's co-rank; keys are distinct, so there are no ties).
__device__ __forceinline__ int64_t co_rank(const uint64_t *A, int64_t la, const uint64_t *B, int64_t lb, int64_t d) {
    int64_t lo = std::max<int64_t>(0, d - lb), hi = std::min<int64_t>(d, la);
    while (lo < hi) {
        const int64_t mid = (lo + hi) >> 1;
        if (A[mid] > B[d - mid - 1]) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// The same by one wave: its lanes probe 64 ascending points of the range at once, three rounds of
// dependent loads for runs of 65536 where halving takes 17.
__device__ __forceinline__ int64_t co_rank_wave(const uint64_t *A, int64_t la, const uint64_t *B, int64_t lb, int64_t d) {
    const int lane = threadIdx.x % kWaveSize;
    int64_t lo = std::max<int64_t>(0, d - lb), hi = std::min<int64_t>(d, la);
    while (lo < hi) {
        const int64_t span = hi - lo, mid = lo + span * lane / kWaveSize;  // in [lo, hi - 1]
        const int t = __builtin_popcountll(__ballot(A[mid] > B[d - mid - 1]));  // true up to the answer
        const int64_t l = lo;
        if (t > 0) lo = l + span * (t - 1) / kWaveSize + 1;
        if (t < kWaveSize) hi = l + span * t / kWaveSize;
    }
    return lo;
}

// One merge pass: in every lane, runs [base, base + w) and [base + w, base + 2w) (clipped to n)
// into one run of `dst`. A workgroup makes kMergeTile consecutive outputs (kMergeTile divides 2w,
// so they come from one pair of runs): two co-ranks in global memory bound the A and B windows
// that feed them, both windows are staged into LDS with coalesced loads, each thread merges its
// kMergeItems outputs from LDS (its own co-rank by a search in LDS), and the tile is written back
// coalesced (the windows and then the outputs in one 16 KB array, eight workgroups per CU, the
// co-ranks' dependent loads being what a workgroup waits for: a pass over [64, 128256] 65 -> 35.9 us).
// If LAST, the outputs are the values and positions instead of keys.
template <bool LAST>
__global__ __launch_bounds__(kMergeThreads) void k_merge(SortP p, const uint64_t *src, uint64_t *dst, int64_t w,
                                                         int64_t tiles_per_lane) {
    __shared__ uint64_t sk[kMergeTile];  // the A window, then the B window; then the outputs
    __shared__ int64_t cr[2];
    const int tid = threadIdx.x;
    const int64_t lane = blockIdx.x / tiles_per_lane;
    const int64_t n = p.n;
    const int64_t o0 = (blockIdx.x - lane * tiles_per_lane) * kMergeTile;
    const int64_t o1 = std::min<int64_t>(n, o0 + kMergeTile);
    const int64_t base = o0 / (2 * w) * (2 * w);
    const int64_t la = std::min<int64_t>(w, n - base);
    const int64_t lb = std::max<int64_t>(0, std::min<int64_t>(w, n - base - la));
    const uint64_t *A = src + lane * n + base;
    const uint64_t *B = A + la;
    const int64_t d0 = o0 - base, d1 = o1 - base;
    if (p.wide) {
        const int wave = tid / kWaveSize;
        if (wave < 2) {
            const int64_t c = co_rank_wave(A, la, B, lb, wave == 0 ? d0 : d1);
            if (tid % kWaveSize == 0) cr[wave] = c;
        }
    } else if (tid < 2) {
        cr[tid] = co_rank(A, la, B, lb, tid == 0 ? d0 : d1);
    }
    __syncthreads();
    const int64_t a0 = cr[0], b0 = d0 - cr[0];
    const int na = int(cr[1] - cr[0]), nb = int((d1 - cr[1]) - b0);
    const int total = na + nb;
#pragma unroll
    for (int q = 0; q < kMergeItems; q++) {
        const int e = tid + q * kMergeThreads;
        if (e < total) sk[e] = e < na ? A[a0 + e] : B[b0 + e - na];
    }
    __syncthreads();
    const uint64_t *sa = sk, *sb = sk + na;
    const int dl = tid * kMergeItems;
    uint64_t out[kMergeItems];
    if (dl < total) {
        int lo = std::max(0, dl - nb), hi = std::min(dl, na);
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (sa[mid] > sb[dl - mid - 1]) lo = mid + 1;
            else hi = mid;
        }
        int ia = lo, ib = dl - lo;
        // (past a window's end a key of 0, below every real one; the last thread's outputs past
        // `total` are not stored)
        uint64_t ka = ia < na ? sa[ia] : 0, kb = ib < nb ? sb[ib] : 0;
#pragma unroll
        for (int q = 0; q < kMergeItems; q++) {
            const bool from_a = ka > kb;
            out[q] = from_a ? ka : kb;
            if (from_a) ka = ++ia < na ? sa[ia] : 0;
            else kb = ++ib < nb ? sb[ib] : 0;
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kMergeItems; q++)
        if (dl + q < total) sk[dl + q] = out[q];
    __syncthreads();
    const int64_t o = lane / p.inner, i = lane - o * p.inner;
    for (int e = tid; e < total; e += kMergeThreads) {
        const uint64_t c = sk[e];
        if constexpr (LAST) {
            const uint32_t s = key_pos(c);
            const int64_t at = (o * n + o0 + e) * p.inner + i;
            p.vals[at] = key_value(c, p.x, (o * n + s) * p.inner + i);
            p.idx[at] = int32_t(s);
        } else {
            dst[lane * n + o0 + e] = c;
        }
    }
}

}  // namespace
}  // namespace nt

using namespace nt;

extern "C" {

int nt_hip_sort_desc(const float *x, int64_t outer, int64_t n, int64_t inner, float *vals, int32_t *idx) {
    if (outer < 0 || n < 0 || inner < 0) return fail(NT_E_ARG, "sort_desc: negative lanes");
    if (n > int64_t(0x7fffffff)) return fail(NT_E_ARG, "sort_desc: a lane longer than 2^31 - 1 (I32 positions)");
    const int64_t lanes = outer * inner;
    if (lanes == 0 || n == 0) return 0;
    if (!x || !vals || !idx) return fail(NT_E_ARG, "sort_desc: null buffer");
    SortP p{};
    p.x = x;
    p.vals = vals;
    p.idx = idx;
    p.outer = outer;
    p.n = n;
    p.inner = inner;
    p.run = sort_run(lanes, n);
    const int64_t chunks = (n + p.run - 1) / p.run;
    if (lanes * chunks > int64_t(0x7fffffff)) return fail(NT_E_ARG, "sort_desc: too many lanes");
    p.chunks = int32_t(chunks);
    std::unique_lock<std::mutex> lk;
    if (int rc = enter(&lk)) return rc;
    hipStream_t st = ctx().stream;
    if (chunks == 1) {
        launch_runs(p, n, lanes, st);
        return launched("k_sort_runs");
    }
    void *buf[2] = {nullptr, nullptr};
    const size_t bytes = size_t(lanes) * size_t(n) * sizeof(uint64_t);
    if (int rc = scratch_alloc(bytes, &buf[0])) return rc;
    if (int rc = scratch_alloc(bytes, &buf[1])) {
        scratch_release(buf[0]);
        return rc;
    }
    p.runs = static_cast<uint64_t *>(buf[0]);
    launch_runs(p, p.run, lanes * chunks, st);
    int rc = launched("k_sort_runs");
    const int64_t tiles = (n + kMergeTile - 1) / kMergeTile;
    const int64_t blocks = lanes * tiles;
    p.wide = blocks <= kWideMerges;
    if (blocks > int64_t(0x7fffffff)) {
        scratch_release(buf[0]);
        scratch_release(buf[1]);
        return fail(NT_E_ARG, "sort_desc: too many merge tiles");
    }
    int cur = 0;
    for (int64_t w = p.run; !rc && w < n; w *= 2) {
        const uint64_t *src = static_cast<const uint64_t *>(buf[cur]);
        uint64_t *dst = static_cast<uint64_t *>(buf[cur ^ 1]);
        if (2 * w >= n) {
            hipLaunchKernelGGL((k_merge<true>), dim3(unsigned(blocks)), dim3(kMergeThreads), 0, st, p, src, dst, w,
                               tiles);
        } else {
            hipLaunchKernelGGL((k_merge<false>), dim3(unsigned(blocks)), dim3(kMergeThreads), 0, st, p, src, dst, w,
                               tiles);
        }
        rc = launched("k_merge");
        cur ^= 1;
    }
    const int r0 = scratch_release(buf[0]);
    const int r1 = scratch_release(buf[1]);
    return rc ? rc : (r0 ? r0 : r1);
}

}  // extern "C"
