// Batched f32 matmul of a Device::Hip tensor (GpuBackend::matmul, src/tensor/gpu/mod.rs:155-156),
// bit for bit the reference's product. The reference fixes the arithmetic of every output
// (src/tensor/cuda/kernels.rs:14-20, the order of matrixmultiply 0.3.11's sgemm that CpuRef calls
// per batch, src/tensor/kernels.rs:415-420): an fma chain from zero over k in order, closed every
// 256 k; the first block's chain is the total and each later block's chain is added to it.
//
// The chains run on the matrix cores. On gfx950 v_mfma_f32_32x32x2_f32 adds its two products one
// after the other, each with one rounding, subnormals kept: the bits of
// fma(a1, b1, fma(a0, b0, c)) (tests/test_matmul_mfma_gpu.py compares them on normal, subnormal,
// cancelling, overflowing and special operands). So a run of them over ascending k is the
// reference's chain, at twice the rate of v_fma_f32 (157.3 against 78.6 TFLOP/s nominal).
//
// A workgroup computes a 128x128 (eight waves of 2 x 1 MFMA tiles) or 64x64 (four waves of one) tile;
// panels of 32 k go through LDS, double-buffered, one barrier per panel.
// LDS holds 32 k of a row (of A) or column (of B) with each 8 k as [0 2 4 6 | 1 3 5 7]: an MFMA's
// lanes 0-31 take its first k and lanes 32-63 its second, so one 16-byte read per lane holds four
// MFMAs' operands. Rows are 36 words apart: the reads are free of bank conflicts. A panel of 128 x
// 128 costs a wave 12 such reads against 32 MFMAs of 64 cycles, so what bounds a large product is
// the matrix cores' rate: 4096^3 takes 1118 us (123 TFLOP/s; the VALU kernel before it 1920 us, 71.6),
// 2048^3 142 us (251), 1024^3 27.7 us (50.0). Past the last k both operands are padded with -0 and +0, whose product
// -0 leaves every sum as it is (+0 would turn a chain's -0 into +0).
//
// A half product (GpuBackend::matmul_half; HALF) takes the same path: panels of 64 k rounded to bf16 on
// their way into LDS, 16 k per v_mfma_f32_32x32x16_bf16, one accumulator over the whole of k.
// Against the kernel before it, whose loads were branches between whole, unaligned and last panels:
// 1024^3 24.2 -> 12.6 us, 247 x 525 x 914 39.9 -> 9.1, 300 x 3000 x 3000 391 -> 38.7, 2048^3 59.1 -> 35.7.
//
// Workgroups are renumbered so that each of the 8 XCDs (which the hardware deals consecutive
// workgroups to in turn) works on a contiguous run of tiles, whose A panels then stay in that
// XCD's L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <type_traits>

#include "../../include/noetic_hip.h"
#include "../../include/noetic_ops.h"
#include "nt_internal.hpp"
#include "nt_mfma_pipe.hpp"

#ifndef NT_KERNELS_SHA
#define NT_KERNELS_SHA "unknown"
#endif

namespace nt {
namespace {

constexpr int kMmThreads = 256;
constexpr int kKC = 256;   // the chain is closed every kKC k
constexpr int kMaxBatchDims = NT_MAX_RANK - 2;
constexpr int kLdsRow = 36;  // words between LDS rows: a panel's 32 words (128 bytes) and a pad of 4

struct MatmulP {
    const float *a, *b;
    float *c;
    int64_t a_off, b_off;          // element offsets of batch 0
    int64_t a_rs, a_cs, b_rs, b_cs;
    int64_t bshape[kMaxBatchDims]; // the output's batch dimensions
    int64_t a_bs[kMaxBatchDims];   // per batch dimension: A's stride (0 where A broadcasts)
    int64_t b_bs[kMaxBatchDims];
    int64_t blocks;                // splits * batches * tiles_m * tiles_n
    float *slices;                 // split-k: [ceil(k / 256)][batches * m * n], one per 256-k block
    int64_t outputs;               // batches * m * n
    int32_t m, n, k;
    int32_t tm, tn;                // tiles along m and n
    int32_t nbd;                   // batch dimensions
    int32_t kc_per;                // split-k: 256-k blocks per split
};

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// (16-byte loads of elements that are only 4-byte aligned, as rows of an odd length start)
typedef f32x4_t f32x4_any __attribute__((aligned(4)));

// Eight elements k .. k + 7 of one row of A (column of B) at src, `stride` apart (K1: adjacent), into
// two vectors in order: what reorders them waits for the loads, so that is left to the store into LDS.
template <bool K1>
__device__ __forceinline__ void load8(const float *src, int64_t stride, f32x4_t (&x)[2]) {
    if constexpr (K1) {
        x[0] = reinterpret_cast<const f32x4_any *>(src)[0];
        x[1] = reinterpret_cast<const f32x4_any *>(src)[1];
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) x[e / 4][e % 4] = src[e * stride];
    }
}

// The same of the last panel, when K does not end with it: elements at or past `lim` are `pad`.
template <bool K1>
__device__ __forceinline__ void load8_tail(const float *src, int64_t stride, int lim, float pad, f32x4_t (&x)[2]) {
    if (lim >= 8) {
        load8<K1>(src, stride, x);
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) x[e / 4][e % 4] = e < lim ? src[e * stride] : pad;
    }
}

// A tile of NM x NN waves, each WM x WN MFMA tiles of 32 x 32. Two waves per SIMD (eight per 128 x 128
// tile) let one's MFMAs cover the other's waits: 4096^3 in 1118 us (123 TFLOP/s, 78% of the matrix
// cores' 157.3) against 1202 with four waves of 2 x 2 MFMA tiles; 256 x 128 tiles took 1152.
// AHEAD: panels whose loads are in flight beside the one on its way through LDS. The 64 tile's launches
// are the ones too small to fill the chip, where a panel's MFMAs are shorter than its loads' latency
// (f32 128 x 2000 x 300: 20.1 -> 13.2 us with a second panel ahead; a large product gains nothing).
template <int WM_, int WN_, int NM_, int NN_, int AHEAD_>
struct MmTile {
    static constexpr int WM = WM_, WN = WN_, NM = NM_, NN = NN_, kAhead = AHEAD_;
    static constexpr int kTM = 32 * WM * NM, kTN = 32 * WN * NN, kThreads = 64 * NM * NN;
};
using Tile64 = MmTile<1, 1, 2, 2, 2>;     // 64 x 64, 256 threads
using Tile128 = MmTile<2, 1, 2, 4, 1>;    // 128 x 128, 512 threads

// AK: A is contiguous along k (a_cs == 1): a thread loads 8 k of a row as two 16-byte loads, four
// threads a row of the panel. Otherwise a wave's lanes take consecutive rows, a load for each k.
// BN: a wave's lanes take consecutive columns of B; otherwise B is contiguous along k (b_rs == 1) and
// loaded as A is. Consecutive lanes read consecutive addresses when the view is contiguous along
// either dimension.
// SPLIT: the workgroup covers kc_per 256-k blocks of its tile and writes each block's chain to
// that block's slice; k_fold then closes the chains in order (the same arithmetic, more
// workgroups for outputs too few to fill the chip).
template <bool HALF, class C, bool AK, bool BN, bool SPLIT>
__global__ __launch_bounds__(C::kThreads, 2) void k_matmul(MatmulP p) {
    constexpr int WM = C::WM, WN = C::WN, TM = C::kTM, TN = C::kTN, kThreads = C::kThreads;
    static_assert(!HALF || !SPLIT, "a half product keeps one accumulator over the whole of k");
    constexpr int kBK = HALF ? 64 : 32;      // k per panel: 128 bytes of a row in LDS
    constexpr int kGW = HALF ? 4 : 8;        // LDS words of 8 k
    constexpr int GA = TM * kBK / 8 / kThreads, GB = TN * kBK / 8 / kThreads;  // groups of 8 k per thread and panel
    constexpr float kPadA = HALF ? 0.0f : -0.0f;
    __shared__ __attribute__((aligned(16))) float As[2][TM * kLdsRow];
    __shared__ __attribute__((aligned(16))) float Bs[2][TN * kLdsRow];

    const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    int64_t wg = blockIdx.x;
    const int64_t full = p.blocks / 8 * 8;
    if (wg < full) wg = (wg % 8) * (full / 8) + wg / 8;
    const int64_t per_batch = int64_t(p.tm) * p.tn;
    int64_t z = wg / per_batch;  // split * batches + batch
    const int64_t rem = wg - z * per_batch;
    int kbeg = 0, kend = p.k;
    if constexpr (SPLIT) {
        int64_t nbat = 1;
        for (int d = 0; d < p.nbd; d++) nbat *= p.bshape[d];
        const int sp = int(z / nbat);
        z -= int64_t(sp) * nbat;
        kbeg = sp * p.kc_per * kKC;
        kend = min(p.k, kbeg + p.kc_per * kKC);
    }
    const int row0 = int(rem / p.tn) * TM, col0 = int(rem % p.tn) * TN;
    int64_t ao = p.a_off, bo = p.b_off;
    {
        int64_t q = z;
        for (int d = p.nbd - 1; d >= 0; --d) {
            const int64_t i = q % p.bshape[d];
            q /= p.bshape[d];
            ao += i * p.a_bs[d];
            bo += i * p.b_bs[d];
        }
    }
    const int M = p.m, N = p.n, K = p.k;

    // This thread's groups: their row (column) in the tile, first k in the panel, LDS offset and
    // source. A row past the last one reads row 0 (its outputs are not stored).
    const float *asrc[GA], *bsrc[GB];
    int akg[GA], bkg[GB], alds[GA], blds[GB];
#pragma unroll
    for (int q = 0; q < GA; q++) {
        const int g = tid + kThreads * q, r = AK ? g / (kBK / 8) : g % TM;
        akg[q] = 8 * (AK ? g % (kBK / 8) : g / TM);
        alds[q] = r * kLdsRow + akg[q] / 8 * kGW;
        asrc[q] = p.a + ao + int64_t(row0 + r < M ? row0 + r : 0) * p.a_rs + int64_t(akg[q]) * p.a_cs;
    }
#pragma unroll
    for (int q = 0; q < GB; q++) {
        const int g = tid + kThreads * q, c = BN ? g % TN : g / (kBK / 8);
        bkg[q] = 8 * (BN ? g / TN : g % (kBK / 8));
        blds[q] = c * kLdsRow + bkg[q] / 8 * kGW;
        bsrc[q] = p.b + bo + int64_t(col0 + c < N ? col0 + c : 0) * p.b_cs + int64_t(bkg[q]) * p.b_rs;
    }
    constexpr int NS = C::kAhead;
    f32x4_t ra[NS][GA][2], rb[NS][GB][2];
    auto load = [&](int k0, f32x4_t(&xa)[GA][2], f32x4_t(&xb)[GB][2]) {
#pragma unroll
        for (int q = 0; q < GA; q++) load8<AK>(asrc[q] + int64_t(k0) * p.a_cs, p.a_cs, xa[q]);
#pragma unroll
        for (int q = 0; q < GB; q++) load8<!BN>(bsrc[q] + int64_t(k0) * p.b_rs, p.b_rs, xb[q]);
    };
    auto put8 = [&](float *d, const f32x4_t(&x)[2]) {
        if constexpr (HALF) {
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; e++)
                asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(w[e]) : "v"(x[e / 2][2 * (e % 2)]), "v"(x[e / 2][2 * (e % 2) + 1]));
            *reinterpret_cast<uint4 *>(d) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
            reinterpret_cast<f32x4_t *>(d)[0] = f32x4_t{x[0][0], x[0][2], x[1][0], x[1][2]};
            reinterpret_cast<f32x4_t *>(d)[1] = f32x4_t{x[0][1], x[0][3], x[1][1], x[1][3]};
        }
    };
    auto stash = [&](int s, const f32x4_t(&xa)[GA][2], const f32x4_t(&xb)[GB][2]) {
#pragma unroll
        for (int q = 0; q < GA; q++) put8(&As[s][alds[q]], xa[q]);
#pragma unroll
        for (int q = 0; q < GB; q++) put8(&Bs[s][blds[q]], xb[q]);
    };

    // The wave's part: rows wr .. wr + 32 WM - 1, columns wc .. wc + 32 WN - 1 of the tile.
    const int wr = (wave / C::NN) * 32 * WM, wc = (wave % C::NN) * 32 * WN;
    const int aread = (wr + lane % 32) * kLdsRow + 4 * (lane / 32);
    const int bread = (wc + lane % 32) * kLdsRow + 4 * (lane / 32);
    f32x16_t acc[WM][WN], tot[SPLIT || HALF ? 1 : WM][SPLIT || HALF ? 1 : WN];
    auto clear = [&]() {
#pragma unroll
        for (int i = 0; i < WM; i++)
#pragma unroll
            for (int j = 0; j < WN; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
    };
    clear();
    f32x4_t fa[2][WM], fb[2][WN];  // two groups' operands: one in use, the next on its way from LDS
    auto fetch = [&](int s, int kg) {  // a quarter of the panel: its 8 words from 8 kg on, half of them per lane
#pragma unroll
        for (int i = 0; i < WM; i++)
            fa[kg % 2][i] = *reinterpret_cast<const f32x4_t *>(&As[s][aread + 32 * i * kLdsRow + 8 * kg]);
#pragma unroll
        for (int j = 0; j < WN; j++)
            fb[kg % 2][j] = *reinterpret_cast<const f32x4_t *>(&Bs[s][bread + 32 * j * kLdsRow + 8 * kg]);
    };
    auto group = [&](int kg) {  // its 8 k as four MFMAs of two, or 16 k (8 of each lane) as one
#pragma unroll
        for (int e = 0; e < (HALF ? 1 : 4); e++)
#pragma unroll
            for (int i = 0; i < WM; i++)
#pragma unroll
                for (int j = 0; j < WN; j++) {
                    if constexpr (HALF)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8_t, fa[kg % 2][i]), __builtin_bit_cast(bf16x8_t, fb[kg % 2][j]),
                            acc[i][j], 0, 0, 0);
                    else
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[kg % 2][i][e], fb[kg % 2][j][e], acc[i][j],
                                                                         0, 0, 0);
                }
    };
    // Lane l's value v of MFMA tile (i, j): row wr + 32 i + 8 (v / 4) + 4 (l / 32) + v % 4, column
    // wc + 32 j + l % 32: a store instruction writes 32 consecutive columns of two rows.
    auto put = [&](float *c, const f32x16_t &t, int i, int j) {
        const int col = col0 + wc + 32 * j + lane % 32;
        if (col >= N) return;
#pragma unroll
        for (int v = 0; v < 16; v++) {
            const int row = row0 + wr + 32 * i + 8 * (v / 4) + 4 * (lane / 32) + v % 4;
            if (row < M) c[int64_t(row) * N + col] = t[v];
        }
    };

    auto close = [&](int k0) {  // the chain of the 256-k block that k0 lies in ends
        if constexpr (HALF) return;
        if constexpr (SPLIT) {
#pragma unroll
            for (int i = 0; i < WM; i++)
#pragma unroll
                for (int j = 0; j < WN; j++)
                    put(p.slices + int64_t(k0 / kKC) * p.outputs + z * int64_t(M) * N, acc[i][j], i, j);
        } else if constexpr (!HALF) {
            const bool first = k0 < kKC;
#pragma unroll
            for (int i = 0; i < WM; i++)
#pragma unroll
                for (int j = 0; j < WN; j++)
#pragma unroll
                    for (int v = 0; v < 16; v++) tot[i][j][v] = first ? acc[i][j][v] : acc[i][j][v] + tot[i][j][v];
        }
        if constexpr (!HALF) clear();
    };

    // The whole panels. Panel i's iteration finds its group 0 in registers and the panel whole in LDS
    // buffer s. The next panel is written to the other buffer (last read before the previous
    // barrier) ahead of group 2, and the barrier comes between groups 2 and 3, so that group 3's
    // MFMAs cover the next panel's first reads; the panel after it is loaded meanwhile. (No branch:
    // the last iterations load and store the last panel once more.)
    const int kfull = kbeg + (kend - kbeg) / kBK * kBK, klast = kfull - kBK;
    if (kbeg < kfull) {
        load(kbeg, ra[0], rb[0]);
        stash(0, ra[0], rb[0]);
        load(min(kbeg + kBK, klast), ra[NS - 1], rb[NS - 1]);
        if constexpr (NS == 2) load(min(kbeg + 2 * kBK, klast), ra[0], rb[0]);
        __syncthreads();
        fetch(0, 0);
        auto panel = [&](int s, auto t_c, int k0) {
            constexpr int t = decltype(t_c)::value;  // the next panel's registers
            fetch(s, 1);
            __builtin_amdgcn_sched_barrier(0);
            group(0);
            __builtin_amdgcn_sched_barrier(0);
            fetch(s, 2);
            __builtin_amdgcn_sched_barrier(0);
            group(1);
            __builtin_amdgcn_sched_barrier(0);
            fetch(s, 3);
            stash(s ^ 1, ra[t], rb[t]);
            load(min(k0 + (NS + 1) * kBK, klast), ra[t], rb[t]);
            __builtin_amdgcn_sched_barrier(0);
            group(2);
            __builtin_amdgcn_sched_barrier(0);
            __syncthreads();
            fetch(s ^ 1, 0);
            __builtin_amdgcn_sched_barrier(0);
            group(3);
            __builtin_amdgcn_sched_barrier(0);
            if (!HALF && ((k0 + kBK) % kKC == 0 || k0 + kBK == kend)) close(k0);
        };
        if constexpr (NS == 2) {  // (panel i's registers are set i % 2)
            for (int k0 = kbeg; k0 < kfull; k0 += 2 * kBK) {
                panel(0, std::integral_constant<int, 1>{}, k0);
                if (k0 + kBK >= kfull) break;
                panel(1, std::integral_constant<int, 0>{}, k0 + kBK);
            }
        } else {
            int s = 0;
            for (int k0 = kbeg; k0 < kfull; k0 += kBK, s ^= 1) panel(s, std::integral_constant<int, 0>{}, k0);
        }
    }
    if (kfull < kend) {  // the last panel, when K ends inside it
#pragma unroll
        for (int q = 0; q < GA; q++)
            load8_tail<AK>(asrc[q] + int64_t(kfull) * p.a_cs, p.a_cs, K - kfull - akg[q], kPadA, ra[0][q]);
#pragma unroll
        for (int q = 0; q < GB; q++)
            load8_tail<!BN>(bsrc[q] + int64_t(kfull) * p.b_rs, p.b_rs, K - kfull - bkg[q], 0.0f, rb[0][q]);
        if (kbeg < kfull) __syncthreads();  // (the reads of the last whole panel are done)
        stash(0, ra[0], rb[0]);
        __syncthreads();
#pragma unroll
        for (int kg = 0; kg < 4; kg++) {
            if (kfull + kg * (kBK / 4) < kend) {  // (a quarter past k's end holds padding alone)
                fetch(0, kg);
                group(kg);
            }
        }
        close(kfull);
    }
    if constexpr (!SPLIT) {
#pragma unroll
        for (int i = 0; i < WM; i++)
#pragma unroll
            for (int j = 0; j < WN; j++) {
                if constexpr (HALF) {
                    put(p.c + z * int64_t(M) * N, acc[i][j], i, j);
                } else {
                    if (K == 0)
#pragma unroll
                        for (int v = 0; v < 16; v++) tot[i][j][v] = 0.0f;
                    put(p.c + z * int64_t(M) * N, tot[i][j], i, j);
                }
            }
    }
}

// Split-k's closing pass: per output, the first 256-k block's chain is the total and each later
// block's chain is added to it, in order (the unsplit kernel's closure, element for element).
__global__ void k_fold(const float *slices, int64_t outputs, int nkc, float *out) {
    for (int64_t o = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; o < outputs;
         o += int64_t(gridDim.x) * blockDim.x) {
        float t = slices[o];
        for (int j = 1; j < nkc; j++) t = slices[int64_t(j) * outputs + o] + t;
        out[o] = t;
    }
}

// ------------------------------------------------- matmul_half, packed operands (large products)
// The reduced-precision product (GpuBackend::matmul_half, gpu/mod.rs:157-162; the CUDA backend's
// hgemm_bf16_f32acc, cuda/half_gemm.rs:32-...): f32 operands rounded to bf16 (nearest even), products
// summed in f32 on the matrix cores; k_matmul above with HALF, which rounds as it stages. For
// products of many 256 x 256 output tiles the operands are rounded to bf16 once, into the
// matrix cores' fragment order (the row operand A in row groups of 32, the column operand B
// tile-major in tiles of 256 columns; rows, columns and k past the ends are zeros), and each
// workgroup then runs the bf16 MFMA pipeline of nt_mfma_pipe.hpp over one 256 x 256 tile of one
// batch: the same instruction over the same k order from zero as the staged kernel above, so each
// output is the same sum. The packing reads each f32 operand once and writes half its bytes; the
// tiles then read bf16 fragments only, 16 or 32 bytes per lane per load.

// The batch element offsets of A and B for output batch z (broadcast dimensions repeat).
__device__ __forceinline__ void batch_offsets(const MatmulP &p, int64_t z, int64_t *ao, int64_t *bo) {
    int64_t a = p.a_off, b = p.b_off, q = z;
    for (int d = p.nbd - 1; d >= 0; --d) {
        const int64_t i = q % p.bshape[d];
        q /= p.bshape[d];
        a += i * p.a_bs[d];
        b += i * p.b_bs[d];
    }
    *ao = a;
    *bo = b;
}

// Eight f32 at src + e stride (e < 8, those at or past `lim` zero) as eight bf16, nearest even
// (two 16-byte loads when the eight are contiguous and aligned).
__device__ __forceinline__ uint4 pack8(const float *src, int64_t stride, int lim) {
    float x[8];
    if (stride == 1 && lim == 8 && (reinterpret_cast<uintptr_t>(src) & 15) == 0) {
        const float4 u = reinterpret_cast<const float4 *>(src)[0], v = reinterpret_cast<const float4 *>(src)[1];
        x[0] = u.x; x[1] = u.y; x[2] = u.z; x[3] = u.w;
        x[4] = v.x; x[5] = v.y; x[6] = v.z; x[7] = v.w;
    } else {
#pragma unroll
        for (int e = 0; e < 8; e++) x[e] = e < lim ? src[e * stride] : 0.0f;
    }
    uint32_t w[4];
#pragma unroll
    for (int q = 0; q < 4; q++) asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(w[q]) : "v"(x[2 * q]), "v"(x[2 * q + 1]));
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// One batch's A (row-group fragments) and B (tile-major column fragments) in one launch, batch
// z = blockIdx.y; the first `ablocks` blocks of a row of the grid take A's lanes, the rest B's.
// A: fragment (g, s) of G x S at (g S + s) KiB from the batch's start (G S KiB apart); lane l's
// 16 bytes are row 32 g + l % 32, k 16 s + 8 (l / 32) .. + 7.
// B: tile t of T, step s, column group gi at ((t S + s) 8 + gi) KiB from the batch's start
// (T S 8 KiB apart); lane l's 16 bytes are column 32 (8 t + gi) + l % 32, k 16 s + 8 (l / 32) ..
// + 7. One thread per lane of a fragment.
__global__ void k_pack_half(MatmulP p, int G, int T, int S, int ablocks, uint8_t *pa, uint8_t *pb) {
    const int64_t z = blockIdx.y;
    int64_t ao, bo;
    batch_offsets(p, z, &ao, &bo);
    if (int(blockIdx.x) < ablocks) {
        const int64_t total = int64_t(G) * S * 64;
        for (int64_t idx = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; idx < total;
             idx += int64_t(ablocks) * blockDim.x) {
            const int l = int(idx % 64);
            const int64_t q = idx / 64;
            const int s = int(q % S), g = int(q / S);
            const int row = 32 * g + (l & 31), k0 = 16 * s + 8 * (l >> 5);
            const int lim = row < p.m ? min(8, p.k - k0) : 0;
            const uint4 v = pack8(p.a + ao + int64_t(row < p.m ? row : 0) * p.a_rs + int64_t(k0) * p.a_cs, p.a_cs, lim);
            *reinterpret_cast<uint4 *>(pa + (z * G * S + (int64_t(g) * S + s)) * 1024 + l * 16) = v;
        }
    } else {
        const int64_t total = int64_t(T) * S * 8 * 64;
        const int bblocks = int(gridDim.x) - ablocks;
        for (int64_t idx = (blockIdx.x - ablocks) * int64_t(blockDim.x) + threadIdx.x; idx < total;
             idx += int64_t(bblocks) * blockDim.x) {
            const int l = int(idx % 64);
            const int64_t q = idx / 64;  // (t S + s) 8 + gi
            const int gi = int(q % 8);
            const int64_t ts = q / 8;
            const int s = int(ts % S), t = int(ts / S);
            const int col = 32 * (8 * t + gi) + (l & 31), k0 = 16 * s + 8 * (l >> 5);
            const int lim = col < p.n ? min(8, p.k - k0) : 0;
            const uint4 v = pack8(p.b + bo + int64_t(col < p.n ? col : 0) * p.b_cs + int64_t(k0) * p.b_rs, p.b_rs, lim);
            *reinterpret_cast<uint4 *>(pb + (z * T * S * 8 + q) * 1024 + l * 16) = v;
        }
    }
}

// The packed path from this many 256 x 256 output tiles and this k (below them the staged kernel,
// whose operands need no second pass). Measured (us, staged / packed): 4096^3 (256 tiles) 335 / 140.5,
// 2000 x 4000 x 3000 (96) 133 / 96.6, 3000 x 1000 x 2500 (120) 41.9 / 39.0; at 64 tiles 2048^3 35.7 /
// 55.9, 4096 x 1024 x 1024 21.1 / 38.2, 1024 x 4096 x 4096 81.7 / 97.5.
constexpr int64_t kHalfPackedTiles = 96;
constexpr int64_t kHalfPackedK = 256;

// One 256 x 256 output tile (tm_i, tn_i) of batch z per workgroup. Workgroup w is tile
// (w / (tm tn)) of the batches, then row tiles in order within a column tile: consecutive
// workgroups share their B tile, and the 8 XCDs (dealt workgroups in turn) each hold every
// eighth row tile of it.
__global__ __launch_bounds__(256) void k_half_tiles(MatmulP p, const uint8_t *pa, const uint8_t *pb, int G, int T,
                                                     int S) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[pipe::kPipeStages * pipe::kPipeStageBytes];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t wg = blockIdx.x, per_batch = int64_t(p.tm) * p.tn;
    const int64_t z = wg / per_batch;
    const int rem = int(wg - z * per_batch);
    const int tn_i = rem / p.tm, tm_i = rem % p.tm;
    // this tile's row groups of A (rows past the batch's last group read as zeros: the range)
    const int g0 = 8 * tm_i, ng = min(8, G - g0);
    const __amdgpu_buffer_rsrc_t hres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t *>(pa + (z * G + g0) * int64_t(S) * 1024), short(0), ng * S * 1024, pipe::kBufferWord3);
    const int hoff = 2 * wave * S * 1024 + lane * 16, woff = 2 * wave * 1024 + lane * 16;
    const uint64_t wbase = reinterpret_cast<uint64_t>(pb + (z * T + tn_i) * int64_t(S) * 8192);
    const pipe::v4u wrs = {uint32_t(wbase), uint32_t(wbase >> 32), uint32_t(S * 8192), uint32_t(pipe::kBufferWord3)};
    pipe::f32x16_t acc[8][2];
#pragma unroll
    for (int i = 0; i < 8; i++)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
    pipe::MfmaPipe<false> pp;
    pp.run(lds, hres, hoff, wrs, woff, S, wave, lane, acc);
    pp.last_odd_step(S, acc);
    // lane l holds rows 32 i + 8 (v / 4) + 4 (l / 32) + v % 4, column 64 wave + 32 j + l % 32
    float *c = p.c + z * int64_t(p.m) * p.n;
    const int row0 = 256 * tm_i, col0 = 256 * tn_i + 64 * wave + (lane & 31);
#pragma unroll
    for (int j = 0; j < 2; j++) {
        const int col = col0 + 32 * j;
        if (col >= p.n) continue;
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int row = row0 + 32 * i + 8 * (v / 4) + 4 * (lane >> 5) + (v % 4);
                if (row < p.m) c[int64_t(row) * p.n + col] = acc[i][j][v];
            }
    }
}

template <bool HALF, class C, bool SPLIT>
int launch_matmul(const MatmulP &p, hipStream_t s) {
    // A launch holds fewer than 2^32 threads. More blocks, as of millions of small batches, go in halves
    // along the outermost batch dimension that has any.
    if (p.blocks > ((int64_t(1) << 32) - 1) / C::kThreads) {
        int d = 0;
        while (d < p.nbd && p.bshape[d] == 1) d++;
        if (d == p.nbd) return fail(NT_E_ARG, "matmul: too many output tiles");
        int64_t inner = int64_t(p.m) * p.n, tiles = int64_t(p.tm) * p.tn;
        for (int e = d + 1; e < p.nbd; e++) inner *= p.bshape[e], tiles *= p.bshape[e];
        MatmulP q = p;
        q.bshape[d] = p.bshape[d] / 2;
        q.blocks = q.bshape[d] * tiles;
        if (int rc = launch_matmul<HALF, C, SPLIT>(q, s)) return rc;
        q.a_off += q.bshape[d] * p.a_bs[d];
        q.b_off += q.bshape[d] * p.b_bs[d];
        q.c += q.bshape[d] * inner;
        q.bshape[d] = p.bshape[d] - q.bshape[d];
        q.blocks = q.bshape[d] * tiles;
        return launch_matmul<HALF, C, SPLIT>(q, s);
    }
    const dim3 grid(unsigned(p.blocks)), block(C::kThreads);
    const bool ak = p.a_cs == 1, bn = p.b_cs == 1 || p.b_rs != 1;
    if (ak && bn) hipLaunchKernelGGL((k_matmul<HALF, C, true, true, SPLIT>), grid, block, 0, s, p);
    else if (ak) hipLaunchKernelGGL((k_matmul<HALF, C, true, false, SPLIT>), grid, block, 0, s, p);
    else if (bn) hipLaunchKernelGGL((k_matmul<HALF, C, false, true, SPLIT>), grid, block, 0, s, p);
    else hipLaunchKernelGGL((k_matmul<HALF, C, false, false, SPLIT>), grid, block, 0, s, p);
    return launched(HALF ? "k_matmul (half)" : "k_matmul");
}

// 128 x 128 tiles when they give at least `least` workgroups, else 64 x 64; also 64 x 64 where these cover
// the outputs with half the area (a side of at most 64, as of many small batches). Measured (us, 128 / 64):
// 256 batches of 1 x 4096 x 64 291 / 91, 20000 of 4 x 4 x 4 269 / 81, 300 of 100 x 40 x 30 15.3 / 9.5; half, 4096
// of 16 x 16 x 16 34.2 / 17.8, 64 x 256 x 50304 30.7 / 30.9.
int tile_side(int64_t batches, int64_t m, int64_t n, int64_t least) {
    const int64_t big = batches * ((m + 127) / 128) * ((n + 127) / 128);
    const int64_t small = batches * ((m + 63) / 64) * ((n + 63) / 64);
    return big >= least && small > 2 * big ? 128 : 64;
}

template <bool HALF>
int launch_tile(int tile, const MatmulP &p, hipStream_t s) {
    if (tile == 128) return launch_matmul<HALF, Tile128, false>(p, s);
    return launch_matmul<HALF, Tile64, false>(p, s);
}

}  // namespace
}  // namespace nt

using namespace nt;

extern "C" {

int nt_hip_matmul(const float *a, const NtLayout *al, const float *b, const NtLayout *bl, float *out) {
    if (!al || !bl) return fail(NT_E_ARG, "matmul: null layout");
    const int r = al->rank;
    if (r < 2 || r > NT_MAX_RANK || bl->rank != r || al->shape[r - 1] != bl->shape[r - 2])
        return fail(NT_E_ARG, "matmul: shapes [" + std::to_string(r) + "-d] do not multiply (rank >= 2, equal "
                              "ranks, a's last dimension equal to b's second last)");
    for (int d = 0; d < r; d++)
        if (al->shape[d] < 0 || bl->shape[d] < 0 || al->strides[d] < 0 || bl->strides[d] < 0 || al->offset < 0 ||
            bl->offset < 0)
            return fail(NT_E_ARG, "matmul: negative shape, stride or offset");
    MatmulP p{};
    p.nbd = r - 2;
    int64_t nb = 1;
    for (int d = 0; d < r - 2; d++) {
        const int64_t x = al->shape[d], y = bl->shape[d];
        if (x != y && x != 1 && y != 1)
            return fail(NT_E_ARG, "matmul: batch dimension " + std::to_string(d) + " does not broadcast (" +
                                      std::to_string(x) + " against " + std::to_string(y) + ")");
        p.bshape[d] = x == 1 ? y : x;
        p.a_bs[d] = x == 1 ? 0 : al->strides[d];
        p.b_bs[d] = y == 1 ? 0 : bl->strides[d];
        nb *= p.bshape[d];
    }
    const int64_t m = al->shape[r - 2], k = al->shape[r - 1], n = bl->shape[r - 1];
    if (m >= (int64_t(1) << 31) - 256 || n >= (int64_t(1) << 31) - 256 || k >= (int64_t(1) << 31) - 256)
        return fail(NT_E_ARG, "matmul: m, k and n must each be below 2^31 - 256");
    if (nb == 0 || m == 0 || n == 0) return 0;
    if (!a || !b || !out) return fail(NT_E_ARG, "matmul: null buffer");
    p.a = a;
    p.b = b;
    p.c = out;
    p.a_off = al->offset;
    p.b_off = bl->offset;
    p.a_rs = al->strides[r - 2];
    p.a_cs = al->strides[r - 1];
    p.b_rs = bl->strides[r - 2];
    p.b_cs = bl->strides[r - 1];
    p.m = int32_t(m);
    p.n = int32_t(n);
    p.k = int32_t(k);
    // 128x128 tiles when they give every CU of the 256 a workgroup, else 64x64. Measured (us, 128 /
    // 64 tiles): 2048^3 (256 tiles of 128) 142 / 161, 1500 x 700 x 1900 (180) 54.3 / 46.9, 1024^3 (64)
    // 72.7 / 27.7.
    const int T = tile_side(nb, m, n, 256);
    p.tm = int32_t((m + T - 1) / T);
    p.tn = int32_t((n + T - 1) / T);
    const int64_t tiles = nb * p.tm * p.tn;
    p.outputs = nb * m * n;
    // Split k over more workgroups when the tiles alone leave CUs idle: each workgroup takes kc_per
    // of the ceil(k / 256) chains, so that about 512 workgroups run in all. A 64 tile alone on its
    // CU takes 6.3 us per chain, and the slices, their fold and the scratch cost 10-15 us, so at
    // least three chains have to be saved. Measured (us, split / not): 512 x 2048 x 512 (64 tiles)
    // 23.8 / 50.7, 128 x 2000 x 300 (10) 19.8 / 50.2, 64 x 1024 x 2048 (32) 20.4 / 27.1; 247 x 525 x
    // 914 (60, three chains) 20.2 / 16.9, 512 x 512 x 2048 (256) 24.1 / 16.1.
    const int64_t nkc = (k + kKC - 1) / kKC;
    int64_t splits = 1;
    // (the slices take 4 bytes per output and 256-k block; past 1 GiB the tiles run unsplit)
    if (tiles < 256 && nkc > 1 && nkc * p.outputs <= (int64_t(1) << 28)) {
        const int64_t want = (512 + tiles - 1) / tiles;
        const int64_t per = (nkc + std::min(want, nkc) - 1) / std::min(want, nkc);
        if (nkc - per >= 3) {
            p.kc_per = int32_t(per);
            splits = (nkc + per - 1) / per;
        }
    }
    p.blocks = tiles * splits;
    if (p.blocks > int64_t(0x7fffffff)) return fail(NT_E_ARG, "matmul: too many output tiles");
    std::unique_lock<std::mutex> lk;
    if (int rc = enter(&lk)) return rc;
    hipStream_t st = ctx().stream;
    if (splits == 1) return launch_tile<false>(T, p, st);
    void *sl = nullptr;
    if (int rc = scratch_alloc(size_t(nkc) * size_t(p.outputs) * sizeof(float), &sl)) return rc;
    p.slices = static_cast<float *>(sl);
    int rc = launch_matmul<false, Tile64, true>(p, st);  // (fewer than 256 tiles: the 64 ones)
    if (!rc) {
        const int64_t fb = std::min<int64_t>((p.outputs + kMmThreads - 1) / kMmThreads, 4096);
        hipLaunchKernelGGL(k_fold, dim3(unsigned(fb)), dim3(kMmThreads), 0, st, p.slices, p.outputs, int(nkc), out);
        rc = launched("k_fold");
    }
    const int rf = scratch_release(sl);
    return rc ? rc : rf;
}

int nt_hip_matmul_half(const float *a, const NtLayout *al, const float *b, const NtLayout *bl, float *out) {
    if (!al || !bl) return fail(NT_E_ARG, "matmul_half: null layout");
    const int r = al->rank;
    if (r < 2 || r > NT_MAX_RANK || bl->rank != r || al->shape[r - 1] != bl->shape[r - 2])
        return fail(NT_E_ARG, "matmul_half: shapes [" + std::to_string(r) + "-d] do not multiply (rank >= 2, equal "
                              "ranks, a's last dimension equal to b's second last)");
    for (int d = 0; d < r; d++)
        if (al->shape[d] < 0 || bl->shape[d] < 0 || al->strides[d] < 0 || bl->strides[d] < 0 || al->offset < 0 ||
            bl->offset < 0)
            return fail(NT_E_ARG, "matmul_half: negative shape, stride or offset");
    MatmulP p{};
    p.nbd = r - 2;
    int64_t nb = 1;
    for (int d = 0; d < r - 2; d++) {
        const int64_t x = al->shape[d], y = bl->shape[d];
        if (x != y && x != 1 && y != 1)
            return fail(NT_E_ARG, "matmul_half: batch dimension " + std::to_string(d) + " does not broadcast (" +
                                      std::to_string(x) + " against " + std::to_string(y) + ")");
        p.bshape[d] = x == 1 ? y : x;
        p.a_bs[d] = x == 1 ? 0 : al->strides[d];
        p.b_bs[d] = y == 1 ? 0 : bl->strides[d];
        nb *= p.bshape[d];
    }
    const int64_t m = al->shape[r - 2], k = al->shape[r - 1], n = bl->shape[r - 1];
    if (m >= (int64_t(1) << 31) - 256 || n >= (int64_t(1) << 31) - 256 || k >= (int64_t(1) << 31) - 256)
        return fail(NT_E_ARG, "matmul_half: m, k and n must each be below 2^31 - 256");
    if (nb == 0 || m == 0 || n == 0) return 0;
    if (!a || !b || !out) return fail(NT_E_ARG, "matmul_half: null buffer");
    p.a = a;
    p.b = b;
    p.c = out;
    p.a_off = al->offset;
    p.b_off = bl->offset;
    p.a_rs = al->strides[r - 2];
    p.a_cs = al->strides[r - 1];
    p.b_rs = bl->strides[r - 2];
    p.b_cs = bl->strides[r - 1];
    p.m = int32_t(m);
    p.n = int32_t(n);
    p.k = int32_t(k);
    // Packed operands and 256 x 256 tiles for a product of many such tiles (see k_half_tiles);
    // NOETIC_HIP_HALF_GEMM=packed|staged picks one path (a tuning knob). The packed path keeps
    // every offset in 32 bits: k <= 65536, at most 65535 batches and 1 GiB of packed operands.
    {
        const int64_t S = (k + 15) / 16, G = (m + 31) / 32, T256 = (n + 255) / 256, TM = (m + 255) / 256;
        const int64_t tiles = nb * TM * T256;
        const int64_t bytes_a = nb * G * S * 1024, bytes_b = nb * T256 * S * 8192;
        const bool fits = k <= 65536 && nb <= 65535 && bytes_a + bytes_b <= (int64_t(1) << 30) && tiles <= 0x7fffffff;
        bool packed = fits && tiles >= kHalfPackedTiles && k >= kHalfPackedK;
        if (const char *e = std::getenv("NOETIC_HIP_HALF_GEMM")) {
            if (std::strcmp(e, "packed") == 0) packed = fits;
            else if (std::strcmp(e, "staged") == 0) packed = false;
        }
        if (packed) {
            p.tm = int32_t(TM);
            p.tn = int32_t(T256);
            std::unique_lock<std::mutex> lk;
            if (int rc = enter(&lk)) return rc;
            hipStream_t st = ctx().stream;
            void *ws = nullptr;
            if (int rc = scratch_alloc(size_t(bytes_a + bytes_b), &ws)) return rc;
            uint8_t *pa = static_cast<uint8_t *>(ws), *pb = pa + bytes_a;
            // both operands in one launch, blocks in proportion to their fragments
            const int64_t ta = G * S * 64, tb = T256 * S * 8 * 64;
            const int64_t ba = std::min<int64_t>((ta + 255) / 256, 4096), bb = std::min<int64_t>((tb + 255) / 256, 4096);
            hipLaunchKernelGGL(k_pack_half, dim3(unsigned(ba + bb), unsigned(nb)), dim3(256), 0, st, p, int(G),
                               int(T256), int(S), int(ba), pa, pb);
            int rc = launched("k_pack_half");
            if (!rc) {
                hipLaunchKernelGGL(k_half_tiles, dim3(unsigned(tiles)), dim3(256), 0, st, p, pa, pb, int(G),
                                   int(T256), int(S));
                rc = launched("k_half_tiles");
            }
            const int rf = scratch_release(ws);
            return rc ? rc : rf;
        }
    }
    // 128 x 128 tiles from 160 of them on, else 64 x 64. Measured (us, 128 / 64): 1500 x 700 x 1900 (180
    // tiles of 128) 19.5 / 25.2; 4096 x 4096 x 512 (128) 56.7 / 51.2.
    const int T = tile_side(nb, m, n, 160);
    p.tm = int32_t((m + T - 1) / T);
    p.tn = int32_t((n + T - 1) / T);
    p.blocks = nb * p.tm * p.tn;
    if (p.blocks > int64_t(0x7fffffff)) return fail(NT_E_ARG, "matmul_half: too many output tiles");
    std::unique_lock<std::mutex> lk;
    if (int rc = enter(&lk)) return rc;
    return launch_tile<true>(T, p, ctx().stream);
}

int nt_hip_half_gemm_key(char *buf, size_t cap) {
    if (!buf || cap == 0) return fail(NT_E_ARG, "nt_hip_half_gemm_key: empty buffer");
    std::string sha(NT_KERNELS_SHA);
    const std::string key = "gemm-bf16-mfma32x32x16-f32acc-kernels-" + sha.substr(0, 16);
    if (key.size() + 1 > cap) return fail(NT_E_ARG, "nt_hip_half_gemm_key: buffer too small");
    std::snprintf(buf, cap, "%s", key.c_str());
    return 0;
}

}  // extern "C"
