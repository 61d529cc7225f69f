// The reference's Gumbel-max sampler's device code for gfx950 (MI355X), sample_categorical
// (src/nn/rl.rs:488-529) on a Hip tensor. One source for both ways the library builds it:
// compiled ahead of time into libnoetic_hip.so (rl_gumbel.hip includes this file), and compiled
// at run time by hiprtc from the text embedded in the library (rtc.cpp). The algorithm and its
// contract are described in rl_gumbel.hip.
#pragma once

#include "nt_chacha.hpp"
#include "nt_rows.hpp"

namespace nt {
namespace {

constexpr int kGumbelMaxThreads = 1024;

struct GumbelP {
    const void *logits;
    const void *mask;
    int64_t V, ld;
    MaskMap mm;  // the mask row of each logits row
    float tau;
    int tau_one;
    float inv_tau;  // 1 / tau in f32 (1 at tau == 1, and under an additive mask: its values are divided); NaN
                    // where it overflows, up to tau = 2^-128: no bound then skips an element
    ChachaKey key;
    ChachaColumns col;
    uint64_t h;  // pair index of the stream's u64 0: its low word is keystream word 2 h + ODD
    int vec;     // rows (and mask rows) aligned for one vector load per 8 elements
    int32_t *ids;
    uint8_t *status;
    int segs;               // workgroups per row
    struct GumbelRec *rec;  // segs > 1: what each found, [rows][segs]
};

// A segment's largest screened value, its flags and the candidates within the margin of it: screened
// value, tempered logit and element (more than kGumbelRecCand raise flag 4). Greedy: the first maximum.
constexpr int kGumbelRecCand = 16;
struct GumbelRec {
    float a;
    int flags, n, pad;
    float ca[kGumbelRecCand], cz[kGumbelRecCand];
    int cv[kGumbelRecCand];
};

// z_v = tempered_logits (rl.rs:475-486) in f32: x / tau (skipped at tau == 1), then the
// additive f32 mask, or -inf at a token a u8 keep-mask excludes. Without DIV the division is
// left to the caller (with a u8 mask or none it commutes with the exclusion: -inf / tau = -inf).
// moff: the row's mask row (mask_row_at).
template <int DT, int MK, bool DIV = true>
__device__ __forceinline__ float tempered_at(const GumbelP &p, int64_t row, int64_t moff, int64_t v) {
    float x;
    if constexpr (DT == NT_F32) {
        x = static_cast<const float *>(p.logits)[row * p.ld + v];
    } else {
        x = widen16<DT>(uint32_t(static_cast<const uint16_t *>(p.logits)[row * p.ld + v]));
    }
    if (DIV && !p.tau_one) x = x / p.tau;
    if constexpr (MK == NT_MASK_U8) {
        if (static_cast<const uint8_t *>(p.mask)[moff + v] == 0) x = -INFINITY;
    } else if constexpr (MK == NT_MASK_F32) {
        x = x + static_cast<const float *>(p.mask)[moff + v];
    }
    return x;
}

// f32(-ln(-ln u)) of one u64 of the stream, u = ((k >> 11) + 0.5) / 2^53 (rl.rs:490-498): the
// f64 add rounds to nearest even as the host's does, the scale by 2^-53 is exact.
__device__ __forceinline__ float gumbel_f32(uint32_t lo, uint32_t hi) {
    const uint64_t k = ((uint64_t(hi) << 32) | lo) >> 11;
    const double u = (double(k) + 0.5) * 0x1p-53;
    return float(-log(-log(u)));
}

// (value, index) pair order of the first maximum: b replaces a when greater, or equal with a
// smaller index. Candidates are never NaN (a NaN refuses the row).
__device__ __forceinline__ void best_merge(float &a, int &ia, float b, int ib) {
    if (b > a || (b == a && ib < ia)) {
        a = b;
        ia = ib;
    }
}

// A block's 8 logits and mask entries, loaded together (the aligned path).
template <int DT, int MK>
struct GumbelRaw {
    uint32_t x[DT == NT_F32 ? 8 : 4];
    uint32_t m[MK == NT_MASK_F32 ? 8 : (MK == NT_MASK_U8 ? 2 : 1)];
};

template <int DT, int MK>
__device__ __forceinline__ void gumbel_load(GumbelRaw<DT, MK> &r, __amdgpu_buffer_rsrc_t xres,
                                            __amdgpu_buffer_rsrc_t mres, int v0) {
    if constexpr (DT == NT_F32) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const auto a = __builtin_amdgcn_raw_buffer_load_b128(xres, (v0 + 4 * q) * 4, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) r.x[4 * q + i] = a[i];
        }
    } else {
        const auto a = __builtin_amdgcn_raw_buffer_load_b128(xres, v0 * 2, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; i++) r.x[i] = a[i];
    }
    if constexpr (MK == NT_MASK_U8) {
        const auto k = __builtin_amdgcn_raw_buffer_load_b64(mres, v0, 0, 0);
        r.m[0] = k[0];
        r.m[1] = k[1];
    } else if constexpr (MK == NT_MASK_F32) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const auto a = __builtin_amdgcn_raw_buffer_load_b128(mres, (v0 + 4 * q) * 4, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; i++) r.m[4 * q + i] = a[i];
        }
    }
}

// The same of any 8 elements v0 .. v0 + 7 inside the row, at their own alignment.
template <int DT, int MK>
__device__ __forceinline__ void gumbel_load_any(GumbelRaw<DT, MK> &r, const void *xrow, const void *mrow, int64_t v0) {
    if constexpr (DT == NT_F32) {
        const u32x4_f32 *q = reinterpret_cast<const u32x4_f32 *>(static_cast<const float *>(xrow) + v0);
        const u32x4_f32 a = q[0], b = q[1];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            r.x[i] = a[i];
            r.x[4 + i] = b[i];
        }
    } else {
        const u32x4_f16 a = *reinterpret_cast<const u32x4_f16 *>(static_cast<const uint16_t *>(xrow) + v0);
#pragma unroll
        for (int i = 0; i < 4; i++) r.x[i] = a[i];
    }
    if constexpr (MK == NT_MASK_U8) {
        const u32x2_u8 k = *reinterpret_cast<const u32x2_u8 *>(static_cast<const uint8_t *>(mrow) + v0);
        r.m[0] = k[0];
        r.m[1] = k[1];
    } else if constexpr (MK == NT_MASK_F32) {
        const u32x4_f32 *q = reinterpret_cast<const u32x4_f32 *>(static_cast<const float *>(mrow) + v0);
        const u32x4_f32 a = q[0], b = q[1];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            r.m[i] = a[i];
            r.m[4 + i] = b[i];
        }
    }
}

// A loaded block's values. Without DIV, the logits themselves (-inf where a u8 mask excludes: it
// commutes with the division); under an additive mask always the tempered z.
template <int DT, int MK, bool DIV>
__device__ __forceinline__ void gumbel_values(const GumbelRaw<DT, MK> &r, const GumbelP &p, float (&z)[8]) {
#pragma unroll
    for (int j = 0; j < 8; j++) z[j] = logit<DT>(r.x, j);
    if ((DIV || MK == NT_MASK_F32) && !p.tau_one) div_tau<8>(z, p.tau);
#pragma unroll
    for (int j = 0; j < 8; j++) {
        if constexpr (MK == NT_MASK_U8) {
            if (((r.m[j / 4] >> (8 * (j % 4))) & 0xffu) == 0) z[j] = -INFINITY;
        } else if constexpr (MK == NT_MASK_F32) {
            z[j] = z[j] + __uint_as_float(r.m[j]);
        }
    }
}

// The screen (a draw's value in f32 from hardware logarithms): within 1e-5 of gumbel_f32's
// value, and infinite exactly where it is, with no branch and no division. k = (hi:lo) >> 11 and
// u = (k + 0.5) / 2^53. Below u = 1 - 2^-4, t = -ln u from u in f32 (hi's and k's low 21 bits
// converted apart); t >= 0.06 there, so the logarithm's rounding stays a small relative error.
// Above it, t = -ln(1 - d) = d (1 + d/2 + ... + d^5/6) (the next term is below 2^-24 of t) with
// d = 1 - u taken from the integer: 2^53 d = (2^32 - hi) 2^21 - (k mod 2^21) - (k & 1), the f64
// sum k + 0.5 rounding to even from 2^52 on, in one fused multiply-add. d = 0 (k = 2^53 - 1, u
// rounds to 1) gives t = 0 and g = +inf, as the exact value is.
__device__ __forceinline__ float gumbel_screen(uint32_t lo, uint32_t hi) {
    constexpr float kLn2f = 0.69314718055994530942f;
    const uint32_t kl = lo >> 11;  // k's low 21 bits (its high 32 are hi)
    const float u = fmaf(float(hi), 0x1p-32f, fmaf(float(kl), 0x1p-53f, 0x1p-54f));
    const float tl = __builtin_amdgcn_logf(u) * -kLn2f;
    const float d = fmaf(float(kl + (kl & 1u)), -0x1p-53f, float(0u - hi) * 0x1p-32f);
    float ser = fmaf(d, 1.0f / 6.0f, 1.0f / 5.0f);
    ser = fmaf(ser, d, 1.0f / 4.0f);
    ser = fmaf(ser, d, 1.0f / 3.0f);
    ser = fmaf(ser, d, 0.5f);
    ser = fmaf(ser, d, 1.0f);
    const float t = hi >= 0xf0000000u ? d * ser : tl;
    return __builtin_amdgcn_logf(t) * -kLn2f;
}

constexpr int kGumbelCand = 4;         // screened candidates a thread keeps
constexpr int kGumbelQueue = 128;      // a wave's queue of blocks with an allowed element (LDS)
// The queue's dynamic LDS for a launch of `threads` threads: per wave kGumbelQueue block indices
// and their 8 values each, or their loaded words under a u8 mask (72 to 88 KiB at 16 waves).
constexpr int gumbel_queue_words(int dt, int mk) { return dt == NT_F32 && mk == NT_MASK_U8 ? 10 : 8; }
constexpr size_t gumbel_queue_bytes(int threads, bool greedy, int dt, int mk) {
    return greedy ? 0 : size_t(threads / 64) * kGumbelQueue * (1 + gumbel_queue_words(dt, mk)) * sizeof(float);
}
constexpr float kGumbelScreen = 1e-3f;  // the screen's margin, at least: 250 times its error bound

// The lowest screened value kept as a candidate beside a largest screened value x: x less the
// larger of kGumbelScreen and |x| rel. The value compared is z + g rounded to f32, so a screened
// and an exact sum differ by the screen's error and up to an ulp of the sum; with rel = 2^-21
// (four ulps of x) the margin exceeds two such differences at every magnitude, so an element
// below it cannot reach or pass the element at x exactly. A thread keeps its own candidates
// with rel = 2^-20, a superset of the row's. (x = +inf: the candidates are the infinite values.)
__device__ __forceinline__ float screen_floor(float x, float rel) {
    return x == INFINITY ? x : x - fmaxf(kGumbelScreen, fabsf(x) * rel);
}

// An upper bound of a draw's screened value less its logit, at most 1e-3 above g: g from the high word
// alone, u taken at its upper end (hi + 1) / 2^32. In base 2, t2 = -log2 u = 32 - log2(hi + 1), or
// d (1 + d / 2) log2 e with d = 1 - u = (2^32 - 1 - hi) / 2^32 above u = 1 - 2^-5 (the terms left out
// are below d^2 / 3 = 3.3e-4 of t2, and only lower it), and g = -ln 2 log2 t2 - ln ln 2. Two hardware
// logarithms and nine other operations. Below t2 = 0.0458 the first form's rounding is at most 4e-5.
__device__ __forceinline__ float gumbel_bound(uint32_t hi) {
    constexpr float kLog2eF = 1.44269504088896340736f;
    const float ta = 32.0f - __builtin_amdgcn_logf(float(hi) + 1.0f);
    const float d = float(~hi) * 0x1p-32f;
    const float tb = d * fmaf(d, 0.5f * kLog2eF, kLog2eF);
    const float t2 = hi >= 0xf8000000u ? tb : ta;
    return fmaf(__builtin_amdgcn_logf(t2), -0.69314718055994530942f, 0.36651292058166432701f);
}

// What a bound must reach to be looked at, beside a largest screened value x so far: screen_floor, less
// the bound's slack and the rounding of x inv_tau (and no more than 3e38, so that a logit whose
// rounded product is finite where its quotient is infinite is looked at too). A NaN bound reaches
// every floor: with inv_tau NaN each element is divided and screened.
__device__ __forceinline__ float bound_floor(float x) {
    return fminf(screen_floor(x, 0x1p-20f) - fmaxf(2.0f * kGumbelScreen, fabsf(x) * 0x1p-20f), 3e38f);
}

// The row's first maximum of z + g. Past temperature 0 it runs in three steps. Every allowed element
// gets an upper bound of its value (gumbel_bound; the keystream is generated for it). The few whose
// bound comes near the largest value seen by the wave are screened in f32 (gumbel_screen, their
// logit divided by tau), and those within the margin of the thread's largest (screen_floor) are kept.
// Only the kept ones within the margin of the row's largest can be its maximum: a single one is the
// answer; several are evaluated exactly (gumbel_f32, their keystream block generated again). The
// exact maximum is among them, since the margins cover the errors and the rounding of z + g on both
// sides. A thread whose candidates within the margin of its own largest outnumber its slots makes
// the row take the exact evaluation of every element instead.
//
// With p.segs > 1, workgroup `seg` of a row takes the blocks of that segment and leaves its record for
// k_gumbel_finish.
template <int DT, int MK, bool ODD, bool GREEDY>
struct Gumbel {
    const GumbelP &p;
    const int64_t row, moff;  // moff: the row's mask row
    const int64_t V;
    // pair q0 + v holds element v's u64; block b0 + i elements 8 i - r .. 8 i - r + 7 (greedy, which draws
    // nothing: from the row's start, r = 0)
    const uint64_t q0, b0;
    const int r;
    const int wave, nw, lane;
    int flags = 0;  // bit 0: a candidate (z > -inf); bit 1: a NaN; bit 2: a thread's slots overflowed
    int count = 0;  // summed by the reductions
    float best = -INFINITY;
    int bidx = 0x7fffffff;

    __device__ Gumbel(const GumbelP &p_, int64_t row_)
        : p(p_), row(row_), moff(MK != NT_MASK_NONE ? mask_row_at(p_.mm, row_) : 0), V(p_.V),
          q0(GREEDY ? 0 : p_.h + uint64_t(row_) * uint64_t(p_.V)), b0(q0 >> 3), r(int(q0 & 7)), wave(threadIdx.x / 64),
          nw(blockDim.x / 64), lane(threadIdx.x & 63) {}

    __device__ int blocks() const { return int(((q0 + uint64_t(V) - 1) >> 3) - b0) + 1; }

    // fn(i, z) for every block i of [lo, hi), z its 8 values, each thread its own, two loads ahead (greedy
    // rows, whose blocks begin at the row's start: 1000 x 32000 f32 under a u8 mask 40.9 us through walk below,
    // 26.3 so).
    template <class Fn>
    __device__ __forceinline__ void own_blocks(int lo, int hi, Fn &&fn) {
        const int n = blockDim.x;
        const void *xrow = static_cast<const char *>(p.logits) + row * p.ld * Elem<DT>::kBytes;
        const void *mrow =
            MK != NT_MASK_NONE ? static_cast<const char *>(p.mask) + moff * MaskWords<MK>::kBytes : nullptr;
        auto load = [&](Raw<DT, MK> &w, int i) { load_raw<DT, MK, false>(w, xrow, mrow, 8 * int64_t(i), V); };
        auto use = [&](const Raw<DT, MK> &w, int i) {
            float z[8];
            decode<DT, MK>(w, z, 1.0f, true);
            fn(i, z);
        };
        Raw<DT, MK> cur, nxt;
        int i = lo + int(threadIdx.x);
        if (i < hi) load(cur, i);
        if (i + n < hi) load(nxt, i + n);
        for (; i < hi; i += 2 * n) {  // (a set is used, then loaded again)
            use(cur, i);
            if (i + 2 * n < hi) load(cur, i + 2 * n);
            if (i + n >= hi) break;
            use(nxt, i + n);
            if (i + 3 * n < hi) load(nxt, i + 3 * n);
        }
    }

    // fn(i, z) for every block i of [lo, hi) that holds an element not excluded, z its 8 values
    // (gumbel_values; -inf outside the row), the fn calls of a wave together. Where not
    // every block of a wave's step holds one, they go through the wave's queue in LDS and each call
    // takes whichever queued block falls to the lane, so that the keystream is generated by full
    // waves (the order does not matter to the caller: its merges break ties by index). A call is
    // made by every lane of the wave; `have` says whether the lane has a block.
    template <bool DIV, class Fn>
    __device__ __forceinline__ void walk(int lo, int hi, int *gqb, float *gqz, Fn &&fn) {
        const int n = blockDim.x;
        const void *xrow = static_cast<const char *>(p.logits) + row * p.ld * Elem<DT>::kBytes;
        const void *mrow =
            MK != NT_MASK_NONE ? static_cast<const char *>(p.mask) + moff * MaskWords<MK>::kBytes : nullptr;
        const bool aligned = p.vec && r == 0;  // (uniform) a block's elements are one aligned load
        const int Vb = aligned ? int(V) : 0;
        const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<void *>(xrow), short(0), Vb * Elem<DT>::kBytes, kBufferWord3);
        const __amdgpu_buffer_rsrc_t mres =
            MK != NT_MASK_NONE ? __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(mrow), short(0),
                                                                   Vb * MaskWords<MK>::kBytes, kBufferWord3)
                               : xres;
        auto inside = [&](int i) { return 8 * int64_t(i) - r >= 0 && 8 * int64_t(i) - r + 8 <= V; };
        // block i's elements, two steps ahead of their use; a block that crosses an end of the row
        // (its first or last) loads the 8 elements at that end instead and is read again when used
        auto load = [&](GumbelRaw<DT, MK> &w, int i) {
            if (aligned) {
                gumbel_load<DT, MK>(w, xres, mres, 8 * i);
            } else if (V >= 8) {
                int64_t v0 = 8 * int64_t(i) - r;
                v0 = v0 < 0 ? 0 : (v0 + 8 > V ? V - 8 : v0);
                gumbel_load_any<DT, MK>(w, xrow, mrow, v0);
            }
        };
        auto values = [&](const GumbelRaw<DT, MK> &w, int i, float (&z)[8]) {
            gumbel_values<DT, MK, DIV>(w, p, z);
            if (!inside(i)) {
#pragma unroll
                for (int j = 0; j < 8; j++) {
                    const int64_t v = 8 * int64_t(i) - r + j;
                    z[j] = i < hi && v >= 0 && v < V ? tempered_at<DT, MK, DIV || MK == NT_MASK_F32>(p, row, moff, v)
                                                     : -INFINITY;
                }
            }
        };
        // Under a u8 mask the queue holds the loaded words (its test is two words of the mask), decoded
        // when a block is taken; else the values.
        constexpr bool RAWQ = MK == NT_MASK_U8;
        constexpr int XW = Elem<DT>::kWords;
        constexpr int QW = RAWQ ? XW + 2 : 8;  // words per entry
        static_assert(QW <= gumbel_queue_words(DT, MK), "the launch's LDS");
        uint32_t *qw = reinterpret_cast<uint32_t *>(gqz);
        const int qsize = QW * kGumbelQueue;  // a wave's words, [QW][kGumbelQueue]
        int head = 0, queued = 0;             // this wave's first entry and their number (uniform)
        // the queue's first 64 entries, one per lane (lanes without one: block hi - 1, -inf)
        auto take = [&](bool have, int &i, float (&z)[8]) {
            // (every lane's queue writes are in LDS before any lane reads)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            const int e = (head + lane) % kGumbelQueue;
            const uint32_t *q = qw + wave * qsize + e;
            i = have ? gqb[wave * kGumbelQueue + e] : hi - 1;
            if constexpr (RAWQ) {
                GumbelRaw<DT, MK> t;
#pragma unroll
                for (int k = 0; k < XW; k++) t.x[k] = have ? q[k * kGumbelQueue] : 0;
#pragma unroll
                for (int k = 0; k < 2; k++) t.m[k] = have ? q[(XW + k) * kGumbelQueue] : 0;
                if (have) {
                    values(t, i, z);
                } else {
#pragma unroll
                    for (int j = 0; j < 8; j++) z[j] = -INFINITY;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 8; j++) z[j] = have ? __uint_as_float(q[j * kGumbelQueue]) : -INFINITY;
            }
            // (the reads are done before a later write reuses their slots)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_wave_barrier();
            const int took = queued < 64 ? queued : 64;
            head = (head + took) % kGumbelQueue;
            queued -= took;
        };
        GumbelRaw<DT, MK> cur, nxt;
        const int first = lo + 64 * wave;
        if (first < hi) load(cur, first + lane < hi ? first + lane : hi - 1);
        if (first + n < hi) load(nxt, first + n + lane < hi ? first + n + lane : hi - 1);
        bool odd = false;  // (uniform)
        for (int base = first; base < hi || queued > 0;) {
            int i = base + lane;
            float z[8];
            bool have = i < hi, go = false;
            if (base < hi) {
                // two sets of loads in flight: a set is used, then loaded again for the step two ahead
                // (moving one into the other would wait for it)
                const int ib = have ? i : hi - 1, ahead = i + 2 * n < hi ? i + 2 * n : hi - 1;
                const bool more = base + 2 * n < hi;
                base += n;
                auto step = [&](GumbelRaw<DT, MK> &w) {
                    if constexpr (RAWQ) {
                        have &= (w.m[0] | w.m[1]) != 0 || !inside(ib);
                    } else {
                        values(w, ib, z);
                        bool any = false;
#pragma unroll
                        for (int j = 0; j < 8; j++) any |= !(z[j] == -INFINITY);  // (a NaN counts)
                        have &= any;
                    }
                    const uint64_t bal = __ballot(have);
                    if (!RAWQ && queued == 0 && bal == ~uint64_t(0)) {
                        go = bal != 0;
                    } else {
                        if (have) {
                            const int pos = (head + queued + int(__builtin_amdgcn_mbcnt_hi(
                                                                  uint32_t(bal >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(bal), 0u)))) %
                                            kGumbelQueue;
                            uint32_t *q = qw + wave * qsize + pos;
                            gqb[wave * kGumbelQueue + pos] = i;
                            if constexpr (RAWQ) {
#pragma unroll
                                for (int k = 0; k < XW; k++) q[k * kGumbelQueue] = w.x[k];
#pragma unroll
                                for (int k = 0; k < 2; k++) q[(XW + k) * kGumbelQueue] = w.m[k];
                            } else {
#pragma unroll
                                for (int j = 0; j < 8; j++) q[j * kGumbelQueue] = __float_as_uint(z[j]);
                            }
                        }
                        queued += __builtin_popcountll(bal);
                    }
                    if (more) load(w, ahead);
                };
                if (odd) step(nxt);
                else step(cur);
                odd = !odd;
            }
            if (queued >= 64 || (queued > 0 && base >= hi)) {
                have = lane < queued;
                take(have, i, z);
                go = true;
            }
            if (go) fn(have, i, z);
        }
    }

    // The stream words of a block's 8 elements.
    __device__ __forceinline__ void draws(uint64_t b, uint32_t (&lo)[8], uint32_t (&hi)[8]) const {
        uint32_t w[16];
        chacha_block_dev(p.key, p.col, b, w);
        uint32_t next0 = 0;  // word 0 of block b + 1: the high word of pair 7 when ODD
        if constexpr (ODD) {
            uint32_t w2[16];
            chacha_block_dev(p.key, p.col, b + 1, w2);
            next0 = w2[0];
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            lo[j] = ODD ? w[2 * j + 1] : w[2 * j];
            hi[j] = ODD ? (j == 7 ? next0 : w[2 * j + 2]) : w[2 * j + 1];
        }
    }

    // fn(j, z[j], lo[j], hi[j]) for each bit j of the lane's `take`, the lanes in step (one copy of fn's
    // code, the values by selects: an index would go through memory).
    template <class Fn>
    __device__ __forceinline__ void each(uint32_t take, const float (&z)[8], const uint32_t (&lo)[8],
                                         const uint32_t (&hi)[8], Fn &&fn) {
        while (__ballot(take != 0) != 0) {
            if (take != 0) {
                const int j = __builtin_ctz(take);
                take &= take - 1;
                float zj = z[0];
                uint32_t lj = lo[0], hj = hi[0];
#pragma unroll
                for (int e = 1; e < 8; e++) {
                    zj = j == e ? z[e] : zj;
                    lj = j == e ? lo[e] : lj;
                    hj = j == e ? hi[e] : hj;
                }
                fn(j, zj, lj, hj);
            }
        }
    }

    // the exact evaluation of one element, into this thread's first maximum
    __device__ __forceinline__ void exact(int v, float z, uint32_t lo, uint32_t hi) {
        best_merge(best, bidx, z + gumbel_f32(lo, hi), v);
    }

    // the same of a kept candidate, its words generated again
    __device__ __forceinline__ void exact_again(int v, float z) {
        const uint64_t w0 = 2 * (q0 + uint64_t(v)) + (ODD ? 1 : 0);  // its low word
        uint32_t w[16];
        chacha_block_dev(p.key, p.col, w0 >> 4, w);
        uint32_t lo = w[0], hi = w[0];
#pragma unroll
        for (int e = 0; e < 16; e++) {
            if (e == int(w0 & 15)) lo = w[e];
            if (e == int((w0 + 1) & 15)) hi = w[e];
        }
        if ((w0 & 15) == 15) {  // the high word opens the next block
            uint32_t w2[16];
            chacha_block_dev(p.key, p.col, (w0 >> 4) + 1, w2);
            hi = w2[0];
        }
        exact(v, z, lo, hi);
    }

    // every element exactly (into this thread's first maximum; the caller reduces)
    __device__ __forceinline__ void every_exact(int *gqb, float *gqz) {
        best = -INFINITY;
        bidx = 0x7fffffff;
        walk<true>(0, blocks(), gqb, gqz, [&](bool have, int i, const float (&z)[8]) {
            uint32_t lo[8], hi[8], take = 0;
            draws(b0 + uint64_t(i), lo, hi);
#pragma unroll
            for (int j = 0; j < 8; j++) take |= have && z[j] > -INFINITY ? 1u << j : 0u;
            each(take, z, lo, hi, [&](int j, float zj, uint32_t lj, uint32_t hj) { exact(8 * i - r + j, zj, lj, hj); });
        });
    }

    // the workgroup's (best, bidx) first maximum, OR of the flags and sum of the counts: a fixed
    // butterfly inside each wave, then the waves in order (the result in every thread)
    __device__ __forceinline__ void reduce(float *sbest, int *sidx, int *sflags, int *scount) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float ob = __shfl_xor(best, o, 64);
            const int oi = __shfl_xor(bidx, o, 64);
            best_merge(best, bidx, ob, oi);
            flags |= __shfl_xor(flags, o, 64);
            count += __shfl_xor(count, o, 64);
        }
        if (lane == 0) {
            sbest[wave] = best;
            sidx[wave] = bidx;
            sflags[wave] = flags;
            scount[wave] = count;
        }
        __syncthreads();
        float rb = sbest[0];
        int ri = sidx[0], rf = sflags[0], rc = scount[0];
        for (int i = 1; i < nw; i++) {
            best_merge(rb, ri, sbest[i], sidx[i]);
            rf |= sflags[i];
            rc += scount[i];
        }
        __syncthreads();  // (the arrays are written again by a later reduction)
        best = rb;
        bidx = ri;
        flags = rf;
        count = rc;
    }

    // The reference refuses a row whose maximum is NaN (any NaN: max_dim propagates it) or -inf
    // (rl.rs:515-519). One thread.
    __device__ __forceinline__ void write_row() const {
        const bool nan = flags & 2, none = !(flags & 1);
        p.ids[row] = nan || none ? -1 : bidx;
        p.status[row] = uint8_t(nan ? NT_ROW_NAN : (none ? NT_ROW_NO_TOKEN : NT_ROW_OK));
    }
};

template <int DT, int MK, bool ODD, bool GREEDY>
__global__ __launch_bounds__(kGumbelMaxThreads) void k_sample_gumbel(GumbelP p) {
    __shared__ float sbest[kGumbelMaxThreads / 64];
    __shared__ int sidx[kGumbelMaxThreads / 64];
    __shared__ int sflags[kGumbelMaxThreads / 64];
    __shared__ int scount[kGumbelMaxThreads / 64];
    __shared__ int srec;
    // per wave, the queue of blocks to draw: their index and their 8 values ([8][kGumbelQueue]),
    // in dynamic LDS sized by the launch for its waves (gumbel_queue_bytes; none when greedy)
    extern __shared__ __attribute__((aligned(16))) int gdyn[];
    int *const gqb = gdyn;
    float *const gqz = reinterpret_cast<float *>(gdyn + (blockDim.x / 64) * kGumbelQueue);
    int64_t row = blockIdx.x;
    unsigned seg = 0;
    if (p.segs > 1) {
        row = blockIdx.x / unsigned(p.segs);
        seg = blockIdx.x % unsigned(p.segs);
    }
    Gumbel<DT, MK, ODD, GREEDY> g(p, row);
    // the segment's blocks: whole waves of them
    const int nb = g.blocks(), per = p.segs > 1 ? ((nb + p.segs - 1) / p.segs + 63) / 64 * 64 : nb;
    const int lo = min(nb, int(seg) * per), hi = min(nb, lo + per);
    GumbelRec *rec = p.segs > 1 ? p.rec + blockIdx.x : nullptr;
    if constexpr (GREEDY) {
        g.own_blocks(lo, hi, [&](int i, const float (&z)[8]) {
            if (__builtin_isunordered(z[0], z[1]) | __builtin_isunordered(z[2], z[3]) |
                __builtin_isunordered(z[4], z[5]) | __builtin_isunordered(z[6], z[7]))
                g.flags |= 2;
            const float m = max8_hw(z);
            if (m > g.best) {  // strictly greater: the first maximum of this thread's elements
                g.best = m;
                int j = 7;
#pragma unroll
                for (int e = 6; e >= 0; e--) j = z[e] == m ? e : j;
                g.bidx = 8 * i + j;
            }
        });
        if (g.best > -INFINITY) g.flags |= 1;
        g.reduce(sbest, sidx, sflags, scount);
        if (threadIdx.x != 0) return;
        if (!rec) {
            g.write_row();
        } else {
            rec->a = g.best;
            rec->flags = g.flags;
            rec->n = 1;
            rec->cv[0] = g.bidx;
        }
    } else {
        // ---- the thread's largest screened value and its candidates within the margin of it
        // (four slots as separate values: an array here would be indexed through memory)
        static_assert(kGumbelCand == 4, "the four slots below");
        float amax = -INFINITY;
        float near = -INFINITY;  // bound_floor of the wave's largest (uniform)
        float ca0 = -INFINITY, ca1 = -INFINITY, ca2 = -INFINITY, ca3 = -INFINITY;  // screened values
        float cz0 = 0.0f, cz1 = 0.0f, cz2 = 0.0f, cz3 = 0.0f;                       // tempered logits
        int cv0 = 0, cv1 = 0, cv2 = 0, cv3 = 0;                                     // elements
        g.template walk<false>(lo, hi, gqb, gqz, [&](bool have, int i, const float (&x)[8]) {
            uint32_t wlo[8], whi[8];
            float bound[8];
            g.draws(g.b0 + uint64_t(i), wlo, whi);
#pragma unroll
            for (int j = 0; j < 8; j++) bound[j] = fmaf(x[j], p.inv_tau, gumbel_bound(whi[j]));
            const bool nan = __builtin_isunordered(x[0], x[1]) | __builtin_isunordered(x[2], x[3]) |
                             __builtin_isunordered(x[4], x[5]) | __builtin_isunordered(x[6], x[7]);
            const float top = max8_hw(bound);
            if (__ballot(!(top < near) || nan) == 0) return;
            // A new largest bound: what the wave need look at rises at once to that of the largest
            // value a bound assures (a bound is at most 1e-3 and the product's rounding above its
            // value, but for the first 2^12 and last 2^16 high words), so that a wave's first
            // blocks do not look at everything.
            float sure = -INFINITY;
#pragma unroll
            for (int j = 0; j < 8; j++) sure = fmaxf(sure, whi[j] - 0x1000u < 0xfffef000u ? bound[j] : -INFINITY);
            sure = wave_max3_dpp(sure);
            near = fmaxf(near, bound_floor(sure - fmaxf(kGumbelScreen, fabsf(sure) * 0x1p-20f)));
            uint32_t look = 0;
#pragma unroll
            for (int j = 0; j < 8; j++) look |= !(bound[j] < near) && have ? 1u << j : 0u;
            bool moved = false;
            g.each(look, x, wlo, whi, [&](int j, float xj, uint32_t lj, uint32_t hj) {
                const float z = MK == NT_MASK_F32 || p.tau_one ? xj : xj / p.tau;
                if (z == -INFINITY) return;  // excluded, or its quotient by tau is -inf
                if (z != z) {  // (0 / 0 too, where tau is 0 in f32)
                    g.flags |= 2;
                    return;
                }
                g.flags |= 1;
                const float a = z + gumbel_screen(lj, hj);
                moved |= a > amax;
                amax = fmaxf(amax, a);
                const float lo_keep = screen_floor(amax, 0x1p-20f);
                if (a >= lo_keep) {
                    // into the first slot that holds nothing within the margin (slots are reused)
                    const int at = !(ca0 >= lo_keep) ? 0 : (!(ca1 >= lo_keep) ? 1 : (!(ca2 >= lo_keep) ? 2 : (!(ca3 >= lo_keep) ? 3 : 4)));
                    const int v = 8 * i - g.r + j;
                    ca0 = at == 0 ? a : ca0;
                    ca1 = at == 1 ? a : ca1;
                    ca2 = at == 2 ? a : ca2;
                    ca3 = at == 3 ? a : ca3;
                    cz0 = at == 0 ? z : cz0;
                    cz1 = at == 1 ? z : cz1;
                    cz2 = at == 2 ? z : cz2;
                    cz3 = at == 3 ? z : cz3;
                    cv0 = at == 0 ? v : cv0;
                    cv1 = at == 1 ? v : cv1;
                    cv2 = at == 2 ? v : cv2;
                    cv3 = at == 3 ? v : cv3;
                    if (at == 4) g.flags |= 4;
                }
            });
            if (__ballot(moved) != 0) near = fmaxf(near, bound_floor(wave_max3_dpp(amax)));
        });
        // the segment's largest screened value and the flags
        g.best = amax;
        g.bidx = 0;
        g.reduce(sbest, sidx, sflags, scount);
        const float amx = g.best, lo_row = screen_floor(amx, 0x1p-21f);
        if (rec) {
            if (threadIdx.x == 0) srec = 0;
            __syncthreads();
            // (the candidates' order does not matter: what is made of them breaks ties by element)
            auto leave = [&](float ca, float cz, int cv) {
                if (!(ca >= lo_row)) return;
                const int at = atomicAdd(&srec, 1);
                if (at < kGumbelRecCand) {
                    rec->ca[at] = ca;
                    rec->cz[at] = cz;
                    rec->cv[at] = cv;
                }
            };
            leave(ca0, cz0, cv0);
            leave(ca1, cz1, cv1);
            leave(ca2, cz2, cv2);
            leave(ca3, cz3, cv3);
            __syncthreads();
            if (threadIdx.x == 0) {
                rec->a = amx;
                rec->flags = g.flags | (srec > kGumbelRecCand ? 4 : 0);
                rec->n = min(srec, kGumbelRecCand);
            }
            return;
        }
        // the candidates within the row's margin: when there is one, it is the row's exact first
        // maximum (every other element lies below it exactly), and its index is the answer
        g.best = -INFINITY;
        g.bidx = 0x7fffffff;
        g.count = 0;
        auto offer = [&](float ca, int cv) {
            if (ca >= lo_row) {
                best_merge(g.best, g.bidx, ca, cv);
                g.count++;
            }
        };
        offer(ca0, cv0);
        offer(ca1, cv1);
        offer(ca2, cv2);
        offer(ca3, cv3);
        g.reduce(sbest, sidx, sflags, scount);
        if ((g.flags & 2) || !(g.flags & 1) || (g.count == 1 && !(g.flags & 4))) {
            // a refused row (a NaN, or nothing allowed), or bidx is the one candidate's (with no
            // thread's slots overflowed: an element left out of them could lie within the margin)
        } else if (g.flags & 4) {
            g.every_exact(gqb, gqz);  // a thread ran out of slots
            g.reduce(sbest, sidx, sflags, scount);
        } else {
            // the candidates within the margin of the row's largest, exactly (their blocks again)
            g.best = -INFINITY;
            g.bidx = 0x7fffffff;
            auto resolve = [&](float ca, float cz, int cv) {
                const bool take = ca >= lo_row;
                if (__ballot(take) == 0) return;
                if (take) g.exact_again(cv, cz);
            };
            resolve(ca0, cz0, cv0);
            resolve(ca1, cz1, cv1);
            resolve(ca2, cz2, cv2);
            resolve(ca3, cz3, cv3);
            g.reduce(sbest, sidx, sflags, scount);
        }
        if (threadIdx.x == 0) g.write_row();
    }
}

// The rows of a launch with several workgroups per row: a lane of the first wave per segment's record,
// the candidates of the row's margin among theirs as above.
template <int DT, int MK, bool ODD, bool GREEDY>
__global__ __launch_bounds__(kGumbelMaxThreads) void k_gumbel_finish(GumbelP p) {
    __shared__ float sbest[kGumbelMaxThreads / 64];
    __shared__ int sidx[kGumbelMaxThreads / 64];
    __shared__ int sflags[kGumbelMaxThreads / 64];
    __shared__ int scount[kGumbelMaxThreads / 64];
    extern __shared__ __attribute__((aligned(16))) int gdyn[];
    Gumbel<DT, MK, ODD, GREEDY> g(p, blockIdx.x);
    // (every wave reads the records: what follows is then the same in all of them)
    const bool have = g.lane < p.segs;
    const GumbelRec *rec = p.rec + g.row * p.segs + (have ? g.lane : 0);
    const float a = have ? rec->a : -INFINITY;
    int fl = have ? rec->flags : 0, n = have ? rec->n : 0;
    if constexpr (GREEDY) {
        g.best = a;
        g.bidx = have ? rec->cv[0] : 0x7fffffff;
        g.flags = fl;
        g.reduce(sbest, sidx, sflags, scount);
        if (threadIdx.x == 0) g.write_row();
        return;
    }
    const float amx = wave_max(a), lo_row = screen_floor(amx, 0x1p-21f);
    if (!(a >= lo_row)) {  // a segment that ran out of slots matters only if it is near the row's largest
        fl &= ~4;
        n = 0;
    }
    int total = 0, only = 0x7fffffff;
    for (int k = 0; k < n; k++)
        if (rec->ca[k] >= lo_row) {
            total++;
            only = min(only, rec->cv[k]);
        }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        fl |= __shfl_xor(fl, o, 64);
        total += __shfl_xor(total, o, 64);
        only = min(only, __shfl_xor(only, o, 64));
    }
    g.flags = fl;
    g.bidx = only;
    if (!(fl & 2) && (fl & 1) && (total != 1 || (fl & 4))) {
        g.best = -INFINITY;
        g.bidx = 0x7fffffff;
        if (fl & 4) {
            g.every_exact(gdyn, reinterpret_cast<float *>(gdyn + (blockDim.x / 64) * kGumbelQueue));
        } else if (g.wave == 0) {
            for (int k = 0; k < n; k++)
                if (rec->ca[k] >= lo_row) g.exact_again(rec->cv[k], rec->cz[k]);
        }
        g.reduce(sbest, sidx, sflags, scount);
    }
    if (threadIdx.x == 0) g.write_row();
}

}  // namespace
}  // namespace nt
