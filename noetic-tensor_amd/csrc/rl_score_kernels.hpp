// The nn::rl scorer and its fused backward, device code for gfx950 (MI355X): per-token
// log-probabilities, the exact KL to a frozen reference and the entropy in one pass over a row
// (k_score), and the gradient of a weighted sum of the three with respect to the logits
// (k_score_grad). One source for both ways the library builds them: compiled ahead of time into
// libnoetic_hip.so (rl_kernels.hip includes this file), and compiled at run time by hiprtc from
// the text embedded in the library (rtc.cpp), which names each template instance it needs. The
// row layout, arithmetic and determinism rules are described in rl_kernels.hip.
#pragma once

#include "nt_rows.hpp"

namespace nt {
namespace {

// ------------------------------------------------------------------ scorer

struct ScoreP {
    const void *logits;
    const void *ref;
    const void *mask;
    int64_t V, ld;
    MaskMap mm;  // the mask row of each logits row
    float c;
    float tau;
    int tau_one;
    int nc;
    const int32_t *tokens;
    float *logp, *ref_logp, *kl, *ent;
    uint8_t *status;
    float *lse_base, *lse_rest, *ref_lse_base, *ref_lse_rest;
    int batch;            // chunks per batch (at most the kernel's NB)
    int per;              // batches per record
    int recs;             // records per row
    int segs;             // workgroups per row
    struct RowRec *part;  // segs > 1: the records, [rows][recs]
};

// What a wave found in a run of chunks (value space, exponent scale c). Every sum is relative to the
// run's own maxima, so no term cancels against another of size |logit|:
//   S  = sum w,                 w = exp2((v - a) c)
//   H  = sum w (v - a) c                                  (entropy)
//   B  = sum w ((v - a) - (v_ref - a_ref)) c              (exact KL)
//   Sr = sum exp2((v_ref - a_ref) c)                      (reference normaliser)
struct RowRec {
    float a, S, H, B;
    float ar, Sr;
};

// Sums in f64 relative to the maxima af and arf.
struct RowSums {
    double S, H, B, Sr;
};

__device__ __forceinline__ float shift_of(float a) { return a == -INFINITY ? 0.0f : a; }

// Record r's sums, moved to the maxima af and arf (at least its own), added to t.
template <bool REF, bool KL, bool ENT>
__device__ __forceinline__ void rec_add(RowSums &t, const RowRec &r, float af, float arf, float c) {
    if (r.S > 0.0f) {
        const double d = (double(r.a) - double(af)) * double(c), f = exp2(d);
        t.S += f * double(r.S);
        if constexpr (ENT) t.H += f * (double(r.H) + d * double(r.S));
        if constexpr (KL) {
            const double e = (double(r.ar) - double(arf)) * double(c);
            t.B += f * (double(r.B) + (d - e) * double(r.S));
        }
    } else if (!(r.S == r.S)) {
        t.S = NAN;
    }
    if (REF && r.ar != -INFINITY) t.Sr += exp2((double(r.ar) - double(arf)) * double(c)) * double(r.Sr);
}

// Record o added to s (rows of more than kScoreRecs batches: a record then holds several).
template <bool REF, bool KL, bool ENT>
__device__ __forceinline__ void rec_merge(RowRec &s, const RowRec &o, float c) {
    const float a = fmaxf(s.a, o.a), ar = fmaxf(s.ar, o.ar);
    RowSums t{0.0, 0.0, 0.0, 0.0};
    rec_add<REF, KL, ENT>(t, s, a, ar, c);
    rec_add<REF, KL, ENT>(t, o, a, ar, c);
    s = RowRec{a, float(t.S), float(t.H), float(t.B), ar, float(t.Sr)};
}

constexpr int kScoreThreads = 256;
constexpr int kScoreWaves = kScoreThreads / kWave;
constexpr int kScoreRecs = 256;  // records per row, at most

// load_raw for aligned rows through per-row buffer resources (row bytes below 2^31), no bounds
// branch, 32-bit offsets, non-temporal (every input is read once). Past the row's end the
// hardware range check returns zeros (the caller excludes those lanes). A lane's elements in a
// 512-element chunk at c: bf16 c + 8l .. c + 8l + 7 (one 16-byte load per input); f32 two groups,
// c + 4l .. c + 4l + 3 and c + 256 + 4l .. c + 256 + 4l + 3, so that each 16-byte load
// instruction reads one contiguous kilobyte rather than every other 16 bytes of two (measured
// faster with non-temporal loads). e0 is the lane's first element; each group lies wholly inside
// the row or wholly past its end (V % 8 == 0).
template <int DT>
__device__ __forceinline__ int buf_lane_first(int chunk, int lane) {
    return chunk * kChunk + lane * (DT == NT_F32 ? 4 : kEpl);
}

template <int DT, int MK>
__device__ __forceinline__ void load_raw_buf(Raw<DT, MK> &r, __amdgpu_buffer_rsrc_t xres,
                                             __amdgpu_buffer_rsrc_t mres, int e0) {
    constexpr int kHalf = kChunk / 2;
    if constexpr (DT == NT_F32) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const auto a = __builtin_amdgcn_raw_buffer_load_b128(xres, (e0 + q * kHalf) * 4, 0, kCachePolicyNT);
            for (int i = 0; i < 4; i++) r.x[4 * q + i] = a[i];
        }
        if constexpr (MK == NT_MASK_U8) {
            r.m[0] = __builtin_amdgcn_raw_buffer_load_b32(mres, e0, 0, kCachePolicyNT);
            r.m[1] = __builtin_amdgcn_raw_buffer_load_b32(mres, e0 + kHalf, 0, kCachePolicyNT);
        } else if constexpr (MK == NT_MASK_F32) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const auto a = __builtin_amdgcn_raw_buffer_load_b128(mres, (e0 + q * kHalf) * 4, 0, kCachePolicyNT);
                for (int i = 0; i < 4; i++) r.m[4 * q + i] = a[i];
            }
        } else {
            r.m[0] = 0;
        }
    } else {
        const auto a = __builtin_amdgcn_raw_buffer_load_b128(xres, e0 * 2, 0, kCachePolicyNT);
        for (int i = 0; i < 4; i++) r.x[i] = a[i];
        if constexpr (MK == NT_MASK_U8) {
            const auto k = __builtin_amdgcn_raw_buffer_load_b64(mres, e0, 0, kCachePolicyNT);
            r.m[0] = k[0];
            r.m[1] = k[1];
        } else if constexpr (MK == NT_MASK_F32) {
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const auto a = __builtin_amdgcn_raw_buffer_load_b128(mres, e0 * 4 + 16 * q, 0, kCachePolicyNT);
                for (int i = 0; i < 4; i++) r.m[4 * q + i] = a[i];
            }
        } else {
            r.m[0] = 0;
        }
    }
}


// A row's outputs from its merged state: the references af and arf, the sums relative to them in
// f64. One thread.
template <int DT, int MK, bool REF, bool KL, bool ENT>
__device__ __forceinline__ void score_finish(const ScoreP &p, int64_t row, float af, float arf, double S, double H,
                                             double B, double Sr) {
    const bool tau_one = p.tau_one != 0;
    const void *xrow = static_cast<const char *>(p.logits) + row * p.ld * Elem<DT>::kBytes;
    const void *yrow = nullptr;
    if constexpr (REF) yrow = static_cast<const char *>(p.ref) + row * p.ld * Elem<DT>::kBytes;
    const void *mrow = nullptr;
    if constexpr (MK != NT_MASK_NONE) mrow = static_cast<const char *>(p.mask) + mask_row_at(p.mm, row) * MaskWords<MK>::kBytes;
    // The value-space max as the reference's f32 max of the tempered logits.
    auto zmax = [&](float a) -> float {
        if constexpr (MK != NT_MASK_F32) return tau_one ? a : a / p.tau;
        else return a;
    };
    int stt = NT_ROW_OK;
    // (nothing allowed, or every allowed logit below -FLT_MAX T, whose tempered value is -inf)
    if (af == -INFINITY || zmax(af) == -INFINITY) stt = NT_ROW_NO_TOKEN;
    else if (!(S == S)) stt = NT_ROW_NAN;
    const double lnS = log(S);
    // The tempered logit of one token, with the reference's f32 arithmetic.
    auto ztok = [&](const void *rowp, int64_t tok) -> float {
        float x;
        if constexpr (DT == NT_F32) x = static_cast<const float *>(rowp)[tok];
        else x = widen16<DT>(uint32_t(static_cast<const uint16_t *>(rowp)[tok]));
        float z = tau_one ? x : x / p.tau;
        if constexpr (MK == NT_MASK_U8) {
            if (static_cast<const uint8_t *>(mrow)[tok] == 0) z = -INFINITY;
        } else if constexpr (MK == NT_MASK_F32) {
            z = z + static_cast<const float *>(mrow)[tok];
        }
        return z;
    };
    int64_t tok = -1;
    if (p.tokens) {
        tok = p.tokens[row];
        if ((tok < 0 || tok >= p.V) && stt == NT_ROW_OK) stt = kRowBadToken;
    }
    const bool rowok = stt == NT_ROW_OK || stt == kRowBadToken;
    if (p.logp) p.logp[row] = stt == NT_ROW_OK ? float((double(ztok(xrow, tok)) - double(zmax(af))) - lnS) : NAN;
    if (p.ent) p.ent[row] = rowok ? float(lnS - kLn2 * H / S) : NAN;
    // The log-sum-exp as base + rest (z units): the base is the tempered value of the row's
    // final reference, the rest ln of the sum relative to it.
    if (p.lse_base) p.lse_base[row] = rowok ? zmax(af) : NAN;
    if (p.lse_rest) p.lse_rest[row] = rowok ? float(lnS) : NAN;
    if constexpr (REF) {
        const bool rok = arf != -INFINITY && Sr == Sr;
        if (p.ref_lse_base) p.ref_lse_base[row] = rok ? zmax(arf) : NAN;
        if (p.ref_lse_rest) p.ref_lse_rest[row] = rok ? float(log(Sr)) : NAN;
        if (p.ref_logp)
            p.ref_logp[row] = (rok && tok >= 0 && tok < p.V) ? float((double(ztok(yrow, tok)) - double(zmax(arf))) - log(Sr)) : NAN;
        if constexpr (KL) {
            // KL = sum p ((z - m) - (z_ref - m_ref)) - ln S + ln S_ref; the first sum is
            // ln2 * B / S because c ln2 is the value-to-logit scale (1/T, or 1 with an f32 mask).
            if (p.kl) p.kl[row] = (rowok && rok) ? float(kLn2 * B / S - log(S / Sr)) : NAN;
        }
    }
    if (p.status) p.status[row] = uint8_t(stt);
}

// A row from its records, by one wave: each lane adds records lane, lane + 64, .. in f64, then the lanes'
// sums in a fixed tree.
template <int DT, int MK, bool REF, bool KL, bool ENT>
__device__ __forceinline__ void score_row(const ScoreP &p, int64_t row, const RowRec *rec, int lane) {
    RowRec r[kScoreRecs / kWave];
    float af = -INFINITY, arf = -INFINITY;
#pragma unroll
    for (int k = 0; k < kScoreRecs / kWave; k++) {
        r[k] = RowRec{-INFINITY, 0.0f, 0.0f, 0.0f, -INFINITY, 0.0f};
        if (lane + k * kWave < p.recs) r[k] = rec[lane + k * kWave];
        af = fmaxf(af, r[k].a);
        arf = fmaxf(arf, r[k].ar);
    }
    af = wave_max3_dpp(af);
    if constexpr (REF) arf = wave_max3_dpp(arf);
    RowSums t{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int k = 0; k < kScoreRecs / kWave; k++)
        if (k * kWave < p.recs) rec_add<REF, KL, ENT>(t, r[k], af, arf, p.c);
    t.S = readlane_d(wave_scan_dpp(t.S), kWave - 1);
    if constexpr (ENT) t.H = readlane_d(wave_scan_dpp(t.H), kWave - 1);
    if constexpr (KL) t.B = readlane_d(wave_scan_dpp(t.B), kWave - 1);
    if constexpr (REF) t.Sr = readlane_d(wave_scan_dpp(t.Sr), kWave - 1);
    if (lane == 0) score_finish<DT, MK, REF, KL, ENT>(p, row, af, arf, t.S, t.H, t.B, t.Sr);
}

// A row's chunks go in batches of p.batch consecutive ones, its batches in records of p.per consecutive
// ones, the records to the waves of the row's p.segs workgroups in turn. Both numbers depend on the
// vocabulary and the mask's kind alone, and every record is made and merged alike wherever it is made, so
// a row's bits depend neither on the rows beside it nor on the number of workgroups.
//
// A batch is decoded into registers, the wave's next one is loaded, and then its maxima over the wave and
// its sums relative to them are taken: nothing is rescaled, and the folds over the wave come once per
// batch. NB = 4 holds 32 values of each input per lane (139 registers with a reference: three waves per
// SIMD; asking for four spilled, 268 -> 352 us at 8192 x 50304); an f32 mask's words and division take as
// many again, and there, and for rows of up to 32 chunks, NB = 2. Against a running state per lane over the
// whole row (us, before / now): 16384 x 8200 bf16 64.2 / 53.0, 300 x 128256 29.7 / 26.4, 8192 x 50304 with a
// reference 263 / 261, 4096 x 151936 f32 under a u8 mask 453.3 / 450.4.
template <int DT, int MK, bool REF, bool KL, bool ENT, bool AL, int NB = 4>
__global__ __launch_bounds__(kScoreThreads) void k_score(ScoreP p) {
    __shared__ RowRec ws[kScoreRecs];
    int64_t row = blockIdx.x;
    int seg = 0;
    if (p.segs > 1) {
        row = blockIdx.x / unsigned(p.segs);
        seg = int(blockIdx.x % unsigned(p.segs));
    }
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(seg * kScoreWaves + int(threadIdx.x / kWave));  // in the row
    const int nw = p.segs * kScoreWaves;
    const bool tau_one = p.tau_one != 0;
    const float c = p.c;
    const void *xrow = static_cast<const char *>(p.logits) + row * p.ld * Elem<DT>::kBytes;
    const void *yrow = nullptr;
    if constexpr (REF) yrow = static_cast<const char *>(p.ref) + row * p.ld * Elem<DT>::kBytes;
    const void *mrow = nullptr;
    if constexpr (MK != NT_MASK_NONE) mrow = static_cast<const char *>(p.mask) + mask_row_at(p.mm, row) * MaskWords<MK>::kBytes;

    // (used by the aligned path only, whose rows are below 2^31 bytes)
    const int Vb = AL ? int(p.V) : 0;
    const __amdgpu_buffer_rsrc_t xres =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(xrow), short(0), Vb * Elem<DT>::kBytes, kBufferWord3);
    const __amdgpu_buffer_rsrc_t yres =
        REF ? __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(yrow), short(0), Vb * Elem<DT>::kBytes, kBufferWord3)
            : xres;
    const __amdgpu_buffer_rsrc_t mres =
        MK != NT_MASK_NONE ? __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(mrow), short(0),
                                                               Vb * MaskWords<MK>::kBytes, kBufferWord3)
                           : xres;

    // Chunks c0 .. c0 + p.batch - 1: their maxima over the wave, then their sums relative to them. No
    // weight exceeds 1, so the sums cannot overflow, and the finishing differences (ln S - ln2 H / S for
    // the entropy, ln S - ln S_ref for the KL) stay small: no two terms of the size of the logits
    // cancel. (The maxima pass a NaN by; it stays in the sums.)
    Raw<DT, MK> rx[NB];
    Raw<DT, NT_MASK_NONE> ry[REF ? NB : 1];
    auto load = [&](int c0) {
        const int n = min(p.batch, p.nc - c0);  // (chunks past it load nothing)
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const int ch = c0 + b;
            if constexpr (AL) {
                const int e0 = b < n ? buf_lane_first<DT>(ch, lane) : int(p.V);
                load_raw_buf<DT, MK>(rx[b], xres, mres, e0);
                if constexpr (REF) load_raw_buf<DT, NT_MASK_NONE>(ry[b], yres, mres, e0);
            } else {
                const int64_t e0 = b < n ? int64_t(ch) * kChunk + lane * kEpl : p.V;
                load_raw<DT, MK, AL>(rx[b], xrow, mrow, e0, p.V);
                if constexpr (REF) load_raw<DT, NT_MASK_NONE, AL>(ry[b], yrow, nullptr, e0, p.V);
            }
        }
    };
    auto batch = [&](int c0, int next) -> RowRec {
        const int n = min(p.batch, p.nc - c0);
        float v[NB][kEpl], vr[REF ? NB : 1][kEpl];
        float am = -INFINITY, arm = -INFINITY;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (b < n) {
                decode<DT, MK>(rx[b], v[b], p.tau, tau_one);
                // The reference logits take the same temperature and vocabulary mask
                // (reference_kl, rl.rs:347-351).
                if constexpr (REF) decode_words<DT, MK>(ry[b].x, rx[b].m, vr[b], p.tau, tau_one);
                if constexpr (AL) {
                    // buffer loads past the row's end read zeros: only the last chunk can hold such
                    // element groups, which take no part in the sums
                    if (c0 + b == p.nc - 1) {
                        const int e0 = buf_lane_first<DT>(c0 + b, lane);
#pragma unroll
                        for (int j = 0; j < kEpl; j++) {
                            const int e = DT == NT_F32 ? e0 + (j < 4 ? j : kChunk / 2 + j - 4) : e0 + j;
                            if (e >= int(p.V)) {
                                v[b][j] = -INFINITY;
                                if constexpr (REF) vr[b][j] = -INFINITY;
                            }
                        }
                    }
                }
                const float t = max8_hw(v[b]);
                am = max3_hw(am, t, t);
                if constexpr (REF) {
                    const float tr = max8_hw(vr[b]);
                    arm = max3_hw(arm, tr, tr);
                }
            }
        }
        if (next < p.nc) load(next);
        auto larger = [](float x, float y) { return max3_hw(x, y, y); };
        if constexpr (REF) {
            const float both[2] = {am, arm}, m = wave_folds<2>(both, larger);
            am = readlane_f(m, 0);
            arm = readlane_f(m, 1);
        } else {
            const float one[1] = {am};
            am = readlane_f(wave_folds<1>(one, larger), 0);
        }
        const float sh = shift_of(am), shr = REF ? shift_of(arm) : 0.0f;
        float S = 0.0f, H = 0.0f, B = 0.0f, Sr = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            if (b < n) {
#pragma unroll
                for (int j = 0; j < kEpl; j++) {
                    const float d = (v[b][j] - sh) * c;
                    const float w = exp2_hw(d);
                    S += w;
                    if constexpr (ENT) H = fmaf(w, fmaxf(d, -FLT_MAX), H);
                    if constexpr (REF) {
                        const float e = (vr[b][j] - shr) * c;
                        Sr += exp2_hw(e);
                        if constexpr (KL) B = fmaf(w, fmaxf(d - e, -FLT_MAX), B);
                    }
                }
            }
        }
        // the sums asked for, over the lanes: S in lane 0, H, Sr and B in the next ones
        constexpr int kSums = 1 + ENT + REF + KL, kH = 1, kSr = 1 + ENT, kB = 1 + ENT + REF;
        float x[kSums > 2 ? 4 : kSums] = {};
        x[0] = S;
        if constexpr (ENT) x[kH] = H;
        if constexpr (REF) x[kSr] = Sr;
        if constexpr (KL) x[kB] = B;
        const float t = wave_folds(x, [](float a, float b) { return a + b; });
        RowRec r{am, readlane_f(t, 0), 0.0f, 0.0f, arm, 0.0f};
        if constexpr (ENT) r.H = readlane_f(t, kH);
        if constexpr (REF) r.Sr = readlane_f(t, kSr);
        if constexpr (KL) r.B = readlane_f(t, kB);
        return r;
    };

    RowRec *const recs = p.segs > 1 ? p.part + row * p.recs : ws;
    int c0 = wave < p.recs ? wave * p.per * p.batch : p.nc;
    if (c0 < p.nc) load(c0);
    RowRec r;
    for (int i = wave, k = 0; c0 < p.nc;) {
        // the batch after this one: the record's next, or the first of the wave's next record
        int ni = i, nk = k + 1;
        if (nk == p.per || c0 + p.batch >= p.nc) {
            ni = i + nw;
            nk = 0;
        }
        const int next = ni < p.recs ? (ni * p.per + nk) * p.batch : p.nc;
        const RowRec one = batch(c0, next);
        if (k == 0) r = one;
        else rec_merge<REF, KL, ENT>(r, one, c);
        if (nk == 0 && lane == 0) recs[i] = r;
        i = ni;
        k = nk;
        c0 = next;
    }
    if (p.segs > 1) return;  // (k_score_finish takes them)
    __syncthreads();
    if (threadIdx.x < kWave) score_row<DT, MK, REF, KL, ENT>(p, row, ws, lane);
}

// The rows of a launch with several workgroups per row, a wave each.
template <int DT, int MK, bool REF, bool KL, bool ENT>
__global__ __launch_bounds__(kWave) void k_score_finish(ScoreP p) {
    const int64_t row = blockIdx.x;
    score_row<DT, MK, REF, KL, ENT>(p, row, p.part + row * p.recs, threadIdx.x);
}

// ------------------------------------------------------------------ fused backward
//
// dL/dz_v = [v == token] g_logp - pi_v (A + B log pi_v + C log pi_ref,v) with A = g_logp +
// g_kl KL + g_H H, B = g_H - g_kl, C = g_kl (the sum of the three row gradients), and
// dL/dx_v = dL/dz_v / T. The kernel works in base 2: with l_v = log2 pi_v and r_v = log2 pi_ref,v,
// dL/dx_v = [v == token] g_logp / T - pi_v (A' + B' l_v + C' r_v), where A' = A / T,
// B' = B ln2 / T and C' = C ln2 / T are per-row constants. l_v is clamped at -256: an excluded
// (-inf) logit then has pi_v = 0 and a finite sum, so its gradient is exactly zero without a
// select. A refused row (NaN statistics) sets A' to NaN, which makes the whole row NaN, as the
// op sequence's log_softmax does. One block per row; each lane streams 8 elements per step,
// two steps in flight.

struct GradP {
    const void *logits, *ref, *mask;
    int64_t V, ld, gld;
    MaskMap mm;  // the mask row of each logits row
    float tau;
    int tau_one;
    const int32_t *tokens;
    const float *lb, *lr, *rlb, *rlr, *kl, *ent, *glp, *gkl, *gh;
    void *grad;
    int parts;  // workgroups per row: each takes every parts-th step
};

constexpr int kGradThreads = 256;
constexpr int kGradStep = kGradThreads * kEpl;  // elements a block covers per step

// f32 pair -> packed bf16 pair, round to nearest even (lo from a, hi from b).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
    uint32_t r;
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// Two gradients in a 16-bit dtype, a in the low half: bf16 as above, or f16 rounded to nearest
// even (v_cvt_f16_f32 in the default rounding mode; beyond 65504 they round to infinity).
template <int GDT>
__device__ __forceinline__ uint32_t pack16(float a, float b) {
    if constexpr (GDT == NT_BF16) return pack_bf16(a, b);
    else return uint32_t(__builtin_bit_cast(uint16_t, _Float16(a))) | (uint32_t(__builtin_bit_cast(uint16_t, _Float16(b))) << 16);
}

// The per-row constants of the backward (see above).
struct GradRow {
    float lb, l2, rlb, r2, A, B, C, gtok;
    int64_t tok;
};

template <bool KL>
__device__ __forceinline__ GradRow grad_row(const GradP &p, int64_t row) {
    GradRow g;
    const float inv_tau = p.tau_one ? 1.0f : 1.0f / p.tau;
    const float glp = p.glp ? p.glp[row] : 0.0f;
    const float gh = p.gh ? p.gh[row] : 0.0f;
    const float hv = p.gh ? p.ent[row] : 0.0f;
    float gkl = 0.0f, klv = 0.0f;
    g.lb = p.lb[row];
    const float lr = p.lr[row];
    g.l2 = lr * kLog2e;
    g.rlb = 0.0f;
    g.r2 = 0.0f;
    bool refused = !(g.lb == g.lb) || !(lr == lr);
    if constexpr (KL) {
        gkl = p.gkl[row];
        klv = p.kl[row];
        g.rlb = p.rlb[row];
        const float rlr = p.rlr[row];
        g.r2 = rlr * kLog2e;
        refused = refused || !(g.rlb == g.rlb) || !(rlr == rlr);
    }
    const float A = glp + (KL ? gkl * klv : 0.0f) + (p.gh ? gh * hv : 0.0f);
    g.A = refused ? __builtin_nanf("") : A * inv_tau;
    g.B = (gh - gkl) * float(kLn2) * inv_tau;
    g.C = gkl * float(kLn2) * inv_tau;
    g.gtok = glp * inv_tau;
    g.tok = p.glp ? int64_t(p.tokens[row]) : -1;
    return g;
}

// One element's gradient from its tempered logit z (and reference zr).
template <bool KL>
__device__ __forceinline__ float grad_elem(const GradRow &g, float z, float zr) {
    const float l = fmaxf(fmaf(z - g.lb, kLog2e, -g.l2), -256.0f);
    const float pi = exp2_hw(l);
    float t = fmaf(g.B, l, g.A);
    if constexpr (KL) {
        const float r = fmaxf(fmaf(zr - g.rlb, kLog2e, -g.r2), -256.0f);
        t = fmaf(g.C, r, t);
    }
    return fmaf(-pi, t, 0.0f);
}

// The tempered logit as tempered_logits computes it: x / T (an f32 divide), then the mask
// (TAU1: x is already divided, or T is 1).
template <int MK, bool TAU1>
__device__ __forceinline__ float grad_tempered(float x, float tau, uint32_t mword, int j) {
    float z = TAU1 ? x : x / tau;
    if constexpr (MK == NT_MASK_U8) {
        if (((mword >> (8 * (j % 4))) & 0xffu) == 0) z = -INFINITY;
    } else if constexpr (MK == NT_MASK_F32) {
        z = z + __uint_as_float(mword);
    }
    return z;
}

// The token's own term, in the one lane (of one step) that holds it. A lane's 8 elements are
// e0 + j, or with SPLIT two groups of 4: e0 + j (j < 4) and e1 + j - 4 (j >= 4).
template <bool SPLIT>
__device__ __forceinline__ void add_token_term(const GradRow &g, int64_t e0, int64_t e1, float *out) {
    const int64_t d = g.tok - e0;
    if (static_cast<uint64_t>(d) < uint64_t(SPLIT ? 4 : kEpl)) {
#pragma unroll
        for (int j = 0; j < (SPLIT ? 4 : kEpl); j++) out[j] += (j == int(d)) ? g.gtok : 0.0f;
    }
    if constexpr (SPLIT) {
        const int64_t d1 = g.tok - e1;
        if (static_cast<uint64_t>(d1) < 4u) {
#pragma unroll
            for (int j = 0; j < 4; j++) out[4 + j] += (j == int(d1)) ? g.gtok : 0.0f;
        }
    }
}

template <int DT, int MK, bool KL, bool TAU1, bool SPLIT = false>
__device__ __forceinline__ void grad_step(const GradRow &g, float tau, const Raw<DT, MK> &rx,
                                          const Raw<DT, NT_MASK_NONE> &ry, int64_t e0, int64_t e1, float *out) {
    // x / T for the step's 8 elements at once (div_tau: the IEEE quotient, three instructions each
    // where the division takes about ten), then the mask
    float x[kEpl], xr[kEpl];
#pragma unroll
    for (int j = 0; j < kEpl; j++) {
        x[j] = logit<DT>(rx.x, j);
        xr[j] = KL ? logit<DT>(ry.x, j) : 0.0f;
    }
    if constexpr (!TAU1) {
        div_tau<kEpl>(x, tau);
        if constexpr (KL) div_tau<kEpl>(xr, tau);
    }
#pragma unroll
    for (int j = 0; j < kEpl; j++) {
        const uint32_t mword = MK == NT_MASK_U8 ? rx.m[j / 4] : (MK == NT_MASK_F32 ? rx.m[j] : 0u);
        const float z = grad_tempered<MK, true>(x[j], tau, mword, j);
        const float zr = KL ? grad_tempered<MK, true>(xr[j], tau, mword, j) : 0.0f;
        out[j] = grad_elem<KL>(g, z, zr);
    }
    add_token_term<SPLIT>(g, e0, e1, out);
}

// Aligned rows (V % 8 == 0, 16-byte rows, row bytes below 2^31): every access goes through a
// per-row buffer resource. Past the end of the row loads return zeros and stores are dropped by
// the hardware range check, so the loop needs no bounds tests: every lane runs the same number
// of steps. A step covers 2048 elements. With a bf16 gradient lane t owns elements 8t..8t+7 (one
// 16-byte load per input, one 16-byte store). With an f32 gradient (32 bytes per lane) it owns
// 4t..4t+3 and 1024+4t..1024+4t+3 instead, so that each store instruction writes one contiguous
// stretch of whole cache lines rather than every other 16 bytes of them. Either way a group of
// a lane's elements lies wholly inside the row or wholly past it (V % 8 == 0). Every input is
// read once and the gradient written once, so all of them are accessed non-temporally.
template <int DT, int MK, bool KL, int GDT, bool TAU1>
__device__ __forceinline__ void grad_row_aligned(const GradP &p, const GradRow &g, int64_t row, int part) {
    constexpr int XB = Elem<DT>::kBytes, MB = MaskWords<MK>::kBytes, GB = GDT == NT_F32 ? 4 : 2;
    constexpr bool SPLIT = GDT == NT_F32;
    constexpr int kHalf = kGradStep / 2;
    const int V = int(p.V);
    const auto xres = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char *>(static_cast<const char *>(p.logits) + row * p.ld * XB), short(0), V * XB, kBufferWord3);
    __amdgpu_buffer_rsrc_t yres = xres, mres = xres;
    if constexpr (KL)
        yres = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(static_cast<const char *>(p.ref) + row * p.ld * XB), short(0), V * XB, kBufferWord3);
    if constexpr (MK != NT_MASK_NONE)
        mres = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(static_cast<const char *>(p.mask) + mask_row_at(p.mm, row) * MB), short(0), V * MB,
            kBufferWord3);
    const auto gres = __builtin_amdgcn_make_buffer_rsrc(static_cast<char *>(p.grad) + row * p.gld * GB, short(0),
                                                        V * GB, kBufferWord3);
    // 4 elements of one input at element e into words w0.. of dst (f32: 4 words, bf16: 2)
    auto load4 = [&](uint32_t *dst, __amdgpu_buffer_rsrc_t rs, int e) {
        if constexpr (DT == NT_F32) {
            const auto a = __builtin_amdgcn_raw_buffer_load_b128(rs, e * 4, 0, kCachePolicyNT);
            for (int i = 0; i < 4; i++) dst[i] = a[i];
        } else {
            const auto a = __builtin_amdgcn_raw_buffer_load_b64(rs, e * 2, 0, kCachePolicyNT);
            dst[0] = a[0];
            dst[1] = a[1];
        }
    };
    auto load = [&](auto &rx, auto &ry, int e0, int e1) {
        if constexpr (SPLIT) {
            constexpr int H = Elem<DT>::kWords / 2;
            load4(rx.x, xres, e0);
            load4(rx.x + H, xres, e1);
            if constexpr (KL) {
                load4(ry.x, yres, e0);
                load4(ry.x + H, yres, e1);
            }
            if constexpr (MK == NT_MASK_U8) {
                rx.m[0] = __builtin_amdgcn_raw_buffer_load_b32(mres, e0, 0, kCachePolicyNT);
                rx.m[1] = __builtin_amdgcn_raw_buffer_load_b32(mres, e1, 0, kCachePolicyNT);
            } else if constexpr (MK == NT_MASK_F32) {
                const auto a = __builtin_amdgcn_raw_buffer_load_b128(mres, e0 * 4, 0, kCachePolicyNT);
                const auto b = __builtin_amdgcn_raw_buffer_load_b128(mres, e1 * 4, 0, kCachePolicyNT);
                for (int i = 0; i < 4; i++) {
                    rx.m[i] = a[i];
                    rx.m[4 + i] = b[i];
                }
            }
        } else {
            if constexpr (DT == NT_F32) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const auto a = __builtin_amdgcn_raw_buffer_load_b128(xres, e0 * 4 + 16 * q, 0, kCachePolicyNT);
                    for (int i = 0; i < 4; i++) rx.x[4 * q + i] = a[i];
                    if constexpr (KL) {
                        const auto b = __builtin_amdgcn_raw_buffer_load_b128(yres, e0 * 4 + 16 * q, 0, kCachePolicyNT);
                        for (int i = 0; i < 4; i++) ry.x[4 * q + i] = b[i];
                    }
                }
            } else {
                const auto a = __builtin_amdgcn_raw_buffer_load_b128(xres, e0 * 2, 0, kCachePolicyNT);
                for (int i = 0; i < 4; i++) rx.x[i] = a[i];
                if constexpr (KL) {
                    const auto b = __builtin_amdgcn_raw_buffer_load_b128(yres, e0 * 2, 0, kCachePolicyNT);
                    for (int i = 0; i < 4; i++) ry.x[i] = b[i];
                }
            }
            if constexpr (MK == NT_MASK_U8) {
                const auto k = __builtin_amdgcn_raw_buffer_load_b64(mres, e0, 0, kCachePolicyNT);
                rx.m[0] = k[0];
                rx.m[1] = k[1];
            } else if constexpr (MK == NT_MASK_F32) {
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const auto a = __builtin_amdgcn_raw_buffer_load_b128(mres, e0 * 4 + 16 * q, 0, kCachePolicyNT);
                    for (int i = 0; i < 4; i++) rx.m[4 * q + i] = a[i];
                }
            }
        }
    };
    auto store = [&](int e0, int e1, const float *o) {
        if constexpr (GDT == NT_F32) {
            const v4u a = {__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3])};
            const v4u b = {__float_as_uint(o[4]), __float_as_uint(o[5]), __float_as_uint(o[6]), __float_as_uint(o[7])};
            __builtin_amdgcn_raw_buffer_store_b128(a, gres, e0 * 4, 0, kCachePolicyNT);
            __builtin_amdgcn_raw_buffer_store_b128(b, gres, e1 * 4, 0, kCachePolicyNT);
        } else {
            const v4u w = {pack16<GDT>(o[0], o[1]), pack16<GDT>(o[2], o[3]), pack16<GDT>(o[4], o[5]), pack16<GDT>(o[6], o[7])};
            __builtin_amdgcn_raw_buffer_store_b128(w, gres, e0 * 2, 0, kCachePolicyNT);
        }
    };
    const int t = int(threadIdx.x);
    const int first = SPLIT ? 4 * t : kEpl * t;  // the lane's first element in step 0
    // (no overflow: V is below 2^29 and parts at most V / (2 kGradStep), rounded up)
    for (int s0 = 2 * kGradStep * part; s0 < V; s0 += 2 * kGradStep * p.parts) {
        Raw<DT, MK> x0, x1;
        Raw<DT, NT_MASK_NONE> y0, y1;
        const int a0 = s0 + first, a1 = a0 + kGradStep;
        load(x0, y0, a0, a0 + kHalf);
        load(x1, y1, a1, a1 + kHalf);
        float o[kEpl];
        grad_step<DT, MK, KL, TAU1, SPLIT>(g, p.tau, x0, y0, a0, a0 + kHalf, o);
        store(a0, a0 + kHalf, o);
        grad_step<DT, MK, KL, TAU1, SPLIT>(g, p.tau, x1, y1, a1, a1 + kHalf, o);
        store(a1, a1 + kHalf, o);
    }
}

// Any other row layout: loads and stores at the elements' own alignment, element-wise only where a
// lane's 8 elements cross the row's end.
template <int DT, int MK, bool KL, int GDT, bool TAU1>
__device__ __forceinline__ void grad_row_general(const GradP &p, const GradRow &g, int64_t row, int part) {
    const char *xrow = static_cast<const char *>(p.logits) + row * p.ld * Elem<DT>::kBytes;
    const char *yrow = KL ? static_cast<const char *>(p.ref) + row * p.ld * Elem<DT>::kBytes : nullptr;
    const char *mrow = MK != NT_MASK_NONE ? static_cast<const char *>(p.mask) + mask_row_at(p.mm, row) * MaskWords<MK>::kBytes
                                          : nullptr;
    char *grow = static_cast<char *>(p.grad) + row * p.gld * (GDT == NT_F32 ? 4 : 2);
    for (int64_t e0 = int64_t(part) * kGradStep + threadIdx.x * kEpl; e0 < p.V; e0 += int64_t(p.parts) * kGradStep) {
        Raw<DT, MK> rx;
        Raw<DT, NT_MASK_NONE> ry;
        load_raw<DT, MK, false>(rx, xrow, mrow, e0, p.V);
        if constexpr (KL) load_raw<DT, NT_MASK_NONE, false>(ry, yrow, nullptr, e0, p.V);
        float o[kEpl];
        grad_step<DT, MK, KL, TAU1>(g, p.tau, rx, ry, e0, 0, o);
        if (e0 + kEpl <= p.V) {
            if constexpr (GDT == NT_F32) {
                u32x4_f32 *d = reinterpret_cast<u32x4_f32 *>(reinterpret_cast<float *>(grow) + e0);
                d[0] = u32x4_f32{__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3])};
                d[1] = u32x4_f32{__float_as_uint(o[4]), __float_as_uint(o[5]), __float_as_uint(o[6]), __float_as_uint(o[7])};
            } else {
                *reinterpret_cast<u32x4_f16 *>(reinterpret_cast<uint16_t *>(grow) + e0) =
                    u32x4_f16{pack16<GDT>(o[0], o[1]), pack16<GDT>(o[2], o[3]), pack16<GDT>(o[4], o[5]), pack16<GDT>(o[6], o[7])};
            }
            continue;
        }
        for (int j = 0; j < kEpl; j += 2) {
            if constexpr (GDT == NT_F32) {
                if (e0 + j < p.V) reinterpret_cast<float *>(grow)[e0 + j] = o[j];
                if (e0 + j + 1 < p.V) reinterpret_cast<float *>(grow)[e0 + j + 1] = o[j + 1];
            } else {
                const uint32_t w = pack16<GDT>(o[j], o[j + 1]);
                if (e0 + j < p.V) reinterpret_cast<uint16_t *>(grow)[e0 + j] = uint16_t(w);
                if (e0 + j + 1 < p.V) reinterpret_cast<uint16_t *>(grow)[e0 + j + 1] = uint16_t(w >> 16);
            }
        }
    }
}

template <int DT, int MK, bool KL, int GDT, bool AL>
__global__ __launch_bounds__(kGradThreads) void k_score_grad(GradP p) {
    int64_t row = blockIdx.x;
    int part = 0;
    if (p.parts > 1) {
        row = blockIdx.x / unsigned(p.parts);
        part = int(blockIdx.x % unsigned(p.parts));
    }
    const GradRow g = grad_row<KL>(p, row);
    if (p.tau_one) {
        if constexpr (AL) grad_row_aligned<DT, MK, KL, GDT, true>(p, g, row, part);
        else grad_row_general<DT, MK, KL, GDT, true>(p, g, row, part);
    } else {
        if constexpr (AL) grad_row_aligned<DT, MK, KL, GDT, false>(p, g, row, part);
        else grad_row_general<DT, MK, KL, GDT, false>(p, g, row, part);
    }
}

}  // namespace
}  // namespace nt
