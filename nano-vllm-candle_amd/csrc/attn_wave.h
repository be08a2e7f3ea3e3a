// A wave of the paged attention on matrix cores: K/V fragments in registers, online softmax.  Shared by the prompt and decode kernels (kernels.hip) and the resident
// decode step (resident.hip).
#pragma once
#include "device_common.h"

namespace nvllm {

// gfx950, hipcc of ROCm 7.2: a v_mfma_f32_16x16x32_bf8_bf8 that takes as SrcC the result of a v_mfma_f32_16x16x32_f16 issued
// a few instructions earlier read garbage -- the compiler leaves too few wait states between the two MFMA types and the
// hardware does not interlock.  Seen only once the register allocator had no slack (two waves per SIMD, 230-246 registers):
// in roomier builds the scheduler happened to put other fragments' MFMAs in between, which is luck, not a guarantee.  The
// data dependency pins this statement between producer and consumer; 20 wait states cover a 16-pass producer.
__device__ __forceinline__ void mfma_result_settled(f32x4& acc) { asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(acc)); }

// ... of all accumulators of a wave: each statement waits, for the compiler may put a producer between two of them
template <int QT, int DT>
__device__ __forceinline__ void mfma_results_settled(f32x4 (&o)[QT][DT]) {
#pragma unroll
    for (int t = 0; t < QT; ++t)
#pragma unroll
        for (int d = 0; d < DT; d += 4)
            asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" : "+v"(o[t][d]), "+v"(o[t][d + 1]), "+v"(o[t][d + 2]), "+v"(o[t][d + 3]));
}
// eight f16 as bf8 (the B operand of a residual product; two mantissa bits leave that 2^-12-sized term 12 % accurate)
__device__ __forceinline__ long bf8x8(const f16x8& x) {
    int w0 = 0, w1 = 0;
    w0 = __builtin_amdgcn_cvt_pk_bf8_f32((float)x[0], (float)x[1], w0, false);
    w0 = __builtin_amdgcn_cvt_pk_bf8_f32((float)x[2], (float)x[3], w0, true);
    w1 = __builtin_amdgcn_cvt_pk_bf8_f32((float)x[4], (float)x[5], w1, false);
    w1 = __builtin_amdgcn_cvt_pk_bf8_f32((float)x[6], (float)x[7], w1, true);
    return (long)(((unsigned long long)(unsigned)w1 << 32) | (unsigned)w0);
}
// one of the two 8-byte residual fragments in a lane's 16 bytes
__device__ __forceinline__ long bf8_half(const uint4& w, int second) {
    return (long)(second ? ((unsigned long long)w.w << 32) | w.z : ((unsigned long long)w.y << 32) | w.x);
}

// ---------------------------------------------------------------------------------------------------
// A wave of the paged attention: QT sub-tiles of 16 rows (heads x tokens) against 32-token K/V tiles.
// Decode's waves (QT 1) had a form of their own: a maximum across lanes, a rescale of O and a canonicalising exp2f in every tile, and with a 24-bit cache
// 24 waits of 20 states between the residuals' products and the others, 2.4 us a tile where 16 bits took 1.1.  In this form, us a launch by events, 16 heads on 8:
// 24 rows of 48 to 408 with 24 bits 18.5 -> 16.6, with 16 13.6 -> 13.1; 8 x 300 15.4 -> 13.9, 11.4 the same; 64 x 64 to 512 29.7 -> 28.5, 22.3 -> 21.7; 200 x 64 to 1024 133 -> 131,
// 87 the same; over 36 such calls 4.5 and 2 % less, 1 % with 40 heads on 8 and 16 on one.
// ---------------------------------------------------------------------------------------------------
template <int HD, int QT, int VLO>
struct AttnWave {
    static constexpr int DC = HD / 32, DT = HD / 16, DL = VLO ? DT / 2 : 0;
    static constexpr bool KLO = VLO == 2;
    f16x8 qh[QT][DC], ql[QT][DC];   // q as f16 hi + lo
    long q8[QT][KLO ? DC : 1];      // 24-bit K: q as bf8, against the residual bytes
    f32x4 o[QT][DT];                // not normalised yet
    float m[QT], lsum[QT];          // the softmax's reference, this lane's part of its sum
    int my_row[QT], my_pos[QT];     // this lane's rows (-1: none) and their positions
    bool fresh;                     // no tile seen yet

    // the lanes' rows of a q-tile
    __device__ __forceinline__ void rows(const PrefillTile& q, int gqa, int l15) {
        const int tpq = 16 / gqa;
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            const int tok = t * tpq + l15 / gqa;
            const bool valid = (l15 < tpq * gqa) && (tok < q.nrows);
            my_row[t] = valid ? q.row0 + tok : -1;
            my_pos[t] = valid ? q.first + tok : -1;
        }
    }
    // q as it is stored, for begin(): every lane loads, those of no row the tile's first
    __device__ __forceinline__ void load_q(const AttnArgs& a, const PrefillTile& q, int my_head, int grp, float4 (&x)[QT][DC][2]) const {
        const int ldq = a.nh_l * HD;
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            const float4* p = reinterpret_cast<const float4*>(a.q + (size_t)(my_row[t] < 0 ? q.row0 : my_row[t]) * ldq + (size_t)my_head * HD + grp * 8);
#pragma unroll
            for (int c = 0; c < DC; ++c) { x[t][c][0] = p[c * 8]; x[t][c][1] = p[c * 8 + 1]; }
        }
    }
    __device__ __forceinline__ void begin(const float4 (&q)[QT][DC][2]) {
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                const float4 u = q[t][c][0], v = q[t][c][1];
                const float x[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float y = my_row[t] >= 0 ? x[j] : 0.f;
                    const _Float16 h = (_Float16)y;
                    qh[t][c][j] = h;
                    ql[t][c][j] = (_Float16)(y - (float)h);
                }
            }
        start();
    }
    // qh and ql are there, no tile is yet
    __device__ __forceinline__ void start() {
        if constexpr (KLO) {
#pragma unroll
            for (int t = 0; t < QT; ++t)
#pragma unroll
                for (int c = 0; c < DC; ++c) q8[t][c] = bf8x8(qh[t][c]);
        }
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            m[t] = 0.f;
            lsum[t] = 0.f;
#pragma unroll
            for (int d = 0; d < DT; ++d) o[t][d] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        fresh = true;
    }
    // One tile from token T0 on.  fr: its K fragments, the two halves of each in turn; frl: their residuals.  V's fragments are read after scores_made(),
    // which may overwrite K's.
    template <class F>
    __device__ __forceinline__ void tile(int T0, int grp, int first_pos, const uint4 (&fr)[2 * DC], const uint4 (&frl)[KLO ? DC : 1], const uint4 (&fv)[DT],
                                         const uint4 (&fvl)[VLO ? DL : 1], F scores_made) {
        const int tokA = T0 + grp * 4, tokB = T0 + 16 + grp * 4;
        f32x4 sa[QT], sb[QT];
#pragma unroll
        for (int t = 0; t < QT; ++t) { sa[t] = f32x4{-m[t], -m[t], -m[t], -m[t]}; sb[t] = sa[t]; }  // scores come out less the reference
        // Residual bytes are bf8 numbers, operands as they are, and come first: the f16 products wait once for all of them (see
        // mfma_result_settled)
        if constexpr (KLO) {
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                const long la = bf8_half(frl[c >> 1], c & 1), lb = bf8_half(frl[DC / 2 + (c >> 1)], c & 1);
#pragma unroll
                for (int t = 0; t < QT; ++t) {
                    sa[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf8_bf8(la, q8[t][c], sa[t], 0, 0, 0);
                    sb[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf8_bf8(lb, q8[t][c], sb[t], 0, 0, 0);
                }
            }
#pragma unroll
            for (int t = 0; t < QT; ++t) { mfma_result_settled(sa[t]); mfma_result_settled(sb[t]); }
        }
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            const f16x8 fa = __builtin_bit_cast(f16x8, fr[2 * c]), fb = __builtin_bit_cast(f16x8, fr[2 * c + 1]);
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                sa[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa, qh[t][c], sa[t], 0, 0, 0);
                sb[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb, qh[t][c], sb[t], 0, 0, 0);
            }
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                sa[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fa, ql[t][c], sa[t], 0, 0, 0);
                sb[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb, ql[t][c], sb[t], 0, 0, 0);
            }
        }
        scores_made();
        // Online softmax, written for the VALU: this block, not the MFMAs, sets the wave's time.  m is a reference near the row's maximum,
        // not the maximum: it moves only when a score exceeds it by more than kSlack (p stays below 2^kSlack, well inside f16, and
        // p / sum p does not depend on the reference), so the usual tile needs no maximum across lanes, no rescale of O and, the
        // reference being the accumulators' start, no subtraction.  Every row that has a visible token has one in its wave's first tile,
        // where the reference is set.  Raw v_exp_f32 (a flushed denormal is 0 either way), v_maximum3 without the canonicalisation
        // fmaxf() pays per operand, the causal mask only on tiles that reach past the wave's first row.
        constexpr float kSlack = 8.f;
        f16x8 P[QT], Pl[QT];  // P as f16 hi + lo (see attn_paged_kernel): the prompt's own K/V-dependent rows keep 22 bits too
        if (T0 + 31 > first_pos) {
#pragma unroll
            for (int t = 0; t < QT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    sa[t][r] = tokA + r <= my_pos[t] ? sa[t][r] : -1e30f;
                    sb[t][r] = tokB + r <= my_pos[t] ? sb[t][r] : -1e30f;
                }
        }
        float mt[QT];
        bool moves = fresh;
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            mt[t] = max3(sa[t][0], sa[t][1], sa[t][2]);
            mt[t] = max3(mt[t], sa[t][3], sb[t][0]);
            mt[t] = max3(mt[t], sb[t][1], sb[t][2]);
            mt[t] = max3(mt[t], sb[t][3], mt[t]);
            moves = moves || mt[t] > kSlack;
        }
        if (__builtin_amdgcn_ballot_w64(moves) != 0) {
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                float up = max3(mt[t], __shfl_xor(mt[t], 16), mt[t]);
                up = max3(up, __shfl_xor(up, 32), up);      // the row's maximum, the same in its four lanes
                if (!fresh) up = fmaxf(up, 0.f);
                else if (up <= -1e29f) up = 0.f;                // no visible token (and none to come)
                const float alpha = __builtin_amdgcn_exp2f(-up);  // fresh: what it scales is 0
                m[t] += up;
                lsum[t] = fresh ? 0.f : lsum[t] * alpha;
#pragma unroll
                for (int r = 0; r < 4; ++r) { sa[t][r] -= up; sb[t][r] -= up; }
                if (!fresh)
#pragma unroll
                    for (int d = 0; d < DT; ++d) { o[t][d][0] *= alpha; o[t][d][1] *= alpha; o[t][d][2] *= alpha; o[t][d][3] *= alpha; }
            }
            fresh = false;
        }
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            float p[8];
#pragma unroll
            for (int r = 0; r < 4; ++r) { p[r] = __builtin_amdgcn_exp2f(sa[t][r]); p[4 + r] = __builtin_amdgcn_exp2f(sb[t][r]); }
            lsum[t] += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            split_f16x8(p, P[t], Pl[t]);
        }
        if constexpr (VLO != 0) {
            long P8[QT];
#pragma unroll
            for (int t = 0; t < QT; ++t) P8[t] = bf8x8(P[t]);
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int t = 0; t < QT; ++t) o[t][d] = __builtin_amdgcn_mfma_f32_16x16x32_bf8_bf8(bf8_half(fvl[d >> 1], d & 1), P8[t], o[t][d], 0, 0, 0);
            mfma_results_settled(o);
        }
#pragma unroll
        for (int d = 0; d < DT; ++d) {
#pragma unroll
            for (int t = 0; t < QT; ++t) o[t][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, fv[d]), P[t], o[t][d], 0, 0, 0);
#pragma unroll
            for (int t = 0; t < QT; ++t) o[t][d] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, fv[d]), Pl[t], o[t][d], 0, 0, 0);
        }
    }
};

}  // namespace nvllm
