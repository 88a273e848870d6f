// iq_mfma_half.h -- the reference's exact per-lane products on f16 MFMA
// (Q4_K, Q5_K and Q6_K weights): what ml_product (iq_mfma_lanes.h) computes
// on int8, bit for bit, with the lane integers formed in f32 at once.
//
// A scaled quant sc * q of Q4_K (at most 63 * 15) and Q5_K (63 * 31) is an
// integer below 2048, exact in f16, and so are the int8 activations; a
// Q6_K sc * (q - 32) reaches 4096, so it is split into 8 (sc >> 3) (q - 32),
// a multiple of 8, and (sc & 7) (q - 32).  Every product and partial sum of a
// lane's 32 terms is an integer of at most 2^24, so v_mfma_f32_16x16x32_f16
// over K = (c, e) for one reference lane k yields float(isum_k) itself:
// where the int8 form spends two MFMAs, a shift-add and a conversion per
// lane, output and block before the chain's FMA (two in Q6_K's case), only
// the FMA is left.  That matters because of what these cost on gfx950: with
// two waves or more on a SIMD an f32 FMA issues in 2.5 cycles, a conversion,
// shift-add or packed 16-bit operation in 4.2, a 16 x 16 MFMA in 18, a third of
// it under VALU issue.  Per 16 x 16 tile and Q4_K block that is about 460 cycles
// of issue against 900 (what the kernel adds to them: see mh_product).
#pragma once

#include "iq_mfma_lanes.h"

namespace iq {

typedef _Float16 v8h_mh __attribute__((ext_vector_type(8)));
typedef _Float16 v2h_mh __attribute__((ext_vector_type(2)));
typedef float v16f_mh __attribute__((ext_vector_type(16)));

// Activations: per row and block 512 bytes of f16, granule (k, q) of 16
// bytes at 64 k + 16 q holding dword (c, k) for c = 2 q and c = 2 q + 1, the
// four values of a dword in the order 0, 2, 1, 3 (the order in which a
// weight dword's bytes come apart into 16-bit halves).
constexpr int kMhBlock = 512;
// LDS strides of an activation row and of a weight row: 32 mod 64 bytes, on
// which fragment reads (16 rows, four granules each) have no bank conflicts
constexpr int kMhAS = 544;
template <int FMT>
constexpr int kMhBS = FMT == kQ4_K ? 160 : 224;

// Where lane l of a quantising wave (values 4 l .. 4 l + 3 of the block, packed int8) puts them.
__device__ __forceinline__ void mh_store(int8_t* block, int lane, uint32_t packed) {
    const int c = lane >> 3, k = lane & 7;
    const auto h = [&](int i) { return (_Float16)(float)(int8_t)(uint8_t)(packed >> (8 * i)); };
    *(v4h_ml*)(block + 64 * k + 16 * (c >> 1) + 8 * (c & 1)) = v4h_ml{h(0), h(2), h(1), h(3)};
}

template <int FMT, int RT>
struct MhStage {
    static constexpr int R = 16 * RT;
    static constexpr int A = 0;
    static constexpr int B = A + R * kMhAS;
    static constexpr int D = B + kMlCols * kMhBS<FMT>;
    static constexpr int H = D + R * 4;
    static constexpr int END = H + (MlFmt<FMT>::kMins ? R * 32 : 0);
};

__device__ __forceinline__ v2h_mh mh_pair(uint32_t v) { return __builtin_bit_cast(v2h_mh, v); }
__device__ __forceinline__ uint32_t mh_bits(v2h_mh v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ v2h_mh mh_both(float v) {
    const _Float16 h = (_Float16)v;
    return v2h_mh{h, h};
}
// As ml_product (16 RT activation rows x 64 weight rows on a 256-thread
// workgroup, the same result lanes), op.aq the f16 activations above (op.ldq
// bytes a row).
//
// Bound by issue for about half of the time, for the rest by latency that two
// waves per SIMD (224 VGPRs at RT = 2) do not cover: on [512 x 2048] -> 8192
// Q4_K a tile and block take 1125 cycles of a SIMD, VALU active for 600 of them
// (149 instructions), MFMA busy for 160, and a wave waits 28% of its time.
// [512 x 2048] -> 8192 Q4_K 77 -> 60 us, [512 x 4096] -> 2048 Q5_K 50 -> 38, [512
// x 2048] -> 8192 Q6_K 84 -> 78 (its second MFMA and its decode stay), against
// the int8 form.
// Splitting the eight lanes over two waves (128 VGPRs, four waves per SIMD)
// measured 66-71 us for the Q4_K call, 64-row tiles 66: both decode or
// address more per output than the occupancy returns.
template <int FMT, int RT, class ARow, class BRow>
__device__ __forceinline__ void mh_product(const MlOperands& op, ARow arow, BRow brow, uint8_t (*st)[MhStage<FMT, RT>::END],
                                           float (&v)[4 * RT]) {
    using F = MlFmt<FMT>;
    using L = MhStage<FMT, RT>;
    constexpr int NT = 256;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, jj = lane & 15;
    const int nb = op.nb;

    // ---- staging: fixed slots per thread
    constexpr int kAPer = L::R * 32 / NT;  // 16-byte granules
    constexpr int kB = kMlCols * F::NL, kBPer = (kB + NT - 1) / NT;
    uint32_t a_src[kAPer], b_src[kBPer];
    int a_off[kAPer], b_off[kBPer];
    bool b_hi[kBPer], b_last[kBPer];
    const int tid = threadIdx.x;
#pragma unroll
    for (int i = 0; i < kAPer; i++) {
        const int t = tid + NT * i, rr = t >> 5, part = t & 31;
        a_src[i] = (uint32_t)(arow(rr) * op.ldq + 16 * part);
        a_off[i] = L::A + rr * kMhAS + 16 * part;
    }
#pragma unroll
    for (int i = 0; i < kBPer; i++) {
        const int t = min(tid + NT * i, kB - 1);
        const int c2 = t / F::NL, part = t - c2 * F::NL;
        const int po = FMT == kQ6_K && part == F::NL - 1 ? 196 : 16 * part;
        b_hi[i] = c2 >= op.bsplit;
        b_last[i] = part == F::NL - 1;
        b_src[i] = (uint32_t)(brow(c2) * op.brow_bytes + po);
        b_off[i] = tid + NT * i < kB ? L::B + c2 * kMhBS<FMT> + po : -1;
    }
    const int tD = tid, tH = tid - 64;
    const int64_t d_row = arow(tD & (L::R - 1));
    const int64_t h_row = arow((tH >> 1) & (L::R - 1));

    v4i_ml sa[kAPer];
    u32x4 sb[kBPer];
    float sd = 0.f;
    v4i_ml sh16 = {};
    auto issue = [&](int b) {
        const int8_t* abase = op.aq + (int64_t)b * kMhBlock;
#pragma unroll
        for (int i = 0; i < kAPer; i++) sa[i] = *(const v4i_ml*)(abase + a_src[i]);
        const int64_t boff = FMT == kQ6_K ? ((int64_t)b * F::BB) & ~(int64_t)3 : (int64_t)b * F::BB;
#pragma unroll
        for (int i = 0; i < kBPer; i++) sb[i] = *(const u32x4*)((b_hi[i] ? op.b1 : op.b0) + boff + b_src[i]);
        if (tD < L::R) sd = op.ad[d_row * op.ldd + b];
        if constexpr (F::kMins)
            if (tH >= 0 && tH < 2 * L::R) sh16 = *(const v4i_ml*)(op.hs + (h_row * nb + b) * 16 + 8 * (tH & 1));
    };
    auto park = [&](uint8_t* s) {
#pragma unroll
        for (int i = 0; i < kAPer; i++)
            *(v4i_ml*)(s + a_off[i]) = sa[i];
#pragma unroll
        for (int i = 0; i < kBPer; i++)
            if (b_off[i] >= 0) ml_park_b<FMT>(s + b_off[i], sb[i], b_last[i]);
        if (tD < L::R) *(float*)(s + L::D + 4 * tD) = sd;
        if constexpr (F::kMins)
            if (tH >= 0 && tH < 2 * L::R) *(v4i_ml*)(s + L::H + 32 * (tH >> 1) + 16 * (tH & 1)) = sh16;
    };

    const int col = 16 * wave + jj;
    float acc[8][4 * RT], accm[FMT == kQ4_K ? 4 : 1][4 * RT];
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
        for (int r = 0; r < 4 * RT; r++) acc[k][r] = 0.f;
#pragma unroll
    for (int k = 0; k < (FMT == kQ4_K ? 4 : 1); k++)
#pragma unroll
        for (int r = 0; r < 4 * RT; r++) accm[k][r] = 0.f;
    issue(0);
    park(st[0]);
    lds_barrier();
    for (int b = 0; b < nb; b++) {
        const uint8_t* S = st[b & 1];
        if (b + 1 < nb) issue(b + 1);
        const int sh = FMT == kQ6_K ? (int)(((int64_t)b * F::BB) & 3) : 0;
        const uint8_t* bcol = S + L::B + col * kMhBS<FMT>;
        float dd[4 * RT];
        float xd, xdm = 0.f;
        Q4Scales sc{};
        uint32_t qd[8] = {}, qh[8] = {}, q2[8] = {};  // of lane k: Q4_K qs; Q5_K qs, qh; Q6_K ql, ql + 32, qh
        v2h_mh sA{}, cA{}, sB{}, cB{};                   // Q4_K, Q5_K: scales of chunks 2 q, 2 q + 1
        v2h_mh s6h[4] = {}, s6l[4] = {};                 // Q6_K: 8 (sc >> 3) and sc & 7 of scale 4 q + i
        if constexpr (FMT == kQ4_K || FMT == kQ5_K) {
            constexpr int QO = FMT == kQ5_K ? 48 : 16;
            const u32x4a16 hdr = *(const u32x4a16*)bcol;
            xd = f16_to_f32(hdr.x);
            xdm = f16_to_f32(hdr.x >> 16);
            sc = q4_scales(hdr.y, hdr.z, hdr.w);
            const uint32_t sw = q < 2 ? sc.sc_lo : sc.sc_hi;
            const float fa = (float)byte_of(sw, 2 * (q & 1)), fb = (float)byte_of(sw, 2 * (q & 1) + 1);
            // low nibbles are read as 1024 + q, high ones as 1024 + 16 q
            sA = mh_both(fa);
            cA = mh_both(-1024.f * fa);
            sB = mh_both(0.0625f * fb);
            cB = mh_both(-64.f * fb);
            ml_lds_span<8>(bcol, MlShift<0>{}, QO + 32 * q, qd);
            if constexpr (FMT == kQ5_K) ml_lds_span<8>(bcol, MlShift<0>{}, 16, qh);
        } else {
            xd = f16_to_f32(ml_lds_win(bcol, sh, 208) & 0xffffu);
            const uint32_t q6s = ml_lds_win(bcol, sh, 192 + 4 * q);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int scv = (int)(int8_t)(uint8_t)(q6s >> (8 * i));
                s6h[i] = mh_both((float)(scv & ~7));
                s6l[i] = mh_both((float)(scv & 7));
            }
            ml_lds_span<8>(bcol, sh, 64 * (q >> 1), qd);
            ml_lds_span<8>(bcol, sh, 64 * (q >> 1) + 32, q2);
            ml_lds_span<8>(bcol, sh, 128 + 32 * (q >> 1), qh);
        }
#pragma unroll
        for (int t = 0; t < RT; t++) {
            const f32x4 yd = *(const f32x4*)(S + L::D + 4 * (16 * t + 4 * q));
#pragma unroll
            for (int r = 0; r < 4; r++) dd[4 * t + r] = yd[r] * xd;
        }
        constexpr uint32_t kE = 0x64006400u;  // f16 1024: bits under it read 1024 + value
        // masks kept in registers, so that mask and exponent take one v_and_or (one literal an instruction)
        uint32_t mlo = 0x000f000fu, mhi = 0x00f000f0u, mby = 0x00ff00ffu;
        if constexpr (FMT == kQ6_K) asm volatile("" : "+v"(mby));
        else asm volatile("" : "+v"(mlo), "+v"(mhi));
        // the block integers of reference lane k, all tiles
        auto dots = [&](int k, const v8h_mh (&a)[RT], v4f_ml (&o)[RT]) {
            uint32_t w1[4], w2[4] = {};
            if constexpr (FMT == kQ4_K || FMT == kQ5_K) {
                const uint32_t e = qd[k], od = e >> 8;
                uint32_t h0 = kE, h1 = kE, h2 = kE, h3 = kE;
                if constexpr (FMT == kQ5_K) {
                    // the fifth bits of chunks 2 q and 2 q + 1: bits 2 q and 2 q + 1 of the qh bytes
                    const uint32_t he = qh[k] >> (2 * q), ho = he >> 8;
                    h0 |= (he & 0x00010001u) << 4;
                    h1 |= (ho & 0x00010001u) << 4;
                    h2 |= (he & 0x00020002u) << 7;
                    h3 |= (ho & 0x00020002u) << 7;
                }
                w1[0] = mh_bits(__builtin_elementwise_fma(mh_pair((e & mlo) | h0), sA, cA));
                w1[1] = mh_bits(__builtin_elementwise_fma(mh_pair((od & mlo) | h1), sA, cA));
                w1[2] = mh_bits(__builtin_elementwise_fma(mh_pair((e & mhi) | h2), sB, cB));
                w1[3] = mh_bits(__builtin_elementwise_fma(mh_pair((od & mhi) | h3), sB, cB));
            } else {
                // scales 4 q + 2 cc + (k >= 4)
                const v2h_mh off = {(_Float16)-1056.f, (_Float16)-1056.f};
#pragma unroll
                for (int cc = 0; cc < 2; cc++) {
                    const uint32_t l = cc ? q2[k] : qd[k];
                    const uint32_t lo4 = (q & 1) ? ((l >> 4) & 0x0f0f0f0fu) : (l & 0x0f0f0f0fu);
                    const uint32_t u = lo4 | (((qh[k] >> (2 * (2 * (q & 1) + cc))) & 0x03030303u) << 4);
                    const v2h_mh t02 = mh_pair((u & mby) | kE) + off;
                    const v2h_mh t13 = mh_pair(((u >> 8) & mby) | kE) + off;
                    const int si = 2 * cc + (k >= 4);
                    w1[2 * cc] = mh_bits(t02 * s6h[si]);
                    w1[2 * cc + 1] = mh_bits(t13 * s6h[si]);
                    w2[2 * cc] = mh_bits(t02 * s6l[si]);
                    w2[2 * cc + 1] = mh_bits(t13 * s6l[si]);
                }
            }
            const v8h_mh b1 = __builtin_bit_cast(v8h_mh, u32x4{w1[0], w1[1], w1[2], w1[3]});
            const v8h_mh b2 = __builtin_bit_cast(v8h_mh, u32x4{w2[0], w2[1], w2[2], w2[3]});
#pragma unroll
            for (int t = 0; t < RT; t++) {
                const v4f_ml z = {};
                o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], b1, z, 0, 0, 0);
                if constexpr (FMT == kQ6_K) o[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[t], b2, o[t], 0, 0, 0);
            }
        };
        const uint8_t* ap = S + L::A + jj * kMhAS + 16 * q;
        auto frag = [&](int k, v8h_mh (&a)[RT]) {
#pragma unroll
            for (int t = 0; t < RT; t++) a[t] = *(const v8h_mh*)(ap + 16 * t * kMhAS + 64 * k);
        };
        // step k: the fragments of lane k + 2 are read, the dots of lane k + 1
        // issue and the chains of lane k advance under their passes
        v4f_ml cur[RT], nxt[RT];
        v8h_mh a0[RT], a1[RT];
        frag(0, a0);
        frag(1, a1);
        dots(0, a0, cur);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int k = 0; k < 8; k++) {
            if (k + 2 < 8) frag(k + 2, k & 1 ? a1 : a0);
            if (k + 1 < 8) dots(k + 1, k & 1 ? a0 : a1, nxt);
#pragma unroll
            for (int t = 0; t < RT; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[k][4 * t + r] = __builtin_fmaf(dd[4 * t + r], cur[t][r], acc[k][4 * t + r]);
            // advanced here, not sunk, which bounds the live MFMA results
#pragma unroll
            for (int r = 0; r < 4 * RT; r++) asm volatile("" : "+v"(acc[k][r]));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < RT; t++) cur[t] = nxt[t];
        }
        if constexpr (F::kMins) {
            // lane group q supplies mins 2 q, 2 q + 1 against the 16-value sums 4 q .. 4 q + 3
            const uint32_t mwd = q < 2 ? sc.mn_lo : sc.mn_hi;
            const _Float16 mA = (_Float16)(float)byte_of(mwd, 2 * (q & 1));
            const _Float16 mB = (_Float16)(float)byte_of(mwd, 2 * (q & 1) + 1);
            const v4h_ml bm = {mA, mA, mB, mB};
#pragma unroll
            for (int t = 0; t < RT; t++) {
                const v4h_ml am = *(const v4h_ml*)(S + L::H + (16 * t + jj) * 32 + 8 * q);
                const f32x4 yd = *(const f32x4*)(S + L::D + 4 * (16 * t + 4 * q));
                const float dm[4] = {-yd.x * xdm, -yd.y * xdm, -yd.z * xdm, -yd.w * xdm};
                if constexpr (FMT == kQ4_K) {
                    // four 4-deep products: block k is the reference's mins lane k
                    const v16f_mh z = {};
                    const v16f_mh ms = __builtin_amdgcn_mfma_f32_16x16x4f16(am, bm, z, 0, 0, 0);
#pragma unroll
                    for (int k = 0; k < 4; k++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            accm[k][4 * t + r] = __builtin_fmaf(dm[r], ms[4 * k + r], accm[k][4 * t + r]);
                } else {
                    const v4f_ml z = {};
                    const v4f_ml ms = __builtin_amdgcn_mfma_f32_16x16x16f16(am, bm, z, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; r++) accm[0][4 * t + r] = accm[0][4 * t + r] + dm[r] * ms[r];
                }
#pragma unroll
                for (int k = 0; k < (FMT == kQ4_K ? 4 : 1); k++)
#pragma unroll
                    for (int r = 0; r < 4; r++) asm volatile("" : "+v"(accm[k][4 * t + r]));
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        if (b + 1 < nb) park(st[(b + 1) & 1]);
        lds_barrier();
    }
#pragma unroll
    for (int r = 0; r < 4 * RT; r++) {
        v[r] = ((acc[0][r] + acc[4][r]) + (acc[2][r] + acc[6][r])) + ((acc[1][r] + acc[5][r]) + (acc[3][r] + acc[7][r]));
        if constexpr (FMT == kQ5_K) v[r] = v[r] + accm[0][r];  // the mins scalar
        else if constexpr (F::kMins) v[r] = v[r] + ((accm[0][r] + accm[2][r]) + (accm[1][r] + accm[3][r]));
    }
}

}  // namespace iq
