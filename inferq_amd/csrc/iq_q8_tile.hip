// iq_q8_tile.hip -- y = x . W^T for Q8_0 matrices at many input rows (prefill
// widths), in the reference's exact per-lane order (q80_tile,
// src/qgemm.rs:369-397): every output is bitwise the one-row result.
//
// The reference's lane k owns bytes 4k..4k+3 of every 32-value block and
// advances acc_k = fma(f16(dw) * f16(dx), dot4_k, acc_k) once per block; the
// eight lanes meet in hsum_f32_8.  v_mfma_f32_16x16x4_4b_f16 multiplies four
// independent 16 x 4 by 4 x 16 pairs, which is dot4_k of a 16 x 16 tile for
// four lanes k at once: two of them per block give all eight.  The int8
// values are exact in f16, a product is at most 2^14 and a dot at most 2^16,
// so the f32 results are the exact integers, already converted.
//
// What bounds it: the chains.  Each output takes eight FMAs and one scale
// product per 32 values, 9 VALU issues where a dot of 32 values is 1/16 of
// an int8 MFMA; on [512 x 4096] -> 2048 that is 31 us of VALU issue at
// 2.4 GHz, and the MFMAs another 15.
#include "iq_internal.h"
#include "iq_quant.h"

namespace iq {

namespace {

typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kQtCols = 64;  // weight rows per workgroup (16 per wave)
constexpr int kQtRows = 32;  // input rows per workgroup (16 per wave)
constexpr int kQtCB = 4;     // 32-value blocks per LDS stage

struct QtArgs {
    const uint8_t* w;  // [n][row_bytes], 4-byte aligned rows
    int64_t n, row_bytes;
    int nb;            // 32-value blocks per row, a multiple of kQtCB
    const int8_t* q;   // [m][nb * 32] quantised x, natural order
    const float* d;    // [m][nb] block scales
    int m;
    float* y;  // [m][ldy]
    int64_t ldy;
    // a second matrix of the same shape over the same rows (blockIdx.z 1)
    const uint8_t* w2 = nullptr;
    float* y2 = nullptr;
};

// One wave per (row, 256 values): Q8_0 (bit-exact from_float).  The bytes
// are stored + 128, the form bytes_to_f16 takes.
// SWIGLU: of SwiGLU(x, u) instead of x.
template <bool SWIGLU>
__global__ __launch_bounds__(256) void k_qt_quant(const float* __restrict__ x, const float* __restrict__ u, int64_t ldx,
                                                  int64_t m, int64_t k,
                                                  int8_t* __restrict__ q, float* __restrict__ d) {
    const int lane = threadIdx.x & 63;
    const int64_t wid = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    const int ng = (int)((k + 255) / 256);
    if (wid >= m * ng) return;  // uniform per wave
    const int64_t row = wid / ng;
    const int g = (int)(wid - row * ng);
    f32x4 v = q80_vals4_load(x + row * ldx, k, g);
    if constexpr (SWIGLU) {  // v is gate: (gate / (1 + exp(-gate))) * up, as the reference writes it
        const f32x4 up = q80_vals4_load(u + row * ldx, k, g);
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = __fdiv_rn(v[i], 1.f + exp_f32(-v[i])) * up[i];
    }
    const Q80Lane r = quant_q80_core(v);
    const int64_t b = (int64_t)g * 8 + (lane >> 3);
    if (b >= k / 32) return;
    ((uint32_t*)(q + row * k + (int64_t)g * 256))[lane] = r.packed ^ 0x80808080u;
    if ((lane & 7) == 0) d[row * (k / 32) + b] = f16_to_f32(r.dh);
}

// Four bytes u as f16 values u - 128: the bytes under the exponent of 1024, less 1152.
__device__ __forceinline__ u32x2 bytes_to_f16(uint32_t u) {
    const v2h off = {(_Float16)-1152.f, (_Float16)-1152.f};
    const v2h lo = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, u, 0x04010400u)) + off;
    const v2h hi = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, u, 0x04030402u)) + off;
    return u32x2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
}

// LDS stage of kQtCB blocks: A f16 [block][32 rows][64 bytes], B the same of
// the 64 weight rows, D the rows' block scales, W the weight rows'.  The 16
// bytes p of a row's 64 hold the dwords of reference lanes p and p + 4, what
// lane group p of a fragment multiplies.  Block planes are padded so that the
// four blocks one row's threads park go to different banks.
struct QtStage {
    static constexpr int AP = kQtRows * 64 + 16, BP = kQtCols * 64 + 16;
    static constexpr int A = 0;
    static constexpr int B = A + kQtCB * AP;
    static constexpr int D = B + kQtCB * BP;
    static constexpr int W = D + kQtCB * kQtRows * 4;
    static constexpr int END = W + kQtCB * kQtCols * 4;
};

// Grid (n / 64, m / 32): wave w has weight rows 16 (w % 4) .. +15 and input
// rows 16 (w / 4) .. +15.  One 16 x 16 tile per wave (32 chains) leaves four
// waves per SIMD, which VALU issue needs: on this chip a wave alone issues an
// f32 FMA every 5 cycles, two or four of them one every 2.7 together.  [512 x
// 4096] -> 2048 / [200 x 4096] -> 2048 / [333 x 2048] -> 4096: 60 / 37 / 44 us
// (the lane kernel: 243 / 124 / 148); 64 rows per workgroup 61 / 53 / 54; 16
// rows 77 / 44 / 53; two tiles per wave with the MFMAs issued one step ahead,
// two waves per SIMD, 61 / 54 / 56; a second stage of loads in flight the same;
// every thread staging a quarter block (narrower loads, three times as many)
// 68 / 45 / 52.  Four waves per SIMD leave 128 VGPRs, one too few: one is spilled
// (8 bytes of scratch a lane).
__global__ __launch_bounds__(512, 4) void k_qt_mm(QtArgs a) {
    constexpr int R = kQtRows, NT = 512;
    using L = QtStage;
    __shared__ __align__(16) uint8_t st[2][L::END];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int q = lane >> 4, jj = lane & 15;
    const int rbase = (wave >> 2) * 16, cbase = (wave & 3) * 16;
    const int64_t n0 = (int64_t)blockIdx.x * kQtCols;
    const int row0 = (int)blockIdx.y * R;
    const int rows = min(R, a.m - row0);

    // ---- staging, a block of a row per item: the first four waves take the
    // weight rows, the last ones the input rows, in registers of their own
    // (shared ones would make the waves wait for the loads where the
    // branches join)
    constexpr int kB = kQtCols * kQtCB, kA = R * kQtCB;
    static_assert(kB == 256 && kA == 128, "items of whole waves");
    const int tb = threadIdx.x, ta = NT - 1 - (int)threadIdx.x;
    const bool hasb = tb < kB, hasa = ta < kA;
    const int bc = tb & 3, ac = ta & 3, bcl = (tb >> 2) & (kQtCols - 1), arl = (ta >> 2) & (R - 1);
    const uint8_t* bsrc = (blockIdx.z ? a.w2 : a.w) + min(n0 + bcl, a.n - 1) * a.row_bytes + 34 * bc;
    // quants from the aligned dword at or before them: an even block's start
    // two bytes into it (the ninth dword's upper half is the next block's),
    // an odd block's at it
    const int bodd = bc & 1;
    const int64_t arow = row0 + min(arl, rows - 1);
    const int8_t* asrc = a.q + (arow * a.nb + ac) * 32;
    const float* dsrc = a.d + arow * a.nb + ac;

    u32x4 b0 = {}, b1 = {}, a0 = {}, a1 = {};
    uint32_t b2 = 0, bw = 0;  // the ninth dword, the scale
    float ad = 0.f;
    auto issue = [&](int s) {
        if (hasb) {
            const uint8_t* p = bsrc + (int64_t)s * (34 * kQtCB);
            const uint8_t* pq = p + 2 * bodd;
            b0 = *(const u32x4*)pq;
            b1 = *(const u32x4*)(pq + 16);
            b2 = ld32(pq + (bodd ? 28 : 32));
            bw = ld16(p);
        }
        if (hasa) {
            const int8_t* p = asrc + (int64_t)s * (32 * kQtCB);
            a0 = *(const u32x4*)p;
            a1 = *(const u32x4*)(p + 16);
            ad = dsrc[(int64_t)s * kQtCB];
        }
    };
    // 16 bytes p of a row's 64: dwords p and p + 4 as f16
    auto park_block = [&](uint8_t* dst, const uint32_t (&v)[8]) {
#pragma unroll
        for (int p = 0; p < 4; p++) {
            const u32x2 lo = bytes_to_f16(v[p]), hi = bytes_to_f16(v[p + 4]);
            *(u32x4a16*)(dst + 16 * p) = u32x4a16{lo.x, lo.y, hi.x, hi.y};
        }
    };
    auto park = [&](int P) {
        if (hasb) {
            const uint32_t w[9] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w, b2};
            const uint32_t sh = bodd ? 0u : 2u;
            uint32_t v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) v[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], sh) ^ 0x80808080u;
            park_block(st[P] + L::B + bc * L::BP + bcl * 64, v);
            *(float*)(st[P] + L::W + 4 * (bc * kQtCols + bcl)) = f16_to_f32(bw);
        }
        if (hasa) {
            const uint32_t v[8] = {a0.x, a0.y, a0.z, a0.w, a1.x, a1.y, a1.z, a1.w};
            park_block(st[P] + L::A + ac * L::AP + arl * 64, v);
            *(float*)(st[P] + L::D + 4 * (ac * R + arl)) = ad;
        }
    };

    // acc[k][r]: chain of reference lane k, output (row 4 q + r, column jj) of the wave's tile
    float acc[8][4];
#pragma unroll
    for (int k = 0; k < 8; k++)
#pragma unroll
        for (int r = 0; r < 4; r++) acc[k][r] = 0.f;

    const int ns = a.nb / kQtCB;
    issue(0);
    park(0);
    lds_barrier();
    for (int s = 0; s < ns; s++) {
        const uint8_t* S = st[s & 1];
        if (s + 1 < ns) issue(s + 1);
        // A (row jj) and B (column jj) of 16x16x4: lane group q holds the
        // four values of its block q.  A block's operands are read while the
        // one before it is multiplied.
        struct Frag {
            u32x4a16 a, b;
            f32x4 yd;
            float xd;
        };
        auto load = [&](int c) {
            return Frag{*(const u32x4a16*)(S + L::A + c * L::AP + (rbase + jj) * 64 + 16 * q),
                        *(const u32x4a16*)(S + L::B + c * L::BP + (cbase + jj) * 64 + 16 * q),
                        *(const f32x4*)(S + L::D + 4 * (c * R + rbase + 4 * q)),
                        *(const float*)(S + L::W + 4 * (c * kQtCols + cbase + jj))};
        };
        Frag f = load(0);
        if (rbase < rows)  // uniform per wave
#pragma unroll
        for (int c = 0; c < kQtCB; c++) {
            const v16f z = {};
            const v16f d0 = __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(v4h, u32x2{f.a.x, f.a.y}),
                                                                 __builtin_bit_cast(v4h, u32x2{f.b.x, f.b.y}), z, 0, 0, 0);
            const v16f d1 = __builtin_amdgcn_mfma_f32_16x16x4f16(__builtin_bit_cast(v4h, u32x2{f.a.z, f.a.w}),
                                                                 __builtin_bit_cast(v4h, u32x2{f.b.z, f.b.w}), z, 0, 0, 0);
            const float dd[4] = {f.xd * f.yd.x, f.xd * f.yd.y, f.xd * f.yd.z, f.xd * f.yd.w};
            if (c + 1 < kQtCB) f = load(c + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[k][r] = __builtin_fmaf(dd[r], d0[4 * k + r], acc[k][r]);
#pragma unroll
            for (int k = 0; k < 4; k++)
#pragma unroll
                for (int r = 0; r < 4; r++) acc[k + 4][r] = __builtin_fmaf(dd[r], d1[4 * k + r], acc[k + 4][r]);
            // the chains are advanced here, not sunk, which bounds the live MFMA results
#pragma unroll
            for (int k = 0; k < 8; k++)
#pragma unroll
                for (int r = 0; r < 4; r++) asm volatile("" : "+v"(acc[k][r]));
            __builtin_amdgcn_sched_barrier(0);
        }
        if (s + 1 < ns) park((s + 1) & 1);
        lds_barrier();
    }
    const int64_t n = n0 + cbase + jj;
    float* y = blockIdx.z ? a.y2 : a.y;
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const float v = ((acc[0][r] + acc[4][r]) + (acc[2][r] + acc[6][r])) + ((acc[1][r] + acc[5][r]) + (acc[3][r] + acc[7][r]));
        const int rr = rbase + 4 * q + r;
        if (rr < rows && n < a.n) y[(int64_t)(row0 + rr) * a.ldy + n] = v;
    }
}

// ---- 3..8 input rows --------------------------------------------------------
//
// v_mfma_f32_4x4x4_16b_f16 multiplies sixteen 4 x 4 by 4 x 4 pairs: here the
// pairs are the eight reference lanes k times two groups of four input rows,
// over four weight rows, so one instruction yields every lane's dot of a
// block for 8 x 4 outputs and each lane of the wave holds four of them (lane
// 8 k + 4 g + j: reference lane k, input rows 4 g .. 4 g + 3, weight row j).
// A wave advances only four chains a block and decodes a weight once, where
// the GEMV's waves keep eight rows' chains each.  What bounds it: one wave's
// walk along its rows (about 200 cycles a block), and past 16000 rows the
// VALU issue of the decode.  8 rows, GEMV before: [2048 x 4096] 17.2 -> 14.8
// us, [8192 x 2048] 19.0 -> 13.2, [16000 x 4096] 52 -> 32.

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kQfSB = 32;                   // blocks per staged step of a weight row (1088 bytes)
constexpr int kQfStride = 34 * kQfSB + 32;  // LDS row stride: four rows' dwords on distinct banks
constexpr int kQfMaxNb = 128;               // blocks of the widest row (4096)

struct QfArgs {
    const uint8_t* w;  // [n][row_bytes], 16-byte aligned
    int64_t n, row_bytes;
    int nb;            // a multiple of kQfSB
    const uint8_t* q;  // [nb / 2][64 lanes][16]: the lane's four values of two blocks as f16
    const float* d;    // [nb][8] block scales
    int m;
    float* y;
    int64_t ldy;
};

// One wave per (row of 8, 256 values); rows past m are zeros.
__global__ __launch_bounds__(256) void k_qf_quant(const float* __restrict__ x, int64_t ldx, int m, int64_t k,
                                                  uint8_t* __restrict__ q, float* __restrict__ d) {
    const int lane = threadIdx.x & 63;
    const int wid = (int)blockIdx.x * 4 + (int)(threadIdx.x >> 6), ng = (int)(k / 256);
    if (wid >= 8 * ng) return;  // uniform per wave
    const int row = wid / ng, g = wid - row * ng;
    Q80Lane r = {0u, 0};
    if (row < m) r = quant_q80_core(q80_vals4_load(x + row * ldx, k, g));
    const int b = 8 * g + (lane >> 3), kk = lane & 7;
    *(u32x2*)(q + ((int64_t)(b >> 1) * 64 + 8 * kk + row) * 16 + 8 * (b & 1)) = bytes_to_f16(r.packed ^ 0x80808080u);
    if (kk == 0) d[b * 8 + row] = f16_to_f32(r.dh);
}

// Grid n / 8: a workgroup of two waves, four weight rows each.
__global__ __launch_bounds__(128) void k_qf_mm(QfArgs a) {
    __shared__ __align__(16) uint8_t st[2][2][4 * kQfStride];  // [wave][step]
    __shared__ __align__(16) float s_d[kQfMaxNb * 8];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int j = lane & 3, g = (lane >> 2) & 1, k = lane >> 3;
    const int64_t n0 = ((int64_t)blockIdx.x * 2 + wave) * 4;
    // a step's 4 rows x 68 granules of 16 bytes, five loads a lane
    constexpr int kG = 34 * kQfSB / 16, kL = (4 * kG + 63) / 64;
    const uint8_t* src[kL];
    int dst[kL];
#pragma unroll
    for (int i = 0; i < kL; i++) {
        const int t = min(lane + 64 * i, 4 * kG - 1), r = t / kG, part = t - r * kG;
        src[i] = a.w + min(n0 + r, a.n - 1) * a.row_bytes + 16 * part;
        dst[i] = r * kQfStride + 16 * part;
    }
    u32x4 sb[kL];
    auto issue = [&](int s) {
#pragma unroll
        for (int i = 0; i < kL; i++) sb[i] = *(const u32x4*)(src[i] + (int64_t)s * (34 * kQfSB));
    };
    auto park = [&](int p) {
#pragma unroll
        for (int i = 0; i < kL; i++) *(u32x4a16*)(st[wave][p] + dst[i]) = u32x4a16{sb[i].x, sb[i].y, sb[i].z, sb[i].w};
    };
    const int ns = a.nb / kQfSB;
    issue(0);
    u32x4a16 av[2][4];  // the activations of four blocks pairs, two sets
    const uint8_t* aq = a.q + 16 * lane;
    auto fetch = [&](int pair, u32x4a16 (&o)[4]) {  // pairs past the end are never used: clamp
#pragma unroll
        for (int i = 0; i < 4; i++) o[i] = *(const u32x4a16*)(aq + (int64_t)min(pair + i, a.nb / 2 - 1) * 1024);
    };
    fetch(0, av[0]);
    for (int i = threadIdx.x; i < a.nb * 2; i += 128) ((f32x4*)s_d)[i] = ((const f32x4*)a.d)[i];
    park(0);
    __syncthreads();
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < ns; s++) {
        if (s + 1 < ns) issue(s + 1);
        const uint8_t* row = st[wave][s & 1] + j * kQfStride;
        const float* dp = s_d + (s * kQfSB) * 8 + 4 * g;
        // a real loop over halves of a step: unrolled whole, the operands of its 32 blocks were live at once
        // (362 registers a lane against 116, half the waves: [16000 x 2048] at 8 rows 28.5 -> 19.7 us)
#pragma unroll 1
        for (int h = 0; h < kQfSB; h += 16, row += 16 * 34, dp += 16 * 8) {
#pragma unroll
            for (int c = 0; c < 16; c++) {
                if (c % 8 == 0) {
                    __builtin_amdgcn_sched_barrier(0);
                    fetch((s * kQfSB + h + c) / 2 + 4, av[(c / 8 + 1) & 1]);
                }
                const uint32_t lo = *(const uint32_t*)(row + ((34 * c) & ~3) + 4 * k);
                const uint32_t hi = *(const uint32_t*)(row + ((34 * c) & ~3) + 4 * k + 4);
                // quants at 2 (mod 4) in an even block, aligned (the second dword) in an odd one
                const uint32_t v = (c & 1) ? hi : __builtin_amdgcn_alignbyte(hi, lo, 2);
                const float xd = f16_to_f32(*(const uint16_t*)(row + 34 * c));
                const u32x4a16 aw = av[(c / 8) & 1][(c & 7) >> 1];
                const v4h af = __builtin_bit_cast(v4h, (c & 1) ? u32x2{aw.z, aw.w} : u32x2{aw.x, aw.y});
                const v4h bf = __builtin_bit_cast(v4h, bytes_to_f16(v ^ 0x80808080u));
                const v4f z = {};
                const v4f dot = __builtin_amdgcn_mfma_f32_4x4x4f16(af, bf, z, 0, 0, 0);
                const f32x4 yd = *(const f32x4*)(dp + 8 * c);
#pragma unroll
                for (int r = 0; r < 4; r++) acc[r] = __builtin_fmaf(xd * yd[r], dot[r], acc[r]);
            }
        }
        if (s + 1 < ns) park((s + 1) & 1);
        // the step's region is this wave's own
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    // hsum_f32_8 over lanes k (bits 3..5 of the lane)
#pragma unroll
    for (int r = 0; r < 4; r++) {
        float v = acc[r];
        v = v + __shfl_xor(v, 32);
        v = v + __shfl_xor(v, 16);
        v = v + __shfl_xor(v, 8);
        const int rr = 4 * g + r;
        if (k == 0 && rr < a.m && n0 + j < a.n) a.y[(int64_t)rr * a.ldy + n0 + j] = v;
    }
}

constexpr size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace

// From 9 rows, where no GEMV takes the call or the GEMV would be slower: a
// GEMV's time grows with the weight bytes it decodes again for every 8 rows
// (about 0.55 us a MB), the tile's with the blocks of a row while its
// workgroups are few (0.27 us a block: the chain of one 16 x 16 tile).
// Measured, tile / GEMV: [8192 x 2048] at 9 / 16 rows 21.6 / 20.8 and 21.6 /
// 27.1 us, [12288 x 2048] at 9 rows 22 / 32, [4096 x 4096] at 16 rows 37 / 28,
// [8192 x 4096] at 16 rows 40 / 43, [512 x 2048] at 63 rows 20 / 12, [2048 x
// 1024] at 32 / 63 rows 13.2 / 11.3 and 13 / 16, [4096 x 1024] at 16 / 20 rows
// 12.0 / 11.3 and 13.2 / 17.0 (the GEMV's workgroups fill its last round).
bool q8_tile_supported(const WeightView& w, int64_t m) {
    if (w.dtype != kQ8_0 || m < 9 || m > (int64_t)1 << 20 || w.rows < 1 || w.cols % (32 * kQtCB) != 0 ||
        ((uintptr_t)w.w & 3) != 0)
        return false;
    return !gemv_supported(w, m) || (double)(w.rows * w.row_bytes) * (double)m / 8 > 1e6 * (0.4 * (double)(w.cols / 32) - 3.8);
}

namespace {

QtArgs qt_args(const WeightView& w, int64_t m, void* ws) {
    QtArgs a;
    a.w = w.w;
    a.n = w.rows;
    a.row_bytes = w.row_bytes;
    a.nb = (int)(w.cols / 32);
    a.q = (const int8_t*)ws;
    a.d = (const float*)((uint8_t*)ws + align256((size_t)(m * w.cols)));
    a.m = (int)m;
    a.ldy = w.rows;
    return a;
}

template <bool SWIGLU>
hipError_t qt_quant(const QtArgs& a, const float* x, const float* u, int64_t ldx, hipStream_t s) {
    const int64_t k = (int64_t)a.nb * 32, waves = a.m * ((k + 255) / 256);
    hipLaunchKernelGGL((k_qt_quant<SWIGLU>), dim3((unsigned)((waves + 3) / 4)), dim3(256), 0, s, x, u, ldx, (int64_t)a.m, k,
                       (int8_t*)a.q, (float*)a.d);
    return hipGetLastError();
}

hipError_t qt_mm(const QtArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(k_qt_mm, dim3((unsigned)((a.n + kQtCols - 1) / kQtCols), (unsigned)((a.m + kQtRows - 1) / kQtRows),
                                     a.w2 ? 2u : 1u), dim3(512), 0, s, a);
    return hipGetLastError();
}

}  // namespace

hipError_t launch_q8_tile(const WeightView& w, const float* x, int64_t ldx, int64_t m, float* y, int64_t ldy, void* ws,
                          hipStream_t s) {
    if (!q8_tile_supported(w, m)) return hipErrorNotSupported;
    QtArgs a = qt_args(w, m, ws);
    a.y = y;
    a.ldy = ldy;
    if (hipError_t e = qt_quant<false>(a, x, nullptr, ldx, s)) return e;
    return qt_mm(a, s);
}

// Gate and up in one launch: apart, a [512 x 2048] matrix at 512 tokens is 128
// workgroups, half the CUs, and takes as long as both together (19.6 us
// each); x is quantised once, and SwiGLU runs inside the down product's
// quantisation.  Four launches instead of seven: 1100 tokens 693 -> 616 us.
hipError_t launch_q8_swiglu(const WeightView& gate, const WeightView& up, const WeightView& down, const float* x,
                            int64_t m, float* g, float* u, float* out, void* ws, hipStream_t s) {
    if (!q8_tile_supported(gate, m) || !q8_tile_supported(up, m) || !q8_tile_supported(down, m) ||
        gate.rows != up.rows || gate.cols != up.cols || down.cols != gate.rows)
        return hipErrorNotSupported;
    QtArgs a = qt_args(gate, m, ws);
    a.y = g;
    a.w2 = up.w;
    a.y2 = u;
    if (hipError_t e = qt_quant<false>(a, x, nullptr, gate.cols, s)) return e;
    if (hipError_t e = qt_mm(a, s)) return e;
    QtArgs d = qt_args(down, m, ws);
    d.y = out;
    if (hipError_t e = qt_quant<true>(d, g, u, gate.rows, s)) return e;
    return qt_mm(d, s);
}

namespace {

// What k_qf_* can take at any number of rows up to 8.
bool qf_shape(const WeightView& w) {
    return w.dtype == kQ8_0 && w.rows >= 1 && w.rows <= (int64_t)1 << 31 && w.cols >= 1 && w.cols % (32 * kQfSB) == 0 &&
           w.cols / 32 <= kQfMaxNb && ((uintptr_t)w.w & 15) == 0;
}

}  // namespace

// The tile's time hardly depends on the rows; the GEMV's grows with them and
// with the matrix, so the line is a least amount of work that falls with the
// row's length (a chain's walk: 0.09 us a block).  Measured, tile / GEMV in
// us: [2048 x 4096] at 6 / 7 rows 14.9 / 14.5 and 14.8 / 17.2, [4096 x 4096]
// at 3 / 4 rows 17.0 / 15.0 and 17.1 / 18.1, [4096 x 2048] at 4 / 5 rows 11.3
// / 11.0 and 11.4 / 14.5, [2048 x 1024] at 8 rows 7.6 / 7.5, [8192 x 1024] at
// 5 rows 9.4 / 11.5.  From 16384 rows the GEMV's waves fill the chip and it
// reads the matrix at a better rate: [16000 x 2048] at 3 rows 18.1 / 23.3,
// [16384 x 2048] at 3 / 4 / 5 rows 18.4 / 14.8, 18.7 / 17.7 and 18.8 / 21.7
// ([16384 x 1024] at 3 / 4 rows 11.8 / 12.0 and 12.1 / 13.5), [24576 x 2048] at
// 4 / 5 / 6 rows 24.4 / 20.9, 24.6 / 25.2 and 24.8 / 27.2, [32000 x 2048] at 4
// / 6 rows 30.9 / 29.1 and 29.1 / 34.0, [248320 x 2048] at 6 / 8 rows 177 / 163
// and 177 / 199.
// Rows of 6144: 20.4 / 17.9 at 8 rows, so not taken.
bool q8_few_supported(const WeightView& w, int64_t m) {
    if (m < 3 || m > 8 || !qf_shape(w)) return false;
    const int64_t least = w.rows < 16384 ? 3 : w.rows < 24576 ? (w.cols <= 1024 ? 4 : 5) : w.rows <= 65536 ? 6 : 8;
    return m >= least && w.rows * m * (w.cols / 32 + 64) >= 2500000;
}

size_t q8_few_workspace(const WeightView& w, int64_t m) {
    return m >= 3 && qf_shape(w) ? (size_t)w.cols * 17 : 0;
}

hipError_t launch_q8_few(const WeightView& w, const float* x, int64_t ldx, int64_t m, float* y, int64_t ldy, void* ws,
                         hipStream_t s) {
    if (!q8_few_supported(w, m)) return hipErrorNotSupported;
    QfArgs a;
    a.w = w.w;
    a.n = w.rows;
    a.row_bytes = w.row_bytes;
    a.nb = (int)(w.cols / 32);
    a.q = (const uint8_t*)ws;
    a.d = (const float*)((uint8_t*)ws + w.cols * 16);
    a.m = (int)m;
    a.y = y;
    a.ldy = ldy;
    hipLaunchKernelGGL(k_qf_quant, dim3((unsigned)(w.cols / 128)), dim3(256), 0, s, x, ldx, (int)m, w.cols, (uint8_t*)a.q,
                       (float*)a.d);
    if (hipError_t e = hipGetLastError()) return e;
    hipLaunchKernelGGL(k_qf_mm, dim3((unsigned)((a.n + 7) / 8)), dim3(128), 0, s, a);
    return hipGetLastError();
}

}  // namespace iq
