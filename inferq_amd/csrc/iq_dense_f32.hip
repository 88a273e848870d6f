// iq_dense_f32.hip -- y = x . W^T for F32 and BF16 matrices, the MoE router
// among them.  The reference's QuantizedMatrix accepts both (src/gguf.rs:
// 305-317) and multiplies them through candle's f32 matmul, having no
// multi-row kernel for them (src/gguf.rs:533-535, :599); such matrices are
// small (routers, gate vectors), and the product is a plain f32 dot per
// output.
//
// Order: for each (input row, weight row) lane l sums x[k] * w[k] (the
// product rounded, then the add) over k = l + 64 j for j = 0, 1, ... in
// turn, then the 64 lanes meet in a butterfly (xor 32, 16, ..., 1).  BF16
// weights widen to f32 exactly first.  Every pair is formed the same way at
// any row count.
#include <type_traits>

#include "iq_device.h"
#include "iq_internal.h"

namespace iq {

namespace {

template <bool BF16>
__device__ __forceinline__ float float_w(const uint8_t* w, int64_t i) {
    if constexpr (BF16) return __builtin_bit_cast(float, (uint32_t)((const uint16_t*)w)[i] << 16);
    else return ((const float*)w)[i];
}

// Few pairs, or few input rows: one wave per weight row and TT input rows,
// grid (n, ceil(m / TT)).  Latency bound: a 2048-wide row's 32 loads of each
// operand are in flight at once (one round trip), what is left of a row goes
// in passes of 16 and 8 steps and one cut short at its end.  A wave that took
// eight input rows in turn, eight values at a time, made 4 x 8 dependent round
// trips: router [256 x 2048] at 8 rows 18.5 -> 3.5 us, BF16 [64 x 2048] at 8
// rows 14.4 -> 2.6 us; single steps at the end of a row: [2048 x 1024] at 4
// rows 6.6 against 4.8 us.
template <bool BF16, int TT, int UM>
__global__ __launch_bounds__(64) void k_float_pair(const uint8_t* __restrict__ w, int64_t k,
                                                   const float* __restrict__ x, int64_t ldx, int m,
                                                   float* __restrict__ y, int64_t ldy) {
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int t0 = (int)blockIdx.y * TT, nt = min(TT, m - t0);
    const uint8_t* wr = w + row * k * (BF16 ? 2 : 4);
    const float* xr = x + (int64_t)t0 * ldx;
    float part[TT];
#pragma unroll
    for (int i = 0; i < TT; i++) part[i] = 0.f;
    // U steps of the chain from value h on; CUT: the row's last ones, those
    // past its end on its last value and left out
    int64_t h = 0;
    auto pass = [&](auto U_, auto CUT_) {
        constexpr int U = U_;
        constexpr bool CUT = CUT_;
        const int left = CUT ? (int)(k - h) : 0;
        auto at = [&](int j) { return CUT ? min(lane + 64 * j, left - 1) : lane + 64 * j; };
        const uint8_t* wh = wr + h * (BF16 ? 2 : 4);
        float rv[U], xv[U];
#pragma unroll
        for (int j = 0; j < U; j++) rv[j] = float_w<BF16>(wh, at(j));
#pragma unroll
        for (int i = 0; i < TT; i++) {
            if (TT > 1 && i >= nt) break;  // uniform
            const float* xh = xr + i * ldx + h;
#pragma unroll
            for (int j = 0; j < U; j++) xv[j] = xh[at(j)];
#pragma unroll
            for (int j = 0; j < U; j++) {
                const float v = part[i] + xv[j] * rv[j];
                part[i] = !CUT || lane + 64 * j < left ? v : part[i];
            }
        }
        h += 64 * U;
    };
    using std::integral_constant;
    while (k - h >= 64 * UM) pass(integral_constant<int, UM>{}, std::false_type{});
    if (__builtin_expect(k > h, 0)) {  // out of the way of rows that have none: code to fetch is latency here
        if (UM > 16 && k - h >= 64 * 16) pass(integral_constant<int, 16>{}, std::false_type{});
        if (UM > 8 && k - h >= 64 * 8) pass(integral_constant<int, 8>{}, std::false_type{});
        if (k - h > 64 * 4) pass(integral_constant<int, 8>{}, std::true_type{});
        else if (k - h > 64) pass(integral_constant<int, 4>{}, std::true_type{});
        else if (k - h > 0) pass(integral_constant<int, 1>{}, std::true_type{});
    }
#pragma unroll
    for (int i = 0; i < TT; i++) {
        float v = part[i];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) v = v + __shfl_xor(v, off);
        if (lane == 0 && (TT == 1 || i < nt)) y[(t0 + i) * ldy + row] = v;
    }
}

// Butterfly step of N values per lane at distance OFF, halving them: the
// lanes whose OFF bit is clear end with the sums of values 0 .. N/2 - 1, the
// others with those of N/2 .. N - 1.  Each sum is the butterfly's own (own
// value plus the partner's), formed once instead of in both lanes.
template <int OFF, int N>
__device__ __forceinline__ void float_halve(float (&v)[N], float (&o)[N / 2]) {
    const bool up = threadIdx.x & OFF;
#pragma unroll
    for (int i = 0; i < N / 2; i++) {
        if constexpr (OFF == 32 || OFF == 16) {
            const uint32_t a = __builtin_bit_cast(uint32_t, v[i]), b = __builtin_bit_cast(uint32_t, v[i + N / 2]);
            const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(a, b, false, false)
                                     : __builtin_amdgcn_permlane16_swap(a, b, false, false);
            o[i] = __builtin_bit_cast(float, (uint32_t)r[0]) + __builtin_bit_cast(float, (uint32_t)r[1]);
        } else {
            const float keep = up ? v[i + N / 2] : v[i], send = up ? v[i] : v[i + N / 2];
            o[i] = keep + __shfl_xor(send, OFF);
        }
    }
}

// Many pairs: a workgroup of four waves takes 2 ET weight rows x 2 TT input
// rows, a wave ET x TT of them, all in registers; the rows pass through LDS
// 256 values at a time (a lane's four values side by side, so that one
// 16-byte read gives four steps of its chain), the next 256 in flight.
// VALU-bound: a product and an add per value and pair (no FMA, the order
// rounds both), 8.5 us of issue for a [256 x 2048] router at 512 rows.
// Values past the end of a row are read as zeros, whose products leave a
// partial sum as it is (it is never -0).
template <bool BF16, int ET, int TT, int J>
__global__ __launch_bounds__(256) void k_float_tile(const uint8_t* __restrict__ w, int64_t n, int64_t k,
                                                    const float* __restrict__ x, int64_t ldx, int m,
                                                    float* __restrict__ y, int64_t ldy) {
    constexpr int NR = 2 * (ET + TT), PW = ET / 2, PX = TT / 2;  // staged rows; of each kind per wave
    static_assert(ET % 2 == 0 && TT % 2 == 0, "rows per wave");
    __shared__ __align__(16) float st[2][J / 4][NR][256];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t r0 = (int64_t)blockIdx.x * 2 * ET;
    const int t0 = (int)blockIdx.y * 2 * TT;
    // staged rows: the weight rows, then the input rows; this wave's are uniform
    int64_t wsrc[PW], xsrc[PX];
#pragma unroll
    for (int i = 0; i < PW; i++) wsrc[i] = min(r0 + wave * PW + i, n - 1) * k;
#pragma unroll
    for (int i = 0; i < PX; i++) xsrc[i] = (int64_t)min(t0 + wave * PX + i, m - 1) * ldx;
    float g[PW + PX][J];
    auto issue = [&](int64_t h0) {
        if (h0 + 64 * J <= k) {
#pragma unroll
            for (int j = 0; j < J; j++) {
#pragma unroll
                for (int i = 0; i < PW; i++) g[i][j] = float_w<BF16>(w, wsrc[i] + h0 + (lane + 64 * j));
#pragma unroll
                for (int i = 0; i < PX; i++) g[PW + i][j] = x[xsrc[i] + h0 + (lane + 64 * j)];
            }
        } else {
#pragma unroll
            for (int j = 0; j < J; j++) {
                const int64_t h = h0 + lane + 64 * j, hc = min(h, k - 1);
#pragma unroll
                for (int i = 0; i < PW; i++) {
                    const float v = float_w<BF16>(w, wsrc[i] + hc);
                    g[i][j] = h < k ? v : 0.f;
                }
#pragma unroll
                for (int i = 0; i < PX; i++) {
                    const float v = x[xsrc[i] + hc];
                    g[PW + i][j] = h < k ? v : 0.f;
                }
            }
        }
    };
    auto park = [&](int p) {
#pragma unroll
        for (int c = 0; c < J / 4; c++)
#pragma unroll
            for (int i = 0; i < PW + PX; i++)
                *(f32x4*)&st[p][c][i < PW ? wave * PW + i : 2 * ET + wave * PX + i - PW][4 * lane] =
                    f32x4{g[i][4 * c], g[i][4 * c + 1], g[i][4 * c + 2], g[i][4 * c + 3]};
    };
    const int er = (wave & 1) * ET, tr = 2 * ET + (wave >> 1) * TT;
    float part[ET * TT];
#pragma unroll
    for (int i = 0; i < ET * TT; i++) part[i] = 0.f;
    issue(0);
    park(0);
    lds_barrier();
    int p = 0;
    for (int64_t h0 = 0; h0 < k; h0 += 64 * J, p ^= 1) {
        if (h0 + 64 * J < k) issue(h0 + 64 * J);
#pragma unroll
        for (int c = 0; c < J / 4; c++) {
            f32x4 wv[ET];
#pragma unroll
            for (int e = 0; e < ET; e++) wv[e] = *(const f32x4*)&st[p][c][er + e][4 * lane];
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const f32x4 xv = *(const f32x4*)&st[p][c][tr + t][4 * lane];
#pragma unroll
                for (int j = 0; j < 4; j++)
#pragma unroll
                    for (int e = 0; e < ET; e++) part[e * TT + t] = part[e * TT + t] + xv[j] * wv[e][j];
            }
        }
        if (h0 + 64 * J < k) park(p ^ 1);
        lds_barrier();
    }
    // pair i of the lane: bits 5, 4, ... of the lane pick the halves
    const int64_t row0 = r0 + er;
    const int tok0 = t0 + tr - 2 * ET;
    float a[ET * TT / 2], b[ET * TT / 4], c[ET * TT / 8], d[ET * TT / 16];
    float_halve<32>(part, a);
    float_halve<16>(a, b);
    float_halve<8>(b, c);
    float_halve<4>(c, d);
    int i = ((lane >> 5) & 1) * (ET * TT / 2) + ((lane >> 4) & 1) * (ET * TT / 4) + ((lane >> 3) & 1) * (ET * TT / 8) +
            ((lane >> 2) & 1) * (ET * TT / 16);
    float v;
    static_assert(ET * TT == 16 || ET * TT == 32, "pairs per wave");
    if constexpr (ET * TT == 32) {
        float f[1];
        float_halve<2>(d, f);
        v = f[0];
        i += (lane >> 1) & 1;
    } else {
        v = d[0] + __shfl_xor(d[0], 2);
    }
    v = v + __shfl_xor(v, 1);
    const int64_t row = row0 + i / TT;
    const int tok = tok0 + i % TT;
    if ((lane & (ET * TT == 32 ? 1 : 3)) == 0 && row < n && tok < m) y[(int64_t)tok * ldy + row] = v;
}

template <bool BF16, int ET, int TT, int J>
hipError_t launch_tile(const WeightView& w, const float* x, int64_t ldx, int64_t m, float* y, int64_t ldy, hipStream_t s) {
    const dim3 grid((unsigned)((w.rows + 2 * ET - 1) / (2 * ET)), (unsigned)((m + 2 * TT - 1) / (2 * TT)));
    hipLaunchKernelGGL((k_float_tile<BF16, ET, TT, J>), grid, dim3(256), 0, s, w.w, w.rows, w.cols, x, ldx, (int)m, y, ldy);
    return hipGetLastError();
}

template <bool BF16, int TT, int UM>
hipError_t launch_pair(const WeightView& w, const float* x, int64_t ldx, int64_t m, float* y, int64_t ldy, hipStream_t s) {
    const dim3 grid((unsigned)w.rows, (unsigned)((m + TT - 1) / TT));
    hipLaunchKernelGGL((k_float_pair<BF16, TT, UM>), grid, dim3(64), 0, s, w.w, w.cols, x, ldx, (int)m, y, ldy);
    return hipGetLastError();
}

// Up to 8192 pairs one wave each ([256 x 2048] at 32 / 64 rows: pairs 6.5 /
// 10.3 us, tiles 7.0 / 7.4).  Tall matrices at one to three rows stream, a
// wave per weight row for all of them, 16 steps at a time where that leaves
// more waves in flight: a tile multiplies eight input rows whatever the call
// has.  us, streamed / tile: BF16 [32000 x 2048] at 1 / 2 / 3 rows 20.4 / 38.6,
// 25.4 / 38.6, 33.3 / 38.7 (4 rows: 40.9 / 38.7), F32 [8200 x 2048] 12.0 / 18.4,
// 12.9 / 18.8, 13.9 / 19.4; two rows against a wave each [2048 x 2048] 4.8 /
// 4.8, [4096 x 2048] 6.0 / 6.5.  Three rows past 256 MiB, out of the Infinity
// Cache's reach, and of 512 columns take the tile: BF16 [64000 x 4096] 182 /
// 152, [32000 x 512] 14.1 / 13.0.  Tiles of 4 x 4 pairs a wave with 512 values a
// stage while they leave at most two workgroups per CU, whose barriers and
// round trips then cost more than the LDS they take ([64 x 2048] at 512 rows
// 9.4 against 10.3 us with 256; [256 x 2048] at 256 rows 14.6 against 12.4);
// 8 x 4 from four workgroups per CU ([500 x 3001] at 700 rows 84 -> 66 us, [256
// x 2048] at 512 rows the same).
template <bool BF16>
hipError_t launch_bf(const WeightView& w, const float* x, int64_t ldx, int64_t m, float* y, int64_t ldy, hipStream_t s) {
    const int64_t tiles = ((w.rows + 7) / 8) * ((m + 7) / 8), wide = ((w.rows + 15) / 16) * ((m + 7) / 8);
    const bool few = m <= 3 && w.rows < (int64_t)1 << 26;  // a launch has at most 2^32 threads
    if (few && m == 2 && w.rows > 2048) return launch_pair<BF16, 2, 16>(w, x, ldx, m, y, ldy, s);
    if ((few && m == 1) || w.rows * m <= 8192) return launch_pair<BF16, 1, 32>(w, x, ldx, m, y, ldy, s);
    if (few && m == 3 && w.cols >= 1024 && w.rows * w.row_bytes <= (int64_t)256 << 20)
        return launch_pair<BF16, 3, 16>(w, x, ldx, m, y, ldy, s);
    if (tiles <= 512) return launch_tile<BF16, 4, 4, 8>(w, x, ldx, m, y, ldy, s);
    if (wide < 1024) return launch_tile<BF16, 4, 4, 4>(w, x, ldx, m, y, ldy, s);
    return launch_tile<BF16, 8, 4, 4>(w, x, ldx, m, y, ldy, s);
}

}  // namespace

hipError_t launch_float_mm(const WeightView& w, const float* x, int64_t ldx, int64_t m, float* y, int64_t ldy,
                           hipStream_t s) {
    if ((w.dtype != kF32 && w.dtype != kBF16) || m < 1 || w.rows < 1 || w.cols < 1) return hipErrorNotSupported;
    if ((w.rows + 3) / 4 > 0x7fffffff || (m + 7) / 8 > 65535) return hipErrorNotSupported;
    return w.dtype == kBF16 ? launch_bf<true>(w, x, ldx, m, y, ldy, s) : launch_bf<false>(w, x, ldx, m, y, ldy, s);
}

}  // namespace iq
