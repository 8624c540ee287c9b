// qgemm_grp.h -- group-wise MFMA GEMM (gfx950): any code width, type of x and
// K % 64 == 0, with the GEMVs' semantics (the format's exact weights).
//
// y[m, n] = sum over groups g of  s (x . (q - C)) + (b + C s) sum_x,  s, b and
// the sums per (n, g), C = 2^(BITS - 1): the format's definition regrouped as
// the f32 GEMVs do it, with the inner products on the 16-bit matrix cores and
// nothing rounded to 16 bits on the way:
//  * a centred code (at most 8 bits) is a bf16 and an f16 number exactly;
//  * 16-bit x goes in as it is; f32 x is the sum of three bf16 numbers
//    exactly: its leading 8 significant bits, the next 8 and the last 8, each
//    by truncation (so the first never rounds up to infinity).  Below 2^-109
//    the third underflows: a tile with a row of x that has nothing from 2^-100
//    on is run once more, with such rows times 2^24;
//  * a product of the two has at most 19 bits and is exact in the f32
//    accumulator, which is started afresh for every group and then scaled
//    into the f32 sums of y.
// An f32 FMA chain would round once per k; this rounds the partial sums of
// each group, and centring keeps them small (with q itself a random row's
// sums are twice as large and their roundings with them).  (f32 MFMAs,
// v_mfma_f32_32x32x2_f32, run at 1/16 of the bf16 rate per k, 3/16 of three
// bf16 products, and round once per k.)
//
// Block: 8 waves (two per SIMD: one wave alone issues VALU at half rate), 32
// MT rows of x by 128 columns.  Wave (kg, nw) takes columns 64 nw .. +64 (two
// tiles of 32) of all the rows, and the 32 codes of K numbered kg of every
// 128: x is split once per block and shared, a code is converted once per
// block, and the four K parts meet in LDS at the end.  (Waves of 32 columns
// and 64 codes read every x fragment for half as many products: LDS bound.)
// Groups of 64 and 128 are scaled 32 codes at a time like groups of 32.
//
// Each step of 128 k: the matrix products of this step; between them the
// next step's x is split into the three planes of the other LDS stage, with
// its sums over 32 k, and the next codes are copied there; then the x and
// codes of the step after that are loaded into the registers these leave; one
// barrier.  (Two or three steps of loads in flight measured the same.)
// Scales come in windows of 32 bytes per column, 2 to 16 steps.  (Lanes that
// loaded their own columns' codes and scales straight into registers touched
// 1000 cache lines a step and took 1.5 times as long.)
//
// LDS: two stages of x, each one or (f32) three planes of 32 MT rows x 128 k
// in 16 bits (256 bytes a row; 16-byte chunk ch of row r at position ch ^ (r & 15): the
// fragment reads, 32 rows at one chunk, hit all banks evenly) and the sums of
// x, [32 k][row]; two stages of codes, 16 BITS bytes a column; two scale
// windows.  Column rows are padded so that 32 columns spread over the banks.
//
// K is split over `parts` blocks per tile where the tiles alone would leave
// CUs idle; the parts' tiles meet in the workspace (qsplit.h, K parts), where
// the last to arrive adds all of them in part order, four at a time as two
// pairs.
#pragma once
#include <type_traits>

#include "kernels.h"
#include "qcommon.h"
#include "qsplit.h"

namespace lxq {
namespace grp {

// the kernel's lambdas hold register arrays: one left as a call would put them
// in memory
#define LXQ_INLINE __attribute__((always_inline))

typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f4g __attribute__((ext_vector_type(4), aligned(4)));  // x and y may be dword-aligned only
typedef uint32_t u2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4g __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u4h __attribute__((ext_vector_type(4), aligned(2)));  // scale rows of odd length

constexpr int BN = 128, BK = 128, kThreads = 512;
constexpr int kRowBytes = BK * 2;  // one plane's row of a step

template <int MT, int BITS, int P>
struct Lds {
    static constexpr int BM = 32 * MT;
    static constexpr int kPlane = BM * kRowBytes;
    static constexpr int kSums = P * kPlane;               // [4][BM] f32
    static constexpr int kStage = kSums + 4 * BM * 4;
    static constexpr int kCodeRow = 16 * BITS + 16;
    static constexpr int kCodes = 2 * kStage;              // 2 x [128 columns]
    static constexpr int kScaleRow = 36;                   // 32 bytes and a bank
    static constexpr int kWindow = 2 * BN * kScaleRow;     // scales, then biases
    static constexpr int kScales = kCodes + 2 * BN * kCodeRow;
    static constexpr int kOut = BN + 4;                    // floats per row of the output tile
    static constexpr int kTile = BM * kOut * 4;            // two of them at the end (pairs of K parts)
    static constexpr int kRows = 2 * kTile;                // past the tiles: a value per row
    static constexpr int kEnd = kRows + 4 * BM;
    static constexpr int kLoop = kScales + 2 * kWindow;
    static constexpr int kFlag = kLoop > kEnd ? kLoop : kEnd;  // past all of that: a word
    static constexpr int kBytes = kFlag + 16;
    static_assert(kBytes <= 160 * 1024, "LDS");
};

// f32 x runs on the bf16 units, like bf16
template <int TX>
__device__ __forceinline__ f32x16 mfma(const u4& a, const u4& b, const f32x16& c) {
    if constexpr (TX == DT_F16)
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0,
                                                     0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                      0, 0, 0);
}

// the top bit of every code that ends in word i of a run of 16 codes: codes
// with it flipped are q - C in two's complement
template <int BITS>
constexpr uint32_t top_bits(int i) {
    uint32_t m = 0;
    for (int k = 0; k < 16; k++) {
        const int bit = k * BITS + BITS - 1;
        if (bit / 32 == i) m |= 1u << (bit % 32);
    }
    return m;
}

// codes 8 j .. 8 j + 7 of the words w (top bits flipped; j a compile-time
// constant after unrolling) as four packed pairs of the matrix type (both hold
// every q - C exactly)
template <int BITS, int TX>
__device__ __forceinline__ u4 codes8(const uint32_t* w, int j) {
    float q[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const int bit = (8 * j + i) * BITS, wi = bit >> 5, sh = bit & 31;
        const bool straddle = sh + BITS > 32;
        const uint32_t v = straddle ? __builtin_amdgcn_alignbit(w[straddle ? wi + 1 : wi], w[wi], sh) : w[wi];
        q[i] = (float)(int)__builtin_amdgcn_sbfe((int)v, straddle ? 0 : sh, BITS);
    }
    u4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) {
        if constexpr (TX == DT_F16)
            r[i] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(q[2 * i], q[2 * i + 1]));
        else
            r[i] = __builtin_amdgcn_perm(__float_as_uint(q[2 * i + 1]), __float_as_uint(q[2 * i]), 0x07060302u);
    }
    return r;
}

// a thread's 16-byte vectors of the output tile: 4 columns of rows tid / 32 + 16 i
template <int MT>
constexpr int kOutVecs = 32 * MT * BN / 4 / kThreads;
// rows of f32 x whose third terms have underflowed, and what such x is taken times
constexpr float kSmall = 0x1p-100f, kSmallUp = 0x1p24f, kSmallDown = 0x1p-24f;

// One run over steps s0 .. s1 - 1 of the tile at (m0, n0): its sums in o.
// BITS: code width; TX: type of x; SBF: f32 scales (else 16-bit ones, sb_dt
// says which); MT: 32-row tiles.  f32 x: true where a row has nothing from
// kSmall on; run 1 then takes such rows times kSmallUp (bit i of small: the
// thread's load i of x is of one, of rows: its vector i of the output).
template <int BITS, int TX, bool SBF, int MT>
__device__ __forceinline__ bool run_tile(uint8_t* lds, const void* __restrict__ x, const uint32_t* __restrict__ wq,
                                         const void* __restrict__ scales, const void* __restrict__ biases, int M, int K,
                                         int N, int gshift, int sb_dt, int m0, int n0, int s0, int s1, int run,
                                         uint32_t& small, uint32_t& rows, f4 (&o)[kOutVecs<MT>]) {
    constexpr int P = TX == DT_F32 ? 3 : 1;       // planes of x
    using L = Lds<MT, BITS, P>;
    constexpr int BM = L::BM, NT = 2;
    constexpr int XE = TX == DT_F32 ? 4 : 8;      // k per 16-byte load of x
    constexpr int WL = (BITS + 1) / 2;            // code words per lane, tile and step: 16 codes
    constexpr int XL = BM * BK / XE / kThreads;   // 16-byte loads of x per thread and step
    constexpr int CL = (BITS + 3) / 4;            // 16-byte loads of codes per thread and step
    constexpr int XC = BK / XE;                   // loads per row of x
    constexpr int XR = kThreads / XC;             // rows per pass of x loads
    constexpr int kSb = SBF ? 4 : 2;
    constexpr float C = (float)(1 << (BITS - 1));
    int tid = threadIdx.x;
    // Each run works its addresses out anew: kept over both they cost 80
    // registers, and worked out ahead of the loop around the runs they stood in
    // front of the first load (M = 64, K = N = 4096, 4-bit: 20.5 us, so 19.7).
    if constexpr (TX == DT_F32)
        asm volatile("" : "+v"(tid), "+s"(M), "+s"(K), "+s"(N), "+s"(gshift), "+s"(m0), "+s"(n0), "+s"(s0), "+s"(s1));
    tid &= kThreads - 1;  // (what the compiler knew of it)
    const bool again = __builtin_amdgcn_readfirstlane(run) != 0;  // (scalar branches)
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave >> 1, nw = wave & 1;
    const int c = lane & 31, h = lane >> 5;
    const int steps = (K + BK - 1) / BK;

    // x: thread t loads 16 bytes (chunk t % XC) of rows t / XC, + XR, ...; rows
    // past M re-read the last (never stored), k past K are zeros
    const int xc = tid % XC, xr = tid / XC;
    const uint8_t* xp[XL];
#pragma unroll
    for (int i = 0; i < XL; i++)
        xp[i] = static_cast<const uint8_t*>(x) + (size_t)min(m0 + xr + XR * i, M - 1) * K * (16 / XE);
    struct Raw {
        u4 x[XL];
        u4 c[CL];
    };
    auto load_x = [&](Raw& o, int s) LXQ_INLINE {
#pragma unroll
        for (int i = 0; i < XL; i++)
            o.x[i] = *reinterpret_cast<const u4h*>(xp[i] + (size_t)min(s * BK + XE * xc, K - XE) * (16 / XE));
    };
    // the first step's x, ahead of every other address (in the scheduler's
    // order, behind all of them, 20.0 us there)
    Raw next;
    load_x(next, s0);
    __builtin_amdgcn_sched_barrier(0);
    // codes: chunk q = t + 512 i of the block's 128 BITS: column q / BITS, 16
    // bytes q % BITS of its step (columns past N re-read the last; a half
    // step at the end of K reads on into the next row or the readable tail)
    const uint8_t* cp[CL];
    int cd[CL];
#pragma unroll
    for (int i = 0; i < CL; i++) {
        const int q = min(tid + kThreads * i, BN * BITS - 1), col = q / BITS, b = q % BITS * 16;
        cp[i] = reinterpret_cast<const uint8_t*>(wq) + (size_t)min(n0 + col, N - 1) * ((size_t)K * BITS / 8) + b;
        cd[i] = col * L::kCodeRow + b;
    }
    auto load_codes = [&](Raw& o, int s) LXQ_INLINE {
#pragma unroll
        for (int i = 0; i < CL; i++) o.c[i] = *reinterpret_cast<const u4g*>(cp[i] + (size_t)s * (16 * BITS));
    };
    load_codes(next, s0);
    // scales: thread t loads 16 bytes (half t / 256) of the window of column t
    // % 128, scales or biases (t / 128 % 2); a window is 32 / kSb groups
    const int gws = 5 - (SBF ? 2 : 1) + gshift - 7;  // steps per window, log2
    const uint8_t* wp = static_cast<const uint8_t*>((tid >> 7) & 1 ? biases : scales) +
                        (size_t)min(n0 + (tid & 127), N - 1) * (size_t)(K >> gshift) * kSb + (tid >> 8) * 16;
    const int wd = ((tid >> 7) & 1) * (BN * L::kScaleRow) + (tid & 127) * L::kScaleRow + (tid >> 8) * 16;
    // a window past the row's end reads on within the array or its tail
    auto load_win = [&](int win) LXQ_INLINE { return *reinterpret_cast<const u4h*>(wp + (size_t)win * 32); };
    auto store_win = [&](int win, const u4& v) LXQ_INLINE {
        uint32_t* d = reinterpret_cast<uint32_t*>(lds + L::kScales + (win & 1) * L::kWindow + wd);
#pragma unroll
        for (int e = 0; e < 4; e++) d[e] = v[e];
    };

    auto load = [&](Raw& o, int s) LXQ_INLINE {
        load_x(o, s);
        load_codes(o, s);
    };
    auto store_codes = [&](const Raw& o, int stage) LXQ_INLINE {
        uint8_t* d = lds + L::kCodes + stage * (BN * L::kCodeRow);
#pragma unroll
        for (int i = 0; i < CL; i++)
            if (BITS % 4 == 0 || tid + kThreads * i < BN * BITS) *reinterpret_cast<u4*>(d + cd[i]) = o.c[i];
    };
    // load i of step s into the planes of stage st; the sum over the thread's
    // XE k.  fix: an infinity's residue (inf - inf) is 0; a NaN's stays NaN.
    // low: the third terms' bits, of which the last 16 are what it has lost
    auto split = [&](const Raw& o, int s, int i, uint8_t* st, uint32_t& low, auto fix) LXQ_INLINE {
        u4 v = o.x[i];
        if ((s + 1) * BK > K && s * BK + XE * xc >= K) v = u4{0u, 0u, 0u, 0u};
        const int row = xr + XR * i;
        uint8_t* d = st + row * kRowBytes;
        if constexpr (TX == DT_F32) {
            d += (((xc >> 1) ^ (row & 15)) << 4) + (xc & 1) * 8;
            uint32_t p[3][4];
            float f[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                f[e] = __uint_as_float(v[e]);
                p[0][e] = v[e] & 0xffff0000u;
                float r = f[e] - __uint_as_float(p[0][e]);
                if constexpr (decltype(fix)::value) r = __builtin_isinf(f[e]) ? 0.f : r;
                p[1][e] = __float_as_uint(r) & 0xffff0000u;
                p[2][e] = __float_as_uint(r - __uint_as_float(p[1][e]));
                low |= p[2][e];
            }
#pragma unroll
            for (int q = 0; q < 3; q++)
                *reinterpret_cast<u2*>(d + q * L::kPlane) = u2{__builtin_amdgcn_perm(p[q][1], p[q][0], 0x07060302u),
                                                               __builtin_amdgcn_perm(p[q][3], p[q][2], 0x07060302u)};
            return (f[0] + f[1]) + (f[2] + f[3]);
        } else {
            *reinterpret_cast<u4*>(d + ((xc ^ (row & 15)) << 4)) = v;
            float f[4];
#pragma unroll
            for (int e = 0; e < 4; e++)
                f[e] = TX == DT_F16 ? f16_to_f32(v[e] & 0xffffu) + f16_to_f32(v[e] >> 16)
                                    : bf16_to_f32(v[e]) + __uint_as_float(v[e] & 0xffff0000u);
            return (f[0] + f[1]) + (f[2] + f[3]);
        }
    };
    // after the splits of a step: the rare step that may hold an infinity (its
    // third term is a NaN) is split again; the sums over 32 k (32 / XE lanes)
    auto finish = [&](const Raw& o, int s, float (&sum)[XL], uint8_t* st, uint32_t low) LXQ_INLINE {
        if (TX == DT_F32 && __any((low & 0x7f800000u) == 0x7f800000u)) {
#pragma unroll
            for (int i = 0; i < XL; i++) split(o, s, i, st, low, std::true_type{});
        }
#pragma unroll
        for (int i = 0; i < XL; i++) sum[i] += dpp_f<0xB1>(sum[i]);
#pragma unroll
        for (int i = 0; i < XL; i++) sum[i] += dpp_f<0x4E>(sum[i]);
        if constexpr (TX == DT_F32) {
#pragma unroll
            for (int i = 0; i < XL; i++) sum[i] += dpp_f<0x141>(sum[i]);
        }
        constexpr int LG = 32 / XE;
        if (xc % LG == 0) {
#pragma unroll
            for (int i = 0; i < XL; i++)
                *reinterpret_cast<float*>(st + L::kSums + (xc / LG * BM + xr + XR * i) * 4) = sum[i];
        }
    };
    auto sb_f = [&](const uint8_t* p) LXQ_INLINE {
        if constexpr (SBF) return *reinterpret_cast<const float*>(p);
        const uint32_t raw = *reinterpret_cast<const uint16_t*>(p);
        return sb_dt == DT_F16 ? f16_to_f32(raw) : bf16_to_f32(raw);
    };

    auto scale_x = [&](Raw& o) LXQ_INLINE {
        uint32_t m = small;
        asm volatile("" : "+v"(m));  // nothing of this in front of the branch to it
#pragma unroll
        for (int i = 0; i < XL; i++) {
            const float f = (m >> i) & 1u ? kSmallUp : 1.f;
#pragma unroll
            for (int e = 0; e < 4; e++) o.x[i][e] = __float_as_uint(__uint_as_float(o.x[i][e]) * f);
        }
    };
    uint32_t lost = 0;  // the third terms' bits of all steps

    f32x16 acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; i++)
#pragma unroll
        for (int t = 0; t < NT; t++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][t][v] = 0.f;

    u4 win;
    // step s from stage (s - s0) % 2; o holds step s + 1 as loaded (past the
    // last step: the last again, into a stage that nobody reads)
    auto step = [&](int s, Raw& o) LXQ_INLINE {
        if (TX == DT_F32 && again) scale_x(o);
        const int stage = (s - s0) & 1, sn = min(s + 1, s1 - 1);
        const uint8_t* st = lds + stage * L::kStage;
        uint8_t* other = lds + (stage ^ 1) * L::kStage;
        const int wi = s >> gws;
        if (s == s0 || (s & ((1 << gws) - 1)) == 0) win = load_win(min(wi + 1, (steps - 1) >> gws));
        uint32_t w[NT][WL];
        float sc[NT], bi[NT];
#pragma unroll
        for (int t = 0; t < NT; t++) {
            const int col = 64 * nw + 32 * t + c;
            // codes 16 h .. +16 of the wave's 32, in whole words (for odd
            // widths half h = 1 starts 16 bits into its first word)
            const uint32_t* cs = reinterpret_cast<const uint32_t*>(lds + L::kCodes + stage * (BN * L::kCodeRow) +
                                                                   col * L::kCodeRow) + kg * BITS + h * (BITS / 2);
            uint32_t raw[WL];
#pragma unroll
            for (int i = 0; i < WL; i++) raw[i] = cs[i];
#pragma unroll
            for (int i = 0; i < WL; i++) {
                uint32_t v = raw[i];
                if constexpr (BITS % 2 == 1) v = __builtin_amdgcn_alignbit(i + 1 < WL ? raw[i + 1 < WL ? i + 1 : i] : 0u, v, 16 * h);
                w[t][i] = v ^ top_bits<BITS>(i);
            }
            const int g = ((s & ((1 << gws) - 1)) * BK + 32 * kg) >> gshift;  // group within the window
            const uint8_t* ss = lds + L::kScales + (wi & 1) * L::kWindow + col * L::kScaleRow + g * kSb;
            // 32 codes past K (zeros of x): no scale of the next row or the tail
            const bool in = s * BK + 32 * kg < K;
            sc[t] = in ? sb_f(ss) : 0.f;
            bi[t] = in ? fmaf(sc[t], C, sb_f(ss + BN * L::kScaleRow)) : 0.f;
        }
        store_codes(o, stage ^ 1);
        float sum[XL];
        uint32_t low = 0;
        f32x16 g[MT][NT];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            // sub-step j: k 16 h + 8 j .. +8 of the wave's 32 (chunk of the row)
            const int ch = 4 * kg + 2 * h + j;
            u4 a[MT][P], b[NT];
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int q = 0; q < P; q++)
                    a[i][q] = *reinterpret_cast<const u4*>(st + q * L::kPlane + (32 * i + c) * kRowBytes +
                                                           ((ch ^ (c & 15)) << 4));
#pragma unroll
            for (int t = 0; t < NT; t++) b[t] = codes8<BITS, TX>(w[t], j);
#pragma unroll
            for (int q = 0; q < P; q++)
#pragma unroll
                for (int i = 0; i < MT; i++)
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        if (j == 0 && q == 0) {
                            f32x16 z;
#pragma unroll
                            for (int v = 0; v < 16; v++) z[v] = 0.f;
                            g[i][t] = mfma<TX>(a[i][q], b[t], z);
                        } else {
                            g[i][t] = mfma<TX>(a[i][q], b[t], g[i][t]);
                        }
                    }
#pragma unroll
            for (int i = j * XL / 2; i < (j + 1) * XL / 2; i++) sum[i] = split(o, sn, i, other, low, std::false_type{});
        }
        finish(o, sn, sum, other, low);
        lost |= low;
        load(o, min(s + 2, s1 - 1));
        const uint8_t* sums = st + L::kSums + kg * (BM * 4);
#pragma unroll
        for (int i = 0; i < MT; i++)
#pragma unroll
            for (int v4 = 0; v4 < 4; v4++) {
                const f4 xs = *reinterpret_cast<const f4*>(sums + (32 * i + 8 * v4 + 4 * h) * 4);
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int t = 0; t < NT; t++) {
                        const int v = 4 * v4 + e;
                        acc[i][t][v] = fmaf(sc[t], g[i][t][v], fmaf(bi[t], xs[e], acc[i][t][v]));
                    }
            }
        if (((s + 1) & ((1 << gws) - 1)) == 0) store_win(wi + 1, win);
        __syncthreads();
    };

    uint32_t* flag = reinterpret_cast<uint32_t*>(lds + L::kFlag);
    if (TX == DT_F32 && tid == 0) *flag = 0u;
    {
        float sum[XL];
        uint32_t low = 0;
        const u4 w0 = load_win(s0 >> gws);
        if (TX == DT_F32 && again) scale_x(next);
#pragma unroll
        for (int i = 0; i < XL; i++) sum[i] = split(next, s0, i, lds, low, std::false_type{});
        finish(next, s0, sum, lds, low);
        lost |= low;
        store_codes(next, 0);
        load(next, min(s0 + 1, s1 - 1));
        store_win(s0 >> gws, w0);
    }
    __syncthreads();
    for (int s = s0; s < s1; s++) step(s, next);

    // the four K parts meet in LDS, in two [BM][128] tiles (lane: column c of a
    // 32 x 32 tile, register v its row 8 (v / 4) + 4 h + v % 4): parts 0 and 2
    // store, 1 and 3 add theirs
    float* ot = reinterpret_cast<float*>(lds + (kg >> 1) * L::kTile);
    if (TX == DT_F32 && (lost & 0xffffu) != 0u) *flag = 1u;
#pragma unroll
    for (int half = 0; half < 2; half++) {
        if ((kg & 1) == half) {
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (int t = 0; t < NT; t++)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        float* d = ot + (32 * i + 8 * (v >> 2) + 4 * h + (v & 3)) * L::kOut + 64 * nw + 32 * t + c;
                        *d = half ? *d + acc[i][t][v] : acc[i][t][v];
                    }
        }
        __syncthreads();
    }
    const int oc = 4 * (tid & 31), orow = tid >> 5;
#pragma unroll
    for (int i = 0; i < kOutVecs<MT>; i++) {
        const float* d = reinterpret_cast<const float*>(lds) + (orow + 16 * i) * L::kOut + oc;
        o[i] = *reinterpret_cast<const f4*>(d) + *reinterpret_cast<const f4*>(d + L::kTile / 4);
    }
    if constexpr (TX != DT_F32) return false;
    if (again) {
#pragma unroll
        for (int i = 0; i < kOutVecs<MT>; i++)
            if ((rows >> i) & 1u) o[i] *= kSmallDown;
        return false;
    }
    if (__builtin_amdgcn_readfirstlane(*flag) == 0u) return false;
    // bits were lost somewhere (a tail of SiLU or of an exponential will do
    // it): the largest x of each row
    float most[XL];
#pragma unroll
    for (int i = 0; i < XL; i++) most[i] = 0.f;
    for (int s = s0; s < s1; s++) {
        load(next, s);
#pragma unroll
        for (int i = 0; i < XL; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) most[i] = fmaxf(most[i], fabsf(__uint_as_float(next.x[i][e])));
    }
    float* row_most = reinterpret_cast<float*>(lds + L::kRows);
#pragma unroll
    for (int i = 0; i < XL; i++) {
#pragma unroll
        for (int d = 1; d < XC; d <<= 1) most[i] = fmaxf(most[i], __shfl_xor(most[i], d));
        if (xc == 0) row_most[xr + XR * i] = most[i];
        if (most[i] < kSmall) small |= 1u << i;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kOutVecs<MT>; i++)
        if (row_most[orow + 16 * i] < kSmall) rows |= 1u << i;
    const float r = row_most[lane & (BM - 1)];
    __syncthreads();  // the tiles and the rows are read before another run's stages
    return __any(r > 0.f && r < kSmall);
}

template <int BITS, int TX, bool SBF, int MT>
__global__ __launch_bounds__(kThreads, 1) void qgemm_grp_kernel(
    const void* __restrict__ x, const uint32_t* __restrict__ wq, const void* __restrict__ scales,
    const void* __restrict__ biases, void* __restrict__ y, int M, int K, int N, int gshift, int sb_dt, Epilogue ep,
    int mtiles, int each, int longer, void* __restrict__ ws) {
    constexpr int BM = 32 * MT, kVec = kOutVecs<MT>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    // grid: (tiles, parts); the first `longer` parts are each + 1 steps
    // (no divisions where there is one tile of rows: the first loads wait for
    // all of this)
    const int tile = (int)blockIdx.x, part = (int)blockIdx.y;
    const unsigned un = mtiles == 1 ? blockIdx.x : blockIdx.x / (unsigned)mtiles;
    const int m0 = (int)(blockIdx.x - un * (unsigned)mtiles) * BM, n0 = (int)un * BN;
    const int s0 = part * each + min(part, longer), s1 = s0 + each + (part < longer ? 1 : 0);
    f4 o[kVec];
    uint32_t small = 0, rows = 0;
    for (int run = 0; run_tile<BITS, TX, SBF, MT>(lds, x, wq, scales, biases, M, K, N, gshift, sb_dt, m0, n0, s0, s1,
                                                  run, small, rows, o);)
        run = 1;
    const int tid = threadIdx.x, oc = 4 * (tid & 31), orow = tid >> 5;
    constexpr uint32_t kSlot = BM * BN * 4;
    const int tiles = (int)gridDim.x, parts = (int)gridDim.y;
    if (parts > 1) {
        const __amdgpu_buffer_rsrc_t pr = __builtin_amdgcn_make_buffer_rsrc(
            static_cast<uint8_t*>(ws) + split::kPartOffset, 0, (int)((uint32_t)(tiles * parts) * kSlot), 0x00020000);
        const uint32_t first = (uint32_t)(tile * parts) * kSlot;
#pragma unroll
        for (int i = 0; i < kVec; i++)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, o[i]), pr, (uint32_t)(tid * 16),
                                                   first + (uint32_t)part * kSlot + (uint32_t)(i * kThreads * 16),
                                                   split::kCachePolicyDevice);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        uint32_t* word = reinterpret_cast<uint32_t*>(lds);
        if (tid == 0) *word = split::count_part(ws, tile, parts) ? 1u : 0u;
        __syncthreads();
        if (*word == 0u) return;
#pragma unroll
        for (int i = 0; i < kVec; i++) o[i] = f4{0.f, 0.f, 0.f, 0.f};
        // four parts' loads in flight together (past the last part: offsets
        // past the buffer's end, which read zeros; 0 + the sum changes nothing)
        constexpr int kPB = 4;
        for (int p0 = 0; p0 < parts; p0 += kPB) {
            u4 v[kPB][kVec];
#pragma unroll
            for (int p = 0; p < kPB; p++)
#pragma unroll
                for (int i = 0; i < kVec; i++)
                    v[p][i] = __builtin_amdgcn_raw_buffer_load_b128(
                        pr, p0 + p < parts ? (uint32_t)(tid * 16) : 0x80000000u,
                        first + (uint32_t)(p0 + p < parts ? p0 + p : 0) * kSlot + (uint32_t)(i * kThreads * 16),
                        split::kCachePolicyDevice);
            // in pairs: added one by one, 72 parts (M = 13, K = 18496, N = 109,
            // 2-bit, f16 x) were 1.65e-7 off in all, a launch per two rows 1.13e-7
#pragma unroll
            for (int i = 0; i < kVec; i++)
                o[i] += (__builtin_bit_cast(f4, v[0][i]) + __builtin_bit_cast(f4, v[1][i])) +
                        (__builtin_bit_cast(f4, v[2][i]) + __builtin_bit_cast(f4, v[3][i]));
        }
    }
    const bool plain = ep.bias == nullptr && ep.act == ACT_NONE && ep.out_dt == DT_F32 && N % 4 == 0;
#pragma unroll
    for (int i = 0; i < kVec; i++) {
        const int m = m0 + orow + 16 * i, n = n0 + oc;
        if (m >= M) continue;
        if (plain) {
            if (n < N) *reinterpret_cast<f4g*>(static_cast<float*>(y) + (size_t)m * N + n) = o[i];
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < N) store_out<true>(y, (size_t)m * N + n + e, (size_t)(n + e), ep, o[i][e]);
        }
    }
}

template <int BITS, int TX, bool SBF, int MT>
LuxStatus launch_t(const QmmArgs& a, hipStream_t st) {
    using L = Lds<MT, BITS, TX == DT_F32 ? 3 : 1>;
    if (planned(a, "qgemm_grp_kernel")) return LuxStatus::Ok;
    auto kern = qgemm_grp_kernel<BITS, TX, SBF, MT>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, L::kBytes);
    if (attr != hipSuccess) return LuxStatus::Internal;
    const int mtiles = (a.M + L::BM - 1) / L::BM, ntiles = (a.N + BN - 1) / BN;
    const size_t all = (size_t)mtiles * ntiles;
    if (all >= (1ull << 31)) return LuxStatus::NotSupported;
    const int tiles = (int)all, steps = (a.K + BK - 1) / BK;
    // K parts until there is a block per CU, at least two steps each, within
    // the workspace
    int parts = 1;
    if (a.ws != nullptr && tiles <= split::kMaxPartTiles) {
        parts = 256 / tiles;
        parts = parts < steps / 2 ? parts : steps / 2;
        const size_t fit = a.ws_bytes > split::kPartOffset
                               ? (a.ws_bytes - split::kPartOffset) / ((size_t)tiles * L::BM * BN * 4) : 0;
        if ((size_t)parts > fit) parts = (int)fit;
        if (parts < 1) parts = 1;
    }
    const int gshift = a.group_size == 32 ? 5 : a.group_size == 64 ? 6 : 7;
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, (unsigned)parts), dim3(kThreads), L::kBytes, st, a.x, a.wq, a.scales,
                       a.biases, a.y, a.M, a.K, a.N, gshift, a.sb_dtype, a.epi(), mtiles, steps / parts, steps % parts,
                       a.ws);
    return hipGetLastError() == hipSuccess ? LuxStatus::Ok : LuxStatus::Internal;
}

template <int BITS, int TX>
LuxStatus launch_x(const QmmArgs& a, hipStream_t st) {
    if (a.sb_dtype == DT_F32)
        return a.M <= 32 ? launch_t<BITS, TX, true, 1>(a, st) : launch_t<BITS, TX, true, 2>(a, st);
    return a.M <= 32 ? launch_t<BITS, TX, false, 1>(a, st) : launch_t<BITS, TX, false, 2>(a, st);
}

template <int TX>
LuxStatus launch_b(const QmmArgs& a, hipStream_t st) {
    switch (a.bits) {
    case 2: return launch_x<2, TX>(a, st);
    case 3: return launch_x<3, TX>(a, st);
    case 4: return launch_x<4, TX>(a, st);
    case 5: return launch_x<5, TX>(a, st);
    case 6: return launch_x<6, TX>(a, st);
    case 8: return launch_x<8, TX>(a, st);
    default: return LuxStatus::NotSupported;
    }
}

extern template LuxStatus launch_b<DT_F32>(const QmmArgs&, hipStream_t);
extern template LuxStatus launch_b<DT_F16>(const QmmArgs&, hipStream_t);
extern template LuxStatus launch_b<DT_BF16>(const QmmArgs&, hipStream_t);

}  // namespace grp
}  // namespace lxq
