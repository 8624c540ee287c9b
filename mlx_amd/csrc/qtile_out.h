// qtile_out.h -- what the large GEMMs share past their K loops: rows of y
// through the output stage, and K parts: their number, and the launch that
// adds them.
#pragma once
#include <algorithm>

#include "kernels.h"
#include "qcommon.h"
#include "qsplit.h"

namespace lxq {
namespace tileout {

typedef uint32_t t4 __attribute__((ext_vector_type(4), aligned(16)));
constexpr int kCUs = 256;
constexpr size_t kTileBytes = 128 * 1024;  // both GEMMs' tiles hold 32 Ki fp32 sums

// 8 columns n .. n + 7 of rows of y, through the output stage: their biases,
// loaded once, and one (16-bit y) or two (f32) 16-byte stores per row.  Rows
// of any N and y of any alignment its type allows: the stores need no more
// than that.  Only the chunk that N ends in stores value by value.  (As whole
// 16-byte chunks where N allowed them, else value by value, every lane 8
// columns from the next: LDS-dequant GEMM M = 1414, K = 256, N = 4913, 3-bit,
// GELU 34.6 us, so 24.2; M = 215, K = 256, N = 8377, 4-bit, RELU 22.8 and 13.7.)
struct RowOut {
    typedef uint32_t f32x4 __attribute__((ext_vector_type(4), aligned(4)));
    typedef uint32_t u16x8 __attribute__((ext_vector_type(4), aligned(2)));
    void* y;
    int N, n;
    float bias[8];
    __device__ __forceinline__ RowOut(void* y_, int N_, int n_, const Epilogue& ep) : y(y_), N(N_), n(n_) {
#pragma unroll
        for (int e = 0; e < 8; e++) bias[e] = ep.bias ? load_f(ep.bias, (size_t)min(n + e, N - 1), ep.bias_dt) : 0.f;
    }
    template <bool EPI>
    __device__ __forceinline__ void store(int m, float (&o)[8], const Epilogue& ep) const {
        if constexpr (EPI) {
#pragma unroll
            for (int e = 0; e < 8; e++) {
                if (ep.bias) o[e] = o[e] + bias[e];
                o[e] = apply_act(ep.act, o[e]);
            }
        }
        const size_t at = (size_t)m * N + n;
        if (ep.out_dt == DT_F32) {
            float* d = static_cast<float*>(y) + at;
            if (n + 8 <= N) {
#pragma unroll
                for (int e = 0; e < 8; e += 4)
                    *reinterpret_cast<f32x4*>(d + e) = f32x4{__float_as_uint(o[e]), __float_as_uint(o[e + 1]),
                                                             __float_as_uint(o[e + 2]), __float_as_uint(o[e + 3])};
            } else {
#pragma unroll
                for (int e = 0; e < 7; e++)
                    if (n + e < N) d[e] = o[e];
            }
            return;
        }
        u16x8 p;
        if (ep.out_dt == DT_BF16) {
#pragma unroll
            for (int e = 0; e < 8; e += 2) p[e / 2] = pack2<DT_BF16>(o[e], o[e + 1]);
        } else {
#pragma unroll
            for (int e = 0; e < 8; e += 2) p[e / 2] = pack2<DT_F16>(o[e], o[e + 1]);
        }
        uint16_t* d = static_cast<uint16_t*>(y) + at;
        if (n + 8 <= N) {
            *reinterpret_cast<u16x8*>(d) = p;
        } else {
#pragma unroll
            for (int e = 0; e < 7; e++)
                if (n + e < N) d[e] = (uint16_t)(p[e / 2] >> (16 * (e & 1)));
        }
    }
};

// chunks of 8 columns per row of a tile BN wide that has `cols` of them left,
// to the next power of two (a thread keeps its columns from row to row): a
// narrow tile's rows go to all the threads (M = 1182, K = 256, N = 15, 4-bit,
// RELU: as 16 chunks per row, 14 of them idle, 19.6 us, so 9.2)
template <int BN>
__device__ __forceinline__ int row_chunks(int cols) {
    int w = BN / 8;
    while (w > 1 && w * 4 >= cols) w >>= 1;
    return w;
}

// Sum of the K parts: 8 columns of a row per thread, the parts' tiles in part
// order, then the output stage.  (As the last part's own work at M = 509, K =
// 11008, N = 4096, 6-bit, 64 CUs each read 512 KiB and ran every GELU: 84 us
// in all.  As a launch of its own over all the CUs, bound by the partials' 32
// MiB: 69.)
template <int BM, int BN, bool EPI>
__global__ __launch_bounds__(256) void parts_kernel(const void* __restrict__ ws, void* __restrict__ y, int M, int N,
                                                    Epilogue ep, int mtiles, int nsplit) {
    const int chunks = (N + 7) / 8;
    const unsigned id = blockIdx.x * 256u + threadIdx.x;
    const int m = (int)(id / (unsigned)chunks), n = (int)(id % (unsigned)chunks) * 8;
    if (m >= M) return;
    const int tile = n / BN * mtiles + m / BM;
    const float* p = reinterpret_cast<const float*>(static_cast<const uint8_t*>(ws) + split::kPartOffset) +
                     (size_t)tile * nsplit * (BM * BN) + (m % BM) * BN + n % BN;
    const RowOut out(y, N, n, ep);
    float o[8] = {};
#pragma unroll 4
    for (int i = 0; i < nsplit; i++) {
        const t4 a = *reinterpret_cast<const t4*>(p + (size_t)i * (BM * BN));
        const t4 b = *reinterpret_cast<const t4*>(p + (size_t)i * (BM * BN) + 4);
#pragma unroll
        for (int e = 0; e < 4; e++) {
            o[e] += __uint_as_float(a[e]);
            o[4 + e] += __uint_as_float(b[e]);
        }
    }
    out.store<EPI>(m, o, ep);
}

template <int BM, int BN, bool EPI>
void launch_parts(const QmmArgs& a, int mtiles, int nsplit, hipStream_t st) {
    static_assert((size_t)BM * BN * 4 == kTileBytes, "tile of sums");
    const size_t threads = (size_t)a.M * ((a.N + 7) / 8);
    hipLaunchKernelGGL((parts_kernel<BM, BN, EPI>), dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, a.ws,
                       a.y, a.M, a.N, a.epi(), mtiles, nsplit);
}

// What a shape's split costs, in eightieths of a us: a K step; the meeting of
// two halves, and more per tile; the parts' launch, and each part's 128 KiB
// (stored and loaded by all CUs together), up to 128 parts and past them; the
// output stage fused into whole tiles or halves instead of that launch.
struct PartPrice {
    int step, halves, halves_tile, launch, part, part_past, fused;
};
// LDS-dequant GEMM: fitted to 492 launches of 1 to 100 tiles, K = 512 .. 8192,
// 3-bit (0.3 % above the best split of each in the mean), against which a
// price of 20 twentieths a step, 100 for halves, 60 for the launch and 1 per
// part was up to 34 % off.  us, halves or whole tiles / K parts (parts): M =
// 2045, N = 507, K = 768 16.3 / 21.9 (3, not taken), K = 2048 25.6 / 29.2 (4,
// not taken), K = 4096 39.2 / 28.9 (8); M = 1021, N = 2043, K = 3072 34.2 /
// 32.4 (4); M = 253, N = 507, K = 512 14.3 / 13.6 (2); with GELU M = 253, N =
// 2043, K = 512 28.6 / 17.0 (2).
constexpr PartPrice kLdsPrice{68, 320, 5, 160, 7, 2, 240};
// Register-W GEMM (its parts summed by the last to arrive / by the launch):
// 8-bit M = 100, K = 14336, N = 1000 55.2 / 20.8; 4-bit M = 128, K = 14336, N =
// 4096 49.5 / 31.2; M = 80, K = 4096, N = 1000 24.1 / 14.5.
constexpr PartPrice kRwPrice{72, 400, 0, 240, 4, 4, 0};

// K parts for a shape with few tiles (1: none, whole tiles or halves of a
// split round) of KT steps, at most `most`: the cheapest.  Parts are whole
// units of KT / most steps, so counts that do not divide them leave one part
// longer than KT / S: priced at KT / S they took M = 330, K = 1024, N = 1778,
// 6-bit as 3 parts of 1, 1 and 2 units, 19.6 us, against 18.2 as 4; M = 370, K
// = 2048, N = 675, 6-bit 7 parts 20.1, 8 17.4; M = 75, K = 6144, N = 393, 3-bit
// 20 parts 17.6, 24 15.0.
inline int k_parts(int tiles, int KT, int most, bool halves, const PartPrice& c, const QmmArgs& a) {
    if (a.ws == nullptr || 2 * tiles > kCUs) return 1;
    const int cap = std::min(std::min(kCUs / tiles, most),
                             (int)((a.ws_bytes - split::kPartOffset) / ((size_t)tiles * kTileBytes)));
    int best = 1, least = halves && a.epoch != 0u ? c.step * KT / 2 + c.halves + c.halves_tile * tiles : c.step * KT;
    if (a.has_epilogue()) least += c.fused;
    for (int S = 2; S <= cap; S++) {
        const int parts = tiles * S, cost = c.step * (KT / most) * ((most + S - 1) / S) + c.launch +
                                            c.part * std::min(parts, 128) + c.part_past * std::max(parts - 128, 0);
        if (cost < least) { least = cost; best = S; }
    }
    return best;
}

}  // namespace tileout
}  // namespace lxq
