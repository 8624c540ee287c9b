// qgemm_sk.hip -- dispatch of the split-K small-M GEMM (kernel in qgemm_sk.h,
// one translation unit per code width: qgemm_sk_b{2,3,4,5,6,8}.hip).
#include "qgemm_sk.h"

#include <algorithm>

namespace lxq {
namespace sk {

extern template LuxStatus launch_bits<2>(const QmmArgs&, int, hipStream_t);
extern template LuxStatus launch_bits<3>(const QmmArgs&, int, hipStream_t);
extern template LuxStatus launch_bits<4>(const QmmArgs&, int, hipStream_t);
extern template LuxStatus launch_bits<5>(const QmmArgs&, int, hipStream_t);
extern template LuxStatus launch_bits<6>(const QmmArgs&, int, hipStream_t);
extern template LuxStatus launch_bits<8>(const QmmArgs&, int, hipStream_t);

// Measured (K = 4096, 4-bit g64 f16, weights streamed from HBM: eight
// copies in rotation; µs per launch against the W-streaming kernel):
// unsplit, with x read once per 128 columns, this kernel wins on wide N
// (N = 28672 / 32768: M = 64 38.4 / 39.7 against 47.5 / 50.1, M = 32 32.1
// against 37.8, M = 16 31.5 against 37.1); split, the partial sums and the
// last part's fixup add 5-8 µs, and on narrower N it loses (N = 11008
// 3-bit M = 64: 26.2 at best, S = 2, against 23.6; N = 14336 M = 64 26.4
// against 22.9).  So it runs unsplit from kUnsplitTiles tiles on, and split
// only where the W-streaming kernel does not apply (K % 1024 != 0).
constexpr int kUnsplitTiles = 192;
// at most one block per CU; this also bounds the partials: 256 blocks x
// 32 KiB = 8 MiB
constexpr int kMaxBlocks = 256;

bool applies(int M, int K, int N, int bits, int x_dtype) {
    if (M <= 8 || M > 64 || N <= 0 || (x_dtype != DT_F16 && x_dtype != DT_BF16) || K % kSS != 0) return false;
    if (bits != 2 && bits != 3 && bits != 4 && bits != 5 && bits != 6 && bits != 8) return false;
    // buffer offsets are 32-bit
    if ((size_t)M * K * 2 >= (1ull << 31) || (size_t)N * K * bits / 8 >= (1ull << 31) ||
        (size_t)N * (K / 32) * 4 >= (1ull << 31))
        return false;
    // narrow N with K % 1024 == 0: the W-streaming kernel is faster
    return (N + kCols - 1) / kCols >= kUnsplitTiles || K % 1024 != 0;
}

// the number of K parts S: 1 from kUnsplitTiles tiles on; else one block per
// CU, but no more than sqrt(0.9 K / 128) parts (each adds a round trip of its
// sums) of at least 2 super-steps, lowered until the workspace fits `cap`.
// Parts need not be equal.  us per launch, against divisors of K / 128 that
// gave at least kUnsplitTiles blocks: K = 11008 (86 super-steps: 2 parts, 64
// blocks), N = 4096, 4-bit M = 16 / 32 / 64 31.5 / 32.8 / 44.8 -> 16.1 / 17.4 /
// 23.7 (8 parts); K = 13440, N = 1000, 8-bit M = 64 39.7 -> 26; K = 3584, N =
// 4096, 3-bit M = 64 (7 parts) 20.3 -> 18.8 (5); K = 2816, N = 8192, 8-bit M =
// 20 14.7 -> 12.5 (4).  More blocks than CUs lose: K = 13824, N = 5120, M = 64
// 29.2 (6 parts, 240 blocks) against 40.6 (7, 280).
int choose_split(int M, int K, int N, size_t cap) {
    static_assert(kUnsplitTiles <= kMaxSplitTiles, "split tiles have counter slots");
    const int tiles = (N + kCols - 1) / kCols, steps = K / kSS;
    if (tiles >= kUnsplitTiles) return 1;
    int S = std::min(steps / 2, kMaxBlocks / tiles);
    while (S > 1 && (10 * S * S > 9 * steps || ws_bytes(S, M, N) > cap)) S--;
    // two short parts save less than their meeting costs: three, or none (K =
    // 896, N = 300, M = 33: 1 / 2 / 3 parts 9.7 / 10.5 / 9.4)
    if (S == 2 && steps < 12) S = steps >= 6 && 3 * tiles <= kMaxBlocks && ws_bytes(3, M, N) <= cap ? 3 : 1;
    return S < 1 ? 1 : S;
}

}  // namespace sk

size_t qgemm_sk_workspace(int M, int K, int N, int bits, int x_dtype, size_t cap) {
    using namespace sk;
    if (!applies(M, K, N, bits, x_dtype)) return 0;
    const int S = choose_split(M, K, N, cap);
    return S > 1 ? ws_bytes(S, M, N) : 0;
}

LuxStatus launch_qgemm_sk(const QmmArgs& a, hipStream_t st) {
    using namespace sk;
    if (!applies(a.M, a.K, a.N, a.bits, a.x_dtype)) return LuxStatus::NotSupported;
    const size_t cap = a.ws ? a.ws_bytes : 0;
    const int S = choose_split(a.M, a.K, a.N, cap);
    // what the kernel writes when it splits: partials within the workspace,
    // one counter slot per tile
    if (S > 1 && (ws_bytes(S, a.M, a.N) > cap || (a.N + kCols - 1) / kCols > kMaxSplitTiles))
        return LuxStatus::Internal;
    switch (a.bits) {
    case 2: return launch_bits<2>(a, S, st);
    case 3: return launch_bits<3>(a, S, st);
    case 4: return launch_bits<4>(a, S, st);
    case 5: return launch_bits<5>(a, S, st);
    case 6: return launch_bits<6>(a, S, st);
    default: return launch_bits<8>(a, S, st);
    }
}

}  // namespace lxq
