// qgemm_f32.hip -- dispatch of the f32-activation GEMM (kernel in qgemm_f32.h).
#include "qgemm_f32.h"

namespace lxq {

// From 9 rows where the K-split whole-line GEMV takes 4 rows a launch, from 5
// where every row is a launch of its own (3/5/6-bit codes, K it does not
// divide).  g64, f32 scales, 4-bit, us per launch against those kernels: K = N
// = 4096, M = 5 / 8 / 16 / 32 / 64 12.7 / 12.7 / 13.0 / 13.2 / 19.5 against
// 10.9 / 13.2 / 26.3 / 53.3 / 108; K = 4096, N = 14336, M = 8 / 16 / 128 27.8
// / 27.1 / 72.5 against 30.2 / 60.2 / 470; 3-bit K = 14336, N = 4096, M = 16
// 31 against 145; 5-bit K = 640, N = 1000, M = 16 10.4 against 66.7.  The
// whole-line kernel keeps its class of up to 16 rows of 3/5/6-bit codes at K
// <= 4096.
LuxStatus launch_qgemm_f32(const QmmArgs& a, hipStream_t st) {
    if (a.x_dtype != DT_F32 || a.K % 64 != 0) return LuxStatus::NotSupported;
    const bool irregular = a.bits == 3 || a.bits == 5 || a.bits == 6;
    const int mx_step = 16 * (a.K > 8192 ? 16 : a.K > 4096 ? 8 : 4);
    const bool rows = irregular || a.K > 16384 || a.K % mx_step != 0;
    if (a.M < (!rows ? 9 : irregular && a.K <= 4096 ? 17 : 5)) return LuxStatus::NotSupported;
    switch (a.bits) {
    case 2: return f32g::launch_b<2>(a, st);
    case 3: return f32g::launch_b<3>(a, st);
    case 4: return f32g::launch_b<4>(a, st);
    case 5: return f32g::launch_b<5>(a, st);
    case 6: return f32g::launch_b<6>(a, st);
    case 8: return f32g::launch_b<8>(a, st);
    default: return LuxStatus::NotSupported;
    }
}

}  // namespace lxq
