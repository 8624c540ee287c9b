// qgemm_grp.hip -- dispatch of the group-wise GEMM (kernel in qgemm_grp.h, one
// translation unit per type of x: qgemm_grp_{f32,f16,bf16}.hip).
#include "qgemm_grp.h"

namespace lxq {

LuxStatus launch_qgemm_grp(const QmmArgs& a, hipStream_t st) {
    if (a.K % 64 != 0) return LuxStatus::NotSupported;
    switch (a.x_dtype) {
    case DT_F32: return grp::launch_b<DT_F32>(a, st);
    case DT_F16: return grp::launch_b<DT_F16>(a, st);
    default: return grp::launch_b<DT_BF16>(a, st);
    }
}

}  // namespace lxq
