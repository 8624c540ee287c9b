// qgemm_grp_f32.hip -- group-wise GEMM kernels, f32 x.
#include "qgemm_grp.h"

namespace lxq {
namespace grp {
template LuxStatus launch_b<DT_F32>(const QmmArgs&, hipStream_t);
}  // namespace grp
}  // namespace lxq
