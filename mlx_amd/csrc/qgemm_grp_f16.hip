// qgemm_grp_f16.hip -- group-wise GEMM kernels, f16 x.
#include "qgemm_grp.h"

namespace lxq {
namespace grp {
template LuxStatus launch_b<DT_F16>(const QmmArgs&, hipStream_t);
}  // namespace grp
}  // namespace lxq
