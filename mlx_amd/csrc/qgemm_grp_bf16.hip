// qgemm_grp_bf16.hip -- group-wise GEMM kernels, bf16 x.
#include "qgemm_grp.h"

namespace lxq {
namespace grp {
template LuxStatus launch_b<DT_BF16>(const QmmArgs&, hipStream_t);
}  // namespace grp
}  // namespace lxq
