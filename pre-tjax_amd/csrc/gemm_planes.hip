// The fp32 GEMM on operands split ahead of the product (gemm_planes.h).
#include "gemm_tile_launch.h"

namespace ptj_gemm_detail {
int gemm_planes_launch(const GemmArgs& g, char* planes, hipStream_t st) {
    const int rc = gp_launch<false>(g, planes, st);
    if (rc != PTJ_OK || g.splits <= 1 || g.leave_partials) return rc;
    return launch_splitk_reduce<float>(g, g.splits, st);
}
int gemm_planes_mul_launch(const GemmArgs& g, char* planes, hipStream_t st) { return gp_launch<true>(g, planes, st); }
}  // namespace ptj_gemm_detail
