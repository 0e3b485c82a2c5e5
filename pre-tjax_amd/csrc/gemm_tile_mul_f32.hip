// The one-tile-per-workgroup GEMM kernels for fp32 storage (gemm_tile.h), multiplying epilogue with column sums.
#include "gemm_tile_launch.h"

namespace ptj_gemm_detail {
int gemm_tile_mul_launch_f32(const GemmArgs& g, int cfg, int am, int bm, int* mul_rows, hipStream_t st) {
    return gt_dispatch<float, true>(g, cfg, am, bm, mul_rows, st);
}
}  // namespace ptj_gemm_detail
