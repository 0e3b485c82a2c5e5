// The one-tile-per-workgroup GEMM kernels for bf16 storage (gemm_tile.h), multiplying epilogue with column sums.
#include "gemm_tile_launch.h"

namespace ptj_gemm_detail {
int gemm_tile_mul_launch_bf16(const GemmArgs& g, int cfg, int am, int bm, int* mul_rows, hipStream_t st) {
    return gt_dispatch<bf16, true>(g, cfg, am, bm, mul_rows, st);
}
}  // namespace ptj_gemm_detail
