// The one-tile-per-workgroup GEMM kernels for bf16 storage (gemm_tile.h), plain epilogues.
#include "gemm_tile_launch.h"

namespace ptj_gemm_detail {
int gemm_tile_launch_bf16(const GemmArgs& g, int cfg, int am, int bm, hipStream_t st) {
    return gt_dispatch<bf16, false>(g, cfg, am, bm, nullptr, st);
}
}  // namespace ptj_gemm_detail
