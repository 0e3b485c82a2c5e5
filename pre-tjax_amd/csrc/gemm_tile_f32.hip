// The one-tile-per-workgroup GEMM kernels for fp32 storage (gemm_tile.h), plain epilogues.
#include "gemm_tile_launch.h"

namespace ptj_gemm_detail {
int gemm_tile_launch_f32(const GemmArgs& g, int cfg, int am, int bm, hipStream_t st) {
    return gt_dispatch<float, false>(g, cfg, am, bm, nullptr, st);
}
}  // namespace ptj_gemm_detail
