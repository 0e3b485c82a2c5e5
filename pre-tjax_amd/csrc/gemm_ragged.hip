// The bf16 GEMM kernels for operands without 16-byte alignment (gemm_ragged.h).
#include "gemm_core.h"

namespace {
#include "gemm_ragged.h"

typedef GrCfg<128, 128, 2, 2> GrSquare;
typedef GrCfg<64, 64, 2, 2> GrSmall;
}  // namespace

namespace ptj_gemm_detail {
int gemm_ragged_launch_bf16(const GemmArgs& g, int cfg, int am, int bm, hipStream_t st) {
    return cfg == 0 ? gr_launch<GrSquare>(g, am, bm, st) : gr_launch<GrSmall>(g, am, bm, st);
}
}  // namespace ptj_gemm_detail
