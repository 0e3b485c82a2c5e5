// The persistent bf16 GEMM with 256x192 tiles (gemm_ring.h), plain epilogues.
#include "gemm_core.h"

namespace ptj_gemm_detail {
int gemm_ring_narrow_launch(const GemmArgs& g, int am, int bm, hipStream_t st) { return ring_launch<RingNarrow, false>(g, am, bm, st); }
}  // namespace ptj_gemm_detail
