// The tile shapes of gemm_tile.h that are built, by configuration number (costs and choice: gemm_plan.h), for one
// storage type per translation unit.
#pragma once
#include "gemm_core.h"

namespace {

//                      tile     waves K-groups stages chunks per register set
typedef GtCfg<32, 32, 1, 1, 4, 3, 4> GtTiny;        // few rows: four wavefronts share one 32x32 tile along K
typedef GtCfg<64, 64, 1, 2, 2, 3, 4> GtSmall;       // (fp32)
typedef GtCfg<32, 64, 1, 1, 4, 3, 4> GtTinyWide;
typedef GtCfg<64, 64, 2, 2, 2, 4, 4> GtSmall8;      // eight wavefronts
typedef GtCfg<64, 128, 1, 4, 2, 3, 4> GtWide8;      // eight wavefronts
typedef GtCfg<64, 64, 1, 2, 2, 2, 4> GtSmall2;      // two workgroups per CU
typedef GtCfg<64, 128, 1, 4, 1, 3, 4> GtWide;
typedef GtCfg<128, 128, 2, 4, 1, 3, 4> GtSquare;
typedef GtCfg<128, 128, 2, 4, 1, 2, 2> GtSquare2;   // two workgroups per CU
typedef GtCfg<128, 192, 2, 2, 1, 2, 2> GtLarge;     // two workgroups per CU

#include "gemm_split.h"
#include "gemm_planes.h"

typedef GsCfg<128, 128, 4, 2> GsSquare;
typedef GsCfg<64, 64, 2, 2> GsSmall;                // two workgroups per CU

template <typename T, bool MUL, typename C>
int gt_run(const GemmArgs& g, int am, int bm, int* mul_rows, hipStream_t st) {
    if (mul_rows != nullptr) *mul_rows = C::TMW * 32;
    const int rc = gt_launch<T, C, MUL>(g, am, bm, st);
    if (rc != PTJ_OK || g.splits <= 1 || g.leave_partials) return rc;
    return launch_splitk_reduce<T>(g, g.splits, st);
}

template <bool MUL, typename C>
int gs_run(const GemmArgs& g, int am, int bm, int* mul_rows, hipStream_t st) {
    if (mul_rows != nullptr) *mul_rows = C::TMW * 32;
    const int rc = gs_launch<C, MUL>(g, am, bm, st);
    if (rc != PTJ_OK || g.splits <= 1 || g.leave_partials) return rc;
    return launch_splitk_reduce<float>(g, g.splits, st);
}

template <typename T, bool MUL>
int gt_dispatch(const GemmArgs& g, int cfg, int am, int bm, int* mul_rows, hipStream_t st) {
    if constexpr (sizeof(T) == 2) {
        switch (cfg) {
            case 0: return gt_run<T, MUL, GtTiny>(g, am, bm, mul_rows, st);
            case 2: return gt_run<T, MUL, GtWide>(g, am, bm, mul_rows, st);
            case 3: return gt_run<T, MUL, GtSquare>(g, am, bm, mul_rows, st);
            case 8: return gt_run<T, MUL, GtTinyWide>(g, am, bm, mul_rows, st);
            case 9: return gt_run<T, MUL, GtSmall8>(g, am, bm, mul_rows, st);
            case 10: return gt_run<T, MUL, GtWide8>(g, am, bm, mul_rows, st);
            case 4: return gt_run<T, MUL, GtSquare2>(g, am, bm, mul_rows, st);
            default: return gt_run<T, MUL, GtLarge>(g, am, bm, mul_rows, st);
        }
    } else {
        switch (cfg) {
            case 0: return gt_run<T, MUL, GtTiny>(g, am, bm, mul_rows, st);
            case 1: return gt_run<T, MUL, GtSmall>(g, am, bm, mul_rows, st);
            case 2: return gt_run<T, MUL, GtSmall2>(g, am, bm, mul_rows, st);
            case 3: return gt_run<T, MUL, GtWide>(g, am, bm, mul_rows, st);
            case 4: return gs_run<MUL, GsSquare>(g, am, bm, mul_rows, st);
            default: return gs_run<MUL, GsSmall>(g, am, bm, mul_rows, st);
        }
    }
}

}  // namespace
