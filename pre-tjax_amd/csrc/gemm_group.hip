// The weight gradients of several blocks in one launch (internal.h: ptj_weight_grads).
//
// One block's four products have few tiles and a long contraction, the tokens.  Launched one by one they took K splits, whose partial
// sums were written and read once more; beside their dX (gemm_pair.hip) they shared its rounds.  The blocks' products do not depend
// on each other, and nothing in the backward waits for them: what they read is kept and all of them go at once, whole tiles along
// the contraction, in rounds that are full but for the last.  The kernels are those of gemm_ring.h and gemm_split.h with another way
// from a work item to its operands.  Twelve blocks 768 wide, all weight gradients: 16384 tokens bf16 3.30 ms in 48 launches with
// 36 second stages, 2.22 ms (1250 TFLOP/s) in one; 4096 tokens fp32 4.6 -> 4.2 ms.
//
// Taken from a round of tiles on (ptj_weight_grads_fill).  Training steps, each with its dX / together, us: 12 blocks of 768, bf16, 64 tokens
// 1914 / 1686, 512 2469 / 2455, 1536 3663 / 3598, 4096 6437 / 5772, 16384 18165 / 17059, fp32 64 2623 / 2358, 1024 7648 / 6994, 3072 17130 /
// 16500; 12 of 256, 8192 tokens (264 tiles, a second round of 8) 3646 / 3305; 2 of 768, 4096 tokens 1193 / 1151; 24 of 1024, 512 tokens
// 6305 / 6141; no size was slower.
#include "gemm_tile_launch.h"
#include "gemm_plan.h"

namespace {

// Tile shape with the lowest estimate (bf16: of gemm_ring.h), or -1: less than a round of any
int group_config(const PtjGradGroup& p, int dtype) {
    const int cus = num_cus();
    double best = 1e30;
    int cfg = -1;
    for (int i = 0; i < (dtype == PTJ_BF16 ? RING_CONFIGS : 1); ++i) {
        const TileCost& c = dtype == PTJ_BF16 ? RING_COST[i] : GT_COST[1][4];
        int64_t tiles = 0;
        for (int kind = 0; kind < PtjGradGroup::KINDS; ++kind) tiles += gp_ceil(p.n[kind], c.tbm) * gp_ceil(p.m[kind], c.tbn);
        tiles *= p.blocks;
        if (tiles < cus) continue;
        const double us = (double)gp_ceil(tiles, cus) * ((double)gp_ceil(p.k, c.bkt) * gp_step_us(c, tiles, cus) + c.finish);
        if (us < best) {
            best = us;
            cfg = i;
        }
    }
    return cfg;
}

}  // namespace

bool ptj_weight_grads_fill(const PtjGradGroup& p, int dtype) { return group_config(p, dtype) >= 0; }

int ptj_weight_grads(const PtjGradGroup& p, int dtype, hipStream_t st) {
    if (p.blocks < 1 || p.blocks > PtjGradGroup::BLOCKS || p.k < 1) return ptj_set_error(PTJ_ERR_INVALID, "weight_grads: bad group");
    for (int i = 0; i < PtjGradGroup::KINDS; ++i)
        for (int j = 0; j < p.blocks; ++j) PTJ_CHECK_ARG(p.d[i][j] && p.x[i][j] && p.dw[i][j], "weight_grads: null pointer");
    if (dtype != PTJ_BF16) {
        int parts[PtjGradGroup::KINDS];
        for (int i = 0; i < PtjGradGroup::KINDS; ++i) parts[i] = gemm_plan(p.n[i], p.m[i], p.k, 4, (size_t)-1, num_cus()).kps;
        return gs_group_launch<GsSquare>(p, parts, st);
    }
    return group_config(p, dtype) == 0 ? ring_group_launch<RingFull>(p, st) : ring_group_launch<RingNarrow>(p, st);
}
