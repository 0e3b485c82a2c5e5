// The weight gradients of several blocks in one launch (internal.h: ptj_weight_grads).
//
// One block's four products have few tiles and a long contraction, the tokens.  Launched one by one they took K splits, whose partial
// sums were written and read once more; beside their dX (gemm_pair.hip) they shared its rounds.  The blocks' products do not depend
// on each other, and nothing in the backward waits for them: what they read is kept and all of them go at once, whole tiles along
// the contraction, in rounds that are full but for the last.  The kernels are those of gemm_ring.h and gemm_split.h with another way
// from a work item to its operands.  Twelve blocks 768 wide, all weight gradients: 16384 tokens bf16 3.30 ms in 48 launches with
// 36 second stages, 2.22 ms (1250 TFLOP/s) in one and 2.03 in two; 4096 tokens fp32 4.6 -> 4.2 ms.
//
// Taken from a round of tiles on (ptj_weight_grads_blocks).  Training steps, each with its dX / together, us: 12 blocks of 768, bf16, 64 tokens
// 1914 / 1686, 512 2469 / 2455, 1536 3663 / 3598, 4096 6437 / 5772, 16384 18165 / 17059, fp32 64 2634 / 2322, 1024 7757 / 7057, 3072 17255 /
// 16250; 12 of 256, 8192 tokens (264 tiles, a second round of 8) 3646 / 3305; 2 of 768, 4096 tokens 1193 / 1151; 24 of 1024, 512 tokens
// 6305 / 6141; no size was slower.
//
// What the products of a group read is kept for it: 9 values a token and unit of width, beside the 16 of a block's activations.  So a group
// has the fewest blocks whose groups are estimated within GROUP_SLACK of the best: twelve blocks 768 wide in bf16 go as
// five in 2.8 rounds of 256x192 tiles and seven in 2.95 of 256x256, in fp32 as three times four (6.75 rounds, all at once 20.25).  Peak memory
// and time of a training step, all twelve in one launch / so: 16x1024 bf16 10.25 / 9.12 GB, 17.24 / 17.18 ms, 8x512 fp32 6.75 / 5.85 GB,
// 19.8 / 19.6 ms.  Up to GROUP_SPLIT_FROM tokens (28 MB a block in bf16) the further launches cost more than the memory is worth: all / so, us: bf16
// 128 tokens 49 / 60, 512 110 / 112, 1024 176 / 180, 2048 324 / 322, 4096 620 / 608, fp32 128 229 / 245, 512 591 / 623, 1024 1101 / 1100,
// 2048 2139 / 2126, 4096 4256 / 4176.
#include "gemm_tile_launch.h"
#include "gemm_plan.h"

namespace {

constexpr double GROUP_SLACK = 1.02;
constexpr int GROUP_SPLIT_FROM = 2048;

struct GroupPlan { int cfg; double us; };
// Tile shape with the lowest estimate (bf16: of gemm_ring.h); `round`: of those with a round of tiles or more, cfg = -1: none
GroupPlan group_plan(const PtjGradGroup& p, int dtype, bool round) {
    const int cus = num_cus();
    GroupPlan best = {-1, 1e30};
    for (int i = 0; i < (dtype == PTJ_BF16 ? RING_CONFIGS : 1); ++i) {
        const TileCost& c = dtype == PTJ_BF16 ? RING_COST[i] : GT_COST[1][4];
        int64_t tiles = 0;
        for (int kind = 0; kind < PtjGradGroup::KINDS; ++kind) tiles += gp_ceil(p.n[kind], c.tbm) * gp_ceil(p.m[kind], c.tbn);
        tiles *= p.blocks;
        if (round && tiles < cus) continue;
        const double us = c.start + (double)gp_ceil(tiles, cus) * ((double)gp_ceil(p.k, c.bkt) * gp_step_us(c, tiles, cus) + c.finish);
        if (us < best.us) best = {i, us};
    }
    return best;
}

}  // namespace

int ptj_weight_grads_blocks(PtjGradGroup p, int64_t layers, int dtype) {
    double us[PtjGradGroup::BLOCKS + 1] = {}, best = 1e30;
    const int most = layers < PtjGradGroup::BLOCKS ? (int)layers : PtjGradGroup::BLOCKS;
    for (int i = 1; i <= most; ++i) {
        p.blocks = i;
        us[i] = group_plan(p, dtype, false).us;
    }
    auto all = [&](int blocks) { return (double)(layers / blocks) * us[blocks] + us[layers % blocks]; };
    auto fills = [&](int blocks) { p.blocks = blocks; return group_plan(p, dtype, true).cfg >= 0; };
    const int64_t parts = (layers + PtjGradGroup::BLOCKS - 1) / PtjGradGroup::BLOCKS;
    const int equal = (int)((layers + parts - 1) / parts);
    if (!fills(equal)) return 0;                      // (equal parts, so that no launch is left with a few tiles alone)
    if (p.k < GROUP_SPLIT_FROM) return equal;
    for (int i = 1; i <= most; ++i)
        if (fills(i) && all(i) < best) best = all(i);
    for (int i = 1; i <= most; ++i)
        if (fills(i) && all(i) <= GROUP_SLACK * best) return i;
    return 0;
}

int ptj_weight_grads(const PtjGradGroup& p, int dtype, hipStream_t st) {
    if (p.blocks < 1 || p.blocks > PtjGradGroup::BLOCKS || p.k < 1) return ptj_set_error(PTJ_ERR_INVALID, "weight_grads: bad group");
    for (int i = 0; i < PtjGradGroup::KINDS; ++i)
        for (int j = 0; j < p.blocks; ++j) PTJ_CHECK_ARG(p.d[i][j] && p.x[i][j] && p.dw[i][j], "weight_grads: null pointer");
    if (dtype != PTJ_BF16) {
        int parts[PtjGradGroup::KINDS];
        for (int i = 0; i < PtjGradGroup::KINDS; ++i) parts[i] = gemm_plan(p.n[i], p.m[i], p.k, 4, (size_t)-1, num_cus()).kps;
        return gs_group_launch<GsSquare>(p, parts, st);
    }
    return group_plan(p, dtype, false).cfg == 0 ? ring_group_launch<RingFull>(p, st) : ring_group_launch<RingNarrow>(p, st);
}
