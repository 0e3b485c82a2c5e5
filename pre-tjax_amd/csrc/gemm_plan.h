// Which GEMM kernel a product takes.  Two families exist: the persistent kernels of gemm_ring.h (bf16), which stream tile after
// tile of 256x256 or 256x192 through every CU and win when there is about a round of such tiles or more, and the
// one-tile-per-workgroup kernels of gemm_tile.h (fp32: also gemm_split.h, and gemm_planes.h for large products) below that.
//
// The choice minimises a time estimate,
//     start + rounds * (K steps * step + finish)  [+ second stage of a K split],
// where a round is one workgroup in every slot (256 CUs x workgroups per CU).  start, step and finish
// (microseconds) are fitted per kernel to timings of the 12 products of a GPT-2 small block, forward, dX and dW
// (launches replayed from a graph, operands rotating over 200 MB).  bf16: checked on these at eight token counts from 448 to
// 16384, against every kernel and K split within 1.6 times the lowest estimate, the estimate is off by 8 % rms and the pick is
// 0.4 % slower than the best one on average and 11 % at worst.  (Before the configurations for up to a round of tiles, 8 to 10, which are
// fitted to their own sizes below.)
// (64x128 and two 128x128 tiles a CU were fitted again on 1280 to 2048 tokens, where the first was estimated 10 % low and the
// picks had become up to 8 % slower than those before the ring kernels.  Forward before these / now, in turn on one box:
// 1280 tokens 944 / 920 us, 1408 1114 / 1082, 1536 1107 / 1088, 2048 1332 / 1333.)
#pragma once
#include "common.h"

namespace {

struct TileCost {
    int tbm, tbn;        // C tile
    int bkt;             // contraction elements per K step (panels of 128 bytes x K groups)
    int per_cu;          // workgroups per CU
    double start, step, finish;   // us
    double shared;       // step time with every slot of a CU taken, relative to one workgroup per CU
    double crowd;        // growth of the step time from half the CUs busy (0) to all of them
};

// bf16 / fp32; the index is the configuration number of gemm_tile_launch (bf16: 1 is gemm_pair.hip's alone)
// operands without 16-byte alignment: the configurations from here on (bf16: gemm_ragged.h; fp32: gemm_split.h)
constexpr int RAGGED_FIRST[2] = {6, 4}, RAGGED_END[2] = {8, 6};
// The last three of bf16 are for up to a round of tiles: a chain of K steps whose copies are on their way for 0.7-1.1 us.  Eight wavefronts
// and four stages of 64x64 leave 0.4 us less around the loop than four and three (which they replace); 32x64 tiles put twice as many
// CUs to work; 64x128 with two K groups has half the steps.  One product, us, the best of the others / these: 512x768x768 6.5 / 5.4,
// 512x768x2304 10.5 / 8.7, 512x768x3072 12.6 / 10.1 (K split in two with its second stage 12.7), 256x2304x768 6.5 / 6.2, 512x2304x768 8.5 /
// 8.0, 1536x768x768 8.5 / 8.0, 1536x768x2304 15.3 / 13.9, 1536x768x3072 19 / 17; four and five stages of 128x128, 64x64 and 32x32: no faster.
// 32x64 and 64x128 with two K groups take no K split: their staging of partial sums costs more than the estimate knows (forward of 512
// tokens with 64x128 in five 685 us, with 32x64 whole 645; of 1024 tokens with 64x128 in two 962, with 64x64 whole 943).
// `along` below: 32x32 tiles of operands that both run along the contraction take whole lines of either, and go faster than estimated, where
// the panels of an operand across it come in half lines.  So there a K split of 64x64 tiles has to start as late as that of the four
// wavefronts before.  us, operands from memory, 32x32 / 64x64 in parts: along 2183x64x2624 9.9 / 11.9, 700x192x2624 9.1 / 11.2, 312x64x1280 5.3 /
// 6.6, 814x320x1920 9.7 / 11.6, 526x640x3584 14.0 / 15.6; across 192x768x3072 13.0 / 11.6, 256x768x3072 13.0 / 11.8, 982x256x3456 13.8 / 12.4.
// (Partial sums that the next norm adds up have a cost of their own, fitted with these tiles.)
constexpr double SMALL8_SPLIT = 0.92;
constexpr int GT_END[2] = {11, 6};
inline bool gt_plain(int type, int i) { return type == 1 || (i != 1 && (i < RAGGED_FIRST[0] || i >= RAGGED_END[0])); }
constexpr TileCost GT_COST[2][11] = {
    {{32, 32, 256, 1, 2.08, 0.571, 1.33, 1.0, 0.0},
     {64, 64, 128, 1, 3.62, 0.341, 1.57, 1.0, 0.0},
     {64, 128, 64, 2, 4.50, 0.300, 1.12, 1.87, 0.10},
     {128, 128, 64, 1, 4.59, 0.384, 1.68, 1.0, 0.34},
     {128, 128, 64, 2, 4.25, 0.632, 2.01, 1.33, 0.23},
     {128, 192, 64, 2, 5.57, 0.587, 3.93, 1.32, 0.91},
     {128, 128, 64, 2, 4.32, 0.765, 5.66, 1.57, 0.0},
     {64, 64, 64, 2, 4.51, 0.471, 1.01, 1.08, 0.0},
     {32, 64, 256, 1, 2.85, 0.530, 1.70, 1.0, 0.0},
     {64, 64, 128, 1, 2.70, 0.364, 1.90, 1.0, 0.0},
     {64, 128, 128, 1, 2.50, 0.487, 3.20, 1.0, 0.0}},
    // fp32: the last two multiply on the bf16 pipe (gemm_split.h)
    {{32, 32, 128, 1, 3.25, 0.663, 1.67, 1.0, 0.0},
     {64, 64, 64, 1, 3.56, 1.077, 2.37, 1.0, 0.0},
     {64, 64, 64, 2, 4.16, 1.326, 1.45, 1.51, 0.0},
     {64, 128, 32, 2, 6.44, 1.035, 0.56, 1.88, 0.0},
     {128, 128, 32, 1, 3.10, 1.218, 3.22, 1.0, 0.0},
     {64, 64, 32, 2, 5.87, 0.640, 0.00, 1.32, 0.0}},
};

enum { ALIGNED = 0, LOOSE_OUTPUT = 1, LOOSE_OPERAND = 2 };   // what of a product does not come in aligned 16-byte vectors

// gemm_ring.h, configurations from RING_FIRST on
constexpr int RING_FIRST = 16, RING_CONFIGS = 2;
constexpr TileCost RING_COST[RING_CONFIGS] = {
    {256, 256, 64, 1, 5.83, 1.261, 8.85, 1.0, 0.11},
    {256, 192, 64, 1, 4.53, 1.030, 7.65, 1.0, 0.07},
};

// gemm_planes.h (fp32): start and step of the product with the launch of the split in the start; the split itself moves 10 bytes
// an element.  Fitted to the same products at 256 to 8192 tokens (6 % rms; with it the picks are 0.5 % slower than the best).
// Below about 2000 tokens, and for 768-wide outputs below 8192, the split costs more than it saves.
constexpr int PLANES_CFG = 32;
constexpr TileCost PLANES_COST = {128, 128, 16, 2, 8.66, 0.581, 0.0, 1.90, 0.0};
inline size_t gp_planes_bytes(int64_t n, int64_t m, int64_t k) {
    return ((size_t)(n + 31) / 32 + (size_t)(m + 31) / 32) * ((size_t)(k + 15) / 16) * 3072;
}

struct GemmPlan {
    int cfg;      // configuration of gemm_tile.h, gemm_ring.h or gemm_planes.h, or -1: the kernels for operands of any strides
    int splits;   // K splits
    int kps;      // contraction elements per split (a multiple of bkt)
    int tail_first, tail_splits, tail_kps;   // gemm_ring.h: the tiles from tail_first on (0: none) are K-split
    double us;
};

// kernels a product may take
enum { ANY_KERNEL = 0, RING_ONLY = 1 };

inline int64_t gp_ceil(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Second stage of a K split: its launch, and the partial sums written and read once more.  (bf16: 4.9 us and 0.23 fit best; the
// launch is taken lower because behind a feed-forward block the next norm adds up the partial sums without one.)
// `later`, bf16: it does, and pays 1.6 us and some more for the bytes.  Second feed-forward product in a forward: 512 tokens
// in two parts of 64x64 685 us, with 32x64 tiles whole 645; 1536 tokens in three of 128x128 1113, with 64x128 whole 1132.  A
// product with a bias that runs its second stage itself is planned at the full cost: 750x768x3072 15.6 us with the cost of `later`, 12.3 with
// the full one, 1450x768x3072 20.1 / 16.9.
inline double gp_reduce_us(int64_t n, int64_t m, int splits, int elt, bool later = false) {
    if (splits <= 1) return 0.0;
    const double bytes = 4.0 * (double)splits * (double)n * (double)m;
    if (later && elt == 2) return 1.6 + 0.12e-6 * bytes;
    return 2.6 + (elt == 2 ? 0.24e-6 : 0.35e-6) * bytes;
}
// a K step of one workgroup when `work` of them share the chip
inline double gp_step_us(const TileCost& c, int64_t work, int cus) {
    const double busy = work < cus ? (double)work / (double)cus : 1.0;
    return c.step * (1.0 + (busy > 0.5 ? c.crowd * 2.0 * (busy - 0.5) : 0.0));
}

inline double gp_tile_us(const TileCost& c, int64_t n, int64_t m, int64_t k, int elt, int splits, int cus, bool later) {
    const int64_t work = gp_ceil(n, c.tbm) * gp_ceil(m, c.tbn) * splits;
    const int64_t steps = gp_ceil(gp_ceil(k, splits), c.bkt);
    const double step = gp_step_us(c, work, cus);
    const int64_t slots = (int64_t)cus * c.per_cu, full = work / slots, rem = work % slots;
    double t = c.start + (double)full * ((double)steps * step * c.shared + c.finish);
    if (rem) t += (double)steps * step * (rem > cus ? c.shared : 1.0) + c.finish;
    // bf16: a chip that stays full over several rounds shares the path from L2: measured 10 % at 1.5 rounds, 30 % at many
    const double rounds = (double)work / (double)slots;
    if (elt == 2 && rounds > 1.0) t *= 1.0 + 0.3 * (1.0 - 1.0 / rounds);
    return t + gp_reduce_us(n, m, splits, elt, later);
}

// The persistent kernels.  A last round that is not full costs its steps whole, but its stores only by their share; cut into
// tail_splits K slices per tile (*tail) it costs the steps of a slice, and fp32 partial tiles written and read once.
inline double gp_ring_us(const TileCost& c, int64_t n, int64_t m, int64_t k, int splits, int cus, bool later) {
    const int64_t work = gp_ceil(n, c.tbm) * gp_ceil(m, c.tbn) * splits, steps = gp_ceil(gp_ceil(k, splits), 64);
    const int64_t full = work / cus, rem = work % cus;
    const double tile = (double)steps * gp_step_us(c, work, cus);
    return c.start + (double)full * (tile + c.finish) + (rem ? tile + c.finish * (double)rem / (double)cus : 0.0) +
           gp_reduce_us(n, m, splits, 2, later);
}
inline double gp_ring_tail_us(const TileCost& c, int64_t n, int64_t m, int64_t k, int tail_splits, int cus) {
    const int64_t work = gp_ceil(n, c.tbm) * gp_ceil(m, c.tbn), full = work / cus, items = work % cus * tail_splits;
    const double steps = (double)gp_ceil(k, 64), part = (double)gp_ceil((int64_t)steps, tail_splits), step = gp_step_us(c, cus, cus);
    return c.start + (double)full * (steps * step + c.finish) + (double)gp_ceil(items, cus) * part * step +
           c.finish * (double)items / (double)cus + gp_reduce_us(c.tbm, c.tbn, (int)items, 2);
}

// `ws_bytes`: workspace for fp32 partial sums.  Contractions shorter than 1024 are not split, so that a product and the same
// product with another epilogue add in the same order.  `loose`: operands or outputs that do not come in aligned
// 16-byte vectors; the ring kernels take such operands not at all and write such outputs element by element (twice the
// time at k = 768), the tile kernels write any.
// `later`: the consumer adds up the partial sums of a K split (PTJ_EPI_BIAS_NORM).  `along`: both operands run along the contraction.
// `planes_ws`: workspace for operands split ahead of a product without a K split, where partial sums may not take any.
inline GemmPlan gemm_plan(int64_t n, int64_t m, int64_t k, int elt, size_t ws_bytes, int cus, int loose = ALIGNED,
                          int kernels = ANY_KERNEL, size_t planes_ws = 0, bool later = false, bool along = false) {
    const bool ragged = loose == LOOSE_OPERAND;
    GemmPlan best = {-1, 1, (int)k, 0, 1, 0, 1e30};
    const int type = elt == 2 ? 0 : 1;
    auto fits = [&](double bytes) { return bytes <= (double)ws_bytes; };
    if (kernels != RING_ONLY)
        for (int i = ragged ? RAGGED_FIRST[type] : 0; i < (ragged ? RAGGED_END[type] : GT_END[type]); ++i) {
            if (!ragged && !gt_plain(type, i)) continue;
            const TileCost& c = GT_COST[type][i];
            for (int s = 1; s <= (type == 0 && (i == 8 || i == 10) ? 1 : 16); ++s) {
                if (s > 1 && (k < 1024 || k / s < 256 || !fits(4.0 * s * (double)n * (double)m))) break;
                const int64_t kps = gp_ceil(gp_ceil(k, s), c.bkt) * c.bkt;
                if (s > 1 && gp_ceil(k, kps) != s) continue;
                const double us = gp_tile_us(c, n, m, k, elt, s, cus, later) + (type == 0 && i == 9 && s > 1 && along && !later ? SMALL8_SPLIT : 0.0);
                if (us < best.us) best = {i, s, (int)(s > 1 ? kps : k), 0, 1, 0, us};
            }
        }
    if (elt == 4 && kernels == ANY_KERNEL) {
        const double planes = (double)gp_planes_bytes(n, m, k), split = 1e-6 * (double)(n + m) * (double)k;
        for (int s = 1; s <= 16; ++s) {
            if (s > 1 && (k < 1024 || k / s < 256)) break;
            if (!fits(planes + (s > 1 ? 4.0 * s * (double)n * (double)m : 0.0)) && !(s == 1 && planes <= (double)planes_ws)) break;
            const int64_t kps = gp_ceil(gp_ceil(k, s), 32) * 32;
            if (s > 1 && gp_ceil(k, kps) != s) continue;
            const double us = gp_tile_us(PLANES_COST, n, m, k, elt, s, cus, later) + split;
            if (us < best.us) best = {PLANES_CFG, s, (int)(s > 1 ? kps : k), 0, 1, 0, us};
        }
    }
    if (elt != 2 || ragged) return best;
    for (int i = 0; i < RING_CONFIGS; ++i) {
        const TileCost& c = RING_COST[i];
        const double slow = loose == LOOSE_OUTPUT ? 2.0 : 1.0;
        const int64_t tiles = gp_ceil(n, c.tbm) * gp_ceil(m, c.tbn), full = tiles / cus * cus;
        for (int s = 1; s <= 32; ++s) {
            if (s > 1 && (k < 1024 || k / s < 256 || tiles >= 2 * cus || !fits(4.0 * s * (double)n * (double)m))) break;
            const int64_t kps = gp_ceil(gp_ceil(k, s), 64) * 64;
            if (s > 1 && gp_ceil(k, kps) != s) continue;
            const double us = slow * gp_ring_us(c, n, m, k, s, cus, later);
            if (us < best.us) best = {RING_FIRST + i, s, (int)(s > 1 ? kps : k), 0, 1, 0, us};
        }
        for (int s = 2; s <= 32 && full > 0 && tiles > full && k >= 1024; ++s) {
            const int64_t kps = gp_ceil(gp_ceil(k, s), 64) * 64;
            if (k / s < 256 || !fits(4.0 * s * (double)(tiles - full) * c.tbm * c.tbn)) break;
            if (gp_ceil(k, kps) != s) continue;
            const double us = slow * gp_ring_tail_us(c, n, m, k, s, cus);
            if (us < best.us) best = {RING_FIRST + i, 1, (int)k, (int)full, s, (int)kps, us};
        }
    }
    return best;
}

// workspace that a plan takes: split operands, then partial sums
inline size_t gp_workspace_bytes(const GemmPlan& p, int64_t n, int64_t m, int64_t k) {
    const size_t planes = p.cfg == PLANES_CFG ? gp_planes_bytes(n, m, k) : 0;
    if (planes > 0 || p.splits > 1) return planes + (p.splits > 1 ? (size_t)p.splits * (size_t)n * (size_t)m * sizeof(float) : 0);
    if (p.tail_splits <= 1) return 0;
    const TileCost& c = RING_COST[p.cfg - RING_FIRST];
    return (size_t)(gp_ceil(n, c.tbm) * gp_ceil(m, c.tbn) - p.tail_first) * p.tail_splits * c.tbm * c.tbn * sizeof(float);
}

}  // namespace
