// Which GEMM kernel a product takes.  Two families exist: the persistent 256x192 kernels (gemm_core.h,
// gemm_direct.h), which stream tile after tile through every CU and win when there are several rounds of
// tiles, and the one-tile-per-workgroup kernels of gemm_tile.h, which win when the 256x192 tiles would
// leave CUs idle or when a border would take the slow element-wise loader.
//
// The choice minimises a time estimate,
//     start + rounds * (K steps * step + finish)  [+ second stage of a K split],
// where a round is one workgroup in every slot (256 CUs x workgroups per CU).  start, step and finish
// (microseconds) are fitted per kernel to timings of the 11 products of a GPT-2 small block, forward, dX and dW
// (launches replayed from a graph, operands rotating over 200 MB).  Checked on these at eight token counts from 64
// to 8192 and both storage types, against every kernel and K split within twice the lowest estimate: the estimate
// is off by 7 % (bf16) and 6 % (fp32) on average, and the pick is 0.4 % slower than the best one on average and
// 8 % at worst.  The kernels for unaligned bf16 operands are fitted to products with odd sizes up to 4001.
#pragma once
#include "common.h"

namespace {

struct TileCost {
    int tbm, tbn;        // C tile
    int bkt;             // contraction elements per K step (panels of 128 bytes x K groups)
    int per_cu;          // workgroups per CU
    double start, step, finish;   // us
    double shared;       // step time with every slot of a CU taken, relative to one workgroup per CU
};

// bf16 / fp32; the index is the configuration number of gemm_tile_launch
constexpr int GT_CONFIGS[2] = {7, 6};
// operands without 16-byte alignment: the configurations from here on (bf16: gemm_ragged.h; fp32: gemm_split.h)
constexpr int RAGGED_FIRST[2] = {7, 4}, RAGGED_END[2] = {9, 6};
constexpr TileCost GT_COST[2][9] = {
    {{32, 32, 256, 1, 2.03, 0.522, 1.24, 1.0},
     {64, 64, 128, 1, 2.49, 0.372, 1.81, 1.0},
     {64, 128, 64, 2, 3.49, 0.299, 1.21, 1.89},
     {128, 128, 64, 1, 1.84, 0.402, 3.18, 1.0},
     {128, 128, 64, 2, 2.73, 0.714, 1.88, 1.39},
     {128, 192, 64, 2, 2.45, 0.922, 5.00, 1.50},
     {256, 192, 64, 1, 2.00, 1.250, 8.00, 1.0},
     {128, 128, 64, 2, 4.32, 0.765, 5.66, 1.57},
     {64, 64, 64, 2, 4.51, 0.471, 1.01, 1.08}},
    // fp32: the last two multiply on the bf16 pipe (gemm_split.h)
    {{32, 32, 128, 1, 3.25, 0.663, 1.67, 1.0},
     {64, 64, 64, 1, 3.56, 1.077, 2.37, 1.0},
     {64, 64, 64, 2, 4.16, 1.326, 1.45, 1.51},
     {64, 128, 32, 2, 6.44, 1.035, 0.56, 1.88},
     {128, 128, 32, 1, 3.10, 1.218, 3.22, 1.0},
     {64, 64, 32, 2, 5.87, 0.640, 0.00, 1.32}},
};

enum { ALIGNED = 0, LOOSE_OUTPUT = 1, LOOSE_OPERAND = 2 };   // what of a product does not come in aligned 16-byte vectors

struct GemmPlan {
    int cfg;      // configuration of gemm_tile.h, or -1: the persistent kernels with their own K split
    int splits;   // K splits of cfg >= 0
    int kps;      // contraction elements per split (a multiple of bkt)
};

inline int64_t gp_ceil(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Second stage of a K split: its launch, and the partial sums written and read once more.
inline double gp_reduce_us(int64_t n, int64_t m, int splits) {
    return splits > 1 ? 2.6 + 0.35e-6 * 4.0 * (double)splits * (double)n * (double)m : 0.0;
}

inline double gp_tile_us(const TileCost& c, int64_t n, int64_t m, int64_t k, int elt, int splits, int cus) {
    const int64_t work = gp_ceil(n, c.tbm) * gp_ceil(m, c.tbn) * splits;
    const int64_t steps = gp_ceil(gp_ceil(k, splits), c.bkt);
    const int64_t slots = (int64_t)cus * c.per_cu, full = work / slots, rem = work % slots;
    double t = c.start + (double)full * ((double)steps * c.step * c.shared + c.finish);
    if (rem) t += (double)steps * c.step * (rem > cus ? c.shared : 1.0) + c.finish;
    // bf16: a chip that stays full over several rounds shares the path from L2: measured 10 % at 1.5 rounds, 30 % at many
    const double rounds = (double)work / (double)slots;
    if (elt == 2 && rounds > 1.0) t *= 1.0 + 0.3 * (1.0 - 1.0 / rounds);
    return t + gp_reduce_us(n, m, splits);
}

// The persistent bf16 kernels: 20 us per round of 256x192 tiles at k = 768; a partial panel along K goes through the
// element-wise loader.
inline double gp_persistent_us(int64_t n, int64_t m, int64_t k, int splits, int cus) {
    const int64_t work = gp_ceil(n, 256) * gp_ceil(m, 192) * splits, steps = gp_ceil(gp_ceil(k, splits), 64);
    const int64_t full = work / cus, rem = work % cus;
    const double rounds = (double)full + (rem ? 0.35 + 0.65 * (double)rem / cus : 0.0);
    double t = 7.0 + rounds * (1.2 * (double)steps + 4.3);
    if (n % 256 != 0 || m % 192 != 0) t += 8.0;
    if (k % 64 != 0) t += 20.0;
    return t + gp_reduce_us(n, m, splits);
}

// `persistent_splits`: what choose_splits gives the persistent kernels; `ws_bytes`: workspace for fp32 partial sums.
// Contractions shorter than 1024 are not split, so that a product and the same product with another epilogue
// add in the same order.  `loose`: the persistent kernels read operands without 16-byte alignment element by element (an
// order of magnitude slower) and write such outputs so (twice the time at k = 768); the tile kernels write any.
inline GemmPlan gemm_plan(int64_t n, int64_t m, int64_t k, int elt, size_t ws_bytes, int persistent_splits, int cus,
                          int loose = ALIGNED) {
    const bool ragged = loose == LOOSE_OPERAND;
    GemmPlan best = {-1, 1, (int)k};
    // within 8 % the persistent kernels are kept: in a training step their loads run on from product to product.  In fp32 they
    // are never the fastest (158 us against 120 for 4096x3072x768): they serve what the tile kernels do not take (operands
    // without a unit stride, overlapping rows, pitches from 2^21 elements, or below 8 off the vector grid), and every other
    // fp32 product gets a configuration.
    double best_us = ragged || elt != 2 ? 1e30 : (loose ? 2.0 : 0.92) * gp_persistent_us(n, m, k, persistent_splits, cus);
    const int type = elt == 2 ? 0 : 1;
    for (int i = ragged ? RAGGED_FIRST[type] : 0; i < (ragged ? RAGGED_END[type] : GT_CONFIGS[type]); ++i) {
        const TileCost& c = GT_COST[type][i];
        for (int s = 1; s <= 16; ++s) {
            if (s > 1 && (k < 1024 || k / s < 256 || (size_t)s * (size_t)n * (size_t)m * sizeof(float) > ws_bytes)) break;
            const int64_t kps = gp_ceil(gp_ceil(k, s), c.bkt) * c.bkt;
            if (s > 1 && gp_ceil(k, kps) != s) continue;
            const double us = gp_tile_us(c, n, m, k, elt, s, cus);
            if (us < best_us) {
                best_us = us;
                best = {i, s, (int)(s > 1 ? kps : k)};
            }
        }
    }
    return best;
}

}  // namespace
