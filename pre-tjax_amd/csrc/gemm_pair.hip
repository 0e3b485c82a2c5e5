// The two products of a linear layer's backward (internal.h: ptj_linear_bwd) in one launch.
//
// At a few hundred tokens each of the two takes 7-13 us, most of it the latency of a launch, of the first panels
// (weights that the optimizer pass has pushed out of every cache) and of the write-back, on a quarter to a half of
// the CUs.  Side by side they cost about what the longer one costs alone.  At some thousand tokens they make between one and
// three rounds of tiles, and share the rounds: the product whose tiles take longer comes first in the grid and the shorter
// tiles of the other fill the CUs as they fall free (dx: m contraction elements a tile, dw: n).  With dx first / with dw first, us:
// 3136 tokens proj 20.4 / 19.7, 6000 tokens ffn2 with its multiplier 95.6 / 84.5, 8192 tokens qkv 79.9 / 66.2, ffn1 115.1 / 90.5.
#include "gemm_core.h"
#include "gemm_plan.h"
#include "internal.h"

namespace {

typedef GtCfg<64, 64, 1, 2, 2, 3, 4> PairSmall;      // gemm_tile_launch.h: configurations 1, 2, 3 of the bf16 table
typedef GtCfg<64, 128, 1, 4, 1, 3, 4> PairWide;
typedef GtCfg<128, 128, 2, 4, 1, 3, 4> PairSquare;

constexpr int max_int(int a, int b) { return a > b ? a : b; }

template <typename CX, typename CW, bool MUL>
__global__ __launch_bounds__(CX::THREADS, CX::WAVES_EU < CW::WAVES_EU ? CX::WAVES_EU : CW::WAVES_EU) void gemm_pair_kernel(
    const GemmArgs gx, const GemmArgs gw, int nx, int nw, bool dw_first) {
    static_assert(CX::THREADS == CW::THREADS, "one workgroup size");
    __shared__ __attribute__((aligned(1024))) char smem[max_int(CX::SMEM, CW::SMEM)];
    const int x = (int)blockIdx.x - (dw_first ? nw : 0), w = (int)blockIdx.x - (dw_first ? 0 : nx);
    if (x >= 0 && x < nx) gt_tile<bf16, KMAJOR, MNMAJOR, CX, MUL>(gx, x, smem);
    else gt_tile<bf16, MNMAJOR, MNMAJOR, CW, false>(gw, w, smem);
}

template <typename CX, typename CW>
int launch_pair(const GemmArgs& gx, const GemmArgs& gw, bool mul, bool dw_first, hipStream_t st) {
    const int nx = ((gx.n + CX::TBM - 1) / CX::TBM) * ((gx.m + CX::TBN - 1) / CX::TBN);
    const int nw = ((gw.n + CW::TBM - 1) / CW::TBM) * ((gw.m + CW::TBN - 1) / CW::TBN);
    const dim3 grid(nx + nw), block(CX::THREADS);
    if (mul) hipLaunchKernelGGL((gemm_pair_kernel<CX, CW, true>), grid, block, 0, st, gx, gw, nx, nw, dw_first);
    else hipLaunchKernelGGL((gemm_pair_kernel<CX, CW, false>), grid, block, 0, st, gx, gw, nx, nw, dw_first);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

// Time of n1 tiles of t1, then n2 of t2 <= t1, on `slots` workgroups that take the next tile as they end one.
double pair_makespan(int64_t n1, double t1, int64_t n2, double t2, int64_t slots) {
    const int64_t full = n1 / slots, rest = n1 % slots;
    const double first = (double)(full + (rest > 0)) * t1;
    auto holds = [&](double t) {          // tiles of t2 that end by t
        const double late = t - (double)(full + 1) * t1, early = t - (double)full * t1;
        return (double)rest * floor((late > 0 ? late : 0.0) / t2 + 1e-9) + (double)(slots - rest) * floor((early > 0 ? early : 0.0) / t2 + 1e-9);
    };
    if (holds(first) >= (double)n2) return first;
    double lo = first, hi = first + (double)(n2 / slots + 2) * t2;
    for (int i = 0; i < 30; ++i) {
        const double mid = 0.5 * (lo + hi);
        if (holds(mid) >= (double)n2) hi = mid;
        else lo = mid;
    }
    return hi;
}

// Estimated time of a pair (us) with configurations ix, iw of the bf16 table.  Fitted to the pairs themselves: the four layers of a GPT-2
// small block, every choice here and two launches (estimated by gemm_plan; SEPARATE and, with a multiplier, SEPARATE_MUL times
// that), alone at 25 token counts from 256 to 16384 and inside a training step at 12.  The pick is 1.6 % slower than the
// best of them on average; the estimates of gemm_plan, and dx always first, picked 7 % above it.  Training step, before / now, us:
// 512 tokens 2690 / 2678, 1024 3785 / 3659, 2560 5376 / 5290, 3136 5804 / 5567, 3584 6599 / 6451, 6144 9925 / 9293, 12288 the same.
struct PairCost { double step, finish, crowd, dw; };      // us; crowd: growth of a step from half the CUs busy to all; dw: its steps
constexpr PairCost PAIR_COST[4] = {{}, {0.21, 1.75, 0.31, 0.88}, {0.19, 1.59, 0.49, 1.07}, {0.33, 3.52, 0.15, 0.97}};
constexpr double PAIR_START = 3.2, PAIR_MUL = 0.48, PAIR_ROUNDS = 0.55, SEPARATE = 0.95, SEPARATE_MUL = 1.22;
constexpr double PAIR_ALONE = 0.84;                       // wide tiles, one a CU because of the small ones beside them
constexpr double PAIR_SHARED = 2.01, PAIR_FLOWS = 0.7;    // wide tiles, two a CU: where one ends early, the other goes on faster
// Layers narrower than the fitted ones: few tiles share a panel and dW's chain of n / 64 steps is what the pair waits for, 0.20-0.25 us a step
// where the fit has 0.18.  256 wide, two launches / the pair that the fit alone took, us: ffn2 12288 tokens 38.3 / 52.9, ffn1 8192 22.2 / 29.8,
// qkv 6000 18.9 / 20.8; 320 wide, ffn2 6000 32.2 / 41.4, 8192 38.1 / 49.7.  Over widths of 256 to 2048 and 256 to 12288 tokens the pick is then 2.6 %
// slower than the best choice on average (256 wide 3.0, 4.6 without it), the picks of the estimate of gemm_plan 5.9 %.
constexpr double PAIR_NARROW = 0.3;
constexpr int64_t PAIR_FITTED = 768;

double pair_us(const PtjLinearBwd& p, int ix, int iw, int cus, bool* dw_first) {
    const TileCost &cx = GT_COST[0][ix], &cw = GT_COST[0][iw];
    const int64_t nx = gp_ceil(p.n, cx.tbm) * gp_ceil(p.k, cx.tbn), nw = gp_ceil(p.m, cw.tbm) * gp_ceil(p.k, cw.tbn), all = nx + nw;
    const int64_t slots = (int64_t)cus * (cx.per_cu < cw.per_cu ? cx.per_cu : cw.per_cu);
    const bool two = slots > cus;
    const double busy = all < cus ? (double)all / (double)cus : 1.0, over = all > cus ? (double)(all - cus) / (double)cus : 0.0;
    const double shared = two ? 1.0 + (PAIR_SHARED - 1.0) * (over < 1.0 ? over : 1.0) : 1.0;
    auto tile = [&](int i, int64_t k, bool dw) {
        const PairCost& c = PAIR_COST[i];
        const double step = c.step * (1.0 + (busy > 0.5 ? c.crowd * 2.0 * (busy - 0.5) : 0.0)) * (dw ? c.dw : 1.0);
        return (double)gp_ceil(k, GT_COST[0][i].bkt) * step * (i == 2 && !two ? PAIR_ALONE : shared) + c.finish;
    };
    const int64_t width = p.m < p.k ? p.m : p.k;
    const double narrow = 1.0 + (width < PAIR_FITTED ? PAIR_NARROW * (double)(PAIR_FITTED - width) / 512.0 : 0.0);
    const double tx = tile(ix, p.m, false) + (p.mul ? PAIR_MUL : 0.0), tw = tile(iw, p.n, true);
    *dw_first = tw > tx;
    if (all <= slots) return (PAIR_START + (tw > tx ? tw : tx)) * narrow;
    double t = tw > tx ? pair_makespan(nw, tw, nx, tx, slots) : pair_makespan(nx, tx, nw, tw, slots);
    if (two) t += PAIR_FLOWS * (((double)nx * tx + (double)nw * tw) / (double)slots - t);
    return (PAIR_START + t) * (1.0 + PAIR_ROUNDS * (1.0 - (double)slots / (double)all)) * narrow;
}

double single_us(int64_t n, int64_t m, int64_t k, bool may_split, int cus) {
    return gemm_plan(n, m, k, 2, may_split ? (size_t)-1 : 0, cus).us;
}

// config 0: two launches; else 1 + 3 * ix + iw over {small, wide, square}
struct PairChoice { int config; bool dw_first; };
PairChoice choose_pair(const PtjLinearBwd& p) {
    struct Entry { int64_t n, m, k; int mul, cus; PairChoice choice; };
    static thread_local Entry table[32] = {};
    const int cus = num_cus(), mul = p.mul != nullptr;
    Entry& e = table[((uint64_t)p.n * 0x9E3779B97F4A7C15ull + (uint64_t)p.m * 0xC2B2AE3D27D4EB4Full + (uint64_t)p.k * 31 + mul) >> 40 & 31];
    if (e.n == p.n && e.m == p.m && e.k == p.k && e.mul == mul && e.cus == cus) return e.choice;
    double best = (mul ? SEPARATE_MUL : SEPARATE) * (single_us(p.n, p.k, p.m, !mul, cus) + single_us(p.m, p.k, p.n, true, cus));
    PairChoice choice = {0, false};
    for (int ix = 1; ix <= 3; ++ix)
        for (int iw = 1; iw <= 3; ++iw) {
            if ((ix == 3) != (iw == 3)) continue;
            bool dw_first;
            const double us = pair_us(p, ix, iw, cus, &dw_first);
            if (us < best) {
                best = us;
                choice = {1 + 3 * (ix - 1) + (iw - 1), dw_first};
            }
        }
    e = {p.n, p.m, p.k, mul, cus, choice};
    return choice;
}

GemmArgs args_of(const void* a, const void* b, void* c, int64_t n, int64_t m, int64_t k, int64_t a_row, int64_t a_k) {
    GemmArgs g{};
    g.a = a; g.b = b; g.c = c;
    g.n = (int)n; g.m = (int)m; g.k = (int)k;
    g.a_row = a_row; g.a_k = a_k;
    g.b_row = 1; g.b_k = m;
    g.c_rs = m;
    g.k_per_split = (int)k;
    g.splits = g.tail_splits = 1;
    g.vec_out = m % 8 == 0 && ptj_aligned16(c);
    g.epilogue = PTJ_EPI_NONE;
    return g;
}

}  // namespace

int ptj_linear_bwd(const PtjLinearBwd& p, void* scratch, size_t scratch_bytes, int dtype, PtjPartialSums* later, hipStream_t st) {
    const int64_t n = p.n, m = p.m, k = p.k;
    if (dtype == PTJ_BF16 && !p.dx_only && n < (1 << 20) && m < (1 << 20) && k < (1 << 20)) {
        GemmArgs gx = args_of(p.d, p.w, p.dx, n, k, m, m, 1), gw = args_of(p.d, p.x, p.dw, m, k, n, 1, m);
        gx.mul = p.mul; gx.mul_rs = k; gx.colpart = p.colpart;
        if (p.mul) gx.vec_out = gx.vec_out && ptj_aligned16(p.mul);
        const bool ok = p.d && p.w && p.x && p.dx && p.dw && pick_mode<bf16>(gx.a, gx.a_row, gx.a_k) == KMAJOR &&
                        pick_mode<bf16>(gx.b, gx.b_row, gx.b_k) == MNMAJOR &&
                        pick_mode<bf16>(gw.a, gw.a_row, gw.a_k) == MNMAJOR && pick_mode<bf16>(gw.b, gw.b_row, gw.b_k) == MNMAJOR &&
                        gt_eligible(gx, KMAJOR, MNMAJOR) && gt_eligible(gw, MNMAJOR, MNMAJOR);
        const PairChoice choice = ok ? choose_pair(p) : PairChoice{0, false};
        if (choice.config != 0) {
            const bool mul = p.mul != nullptr;
            int rc;
            switch (choice.config) {
                case 1: rc = launch_pair<PairSmall, PairSmall>(gx, gw, mul, choice.dw_first, st); break;
                case 2: rc = launch_pair<PairSmall, PairWide>(gx, gw, mul, choice.dw_first, st); break;
                case 4: rc = launch_pair<PairWide, PairSmall>(gx, gw, mul, choice.dw_first, st); break;
                case 5: rc = launch_pair<PairWide, PairWide>(gx, gw, mul, choice.dw_first, st); break;
                default: rc = launch_pair<PairSquare, PairSquare>(gx, gw, mul, choice.dw_first, st); break;
            }
            if (rc != PTJ_OK || !mul) return rc;
            if (!later->add(p.colpart, p.colsum, (n + 63) / 64, k, k))
                return ptj_set_error(PTJ_ERR_INVALID, "linear_bwd: too many pending sums");
            return PTJ_OK;
        }
    }
    if (!p.dx_only) {
        const int rc = ptj_gemm(p.d, p.x, p.dw, nullptr, m, k, n, 1, m, k, 1, k, PTJ_EPI_NONE, nullptr, 0, scratch, scratch_bytes, dtype, st);
        if (rc != PTJ_OK) return rc;
    }
    if (p.mul)
        return ptj_gemm_mul_colsum_later(p.d, p.w, p.mul, p.dx, p.colsum, n, k, m, m, 1, k, 1, k, k, p.colpart,
                                         ptj_gemm_mul_colsum_workspace_bytes(n, k), scratch, scratch_bytes, dtype, later, st);
    return ptj_gemm(p.d, p.w, p.dx, nullptr, n, k, m, m, 1, k, 1, k, PTJ_EPI_NONE, nullptr, 0, scratch, scratch_bytes, dtype, st);
}

extern "C" int ptj_linear_bwd_choice(int64_t n, int64_t m, int64_t k, int multiplied, int* dw_first) {
    PTJ_CHECK_ARG(n >= 1 && m >= 1 && k >= 1 && n < (1 << 20) && m < (1 << 20) && k < (1 << 20) && dw_first, "linear_bwd_choice: bad shape");
    PtjLinearBwd p{};
    p.n = n; p.m = m; p.k = k;
    if (multiplied) p.mul = dw_first;      // (looked at for null only)
    const PairChoice c = choose_pair(p);
    *dw_first = c.dw_first;
    return c.config;
}
