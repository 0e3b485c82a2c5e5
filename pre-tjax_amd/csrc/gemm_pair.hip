// The two products of a linear layer's backward (internal.h: ptj_linear_bwd) in one launch.
//
// At a few hundred tokens each of the two takes 7-13 us, most of it the latency of a launch, of the first panels
// (weights that the optimizer pass has pushed out of every cache) and of the write-back, on a quarter to a half of
// the CUs.  Side by side they cost about what the longer one costs alone: the workgroups of dx come first in the
// grid (the next step of the backward waits for it), those of dw behind them.
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
    const GemmArgs gx, const GemmArgs gw, int nx) {
    static_assert(CX::THREADS == CW::THREADS, "one workgroup size");
    __shared__ __attribute__((aligned(1024))) char smem[max_int(CX::SMEM, CW::SMEM)];
    const int b = (int)blockIdx.x;
    if (b < nx) gt_tile<bf16, KMAJOR, MNMAJOR, CX, MUL>(gx, b, smem);
    else gt_tile<bf16, MNMAJOR, MNMAJOR, CW, false>(gw, b - nx, smem);
}

template <typename CX, typename CW>
int launch_pair(const GemmArgs& gx, const GemmArgs& gw, bool mul, hipStream_t st) {
    const int nx = ((gx.n + CX::TBM - 1) / CX::TBM) * ((gx.m + CX::TBN - 1) / CX::TBN);
    const int nw = ((gw.n + CW::TBM - 1) / CW::TBM) * ((gw.m + CW::TBN - 1) / CW::TBN);
    if (mul) hipLaunchKernelGGL((gemm_pair_kernel<CX, CW, true>), dim3(nx + nw), dim3(CX::THREADS), 0, st, gx, gw, nx);
    else hipLaunchKernelGGL((gemm_pair_kernel<CX, CW, false>), dim3(nx + nw), dim3(CX::THREADS), 0, st, gx, gw, nx);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

// Estimated time of a pair with configurations ix, iw of the bf16 table: both resident at once -> the longer one; more
// workgroups than slots -> the slots shared out over the work, plus half a workgroup of imbalance.
double pair_us(const PtjLinearBwd& p, int ix, int iw, int cus) {
    const TileCost &cx = GT_COST[0][ix], &cw = GT_COST[0][iw];
    const int64_t nx = gp_ceil(p.n, cx.tbm) * gp_ceil(p.k, cx.tbn), nw = gp_ceil(p.m, cw.tbm) * gp_ceil(p.k, cw.tbn);
    const int per_cu = cx.per_cu < cw.per_cu ? cx.per_cu : cw.per_cu;
    const int64_t slots = (int64_t)cus * per_cu;
    const bool packed = nx + nw > cus;                     // CUs with two workgroups: their steps take longer
    const double tx = (double)gp_ceil(p.m, cx.bkt) * gp_step_us(cx, nx + nw, cus) * (packed ? cx.shared : 1.0) + cx.finish;
    const double tw = (double)gp_ceil(p.n, cw.bkt) * gp_step_us(cw, nx + nw, cus) * (packed ? cw.shared : 1.0) + cw.finish;
    const double start = cx.start > cw.start ? cx.start : cw.start, longest = tx > tw ? tx : tw;
    if (nx + nw <= slots) return start + longest;
    return start + ((double)nx * tx + (double)nw * tw) / (double)slots + 0.5 * longest;
}

double single_us(int64_t n, int64_t m, int64_t k, bool may_split, int cus) {
    return gemm_plan(n, m, k, 2, may_split ? (size_t)-1 : 0, cus).us;
}

// 0: two launches; else 1 + 3 * ix + iw over {small, wide, square}
int choose_pair(const PtjLinearBwd& p) {
    struct Entry { int64_t n, m, k; int mul, cus, choice; };
    static thread_local Entry table[32] = {};
    const int cus = num_cus(), mul = p.mul != nullptr;
    Entry& e = table[((uint64_t)p.n * 0x9E3779B97F4A7C15ull + (uint64_t)p.m * 0xC2B2AE3D27D4EB4Full + (uint64_t)p.k * 31 + mul) >> 40 & 31];
    if (e.n == p.n && e.m == p.m && e.k == p.k && e.mul == mul && e.cus == cus) return e.choice;
    double best = 0.95 * (single_us(p.n, p.k, p.m, !mul, cus) + single_us(p.m, p.k, p.n, true, cus));
    int choice = 0;
    for (int ix = 1; ix <= 3; ++ix)
        for (int iw = 1; iw <= 3; ++iw) {
            if ((ix == 3) != (iw == 3)) continue;
            const double us = pair_us(p, ix, iw, cus);
            if (us < best) {
                best = us;
                choice = 1 + 3 * (ix - 1) + (iw - 1);
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
    if (dtype == PTJ_BF16 && n < (1 << 20) && m < (1 << 20) && k < (1 << 20)) {
        GemmArgs gx = args_of(p.d, p.w, p.dx, n, k, m, m, 1), gw = args_of(p.d, p.x, p.dw, m, k, n, 1, m);
        gx.mul = p.mul; gx.mul_rs = k; gx.colpart = p.colpart;
        if (p.mul) gx.vec_out = gx.vec_out && ptj_aligned16(p.mul);
        const bool ok = pick_mode<bf16>(gx.a, gx.a_row, gx.a_k) == KMAJOR && pick_mode<bf16>(gx.b, gx.b_row, gx.b_k) == MNMAJOR &&
                        pick_mode<bf16>(gw.a, gw.a_row, gw.a_k) == MNMAJOR && pick_mode<bf16>(gw.b, gw.b_row, gw.b_k) == MNMAJOR &&
                        gt_eligible(gx, KMAJOR, MNMAJOR) && gt_eligible(gw, MNMAJOR, MNMAJOR);
        const int choice = ok ? choose_pair(p) : 0;
        if (choice != 0) {
            const bool mul = p.mul != nullptr;
            int rc;
            switch (choice) {
                case 1: rc = launch_pair<PairSmall, PairSmall>(gx, gw, mul, st); break;
                case 2: rc = launch_pair<PairSmall, PairWide>(gx, gw, mul, st); break;
                case 4: rc = launch_pair<PairWide, PairSmall>(gx, gw, mul, st); break;
                case 5: rc = launch_pair<PairWide, PairWide>(gx, gw, mul, st); break;
                default: rc = launch_pair<PairSquare, PairSquare>(gx, gw, mul, st); break;
            }
            if (rc != PTJ_OK || !mul) return rc;
            if (!later->add(p.colpart, p.colsum, (n + 63) / 64, k, k))
                return ptj_set_error(PTJ_ERR_INVALID, "linear_bwd: too many pending sums");
            return PTJ_OK;
        }
    }
    int rc = ptj_gemm(p.d, p.x, p.dw, nullptr, m, k, n, 1, m, k, 1, k, PTJ_EPI_NONE, nullptr, 0, scratch, scratch_bytes, dtype, st);
    if (rc != PTJ_OK) return rc;
    if (p.mul)
        return ptj_gemm_mul_colsum_later(p.d, p.w, p.mul, p.dx, p.colsum, n, k, m, m, 1, k, 1, k, k, p.colpart,
                                         ptj_gemm_mul_colsum_workspace_bytes(n, k), scratch, scratch_bytes, dtype, later, st);
    return ptj_gemm(p.d, p.w, p.dx, nullptr, n, k, m, m, 1, k, 1, k, PTJ_EPI_NONE, nullptr, 0, scratch, scratch_bytes, dtype, st);
}
