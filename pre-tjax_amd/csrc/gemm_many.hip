// ptj_gemm_many: several products that do not depend on each other, as one launch of 128x128 tiles where each alone would leave CUs
// idle: dW1, dW2 and dX of a feed-forward block of 3001 tokens have 144 tiles each, 56 % of a round, and 1.7 rounds together.  The
// longest tiles go first.  One launch or one product after the other is chosen by estimate (together): the time of all tiles on CUs
// that take the next one as they end one, against the estimates of gemm_plan.  Feed-forward block, forward and backward, 768 wide, three
// launches / chosen, us: bf16 777 tokens 97.8 / 92.1, 1500 140.3 / 124.8, 3001 185.5 / 167.2, 4096 205.9 / 190.1, 8192 379 / 353, 11000 478 / 464,
// 16384 (apart; together 648) 608; fp32 64 (apart; together 155) 102, 1500 416 / 389, 3001 720 / 689, 4096 872 / 857, 6000 1324 / 1317, 1000
// and 8192 apart; bf16 3001 tokens 512 wide 119 / 106, 1600 wide 504 / 491; nowhere slower by more than what two runs differ by.
#include "gemm_tile_launch.h"
#include "gemm_plan.h"

#include <string.h>

namespace {

constexpr int MANY = 4;      // products of a launch
struct ManyArgs {
    GemmArgs g[MANY];
    int first[MANY + 1];     // tiles in front of each product
    int modes[MANY];         // operand layouts
    int chain[MANY];         // fp32: gemm_split.h
    int count;
};

template <typename T, typename C>
constexpr int many_smem() {
    if constexpr (sizeof(T) == 2) return C::SMEM;
    else return gs_chain_smem<C>;
}
// One tile of one of the products; operands along the contraction and across it (dX), or both across it (dW)
template <typename T, typename C>
__global__ __launch_bounds__(C::THREADS, C::WAVES_EU) void gemm_many_kernel(const ManyArgs a) {
    __shared__ __attribute__((aligned(1024))) char smem[many_smem<T, C>()];
    int i = 0;
#pragma unroll
    for (int j = 1; j < MANY; ++j) i += j < a.count && (int)blockIdx.x >= a.first[j];
    const GemmArgs& g = a.g[i];
    const int pid = (int)blockIdx.x - a.first[i];
    auto tile = [&](auto am, auto bm) __attribute__((always_inline)) {
        if constexpr (sizeof(T) == 2) {
            gt_tile<T, am, bm, C, false>(g, pid, smem);
        } else {
            int tile_m, tile_n, z;
            gt_item(g, pid, (g.n + C::TBM - 1) / C::TBM, (g.m + C::TBN - 1) / C::TBN, tile_m, tile_n, z);
            gs_tile<am, bm, C, false, true>(g, tile_m, tile_n, z, smem, a.chain[i]);
        }
    };
    constexpr std::integral_constant<int, KMAJOR> K{};
    constexpr std::integral_constant<int, MNMAJOR> M{};
    if (a.modes[i] == KMAJOR * 3 + MNMAJOR) tile(K, M);
    else tile(M, M);
}

template <typename T, typename C>
int launch_many(const ManyArgs& a, hipStream_t st) {
    hipLaunchKernelGGL((gemm_many_kernel<T, C>), dim3((unsigned)a.first[a.count]), dim3(C::THREADS), 0, st, a);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

// fp32: a step with the totals of gs_tile beside it, relative to one without (3001 to 8192 rows: 1.04 to 1.06)
constexpr double MANY_CHAINS = 1.05;

// Time of the tiles of all products, in the order of the grid, on CUs that take the next one as they end one
double makespan(const ManyArgs& a, const TileCost& c, int cus, double slower) {
    struct Group { double at; int64_t count; };           // CUs that are free from then on, in order of time
    Group free[MANY + 2] = {{0.0, cus}};                  // (a product takes whole groups and part of one more)
    int groups = 1;
    const double step = gp_step_us(c, a.first[a.count], cus) * slower;
    double last = 0.0;
    for (int i = 0; i < a.count; ++i) {
        const double tile = (double)gp_ceil(a.g[i].k, c.bkt) * step + c.finish;
        for (int64_t left = a.first[i + 1] - a.first[i]; left > 0;) {
            const Group g = {free[0].at + tile, free[0].count < left ? free[0].count : left};
            int at = 0;
            if (g.count == free[0].count) {
                for (; at + 1 < groups && free[at + 1].at <= g.at; ++at) free[at] = free[at + 1];
            } else {
                free[0].count -= g.count;
                for (at = groups++; free[at - 1].at > g.at; --at) free[at] = free[at - 1];
            }
            free[at] = g;
            last = g.at > last ? g.at : last;
            left -= g.count;
        }
    }
    return c.start + last;
}

// Whether one launch is estimated to be faster, and its chains of additions; kept for the sizes asked for last
bool together(ManyArgs& a, int elt) {
    struct Key { int n[MANY], m[MANY], k[MANY], count, elt, cus; };
    static thread_local Key last = {};
    static thread_local bool answer = false;
    static thread_local int chain[MANY] = {};
    const int cus = num_cus();
    Key key = {};
    key.count = a.count; key.elt = elt; key.cus = cus;
    for (int i = 0; i < a.count; ++i) { key.n[i] = a.g[i].n; key.m[i] = a.g[i].m; key.k[i] = a.g[i].k; }
    if (memcmp(&key, &last, sizeof(key)) != 0) {
        double apart = 0.0;
        for (int i = 0; i < a.count; ++i) {
            const GemmPlan p = gemm_plan(a.g[i].n, a.g[i].m, a.g[i].k, elt, (size_t)-1, cus);
            apart += p.us;
            chain[i] = gs_chain(p.kps, a.g[i].k);
        }
        // (fp32: launches that follow each other do not wait for their start twice: 1000 rows apart 119 us, estimated 129, together 129)
        answer = elt == 2 ? makespan(a, GT_COST[0][3], cus, 1.0) < apart
                          : makespan(a, GT_COST[1][4], cus, MANY_CHAINS) < apart - (a.count - 1) * GT_COST[1][4].start;
        last = key;
    }
    memcpy(a.chain, chain, sizeof(chain));
    return answer;
}

}  // namespace

extern "C" {

size_t ptj_gemm_many_workspace_bytes(const ptj_product* p, int64_t count, int dtype) {
    size_t need = 0;
    for (int64_t i = 0; p && i < count; ++i) {
        const size_t w = ptj_gemm_workspace_bytes(p[i].n, p[i].m, p[i].k, dtype);
        need = w > need ? w : need;
    }
    return need;
}

int ptj_gemm_many(const ptj_product* p, int64_t count, void* workspace, size_t workspace_bytes, int dtype, void* stream) {
    PTJ_CHECK_ARG(count >= 0 && (count == 0 || p), "gemm_many: null pointer");
    PTJ_CHECK_ARG(dtype == PTJ_F32 || dtype == PTJ_BF16, "gemm_many: unknown dtype %d", dtype);
    const int elt = dtype == PTJ_BF16 ? 2 : 4;
    const int64_t most = 1 << 20;
    ManyArgs a = {};
    bool ok = count >= 2 && count <= MANY;
    int order[MANY] = {};                                  // the longest tiles first
    for (int i = 0; ok && i < count; ++i) {
        int at = i;
        for (; at > 0 && p[order[at - 1]].k < p[i].k; --at) order[at] = order[at - 1];
        order[at] = i;
    }
    for (int64_t i = 0; ok && i < count; ++i) {
        const ptj_product& q = p[order[i]];
        GemmArgs& g = a.g[i];
        ok = q.n > 0 && q.m > 0 && q.k > 0 && q.n < most && q.m < most && q.k < most && q.a && q.b && q.c && q.c_rs >= q.m;
        if (!ok) break;
        g.a = q.a; g.b = q.b; g.c = q.c;
        g.n = (int)q.n; g.m = (int)q.m; g.k = g.k_per_split = (int)q.k;
        g.a_row = q.a_rs; g.a_k = q.a_cs;
        g.b_row = q.b_cs; g.b_k = q.b_rs;
        g.c_rs = q.c_rs;
        g.splits = g.tail_splits = 1;
        g.vec_out = ptj_aligned16(q.c) && q.c_rs % (16 / elt) == 0;
        g.epilogue = PTJ_EPI_NONE;
        const int am = elt == 2 ? pick_mode<bf16>(q.a, g.a_row, g.a_k) : pick_mode<float>(q.a, g.a_row, g.a_k);
        const int bm = elt == 2 ? pick_mode<bf16>(q.b, g.b_row, g.b_k) : pick_mode<float>(q.b, g.b_row, g.b_k);
        a.modes[i] = am * 3 + bm;
        ok = bm == MNMAJOR && am != GENERIC && gt_eligible(g, am, bm);
        a.first[i + 1] = a.first[i] + ((g.n + 127) / 128) * ((g.m + 127) / 128);
    }
    a.count = (int)count;
    if (ok && together(a, elt))
        return elt == 2 ? launch_many<bf16, GtSquare>(a, (hipStream_t)stream) : launch_many<float, GsSquare>(a, (hipStream_t)stream);
    for (int64_t i = 0; i < count; ++i) {
        const ptj_product& q = p[i];
        const int rc = ptj_gemm(q.a, q.b, q.c, nullptr, q.n, q.m, q.k, q.a_rs, q.a_cs, q.b_rs, q.b_cs, q.c_rs, PTJ_EPI_NONE, nullptr, 0,
                                workspace, workspace_bytes, dtype, stream);
        if (rc != PTJ_OK) return rc;
    }
    return PTJ_OK;
}

}  // extern "C"
