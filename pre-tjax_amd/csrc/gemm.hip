// ptj_gemm: C = A.B (+bias) (gelu) for every operand layout; kernels and launch logic in gemm_core.h.  The bf16
// kernels are instantiated here, the fp32 ones in gemm_f32.hip (the two compile side by side).
#include "gemm_core.h"
#include "gemm_plan.h"
#include "internal.h"

namespace {

uint64_t plan_hash(int64_t n, int64_t m, int64_t k) {
    return ((uint64_t)n * 0x9E3779B97F4A7C15ull) ^ ((uint64_t)m * 0xC2B2AE3D27D4EB4Full) ^ ((uint64_t)k * 0x165667B19E3779F9ull);
}

// gemm_plan through a small per-thread table: a training loop asks for the same few dozen products again and again,
// and the estimate over all tile shapes and splits takes a microsecond.
GemmPlan cached_plan(int64_t n, int64_t m, int64_t k, int elt, size_t ws_bytes, int loose, int kernels = ANY_KERNEL, bool later = false,
                     bool along = false) {
    struct Entry { int64_t n, m, k; size_t ws; int elt, cus, loose, kernels, later, along; GemmPlan plan; };
    constexpr int ENTRIES = 128;
    static thread_local Entry table[ENTRIES] = {};
    const int cus = num_cus();
    const uint64_t kind = ((((uint64_t)loose * 2 + kernels) * 2 + later) * 2 + along) * 2 + (elt == 2);
    const uint64_t h = plan_hash(n, m, k) ^ (((uint64_t)ws_bytes * 64 + kind) * 0xD6E8FEB86659FD93ull);
    Entry& e = table[(h >> 40) % ENTRIES];
    if (e.n != n || e.m != m || e.k != k || e.ws != ws_bytes || e.elt != elt || e.cus != cus || e.loose != loose ||
        e.kernels != kernels || e.later != later || e.along != along)
        e = {n, m, k, ws_bytes, elt, cus, loose, kernels, later, along, gemm_plan(n, m, k, elt, ws_bytes, cus, loose, kernels, 0, later, along)};
    return e.plan;
}

// ptj_gemm.  `later`: a K split of the tile kernels leaves its partial sums to the caller, who finds them there.
int gemm_any(const void* a, const void* b, void* c, const void* bias, int64_t n, int64_t m, int64_t k, int64_t a_rs, int64_t a_cs,
             int64_t b_rs, int64_t b_cs, int64_t c_rs, int epilogue, void* c_pre, int64_t c_pre_rs, void* workspace,
             size_t workspace_bytes, int dtype, void* stream, PtjPartialProduct* later) {
    PTJ_CHECK_ARG(n >= 0 && m >= 0 && k >= 0, "gemm: negative dimension");
    PTJ_CHECK_ARG(n < (1ll << 31) && m < (1ll << 31) && k < (1ll << 31), "gemm: dimension exceeds 31 bits");
    PTJ_CHECK_ARG(epilogue >= PTJ_EPI_NONE && epilogue <= PTJ_EPI_BIAS_NORM, "gemm: unknown epilogue %d", epilogue);
    const bool norm = epilogue == PTJ_EPI_BIAS_NORM;
    if (norm) epilogue = PTJ_EPI_BIAS;
    PTJ_CHECK_ARG(epilogue != PTJ_EPI_BIAS_GELU_DERIV || c_pre, "gemm: the derivative epilogue needs its second output");
    PTJ_CHECK_ARG(epilogue == PTJ_EPI_NONE || epilogue == PTJ_EPI_ACCUMULATE || bias, "gemm: epilogue %d needs a bias", epilogue);
    PTJ_CHECK_ARG(epilogue != PTJ_EPI_ACCUMULATE || (!bias && !c_pre && dtype == PTJ_BF16),
                  "gemm: the accumulating epilogue takes no bias and no second output, 2-byte storage only");
    PTJ_CHECK_ARG(dtype == PTJ_F32 || dtype == PTJ_BF16, "gemm: unknown dtype %d", dtype);
    if (n == 0 || m == 0) return PTJ_OK;
    PTJ_CHECK_ARG(c && (k == 0 || (a && b)), "gemm: null pointer");
    PTJ_CHECK_ARG(c_rs >= m, "gemm: c row stride %lld < m %lld", (long long)c_rs, (long long)m);
    PTJ_CHECK_ARG(!c_pre || ((epilogue == PTJ_EPI_BIAS_GELU || epilogue == PTJ_EPI_BIAS_GELU_DERIV) && c_pre_rs >= m),
                  "gemm: c_pre needs a bias+GELU epilogue and a row stride >= m");
    const int elt = dtype == PTJ_BF16 ? 2 : 4;
    const int bk = BKB / elt;
    GemmArgs g;
    g.a = a; g.b = b; g.c = c; g.bias = bias;
    g.n = (int)n; g.m = (int)m; g.k = (int)k;
    g.a_row = a_rs; g.a_k = a_cs;
    g.b_row = b_cs; g.b_k = b_rs;
    g.c_rs = c_rs;
    g.c_aux = c_pre;
    g.c_aux_rs = c_pre_rs;
    g.epilogue = epilogue;
    g.mul = nullptr; g.mul_rs = 0; g.colpart = nullptr;
    g.leave_partials = 0;
    int am = elt == 2 ? pick_mode<bf16>(a, a_rs, a_cs) : pick_mode<float>(a, a_rs, a_cs);
    int bm = elt == 2 ? pick_mode<bf16>(b, b_cs, b_rs) : pick_mode<float>(b, b_cs, b_rs);
    const bool ragged = am == GENERIC || bm == GENERIC;
    if (ragged) {
        am = stride_mode(a_rs, a_cs);
        bm = stride_mode(b_cs, b_rs);
    }
    const int64_t v = 16 / elt;
    bool outputs_aligned = ptj_aligned16(c) && c_rs % v == 0;
    if (c_pre) outputs_aligned = outputs_aligned && ptj_aligned16(c_pre) && c_pre_rs % v == 0;
    if (bias) outputs_aligned = outputs_aligned && (reinterpret_cast<uintptr_t>(bias) % (4 * (size_t)elt)) == 0;
    const bool aligned_ws = workspace && ptj_aligned16(workspace);
    const int loose = ragged ? LOOSE_OPERAND : outputs_aligned ? ALIGNED : LOOSE_OUTPUT;
    // (whether this caller leaves the partial sums or adds them up does not count: the bits of a product depend on its plan)
    const bool left = norm && !ragged && m % 4 == 0;
    GemmPlan plan = {-1, 1, 0, 0, 1, 0, 0.0};
    if (epilogue == PTJ_EPI_ACCUMULATE) {
        // only the ring kernels start their accumulators from the stored C
        if (ragged || (am == KMAJOR && bm == KMAJOR) || !outputs_aligned || k == 0 || k % 64 != 0 || !ring_eligible(g, am, bm))
            return ptj_set_error(PTJ_ERR_INVALID, "gemm: the accumulating epilogue needs a transposed 16-byte aligned "
                                 "operand layout, k a multiple of 64 and vector-aligned C");
        plan = cached_plan(n, m, k, elt, 0, loose, RING_ONLY);
    } else if (gt_eligible(g, am, bm, ragged ? 8 : 1)) {
        plan = cached_plan(n, m, k, elt, aligned_ws ? workspace_bytes : 0, loose, ANY_KERNEL, left, am == KMAJOR && bm == KMAJOR);
    } else if (elt == 2 && !ragged && ring_eligible(g, am, bm)) {
        plan = cached_plan(n, m, k, elt, aligned_ws ? workspace_bytes : 0, loose, RING_ONLY, left);
    }
    int splits = plan.splits;
    int64_t kps = plan.cfg >= 0 ? plan.kps : k;
    g.tail_first = plan.tail_first; g.tail_splits = plan.tail_splits; g.tail_kps = plan.tail_kps;
    if (plan.cfg < 0) {
        splits = workspace ? choose_splits(n, m, k, elt, workspace_bytes) : 1;
        if (splits > 1) {
            kps = ((k + splits - 1) / splits + bk - 1) / bk * bk;
            splits = (int)((k + kps - 1) / kps);
        } else if (aligned_ws) {
            choose_tail_split(n, m, k, elt, workspace_bytes, &g.tail_first, &g.tail_splits, &g.tail_kps);
        }
    }
    if (kps < 1) kps = bk;  // k == 0: one empty pass writes bias / zeros
    g.k_per_split = (int)kps;
    g.splits = splits;
    g.vec_out = outputs_aligned && (splits <= 1 || (ptj_aligned16(workspace) && m % 4 == 0)) ? 1 : 0;
    const size_t planes = plan.cfg == PLANES_CFG ? gp_planes_bytes(n, m, k) : 0;
    g.partial = (splits > 1 || g.tail_splits > 1) ? (float*)((char*)workspace + planes) : nullptr;
    hipStream_t st = (hipStream_t)stream;
    if (plan.cfg >= 0) {
        g.stream = 0;
        g.leave_partials = later != nullptr && !ragged && splits > 1 && m % 4 == 0;
        if (g.leave_partials) {
            later->part = g.partial;
            later->splits = splits;
        }
        if (plan.cfg == PLANES_CFG) return ptj_gemm_detail::gemm_planes_launch(g, (char*)workspace, st);
        if (plan.cfg == RING_FIRST) return ptj_gemm_detail::gemm_ring_full_launch(g, am, bm, st);
        if (plan.cfg == RING_FIRST + 1) return ptj_gemm_detail::gemm_ring_narrow_launch(g, am, bm, st);
        if (ragged && dtype == PTJ_BF16)
            return ptj_gemm_detail::gemm_ragged_launch_bf16(g, plan.cfg - RAGGED_FIRST[0], am, bm, st);
        return dtype == PTJ_F32 ? ptj_gemm_detail::gemm_tile_launch_f32(g, plan.cfg, am, bm, st)
                                : ptj_gemm_detail::gemm_tile_launch_bf16(g, plan.cfg, am, bm, st);
    }
    // streamed tiles need whole, evenly many K panels (the two-step loop body) and vector-aligned outputs
    g.stream = (splits == 1 && g.vec_out && k >= 2 * bk && k % bk == 0) ? 1 : 0;
    return dtype == PTJ_F32 ? ptj_gemm_detail::launch_plain_f32(g, splits, st) : gemm_impl<bf16>(g, splits, st);
}

}  // namespace

extern "C" {

// Every wrapper asks before it launches, so the answers are kept, per thread: worked out again for each product they took 5-10 us
// (some dozen plans), looked up 0.2.
size_t ptj_gemm_workspace_bytes(int64_t n, int64_t m, int64_t k, int dtype) {
    if (n <= 0 || m <= 0 || k <= 0) return 0;
    struct Entry { int64_t n, m, k; int elt, cus; size_t need; };
    constexpr int ENTRIES = 128;
    static thread_local Entry table[ENTRIES] = {};
    const int elt = dtype == PTJ_BF16 ? 2 : 4, cus = num_cus();
    Entry& e = table[(plan_hash(n, m, k) + (uint64_t)elt * 0xD6E8FEB86659FD93ull) >> 40 & (ENTRIES - 1)];
    if (e.n == n && e.m == m && e.k == k && e.elt == elt && e.cus == cus) return e.need;
    // which kernels run depends on the operands' strides and alignment as well: enough for any
    const int s = choose_splits(n, m, k, elt, (size_t)-1);
    int first, ts, tkps;
    size_t need = s > 1 ? (size_t)s * n * m * sizeof(float) : choose_tail_split(n, m, k, elt, (size_t)-1, &first, &ts, &tkps);
    for (const int loose : {ALIGNED, LOOSE_OUTPUT, LOOSE_OPERAND})
        for (const int kernels : {ANY_KERNEL, RING_ONLY})
            for (const int sums : {0, 1, 2}) {                                  // neither, left to the next norm, operands along
                if (elt != 2 && (sums || kernels == RING_ONLY)) continue;       // bf16 alone tells these apart
                const size_t bytes = gp_workspace_bytes(gemm_plan(n, m, k, elt, (size_t)-1, cus, loose, kernels, 0, sums == 1, sums == 2), n, m, k);
                if (bytes > need) need = bytes;
            }
    e = {n, m, k, elt, cus, need};
    return need;
}

int ptj_gemm(const void* a, const void* b, void* c, const void* bias, int64_t n, int64_t m, int64_t k, int64_t a_rs,
             int64_t a_cs, int64_t b_rs, int64_t b_cs, int64_t c_rs, int epilogue, void* c_pre, int64_t c_pre_rs,
             void* workspace, size_t workspace_bytes, int dtype, void* stream) {
    return gemm_any(a, b, c, bias, n, m, k, a_rs, a_cs, b_rs, b_cs, c_rs, epilogue, c_pre, c_pre_rs, workspace, workspace_bytes,
                    dtype, stream, nullptr);
}

}  // extern "C"

int ptj_gemm_partial(const void* a, const void* b, void* c, const void* bias, int64_t n, int64_t m, int64_t k, int64_t a_rs,
                     int64_t a_cs, int64_t b_rs, int64_t b_cs, void* workspace, size_t workspace_bytes, int dtype,
                     hipStream_t st, PtjPartialProduct* out) {
    *out = {c, nullptr, 0, bias};
    return gemm_any(a, b, c, bias, n, m, k, a_rs, a_cs, b_rs, b_cs, m, bias ? PTJ_EPI_BIAS_NORM : PTJ_EPI_NONE, nullptr, 0, workspace,
                    workspace_bytes, dtype, (void*)st, out);
}
