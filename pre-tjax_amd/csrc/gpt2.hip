// The transformer stack between the token ids and the final LayerNorm's output, forward and backward, as one
// call each: the sequence of launches that model_triton.py strings together per layer (:2214-2223, :2291-2299,
// :2334-2351, :2583-2593), issued from native code.
//
// Nothing here computes: every step is an entry point of the C ABI or its twin in internal.h (attention on keep bits that
// one launch makes for all layers, the two products of a linear layer's backward side by side, the second stages of all
// column sums in one launch at the end).  What this file is for is the host's time.  A step of a 12-layer model is about 300
// launches; issued one wrapper call at a time (allocation, pointer and stride queries, argument conversion) they
// took 14 us each, 1.6 ms for a forward of 64 tokens and 5.1 ms for a training step of 512, several times what
// the kernels need.  Activations live in one buffer laid out by `Layout`, temporaries in the workspace.
#include "common.h"
#include "internal.h"

#include <math.h>
#include <string.h>
#include <initializer_list>

namespace {

constexpr int64_t ALIGN = 256;
inline int64_t up(int64_t x) { return (x + ALIGN - 1) / ALIGN * ALIGN; }

// Byte offsets inside the activation buffer.
struct Layout {
    int64_t x0, h0, keepbits, first_layer;                      // embedding output, its norm, keep-bit lines
    int64_t qkv, o, ms, ls, xmid, h2, f1, g1, keep1, keep2, xout, hnext;   // relative to a layer's block
    int64_t layer_stride, total;
};

inline int elt_of(const ptj_gpt2_shape& s) { return s.dtype == PTJ_BF16 ? 2 : 4; }
inline bool has_keep(const ptj_gpt2_shape& s) { return s.train && s.dim % 8 == 0; }

// keep: all layers' activations stay (for the backward); else one block serves every layer in turn.
Layout make_layout(const ptj_gpt2_shape& s, bool keep) {
    const int64_t N = s.batch * s.seq, e = elt_of(s), nd = up(N * s.dim * e), nf = up(N * s.ffn * e);
    const int64_t stat = up(s.batch * s.heads * s.seq * 4), kb = has_keep(s) ? up(N * s.dim / 8) : 0;
    Layout l = {};
    int64_t at = 0;
    auto take = [&](int64_t bytes) { const int64_t o = at; at += bytes; return o; };
    l.x0 = take(nd);
    l.h0 = take(nd);
    l.keepbits = take(s.train ? up(s.layers * s.batch * s.heads * ptj_attn_bitwords(s.seq) * 4) : 0);
    l.first_layer = at;
    at = 0;
    l.qkv = take(up(N * 3 * s.dim * e));
    l.o = take(nd);
    l.ms = take(stat);
    l.ls = take(stat);
    l.xmid = take(nd);
    l.h2 = take(nd);
    l.f1 = take(keep ? nf : 0);
    l.g1 = take(nf);
    l.keep1 = take(kb);
    l.keep2 = take(kb);
    l.xout = take(nd);
    l.hnext = take(nd);
    l.layer_stride = keep ? at : 0;
    l.total = l.first_layer + (keep ? s.layers : 1) * at;
    return l;
}

size_t max2(size_t a, size_t b) { return a > b ? a : b; }

size_t gemm_scratch(const ptj_gpt2_shape& s, bool backward) {
    const int64_t N = s.batch * s.seq, D = s.dim, F = s.ffn;
    const int dt = (int)s.dtype;
    size_t w = 0;
    auto want = [&](int64_t n, int64_t m, int64_t k) { w = max2(w, ptj_gemm_workspace_bytes(n, m, k, dt)); };
    want(N, 3 * D, D); want(N, D, D); want(N, F, D); want(N, D, F);
    if (backward) {
        want(D, F, N); want(F, D, N); want(D, D, N); want(3 * D, D, N); want(N, D, 3 * D);
    }
    return w;
}

// Temporaries of the two directions in front of the scratch area that the single steps share.
struct Temps {
    int64_t t1, dxm, dx[2], delta, ln_parts, mul_parts, scratch;   // partial rows: one slot per sum
    int64_t group;                            // blocks whose weight gradients share a launch (0: each with its dX)
    int64_t df1, dqkv, dm, block;             // what a block's weight gradients read, and from one block's to the next
    int64_t dr, dr_slots;                     // the gradient that enters a block, dropped
    size_t ln_slot, mul_slot, scratch_bytes, total;
};

// The weight gradients of a block: d^T.x with d [tokens, outputs], x [tokens, inputs]
enum { W_FFN2, W_FFN1, W_OUT, W_QKV };
PtjGradGroup grad_group(const ptj_gpt2_shape& s, int64_t blocks) {
    PtjGradGroup g = {};
    g.k = (int)(s.batch * s.seq);
    g.blocks = (int)blocks;
    const int64_t D = s.dim, F = s.ffn, n[4] = {D, F, D, 3 * D}, m[4] = {F, D, D, D};
    for (int i = 0; i < PtjGradGroup::KINDS; ++i) {
        g.n[i] = (int)n[i];
        g.m[i] = (int)m[i];
    }
    return g;
}
// How many blocks' weight gradients are formed in one launch (gemm_group.hip), 0: none.  A single block stays with the pairs: a round of
// its tiles takes a width of 1024.
int64_t grad_group_blocks(const ptj_gpt2_shape& s) {
    const int64_t N = s.batch * s.seq, D = s.dim, F = s.ffn, most = 1 << 20;
    if (s.layers < 2 || N >= most || F >= most || 3 * D >= most || F % 8 != 0) return 0;
    return ptj_weight_grads_blocks(grad_group(s, 1), s.layers, (int)s.dtype);
}

// `together`: weight gradients in groups where grad_group_blocks says so
Temps make_temps(const ptj_gpt2_shape& s, bool backward, bool together = true) {
    // the split counts behind the scratch size take some twenty estimates: kept for the shape asked for last
    static thread_local ptj_gpt2_shape last[3] = {};
    static thread_local Temps kept[3] = {};
    const int dir = backward ? 1 + together : 0;
    if (memcmp(&last[dir], &s, sizeof(s)) == 0) return kept[dir];
    const int64_t N = s.batch * s.seq, e = elt_of(s), nd = up(N * s.dim * e);
    Temps t = {};
    int64_t at = 0;
    auto take = [&](int64_t bytes) { const int64_t o = at; at += bytes; return o; };
    t.t1 = take(nd);
    if (backward) {
        t.dxm = take(nd);
        for (int i = 0; i < 2; ++i) t.dx[i] = take(nd);
        t.group = together ? grad_group_blocks(s) : 0;
        const int64_t first = at;
        t.df1 = take(up(N * s.ffn * e));
        t.dqkv = take(up(N * 3 * s.dim * e));
        t.dm = take(nd);
        t.block = at - first;
        if (t.group) take((t.group - 1) * t.block);
        t.dr_slots = t.group > 2 ? t.group : 2;      // (a block's is formed while the one before it is in use)
        t.dr = take(t.dr_slots * nd);
        t.delta = take(up(s.batch * s.heads * s.seq * 4));
        t.ln_slot = (size_t)up((int64_t)ptj_layernorm_bwd_parts_bytes(N, s.dim));
        t.mul_slot = (size_t)up((int64_t)ptj_gemm_mul_colsum_workspace_bytes(N, s.ffn));
        t.ln_parts = take((2 * s.layers + 1) * (int64_t)t.ln_slot);
        t.mul_parts = take(s.layers * (int64_t)t.mul_slot);
    }
    t.scratch = at;
    t.scratch_bytes = gemm_scratch(s, backward);
    t.total = (size_t)at + t.scratch_bytes;
    last[dir] = s;
    kept[dir] = t;
    return t;
}

int check_shape(const char* what, const ptj_gpt2_shape* s) {
    if (!s) return ptj_set_error(PTJ_ERR_INVALID, "%s: null shape", what);
    if (s->layers < 1 || s->batch < 1 || s->seq < 1 || s->dim < 1 || s->heads < 1 || s->ffn < 1 || s->vocab < 1)
        return ptj_set_error(PTJ_ERR_INVALID, "%s: sizes must be positive", what);
    if (s->dim != s->heads * 64)
        return ptj_set_error(PTJ_ERR_INVALID, "%s: head dimension 64 only (dim %lld, heads %lld)", what, (long long)s->dim,
                             (long long)s->heads);
    if (s->dtype != PTJ_F32 && s->dtype != PTJ_BF16)
        return ptj_set_error(PTJ_ERR_INVALID, "%s: unknown dtype %lld", what, (long long)s->dtype);
    return PTJ_OK;
}

enum { P_LN1G, P_LN1B, P_WQKV, P_WO, P_LN2G, P_LN2B, P_W1, P_B1, P_W2, P_B2, P_BLOCK };
constexpr int P_FIRST = 3;   // table, its bias, positions

// Whether these entries of every block are there.  A missing one is refused before the first launch: the launches that several
// products share see no single call's checks.
bool all_given(const void* const* nest, int64_t layers, std::initializer_list<int> entries) {
    for (int64_t i = 0; i < layers; ++i)
        for (const int p : entries)
            if (!nest[P_FIRST + i * P_BLOCK + p]) return false;
    return true;
}

// Dropout decisions recorded by the forward (one byte per 8 columns) for the LayerNorm backward.  The vector kernels do
// that only: fp32 norms off the 16-byte grid recompute the decisions, bf16 ones are refused as in the single calls.
bool keeps_bytes(const ptj_gpt2_shape& s, const void* const* params) {
    if (!has_keep(s) || s.dtype == PTJ_BF16) return has_keep(s);
    const void* const* fin = params + P_FIRST + s.layers * P_BLOCK;
    bool ok = ptj_aligned16(fin[0]) && ptj_aligned16(fin[1]);
    for (int64_t i = 0; i < s.layers; ++i) {
        const void* const* w = params + P_FIRST + i * P_BLOCK;
        for (const int p : {P_LN1G, P_LN1B, P_LN2G, P_LN2B}) ok = ok && ptj_aligned16(w[p]);
    }
    return ok;
}

#define STEP(CALL)                        \
    do {                                  \
        const int rc__ = (CALL);          \
        if (rc__ != PTJ_OK) return rc__;  \
    } while (0)

}  // namespace

extern "C" {

size_t ptj_gpt2_acts_bytes(const ptj_gpt2_shape* s, int keep) {
    return check_shape("gpt2_acts_bytes", s) == PTJ_OK ? (size_t)make_layout(*s, keep != 0).total : 0;
}

size_t ptj_gpt2_workspace_bytes(const ptj_gpt2_shape* s, int backward) {
    return check_shape("gpt2_workspace_bytes", s) == PTJ_OK ? make_temps(*s, backward != 0, backward != 2).total : 0;
}

int ptj_gpt2_fwd(const ptj_gpt2_shape* sp, const void* const* params, const int64_t* tokens, const uint32_t* mask,
                 const int64_t* seeds, void* acts, size_t acts_bytes, int keep, void* x_last, void* h, void* workspace,
                 size_t workspace_bytes, void* stream) {
    STEP(check_shape("gpt2_fwd", sp));
    const ptj_gpt2_shape& s = *sp;
    PTJ_CHECK_ARG(params && tokens && acts && x_last && h && (!s.train || seeds), "gpt2_fwd: null pointer");
    PTJ_CHECK_ARG(all_given(params, s.layers, {P_LN1G, P_LN1B, P_WQKV, P_WO, P_LN2G, P_LN2B, P_W1, P_B1, P_W2}) &&
                      params[P_FIRST + s.layers * P_BLOCK] && params[P_FIRST + s.layers * P_BLOCK + 1],
                  "gpt2_fwd: null parameter");
    const Layout l = make_layout(s, keep != 0);
    const Temps t = make_temps(s, false);
    if (acts_bytes < (size_t)l.total || !workspace || workspace_bytes < t.total)
        return ptj_set_error(PTJ_ERR_WORKSPACE, "gpt2_fwd: %zu / %zu bytes of activations / workspace, %zu / %zu needed",
                             acts_bytes, workspace_bytes, (size_t)l.total, t.total);
    const int64_t B = s.batch, T = s.seq, D = s.dim, H = s.heads, F = s.ffn, N = B * T;
    const int dt = (int)s.dtype, train = s.train != 0;
    hipStream_t st = (hipStream_t)stream;
    char* const base = (char*)acts;
    char* const ws = (char*)workspace;
    void* const scratch = ws + t.scratch;
    const size_t sb = t.scratch_bytes;
    uint32_t* const bits = train ? (uint32_t*)(base + l.keepbits) : nullptr;
    const int64_t bitlen = B * H * ptj_attn_bitwords(T);
    const void* const* fin = params + P_FIRST + s.layers * P_BLOCK;

    STEP(ptj_embed_fwd(params[0], params[2], tokens, base + l.x0, N, D, T, s.vocab, sqrtf((float)D), train, train ? seeds[0] : 0,
                       dt, stream));
    if (train) STEP(ptj_attn_keepbits_many(bits, s.layers, seeds + 1, 3, B * H, T, st));
    STEP(ptj_layernorm_fwd(base + l.x0, params[P_FIRST + P_LN1G], params[P_FIRST + P_LN1B], base + l.h0, N, D, D, D, dt, stream));
    const bool kb = keeps_bytes(s, params);
    const char* x = base + l.x0;
    const char* hn = base + l.h0;
    // few rows, and neither decisions nor activations to keep: each norm inside the product that reads it (gemm_norm.hip)
    bool inside = !keep && !train && ptj_norm_product_fits(N, D, F, dt, false) && ptj_aligned16(acts) && ptj_aligned16(workspace);
    for (int64_t i = P_FIRST; inside && i < P_FIRST + s.layers * P_BLOCK; ++i) inside = ptj_aligned16(params[i]);
    PtjNormProduct entry = {};         // the norm that enters a block, with the block's input
    for (int64_t i = 0; i < s.layers; ++i) {
        const void* const* w = params + P_FIRST + i * P_BLOCK;
        char* const a = base + l.first_layer + i * l.layer_stride;
        const bool last = i + 1 == s.layers;
        const int64_t s1 = train ? seeds[2 + 3 * i] : 0, s2 = train ? seeds[3 + 3 * i] : 0;
        if (entry.res) {
            entry.w = w[P_WQKV];
            entry.c = a + l.qkv;
            STEP(ptj_norm_product(entry, N, D, 3 * D, dt, st));
            entry.res = nullptr;
        } else {
            STEP(ptj_gemm(hn, w[P_WQKV], a + l.qkv, nullptr, N, 3 * D, D, D, 1, 1, D, 3 * D, PTJ_EPI_NONE, nullptr, 0, scratch, sb, dt,
                          stream));
        }
        STEP(ptj_attn_fwd_packed(a + l.qkv, mask, a + l.o, (float*)(a + l.ms), (float*)(a + l.ls), bits ? bits + i * bitlen : nullptr,
                                 B, H, T, train, dt, st));
        STEP(ptj_gemm(a + l.o, w[P_WO], ws + t.t1, nullptr, N, D, D, D, 1, 1, D, D, PTJ_EPI_NONE, nullptr, 0, scratch, sb, dt, stream));
        if (inside) {
            STEP(ptj_norm_product({{ws + t.t1, nullptr, 0, nullptr}, x, w[P_LN2G], w[P_LN2B], w[P_W1], w[P_B1], a + l.xmid, a + l.g1, 1}, N, D, F,
                                  dt, st));
        } else {
            STEP(ptj_dropout_add_layernorm_of({ws + t.t1, nullptr, 0, nullptr}, x, w[P_LN2G], w[P_LN2B], a + l.xmid, a + l.h2,
                                              kb ? a + l.keep1 : nullptr, N, D, train, s1, dt, st));
            STEP(ptj_gemm(a + l.h2, w[P_W1], a + l.g1, w[P_B1], N, F, D, D, 1, 1, D, F,
                          keep ? PTJ_EPI_BIAS_GELU_DERIV : PTJ_EPI_BIAS_GELU, keep ? a + l.f1 : nullptr, keep ? F : 0, scratch, sb, dt,
                          stream));
        }
        char* const xo = last ? (char*)x_last : a + l.xout;
        char* const ho = last ? (char*)h : a + l.hnext;
        const void* const* nx = last ? fin : w + P_BLOCK;   // the norm that reads this block's output
        // a K split's partial sums are added up by the norm, which reads them as vectors
        PtjPartialProduct f2 = {ws + t.t1, nullptr, 0, nullptr};
        bool vectors = true;
        for (const void* p : {w[P_B2], nx[0], nx[1], (const void*)xo, (const void*)ho}) vectors = vectors && ptj_aligned16(p);
        if (vectors)
            STEP(ptj_gemm_partial(a + l.g1, w[P_W2], ws + t.t1, w[P_B2], N, D, F, F, 1, 1, F, scratch, sb, dt, st, &f2));
        else
            STEP(ptj_gemm(a + l.g1, w[P_W2], ws + t.t1, w[P_B2], N, D, F, F, 1, 1, F, D, PTJ_EPI_BIAS_NORM, nullptr, 0, scratch, sb,
                          dt, stream));
        if (inside && !last && ptj_norm_product_fits(N, D, 3 * D, dt, f2.part != nullptr)) entry = {f2, a + l.xmid, nx[0], nx[1], nullptr, nullptr, xo, nullptr, 0};
        else
            STEP(ptj_dropout_add_layernorm_of(f2, a + l.xmid, nx[0], nx[1], xo, ho, kb ? a + l.keep2 : nullptr, N, D, train, s2, dt,
                                          st));
        x = xo;
        hn = ho;
    }
    return PTJ_OK;
}

int ptj_gpt2_bwd(const ptj_gpt2_shape* sp, const void* const* params, const uint32_t* mask, const int64_t* seeds,
                 const void* acts, size_t acts_bytes, const void* x_last, const void* dh, void* const* grads, void* demb,
                 void* workspace, size_t workspace_bytes, void* stream) {
    STEP(check_shape("gpt2_bwd", sp));
    const ptj_gpt2_shape& s = *sp;
    PTJ_CHECK_ARG(params && acts && x_last && dh && grads && demb && (!s.train || seeds), "gpt2_bwd: null pointer");
    PTJ_CHECK_ARG(all_given(params, s.layers, {P_LN1G, P_WQKV, P_WO, P_LN2G, P_W1, P_W2}) && params[P_FIRST + s.layers * P_BLOCK],
                  "gpt2_bwd: null parameter");
    PTJ_CHECK_ARG(all_given(grads, s.layers, {P_WQKV, P_WO, P_W1, P_B1, P_W2}), "gpt2_bwd: null gradient of a weight or of the first bias");
    const Layout l = make_layout(s, true);
    Temps t = make_temps(s, true);
    bool aligned = ptj_aligned16(acts) && ptj_aligned16(workspace);
    for (int64_t i = 0; i < s.layers; ++i)
        for (const int p : {P_W2, P_W1, P_WO, P_WQKV}) aligned = aligned && ptj_aligned16(grads[P_FIRST + i * P_BLOCK + p]);
    if (t.group && (!aligned || workspace_bytes < t.total)) t = make_temps(s, true, false);   // (a workspace for one block's at a time will do)
    if (acts_bytes < (size_t)l.total || !workspace || workspace_bytes < t.total)
        return ptj_set_error(PTJ_ERR_WORKSPACE, "gpt2_bwd: %zu / %zu bytes of activations / workspace, %zu / %zu needed",
                             acts_bytes, workspace_bytes, (size_t)l.total, t.total);
    const int64_t B = s.batch, T = s.seq, D = s.dim, H = s.heads, F = s.ffn, N = B * T;
    const int dt = (int)s.dtype, train = s.train != 0;
    hipStream_t st = (hipStream_t)stream;
    const char* const base = (const char*)acts;
    char* const ws = (char*)workspace;
    void* const scratch = ws + t.scratch;
    const size_t sb = t.scratch_bytes;
    const uint32_t* const bits = train ? (const uint32_t*)(base + l.keepbits) : nullptr;
    const int64_t bitlen = B * H * ptj_attn_bitwords(T);
    const int64_t L = s.layers;
    const bool kb = keeps_bytes(s, params);
    const void* const* fin = params + P_FIRST + L * P_BLOCK;
    void* const* gfin = grads + P_FIRST + L * P_BLOCK;
    auto block = [&](int64_t i) { return base + l.first_layer + i * l.layer_stride; };
    auto seed = [&](int64_t i) { return train ? seeds[i] : (int64_t)0; };

    // Every dropout backward acts on a gradient that a LayerNorm backward has just produced, so each of those also
    // writes the dropped copy its consumer needs, and the column sums that are the bias gradient behind it.
    // The second stages of all column sums wait in `sums` for one launch at the end (beyond some 80 layers: several).
    PtjPartialSums sums;
    auto ln_bwd = [&](int64_t slot, const void* dy, const void* x, const void* const* gb, const void* res, void* dx, void* const* dgb,
                      void* dropped, void* dropped_sum, int64_t sd, const void* keep) {
        if (sums.count + 8 > PtjPartialSums::MAX) {
            STEP(ptj_partial_sums(sums, dt, st));
            sums.count = 0;
        }
        return ptj_layernorm_bwd_later(dy, x, gb[0], res, dx, dgb[0], dgb[1], dropped, dropped_sum, train, sd, keep,
                                       ws + t.ln_parts + slot * (int64_t)t.ln_slot, t.ln_slot, N, D, dt, &sums, st);
    };
    auto entering = [&](int64_t i) { return ws + t.dr + i % t.dr_slots * up(N * D * elt_of(s)); };
    PtjGradGroup group = grad_group(s, 0);
    int cur = 0;
    STEP(ln_bwd(2 * L, dh, x_last, fin, nullptr, ws + t.dx[0], gfin, entering(L - 1), grads[P_FIRST + (L - 1) * P_BLOCK + P_B2],
                seed(3 * L), kb ? block(L - 1) + l.keep2 : nullptr));
    for (int64_t i = L - 1; i >= 0; --i) {
        const void* const* w = params + P_FIRST + i * P_BLOCK;
        void* const* g = grads + P_FIRST + i * P_BLOCK;
        const char* const a = block(i);
        const char* const x_in = i ? block(i - 1) + l.xout : base + l.x0;
        const char* const h1 = i ? block(i - 1) + l.hnext : base + l.h0;
        const char* const dx = ws + t.dx[cur];
        const int64_t own = t.group ? i % t.group * t.block : 0;
        char *const df1 = ws + t.df1 + own, *const dqkv = ws + t.dqkv + own, *const dm = ws + t.dm + own;
        const char* const d = entering(i);
        char* const t1 = ws + t.t1;
        float* const colpart = (float*)(ws + t.mul_parts + i * (int64_t)t.mul_slot);
        // dX, and dW with it or later with the others of its group
        auto linear = [&](int kind, PtjLinearBwd p) {
            if (t.group) {
                group.d[kind][group.blocks] = p.d;
                group.x[kind][group.blocks] = p.x;
                group.dw[kind][group.blocks] = p.dw;
                p.dx_only = true;
            }
            return ptj_linear_bwd(p, scratch, sb, dt, &sums, st);
        };
        // x_out = x_mid + dropout(ffn(ln2(x_mid)))
        STEP(linear(W_FFN2, {d, w[P_W2], a + l.g1, df1, g[P_W2], N, D, F, a + l.f1, colpart, g[P_B1]}));
        STEP(linear(W_FFN1, {df1, w[P_W1], a + l.h2, t1, g[P_W1], N, F, D, nullptr, nullptr, nullptr}));
        STEP(ln_bwd(2 * i + 1, t1, a + l.xmid, w + P_LN2G, dx, ws + t.dxm, g + P_LN2G, dm, nullptr, seed(2 + 3 * i),
                    kb ? a + l.keep1 : nullptr));
        // x_mid = x_in + dropout(attn(ln1(x_in)))
        STEP(linear(W_OUT, {dm, w[P_WO], a + l.o, t1, g[P_WO], N, D, D, nullptr, nullptr, nullptr}));
        STEP(ptj_attn_bwd_packed(t1, a + l.qkv, a + l.o, (const float*)(a + l.ms), (const float*)(a + l.ls), mask, dqkv,
                                 (float*)(ws + t.delta), bits ? bits + i * bitlen : nullptr, B, H, T, train, dt, st));
        STEP(linear(W_QKV, {dqkv, w[P_WQKV], h1, t1, g[P_WQKV], N, 3 * D, D, nullptr, nullptr, nullptr}));
        if (t.group) {
            ++group.blocks;
            if (i % t.group == 0) {      // the next block's gradients take these ones' place
                STEP(ptj_weight_grads(group, dt, st));
                group.blocks = 0;
            }
        }
        // the dropped copy feeds block i - 1 (its feed-forward dropout) or the embedding
        const bool first = i == 0;
        STEP(ln_bwd(2 * i, t1, x_in, w + P_LN1G, ws + t.dxm, ws + t.dx[cur ^ 1], g + P_LN1G, first ? demb : entering(i - 1),
                    first ? nullptr : grads[P_FIRST + (i - 1) * P_BLOCK + P_B2], seed(3 * i),
                    kb && !first ? block(i - 1) + l.keep2 : nullptr));
        cur ^= 1;
    }
    return ptj_partial_sums(sums, dt, st);
}

}  // extern "C"
