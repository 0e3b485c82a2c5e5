// Entry points that the library's own composites use besides the C ABI of include/ptj.h.
#pragma once
#include "common.h"

// Words per batch-head of the attention dropout's keep-bit line.
inline int64_t ptj_attn_bitwords(int64_t T) { return 2 * T / 32 + 2; }

// The keep-bit lines of `count` attention calls (seed seeds[i * stride]) in one launch: bits[i][B*H][bitwords].
int ptj_attn_keepbits_many(uint32_t* bits, int64_t count, const int64_t* seeds, int64_t stride, int64_t BH, int64_t T,
                           hipStream_t st);

// ptj_attn_fwd / ptj_attn_bwd on keep bits that are there already (nullptr: generated into the workspace).  Q, K, V
// (dQ, dK, dV) are the column slices of [B*T, H*3*64], O (dO) is [B*T, H*64].
int ptj_attn_fwd_packed(const void* qkv, const uint32_t* mask, void* o, float* ms, float* ls, const uint32_t* bits, int64_t B,
                        int64_t H, int64_t T, int train, int dtype, hipStream_t st);
int ptj_attn_bwd_packed(const void* d_o, const void* qkv, const void* o, const float* ms, const float* ls,
                        const uint32_t* mask, void* dqkv, float* delta, const uint32_t* bits, int64_t B, int64_t H, int64_t T,
                        int train, int dtype, hipStream_t st);

// A column sum over partial rows that is still to be formed: out[c] = sum_p part[p * stride + c], in a fixed order.
// Producers that take a list append to it instead of launching their second stage, and ptj_partial_sums forms the
// sums of a whole list in one launch (a launch per bias or norm gradient is 3-5 us of latency for 0.2 us of work).
struct PtjPartialSum {
    const float* part;
    void* out;
    int64_t nparts, cols, stride;
};
struct PtjPartialSums {
    static constexpr int MAX = 512;
    PtjPartialSum it[MAX];
    int count = 0;
    bool add(const float* part, void* out, int64_t nparts, int64_t cols, int64_t stride) {
        if (count == MAX) return false;
        it[count++] = {part, out, nparts, cols, stride};
        return true;
    }
};
int ptj_partial_sums(const PtjPartialSums& sums, int dtype, hipStream_t st);

// ptj_layernorm_bwd_dropout whose second stage goes to `later` (nullptr: launched at once, as in the C ABI).
int ptj_layernorm_bwd_later(const void* dy, const void* x, const void* gamma, const void* residual, void* dx, void* dgamma,
                            void* dbeta, void* dropped, void* dropped_colsum, int drop_train, int64_t drop_seed,
                            const void* keep_bytes, void* workspace, size_t workspace_bytes, int64_t rows, int64_t cols,
                            int dtype, PtjPartialSums* later, hipStream_t st);

// Workspace that one such call fills: the partial rows, three sums of them.
inline size_t ptj_layernorm_bwd_parts_bytes(int64_t rows, int64_t cols) {
    const int64_t per = cols <= 1024 ? (rows + 7) / 8 : rows;     // rows of up to 1024 columns: eight per workgroup
    return (size_t)((per < 512 ? per : 512) * 3 * cols) * sizeof(float);
}

// ptj_gemm_mul_colsum whose second stage goes to `later`.
int ptj_gemm_mul_colsum_later(const void* a, const void* b, const void* mul, void* c, void* colsum, int64_t n, int64_t m,
                              int64_t k, int64_t a_rs, int64_t a_cs, int64_t b_rs, int64_t b_cs, int64_t mul_rs, int64_t c_rs,
                              void* workspace, size_t workspace_bytes, void* scratch, size_t scratch_bytes, int dtype,
                              PtjPartialSums* later, hipStream_t st);

// A product [n, m] as stored in `c`, or, where `part` is set, as fp32 partial sums of a K split that its consumer adds up:
// round(sum_z part[z][n][m] + bias), in the order of z.
struct PtjPartialProduct {
    const void* c;
    const float* part;
    int splits;
    const void* bias;
};
// ptj_gemm(A.B (+ bias)) into contiguous rows whose K split, if it takes one, leaves the second stage to the consumer; the
// partial sums lie in `workspace`.
int ptj_gemm_partial(const void* a, const void* b, void* c, const void* bias, int64_t n, int64_t m, int64_t k, int64_t a_rs,
                     int64_t a_cs, int64_t b_rs, int64_t b_cs, void* workspace, size_t workspace_bytes, int dtype,
                     hipStream_t st, PtjPartialProduct* out);
// ptj_dropout_add_layernorm of such a product.
int ptj_dropout_add_layernorm_of(const PtjPartialProduct& x, const void* res, const void* gamma, const void* beta, void* y,
                                 void* h, void* keep_bytes, int64_t rows, int64_t cols, int train, int64_t seed, int dtype,
                                 hipStream_t st);

// y = res + dropout(x) without decisions (x * 0.9) and c = layernorm(y) . w^T (+ bias) (GELU), w [m, dim], in one launch for few rows:
// the same arithmetic as ptj_dropout_add_layernorm_of and ptj_gemm; the norm itself is not stored.  y and c may overlap no operand.
struct PtjNormProduct {
    PtjPartialProduct x;
    const void *res, *gamma, *beta, *w, *bias;
    void *y, *c;
    int gelu;
};
// Whether sizes and type are taken (`partial`: x as partial sums); all pointers have to lie on the 16-byte grid.
bool ptj_norm_product_fits(int64_t rows, int64_t dim, int64_t m, int dtype, bool partial);
int ptj_norm_product(const PtjNormProduct& p, int64_t rows, int64_t dim, int64_t m, int dtype, hipStream_t st);

// The two products of a linear layer's backward, which do not depend on each other: dx = d.w and dw = d^T.x with d [n, m],
// w [m, k], x [n, k] row-major and contiguous.  In one launch where each alone would leave the chip half empty, else one
// after the other.  With `mul` [n, k]: dx = round(d.w) * mul and its column sums to `colsum` (ptj_gemm_mul_colsum; the
// partial rows in `colpart`, ptj_gemm_mul_colsum_workspace_bytes(n, k) bytes, the sums appended to `later`).
struct PtjLinearBwd {
    const void *d, *w, *x;
    void *dx, *dw;
    int64_t n, m, k;
    const void* mul;
    float* colpart;
    void* colsum;
    bool dx_only = false;      // dw is not formed
};
int ptj_linear_bwd(const PtjLinearBwd& p, void* scratch, size_t scratch_bytes, int dtype, PtjPartialSums* later, hipStream_t st);

// The weight gradients of several blocks in one launch: dw[kind][block] = d^T.x with d [k, n[kind]], x [k, m[kind]] and dw
// [n[kind], m[kind]] row-major and contiguous, all of one storage type and on the 16-byte grid, widths multiples of 8.
struct PtjGradGroup {
    static constexpr int KINDS = 4, BLOCKS = 16;
    int k, blocks;
    int n[KINDS], m[KINDS];
    const void *d[KINDS][BLOCKS], *x[KINDS][BLOCKS];
    void* dw[KINDS][BLOCKS];
};
int ptj_weight_grads(const PtjGradGroup& p, int dtype, hipStream_t st);
// How many blocks of `layers` to form in one launch (sizes alone count): the fewest whose launches, of so many blocks and one of the
// rest, take no longer than larger ones; 0: no launch would have a round of tiles.
int ptj_weight_grads_blocks(PtjGradGroup p, int64_t layers, int dtype);
