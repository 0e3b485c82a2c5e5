// Token + position embedding, forward and backward, as single passes.
//
// Forward: out[i] = dropout(round(wemb[token_i] * scale) + pos[i mod seq]) -- the gather,
// the scaling, the position add and the embedding dropout of the model's first step, with
// the storage rounding after each of them that separate kernels would apply.
//
// Backward: dwemb[tok] += scale * sum_{i: token_i = tok} d[i].  The workgroup on the first
// position of a token sums the gradient rows of all its positions in fp32 in order of
// position (four row slots folded through LDS in slot order) and updates that table
// row in place, so the result is deterministic and no [vocab, dim] scratch is touched.
// Up to EMB_SCAN_MAX positions a workgroup finds the equal tokens by comparison; beyond, the
// caller passes the token ids sorted (stable) together with the sorting permutation.
#include "common.h"

namespace {

constexpr int EMB_COLT = 128;            // column threads (one 16-byte vector each per sweep)
constexpr int EMB_SLOTS = 4;             // row slots of the backward workgroup
constexpr int EMB_BWD_THREADS = EMB_COLT * EMB_SLOTS;
constexpr int EMB_SCAN_MAX = PTJ_EMBED_SCAN_MAX;       // positions that embed_bwd_scan_kernel takes

template <typename T, int VEC>
__global__ __launch_bounds__(256) void embed_fwd_kernel(const T* __restrict__ wemb, const T* __restrict__ pos,
                                                         const int64_t* __restrict__ tokens, T* __restrict__ out,
                                                         int64_t n, int dim, int64_t seq, int64_t vocab, float scale,
                                                         int train, uint64_t seed) {
#pragma clang fp contract(off)   // product and sum are rounded separately, as two kernels would
    const int vpr = dim / VEC;
    const int64_t total = n * vpr;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t row = (int64_t)((uint64_t)i / (uint32_t)vpr);
        const int c0 = (int)(i - row * vpr) * VEC;
        int64_t tok = tokens[row];
        tok = tok < 0 ? 0 : (tok >= vocab ? vocab - 1 : tok);   // ids are required to be in range; never read outside the table
        float w[VEC], p[VEC];
        load_vec<T, VEC>(wemb + tok * dim + c0, w);
        load_vec<T, VEC>(pos + (row % seq) * dim + c0, p);
        const uint64_t s = seed + (uint64_t)row;
        const uint32_t k0 = (uint32_t)s, k1 = (uint32_t)(s >> 32);
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            float v = to_f32(from_f32<T>(w[j] * scale));
            v = to_f32(from_f32<T>(v + p[j]));
            if (train) v = philox_keep((uint32_t)(c0 + j), k0, k1) ? v : 0.f;
            else v *= 0.9f;
            w[j] = v;
        }
        store_vec<T, VEC>(out + row * dim + c0, w);
    }
}

// Row of `d` behind sorted position j, clamped so that a bad permutation cannot read outside d.
__device__ __forceinline__ int64_t src_row(const int64_t* __restrict__ order, int64_t j, int64_t n) {
    const int64_t r = order[j];
    return r < 0 ? 0 : (r >= n ? n - 1 : r);
}

// Row `tok` of the table += scale * (the rows row_of(0) .. row_of(count - 1) of d, in this order).  The whole workgroup calls it.
template <typename T, int VEC, typename ROW>
__device__ __forceinline__ void add_run(const T* __restrict__ d, T* __restrict__ dwemb, int64_t tok, int64_t count, int dim, float scale,
                                        float (&red)[EMB_SLOTS][EMB_COLT * VEC], ROW row_of) {
    const int ct = threadIdx.x % EMB_COLT, slot = threadIdx.x / EMB_COLT;
    const int nvec = dim / VEC;
    for (int v0 = 0; v0 < nvec; v0 += EMB_COLT) {
        const int vi = v0 + ct;
        const bool active = vi < nvec;
        float acc[VEC];
#pragma unroll
        for (int j = 0; j < VEC; ++j) acc[j] = 0.f;
        if (active) {
            constexpr int U = 4;
            int64_t j = slot;
            for (; j + (U - 1) * EMB_SLOTS < count; j += U * EMB_SLOTS) {
                float r[U][VEC];
#pragma unroll
                for (int u = 0; u < U; ++u) load_vec<T, VEC>(d + row_of(j + u * EMB_SLOTS) * dim + vi * VEC, r[u]);
#pragma unroll
                for (int u = 0; u < U; ++u)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) acc[e] += r[u][e];
            }
            for (; j < count; j += EMB_SLOTS) {
                float r[VEC];
                load_vec<T, VEC>(d + row_of(j) * dim + vi * VEC, r);
#pragma unroll
                for (int e = 0; e < VEC; ++e) acc[e] += r[e];
            }
#pragma unroll
            for (int e = 0; e < VEC; ++e) red[slot][ct * VEC + e] = acc[e];
        }
        __syncthreads();
        if (active && slot == 0) {
            float row[VEC];
            load_vec<T, VEC>(dwemb + tok * dim + vi * VEC, row);
#pragma unroll
            for (int e = 0; e < VEC; ++e) {
                float s = red[0][ct * VEC + e];
#pragma unroll
                for (int k = 1; k < EMB_SLOTS; ++k) s += red[k][ct * VEC + e];
                row[e] += s * scale;
            }
            store_vec<T, VEC>(dwemb + tok * dim + vi * VEC, row);
        }
        __syncthreads();
    }
}

template <typename T, int VEC>
__global__ __launch_bounds__(EMB_BWD_THREADS) void embed_bwd_kernel(const T* __restrict__ d,
                                                                    const int64_t* __restrict__ sorted_tok,
                                                                    const int64_t* __restrict__ order,
                                                                    T* __restrict__ dwemb, int64_t n, int dim,
                                                                    int64_t vocab, float scale) {
    __shared__ float red[EMB_SLOTS][EMB_COLT * VEC];
    __shared__ int64_t s_end;
    const int64_t first = blockIdx.x;
    const int64_t tok = sorted_tok[first];
    if (first > 0 && sorted_tok[first - 1] == tok) return;      // not the head of a run (uniform)
    if (tok < 0 || tok >= vocab) return;
    if (threadIdx.x == 0) {
        // end of the run: first position after `first` with a different token (binary search)
        int64_t lo = first + 1, hi = n;
        while (lo < hi) {
            const int64_t mid = (lo + hi) >> 1;
            if (sorted_tok[mid] == tok) lo = mid + 1;
            else hi = mid;
        }
        s_end = lo;
    }
    __syncthreads();
    add_run<T, VEC>(d, dwemb, tok, s_end - first, dim, scale, red, [&](int64_t j) { return src_row(order, first + j, n); });
}

// The same without a sort, for n <= EMB_SCAN_MAX: workgroup i compares token i with all of them, ends if an earlier one is equal,
// and lists the equal ones, in order of position, in LDS; so the sums are the same bits.  Every token is read n times from L2
// (8 bytes each, all of a workgroup's at once), where a sort of a few thousand keys is one workgroup's work in several launches.
// us with the sort / without, 768 columns of bf16, ids as in text: 512 tokens 34.0 / 4.1, 2048 41.8 / 8.4,
// 4096 58.0 / 19.9, 8192 66.8 / 56.2; it grows with n^2, and beyond that the sort is faster.  With ids drawn evenly, whose workgroups
// nearly all have a sum of their own, the line lies there: 5000 54.2 / 37.6, 8192 64.3 / 64.2 (fp32 69.6 / 73.1); with half the ids equal,
// 8192, 228 / 145.
template <typename T, int VEC, int PER>
__global__ __launch_bounds__(EMB_BWD_THREADS) void embed_bwd_scan_kernel(const T* __restrict__ d, const int64_t* __restrict__ tokens,
                                                                         T* __restrict__ dwemb, int n, int dim, int64_t vocab,
                                                                         float scale) {
    constexpr int WAVES = EMB_BWD_THREADS / 64;
    __shared__ float red[EMB_SLOTS][EMB_COLT * VEC];
    __shared__ uint16_t list[PER * EMB_BWD_THREADS];
    __shared__ uint16_t counts[PER * WAVES];                 // equal tokens per 64 positions
    const int i = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t tok = tokens[i];
    if (tok < 0 || tok >= vocab) return;
    bool equal[PER];
    int64_t t[PER];
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        const int p = u * EMB_BWD_THREADS + tid;
        t[u] = p < n ? tokens[p] : -1;
    }
    bool earlier = false;
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        equal[u] = t[u] == tok;
        earlier |= equal[u] && u * EMB_BWD_THREADS + tid < i;
        const uint64_t m = __ballot(equal[u]);
        if (lane == 0) counts[u * WAVES + wave] = (uint16_t)__popcll(m);
    }
    if (__syncthreads_or(earlier)) return;                  // not the first of its token
    int before = 0, count = 0;                               // of this lane's position among the equal ones; all of them
#pragma unroll
    for (int u = 0; u < PER; ++u) {
        for (int w = 0; w < WAVES; ++w) {
            if (w == wave) before = count;
            count += counts[u * WAVES + w];
        }
        const uint64_t m = __ballot(equal[u]);
        if (equal[u]) list[before + __popcll(m & ((1ull << lane) - 1))] = (uint16_t)(u * EMB_BWD_THREADS + tid);
    }
    __syncthreads();
    add_run<T, VEC>(d, dwemb, tok, count, dim, scale, red, [&](int64_t j) { return (int64_t)list[j]; });
}

template <typename T>
int embed_fwd_impl(const void* wemb, const void* pos, const int64_t* tokens, void* out, int64_t n, int64_t dim,
                   int64_t seq, int64_t vocab, float scale, int train, int64_t seed, hipStream_t st) {
    constexpr int FV = VecOf<T>::N;
    const bool vok = dim % FV == 0 && ptj_aligned16(wemb) && ptj_aligned16(pos) && ptj_aligned16(out);
    const int64_t work = n * (vok ? dim / FV : dim);
    int64_t blocks = (work + 255) / 256;
    if (blocks > (int64_t)ptj_num_cus() * 16) blocks = (int64_t)ptj_num_cus() * 16;
    if (vok)
        hipLaunchKernelGGL((embed_fwd_kernel<T, FV>), dim3((unsigned)blocks), dim3(256), 0, st, (const T*)wemb, (const T*)pos,
                           tokens, (T*)out, n, (int)dim, seq, vocab, scale, train, (uint64_t)seed);
    else
        hipLaunchKernelGGL((embed_fwd_kernel<T, 1>), dim3((unsigned)blocks), dim3(256), 0, st, (const T*)wemb, (const T*)pos,
                           tokens, (T*)out, n, (int)dim, seq, vocab, scale, train, (uint64_t)seed);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

template <typename T>
int embed_bwd_impl(const void* d, const int64_t* sorted_tok, const int64_t* order, void* dwemb, int64_t n, int64_t dim,
                   int64_t vocab, float scale, hipStream_t st) {
    constexpr int FV = VecOf<T>::N;
    const bool vok = dim % FV == 0 && ptj_aligned16(d) && ptj_aligned16(dwemb);
    if (vok)
        hipLaunchKernelGGL((embed_bwd_kernel<T, FV>), dim3((unsigned)n), dim3(EMB_BWD_THREADS), 0, st, (const T*)d,
                           sorted_tok, order, (T*)dwemb, n, (int)dim, vocab, scale);
    else
        hipLaunchKernelGGL((embed_bwd_kernel<T, 1>), dim3((unsigned)n), dim3(EMB_BWD_THREADS), 0, st, (const T*)d,
                           sorted_tok, order, (T*)dwemb, n, (int)dim, vocab, scale);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

template <typename T>
int embed_bwd_scan_impl(const void* d, const int64_t* tokens, void* dwemb, int64_t n, int64_t dim, int64_t vocab, float scale,
                        hipStream_t st) {
    constexpr int FV = VecOf<T>::N;
    const bool vok = dim % FV == 0 && ptj_aligned16(d) && ptj_aligned16(dwemb);
#define SCAN(VEC_, PER_)                                                                                                     \
    hipLaunchKernelGGL((embed_bwd_scan_kernel<T, VEC_, PER_>), dim3((unsigned)n), dim3(EMB_BWD_THREADS), 0, st, (const T*)d, \
                       tokens, (T*)dwemb, (int)n, (int)dim, vocab, scale)
    // tokens per thread: as few as hold them (4096 positions at 8 and 16: 19.9 and 27.2 us)
    if (n <= 4 * EMB_BWD_THREADS) {
        if (vok) SCAN(FV, 4);
        else SCAN(1, 4);
    } else if (n <= 8 * EMB_BWD_THREADS) {
        if (vok) SCAN(FV, 8);
        else SCAN(1, 8);
    } else {
        if (vok) SCAN(FV, EMB_SCAN_MAX / EMB_BWD_THREADS);
        else SCAN(1, EMB_SCAN_MAX / EMB_BWD_THREADS);
    }
#undef SCAN
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

}  // namespace

extern "C" {

int ptj_embed_fwd(const void* wemb, const void* pos, const int64_t* tokens, void* out, int64_t n, int64_t dim,
                  int64_t seq, int64_t vocab, float scale, int train, int64_t seed, int dtype, void* stream) {
    PTJ_CHECK_ARG(n >= 0 && dim >= 1 && dim < (1ll << 31) && seq >= 1 && vocab >= 1, "embed_fwd: bad shape");
    PTJ_CHECK_ARG(dtype == PTJ_F32 || dtype == PTJ_BF16, "embed_fwd: unknown dtype %d", dtype);
    if (n == 0) return PTJ_OK;
    PTJ_CHECK_ARG(wemb && pos && tokens && out, "embed_fwd: null pointer");
    hipStream_t st = (hipStream_t)stream;
    return dtype == PTJ_F32 ? embed_fwd_impl<float>(wemb, pos, tokens, out, n, dim, seq, vocab, scale, train, seed, st)
                            : embed_fwd_impl<bf16>(wemb, pos, tokens, out, n, dim, seq, vocab, scale, train, seed, st);
}

int ptj_embed_bwd(const void* d, const int64_t* sorted_tokens, const int64_t* order, void* dwemb, int64_t n,
                  int64_t dim, int64_t vocab, float scale, int dtype, void* stream) {
    PTJ_CHECK_ARG(n >= 0 && n < (1ll << 31) && dim >= 1 && dim < (1ll << 31) && vocab >= 1, "embed_bwd: bad shape");
    PTJ_CHECK_ARG(dtype == PTJ_F32 || dtype == PTJ_BF16, "embed_bwd: unknown dtype %d", dtype);
    if (n == 0) return PTJ_OK;
    PTJ_CHECK_ARG(d && sorted_tokens && order && dwemb, "embed_bwd: null pointer");
    hipStream_t st = (hipStream_t)stream;
    return dtype == PTJ_F32 ? embed_bwd_impl<float>(d, sorted_tokens, order, dwemb, n, dim, vocab, scale, st)
                            : embed_bwd_impl<bf16>(d, sorted_tokens, order, dwemb, n, dim, vocab, scale, st);
}

int ptj_embed_bwd_tokens(const void* d, const int64_t* tokens, void* dwemb, int64_t n, int64_t dim, int64_t vocab, float scale,
                         int dtype, void* stream) {
    PTJ_CHECK_ARG(n >= 0 && n <= EMB_SCAN_MAX && dim >= 1 && dim < (1ll << 31) && vocab >= 1, "embed_bwd_tokens: bad shape");
    PTJ_CHECK_ARG(dtype == PTJ_F32 || dtype == PTJ_BF16, "embed_bwd_tokens: unknown dtype %d", dtype);
    if (n == 0) return PTJ_OK;
    PTJ_CHECK_ARG(d && tokens && dwemb, "embed_bwd_tokens: null pointer");
    hipStream_t st = (hipStream_t)stream;
    return dtype == PTJ_F32 ? embed_bwd_scan_impl<float>(d, tokens, dwemb, n, dim, vocab, scale, st)
                            : embed_bwd_scan_impl<bf16>(d, tokens, dwemb, n, dim, vocab, scale, st);
}

}  // extern "C"
