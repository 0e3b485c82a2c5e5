// Residual update, LayerNorm and the product that reads it, as one launch for few rows (internal.h: ptj_norm_product).
//
// What bounds a forward of few tokens is the number of dependent launches: each costs 3.5-5 us, of which 1-2 are work.  A norm of 64
// rows took 4-5 us of launch for 0.1 MB.  Here a workgroup forms the normalised rows of its own tile of the product: every tile of
// a row of tiles reads and normalises the same rows again, while its panel of the weights, whole along the contraction, is on its
// way into LDS.  The first tile of a row of tiles stores the residual stream.  Four groups of wavefronts share the contraction as
// those of the 32x32 tile kernel do, and the norm is that of rowwise.hip.
//
// The repeated norm is the price: 19 vector instructions an element, 3 us for 32 rows of 768 (the compute unit's whole time at two
// wavefronts a SIMD) and 1.6 for 16, so tiles have as few rows as a round of them allows.  64 rows of 768, kernel time of norm + product
// apart / with 32 rows a tile / with 16, us: dense rows 4.0 + 5.3 / 7.7 / 6.4, rows as four partial sums 5.3 + 5.1 / 12.0 / 8.4.
// So partial sums are taken with 16 rows only.  Forward without dropout, 12 blocks of 768, bf16, norms apart / inside: 64 tokens
// 413 / 363 us, 128 566 / 530.  With dropout the decisions of every row would be formed again in every tile (15 us): not taken.  More than
// a round of tiles would normalise everything once more: not taken (ptj_norm_product_fits).
#include "gemm_core.h"
#include "internal.h"

namespace {

struct NormProductArgs {
    const bf16* x;              // the product of the layer before, dense, or part: [splits][rows][dim]
    const float* part;
    const bf16 *xbias, *res, *gamma, *beta, *w, *bias;
    bf16 *y, *c;
    int splits, rows, m, gelu;
};

constexpr int NP_THREADS = 512, NP_WAVES = 8, NP_LDS = 160 * 1024;
constexpr int np_lds(int dim, int tbm, int tbn) {
    const int panels = (tbm + tbn) * dim * 2, out = 4 * tbm * (tbn + 4) * 4;
    return panels > out ? panels : out;
}

// ITERS * 256 columns of a row, four per lane and iteration
template <int ITERS, int TBM, int TBN, bool PARTIAL>
__global__ __launch_bounds__(NP_THREADS, 2) void norm_product_kernel(const NormProductArgs g) {
    constexpr int DIM = ITERS * 256, PANELS = DIM / 64, RPW = TBM / NP_WAVES;
    constexpr int A_PANEL = TBM * BKB, B_PANEL = TBN * BKB;
    __shared__ __attribute__((aligned(1024))) char smem[np_lds(DIM, TBM, TBN)];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int num_m = (g.rows + TBM - 1) / TBM, num_n = (g.m + TBN - 1) / TBN;
    const int idx = xcd_range<false>((int)blockIdx.x, num_m * num_n), tile_n = idx / num_m, tile_m = idx - tile_n * num_m;
    const int row0 = tile_m * TBM + wave * RPW, col0 = tile_n * TBN;
    char* const sB = smem + PANELS * A_PANEL;

    // rows past the end re-read the last one; their results are not stored
    auto row_of = [&](int r) { return (int64_t)(row0 + r < g.rows ? row0 + r : g.rows - 1); };
    Pack<bf16, 4> res[RPW][ITERS], x[RPW][ITERS], gm[ITERS], bt[ITERS], xb[ITERS];
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const int64_t at = row_of(r) * DIM + (it * 64 + lane) * 4;
            if constexpr (!PARTIAL) x[r][it] = *reinterpret_cast<const Pack<bf16, 4>*>(g.x + at);
            res[r][it] = *reinterpret_cast<const Pack<bf16, 4>*>(g.res + at);
        }
    float v[RPW][ITERS][4];
    if constexpr (PARTIAL) {
#pragma unroll
        for (int it = 0; it < ITERS; ++it)
#pragma unroll
            for (int j = 0; j < 4; ++j) xb[it].v[j] = from_f32<bf16>(0.f);
        if (g.xbias != nullptr)
#pragma unroll
            for (int it = 0; it < ITERS; ++it) xb[it] = *reinterpret_cast<const Pack<bf16, 4>*>(g.xbias + (it * 64 + lane) * 4);
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int it = 0; it < ITERS; ++it)
#pragma unroll
                for (int j = 0; j < 4; ++j) v[r][it][j] = 0.f;
        // one split of all rows at a time, requested together
        for (int z = 0; z < g.splits; ++z) {
            const float* pz = g.part + (int64_t)z * g.rows * DIM;
            f32x4 p[RPW][ITERS];
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int it = 0; it < ITERS; ++it) p[r][it] = *reinterpret_cast<const f32x4*>(pz + row_of(r) * DIM + (it * 64 + lane) * 4);
#pragma unroll
            for (int r = 0; r < RPW; ++r)
#pragma unroll
                for (int it = 0; it < ITERS; ++it)
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[r][it][j] += p[r][it][j];
        }
    }
#pragma unroll
    for (int it = 0; it < ITERS; ++it) {
        gm[it] = *reinterpret_cast<const Pack<bf16, 4>*>(g.gamma + (it * 64 + lane) * 4);
        bt[it] = *reinterpret_cast<const Pack<bf16, 4>*>(g.beta + (it * 64 + lane) * 4);
    }
    const int out_c = tid % (TBN / 4) * 4;
    // (without a branch, whose end would wait for everything under way)
    const Pack<bf16, 4> ob = *reinterpret_cast<const Pack<bf16, 4>*>(g.bias != nullptr ? g.bias + (col0 + out_c < g.m ? col0 + out_c : 0) : g.gamma);
    __builtin_amdgcn_sched_barrier(0);
    // The tile's weights: eight rows of a panel of 64 contraction elements per copy; columns of the product past its end read as zero
    {
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(g.w + (int64_t)col0 * DIM), 0, (uint32_t)(g.m - col0) * (uint32_t)(DIM * 2),
                                                            0x00020000);
#pragma unroll
        for (int i = 0; i < PANELS * TBN / 8 / NP_WAVES; ++i) {
            const int inst = i * NP_WAVES + wave, panel = inst / (TBN / 8), r = (inst % (TBN / 8)) * 8 + (lane >> 3);
            const uint32_t voff = (uint32_t)(r * DIM + panel * 64 + ((lane & 7) ^ sw(r)) * 8) * 2u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(sB + inst * 1024), 16, voff, 0, 0, 0);
        }
    }
    // (opaque from here on: the compiler forms the norm ahead of the copies otherwise)
#pragma unroll
    for (int r = 0; r < RPW; ++r)
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            gt_u32x2 t = __builtin_bit_cast(gt_u32x2, res[r][it]);
            asm volatile("" : "+v"(t));
            res[r][it] = __builtin_bit_cast(Pack<bf16, 4>, t);
        }
    Pack<bf16, 4> obias = ob;
    {
        gt_u32x2 t = __builtin_bit_cast(gt_u32x2, ob);
        asm volatile("" : "+v"(t));
        obias = __builtin_bit_cast(Pack<bf16, 4>, t);
    }

    const uint32_t lds_a = gt_lds_addr(smem);
    // dropout_add_layernorm_kernel without dropout (rowwise.hip), all rows side by side
    float mu[RPW], rstd[RPW];
    Pack<bf16, 4> y[RPW][ITERS];
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        float s = 0.f;
#pragma unroll
        for (int it = 0; it < ITERS; ++it)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float a;
                if constexpr (PARTIAL) a = to_f32(from_f32<bf16>(g.xbias != nullptr ? v[r][it][j] + to_f32(xb[it].v[j]) : v[r][it][j]));
                else a = to_f32(x[r][it].v[j]);
                y[r][it].v[j] = from_f32<bf16>(to_f32(res[r][it].v[j]) + to_f32(from_f32<bf16>(a * 0.9f)));
                v[r][it][j] = to_f32(y[r][it].v[j]);
                s += v[r][it][j];
            }
        mu[r] = s;
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r) mu[r] = wave_sum(mu[r]) * (1.0f / (float)DIM);
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        float q = 0.f;
#pragma unroll
        for (int it = 0; it < ITERS; ++it)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const float d = v[r][it][j] - mu[r];
                v[r][it][j] = d;
                q += d * d;
            }
        rstd[r] = q;
    }
#pragma unroll
    for (int r = 0; r < RPW; ++r) rstd[r] = 1.0f / sqrtf(wave_sum(rstd[r]) * (1.0f / (float)(DIM - 1)));
#pragma unroll
    for (int r = 0; r < RPW; ++r) {
        const int row = wave * RPW + r;
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            Pack<bf16, 4> h;
#pragma unroll
            for (int j = 0; j < 4; ++j) h.v[j] = from_f32<bf16>(to_f32(gm[it].v[j]) * (v[r][it][j] * rstd[r]) + to_f32(bt[it].v[j]));
            // columns 4 * (it * 64 + lane) ...: half a 16-byte piece of a panel row
            const int panel = it * 4 + (lane >> 4), piece = (lane >> 1) & 7;
            const uint32_t at = lds_a + (uint32_t)(panel * A_PANEL + row * BKB + ((piece ^ sw(row)) << 4) + (lane & 1) * 8);
            asm volatile("ds_write_b64 %0, %1" ::"v"(at), "v"(__builtin_bit_cast(gt_u32x2, h)) : "memory");
        }
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // Wavefront group kg multiplies the panels kg, kg + 4, ..., two wavefronts the halves of the columns; TBM = 32: MFMAs of 32x32x16,
    // one for 32 columns, TBM = 16: of 16x16x32.
    constexpr int PITCH = TBN + 4, GROUP = TBM * PITCH, CW = TBM == 32 ? 32 : TBN / 2, NT = TBM == 32 ? 1 : CW / 16, LANES = TBM;
    const int kg = wave & 3, wn = wave >> 2, lr = lane & (LANES - 1), lg = lane / LANES;
    const bool active = wn * CW < TBN;
    typedef typename std::conditional<TBM == 32, f32x16, f32x4>::type Acc;
    Acc acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < (int)(sizeof(Acc) / 4); ++e) acc[t][e] = 0.f;
    if (active) {
#pragma unroll
        for (int i = 0; i < ITERS; ++i) {
            const int panel = i * 4 + kg;
            constexpr int CHUNKS = TBM == 32 ? 4 : 2;
#pragma unroll
            for (int ch = 0; ch < CHUNKS; ++ch) {
                const int o = ((ch * (8 / CHUNKS) + lg) ^ sw(lr)) << 4;
                const bf16x8 a = *reinterpret_cast<const bf16x8*>(smem + panel * A_PANEL + lr * BKB + o);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const int row = wn * CW + t * LANES + lr, ob = ((ch * (8 / CHUNKS) + lg) ^ sw(row)) << 4;
                    const bf16x8 b = *reinterpret_cast<const bf16x8*>(sB + panel * B_PANEL + row * BKB + ob);
                    if constexpr (TBM == 32) mma_chunk(acc[t], b, a);
                    else acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, a, acc[t], 0, 0, 0);
                }
            }
        }
    }
    __syncthreads();
    float* const out = (float*)smem;
    if (active) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int q = 0; q < (int)(sizeof(Acc) / 16); ++q)
                *reinterpret_cast<f32x4*>(out + kg * GROUP + lr * PITCH + wn * CW + t * LANES + q * 8 + lg * 4) =
                    f32x4{acc[t][q * 4], acc[t][q * 4 + 1], acc[t][q * 4 + 2], acc[t][q * 4 + 3]};
    }
    __syncthreads();
    if (tile_n == 0) {
#pragma unroll
        for (int r = 0; r < RPW; ++r)
#pragma unroll
            for (int it = 0; it < ITERS; ++it)
                if (row0 + r < g.rows) *reinterpret_cast<Pack<bf16, 4>*>(g.y + (int64_t)(row0 + r) * DIM + (it * 64 + lane) * 4) = y[r][it];
    }
    if (tid < TBM * TBN / 4) {
        const int r = tid / (TBN / 4), c = out_c, row = tile_m * TBM + r, col = col0 + c;
        f32x4 s = *reinterpret_cast<const f32x4*>(out + r * PITCH + c);
#pragma unroll
        for (int k = 1; k < 4; ++k) s += *reinterpret_cast<const f32x4*>(out + k * GROUP + r * PITCH + c);
        if (row < g.rows && col < g.m) {                     // (m is a multiple of 4)
            Pack<bf16, 4> o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (g.bias != nullptr) s[e] += to_f32(obias.v[e]);
                o.v[e] = from_f32<bf16>(g.gelu ? gelu_f(s[e]) : s[e]);
            }
            *reinterpret_cast<Pack<bf16, 4>*>(g.c + (int64_t)row * g.m + col) = o;
        }
    }
}

// A tile's rows and columns; rows = 0: not taken.  The fewest rows whose tiles are at most a round.
struct NpTile { int rows, cols; };
NpTile np_tile(int64_t rows, int64_t dim, int64_t m, int dtype) {
    if (dtype != PTJ_BF16 || rows < 1 || dim < 256 || dim > 1024 || dim % 256 != 0 || m < 4 || m % 4 != 0 || m * dim >= 1ll << 30) return {0, 0};
    for (const NpTile t : {NpTile{16, 32}, NpTile{16, 64}, NpTile{32, 32}, NpTile{32, 64}})
        if ((rows + t.rows - 1) / t.rows * ((m + t.cols - 1) / t.cols) <= num_cus() && np_lds((int)dim, t.rows, t.cols) <= NP_LDS) return t;
    return {0, 0};
}

template <int ITERS, int TBM, int TBN>
void np_launch(const NormProductArgs& g, hipStream_t st) {
    const dim3 grid((unsigned)(((g.rows + TBM - 1) / TBM) * ((g.m + TBN - 1) / TBN)));
    if constexpr (TBM == 16)
        if (g.part != nullptr) {
            hipLaunchKernelGGL((norm_product_kernel<ITERS, TBM, TBN, true>), grid, dim3(NP_THREADS), 0, st, g);
            return;
        }
    hipLaunchKernelGGL((norm_product_kernel<ITERS, TBM, TBN, false>), grid, dim3(NP_THREADS), 0, st, g);
}
template <int ITERS>
void np_launch(const NormProductArgs& g, const NpTile& t, hipStream_t st) {
    if (t.rows == 16) t.cols == 32 ? np_launch<ITERS, 16, 32>(g, st) : np_launch<ITERS, 16, 64>(g, st);
    else if (t.cols == 32) np_launch<ITERS, 32, 32>(g, st);
    else if constexpr (np_lds(ITERS * 256, 32, 64) <= NP_LDS) np_launch<ITERS, 32, 64>(g, st);
}

}  // namespace

bool ptj_norm_product_fits(int64_t rows, int64_t dim, int64_t m, int dtype, bool partial) {
    const int tile_rows = np_tile(rows, dim, m, dtype).rows;
    return tile_rows > 0 && (!partial || tile_rows == 16);
}

int ptj_norm_product(const PtjNormProduct& p, int64_t rows, int64_t dim, int64_t m, int dtype, hipStream_t st) {
    const NpTile t = np_tile(rows, dim, m, dtype);
    PTJ_CHECK_ARG((p.x.part || p.x.c) && p.res && p.gamma && p.beta && p.w && p.y && p.c && (p.bias || !p.gelu), "norm_product: null pointer");
    bool ok = t.rows > 0 && (!p.x.part || t.rows == 16);
    for (const void* q : {p.x.part ? (const void*)p.x.part : p.x.c, p.x.part ? p.x.bias : nullptr, p.res, p.gamma, p.beta, p.w, p.bias, (const void*)p.y,
                          (const void*)p.c})
        ok = ok && ptj_aligned16(q);
    if (!ok) return ptj_set_error(PTJ_ERR_INVALID, "norm_product: %lld rows of %lld, %lld outputs, partial sums or unaligned operands", (long long)rows,
                                  (long long)dim, (long long)m);
    const NormProductArgs g = {(const bf16*)p.x.c, p.x.part, (const bf16*)p.x.bias, (const bf16*)p.res, (const bf16*)p.gamma, (const bf16*)p.beta,
                               (const bf16*)p.w, (const bf16*)p.bias, (bf16*)p.y, (bf16*)p.c, p.x.splits, (int)rows, (int)m, p.gelu};
    switch (dim / 256) {
        case 1: np_launch<1>(g, t, st); break;
        case 2: np_launch<2>(g, t, st); break;
        case 3: np_launch<3>(g, t, st); break;
        default: np_launch<4>(g, t, st); break;
    }
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}
