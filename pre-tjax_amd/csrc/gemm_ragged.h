// bf16 GEMM for operands whose rows are not 16-byte aligned (a row pitch that is no multiple of eight elements, a base
// address between vectors).  Included by gemm_ragged.hip inside its unnamed namespace; fp32 operands of this kind take
// gemm_split.h, whose loads need no more than 4-byte alignment.
//
// The asynchronous copies into LDS of gemm_tile.h need whole aligned vectors; here panels travel through registers, two
// steps ahead, in 16-byte loads at element alignment, and one step is 64 contraction elements.  Every access stays inside
// the operand: row indices past its end are clamped (those rows of C are not stored), and the last step, the only one
// whose vectors could reach past the last element, is fetched element by element with clamped indices and zeros selected
// for what lies past the end of the contraction.  LDS layouts and write-back are those of gemm_tile.h.
//
// Before, such operands went element by element through the loader of mma_tile.h: the LM head's input gradient on 8192
// tokens with logits of pitch 50257 took 6.1 ms, its weight gradient 8.2; now 1.0 and 0.95.
typedef short gr_i16x4 __attribute__((ext_vector_type(4)));

template <int MODE, int ROWS, int NTHREADS>
struct GrOperand {
    static constexpr int BK = 64, VEC = 8;
    static constexpr int BYTES = ROWS * BK * 2;                 // one stage
    static constexpr int PER = ROWS * BK / VEC / NTHREADS;      // vectors per thread and step
    static constexpr int PITCH = ROWS * 2;                      // MNMAJOR: bytes per k-row
    static_assert(PER * NTHREADS * VEC == ROWS * BK, "loads divide evenly among the threads");
    typedef LoosePack<uint16_t, VEC> Vec;
    uint32_t voff[PER];                                         // bytes from `base`
    uint32_t loff[PER];                                         // LDS offset inside a stage
    const char* base;
    int64_t step;
    uint32_t s_k2;                                              // MNMAJOR: bytes per k-row in memory
    int rows;                                                   // rows of the operand from row0 on
    gt_u32x4 r[2][PER];

    __device__ __forceinline__ void init(const void* p, int64_t s_row, int64_t s_k, int row0, int nrows, int kbeg, int tid) {
        base = (const char*)p + 2 * (MODE == KMAJOR ? (int64_t)row0 * s_row + kbeg : (int64_t)kbeg * s_k + row0);
        step = (MODE == KMAJOR ? (int64_t)1 : s_k) * BK * 2;
        s_k2 = (uint32_t)s_k * 2u;
        rows = nrows - row0;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int v = i * NTHREADS + tid;
            if constexpr (MODE == KMAJOR) {
                const int row = v >> 3, ch = v & 7;
                voff[i] = (uint32_t)(row < rows ? row : rows - 1) * (uint32_t)s_row * 2u + (uint32_t)ch * 16u;
                loff[i] = row * BKB + ((ch ^ sw(row)) << 4);
            } else {
                constexpr int VPR = ROWS / VEC;                 // vectors per k-row
                const int kk = v / VPR, rv = v - kk * VPR;
                voff[i] = (uint32_t)kk * s_k2 + (uint32_t)(rv * VEC < rows ? rv : 0) * 16u;
                loff[i] = kk * PITCH + ((rv ^ gt_mn_swz<ROWS>(kk)) << 4);
            }
        }
    }

    // Requests the next step's values into register set SET.  kleft: contraction elements from its first one to the end.
    template <int SET>
    __device__ __forceinline__ void load(int kleft, int tid) {
        if (MODE == KMAJOR ? kleft >= BK : kleft > BK) {
#pragma unroll
            for (int i = 0; i < PER; ++i) r[SET][i] = __builtin_bit_cast(gt_u32x4, *reinterpret_cast<const Vec*>(base + voff[i]));
        } else if (kleft > 0) {
            int t = tid;
            asm volatile("" : "+v"(t));                         // keeps the index arithmetic of this path out of the loop's registers
#pragma unroll
            for (int i = 0; i < PER; ++i) {
                const int v = i * NTHREADS + t;
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    uint32_t off;
                    bool inside;
                    if constexpr (MODE == KMAJOR) {
                        const int ch = v & 7, kk = ch * VEC + e;
                        inside = kk < kleft;
                        off = voff[i] - (uint32_t)ch * 16u + (uint32_t)(inside ? kk : kleft - 1) * 2u;
                    } else {
                        constexpr int VPR = ROWS / VEC;
                        const int kk = v / VPR, row = (v - kk * VPR) * VEC + e;
                        inside = kk < kleft;
                        off = (uint32_t)(inside ? kk : kleft - 1) * s_k2 + (uint32_t)(row < rows ? row : rows - 1) * 2u;
                    }
                    const uint32_t x = *reinterpret_cast<const uint16_t*>(base + off);
                    const uint32_t y = inside ? x << (16 * (e & 1)) : 0u;
                    if (e & 1) r[SET][i][e >> 1] |= y;
                    else r[SET][i][e >> 1] = y;
                }
            }
        }
        base += step;
    }
    template <int SET, int I>
    __device__ __forceinline__ void store(char* __restrict__ lds) const {
        *reinterpret_cast<gt_u32x4*>(lds + loff[I]) = r[SET][I];
    }

    // fragment of MFMA tile t (rows wrow + 32 t ...), contraction chunk c of the step
    __device__ __forceinline__ static bf16x8 frag(const char* __restrict__ lds, int wrow, int t, int c, int lane) {
        if constexpr (MODE == KMAJOR) {
            const int row = wrow + t * 32 + (lane & 31), ch = c * 2 + (lane >> 5);
            return *reinterpret_cast<const bf16x8*>(lds + row * BKB + ((ch ^ sw(row)) << 4));
        } else {
            const int l16 = lane & 15, mhalf = (lane >> 4) & 1, lg = lane >> 5, kq = l16 >> 2;
            const int piece = (wrow >> 3) + t * 4 + 2 * mhalf + ((l16 & 3) >> 1);
            const char* p = lds + (16 * c + 8 * lg + kq) * PITCH + ((piece ^ gt_mn_swz<ROWS>(kq)) << 4) + 8 * (l16 & 1);
            const gr_i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) gr_i16x4*)(p));
            const gr_i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) gr_i16x4*)(p + 4 * PITCH));
            return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
};

template <int TBM_, int TBN_, int WM_, int WN_>
struct GrCfg {
    static constexpr int TBM = TBM_, TBN = TBN_, WM = WM_, WN = WN_, KG = 1;
    static constexpr int NW = WM * WN, THREADS = NW * 64;
    static constexpr int TMW = TBM / WM / 32, TNW = TBN / WN / 32;
    static_assert(TMW * WM * 32 == TBM && TNW * WN * 32 == TBN, "whole MFMA tiles per wavefront");
    static constexpr int CW = TNW * 32;
    static constexpr int STAGE = (TBM + TBN) * BKB;
    static constexpr int OUT_PITCH = CW + 4, OUT_WAVE = 32 * OUT_PITCH * 4;
    static constexpr int SMEM = 2 * STAGE > NW * OUT_WAVE ? 2 * STAGE : NW * OUT_WAVE;
    static constexpr int WAVES_EU = (2 * NW + 3) / 4;           // two workgroups per CU
    static_assert(SMEM <= 81920, "two workgroups per CU");
};

template <int AMODE, int BMODE, typename C>
__global__ __launch_bounds__(C::THREADS, C::WAVES_EU) void gemm_ragged_kernel(const GemmArgs g) {
    constexpr int BK = 64, TMW = C::TMW, TNW = C::TNW;
    __shared__ __attribute__((aligned(1024))) char smem[C::SMEM];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / C::WN, wn = wave - wm * C::WN;
    const int num_m = (g.n + C::TBM - 1) / C::TBM, num_n = (g.m + C::TBN - 1) / C::TBN;
    int tile_m, tile_n, z;
    gt_item(g, blockIdx.x, num_m, num_n, tile_m, tile_n, z);
    const int row0 = tile_m * C::TBM, col0 = tile_n * C::TBN;
    const int kbeg = z * g.k_per_split;
    const int kend = g.splits > 1 && kbeg + g.k_per_split < g.k ? kbeg + g.k_per_split : g.k;
    const int klen = kend - kbeg, nk = (klen + BK - 1) / BK;

    typedef GrOperand<AMODE, C::TBM, C::THREADS> OA;
    typedef GrOperand<BMODE, C::TBN, C::THREADS> OB;
    OA oa;
    OB ob;
    oa.init(g.a, g.a_row, g.a_k, row0, g.n, kbeg, tid);
    ob.init(g.b, g.b_row, g.b_k, col0, g.m, kbeg, tid);
    constexpr int NV = OA::PER + OB::PER;
    char* const sA = smem;
    char* const sB = smem + OA::BYTES;

    f32x16 acc[TNW][TMW];
#pragma unroll
    for (int i = 0; i < TNW; ++i)
#pragma unroll
        for (int j = 0; j < TMW; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    auto put = [&](auto set, auto i, int buf) {
        if constexpr (i < OA::PER) oa.template store<set, i>(sA + buf * C::STAGE);
        else ob.template store<set, i - OA::PER>(sB + buf * C::STAGE);
    };
    auto load = [&](auto set, int kleft) {
        oa.template load<set>(kleft, tid);
        ob.template load<set>(kleft, tid);
    };
    constexpr std::integral_constant<int, 0> I0{};
    constexpr std::integral_constant<int, 1> I1{};
    // Step kt (stage kt & 1) while the values of step kt + 1 (register set (kt + 1) & 1) go into the other stage; the set
    // is then refilled with step kt + 3.
    auto step = [&](auto par, int kt) {
        constexpr std::integral_constant<int, 1 - par> NEXT{};
        gt_unroll<0, 4>([&](auto c) {
            bf16x8 fa[TMW], fb[TNW];
#pragma unroll
            for (int t = 0; t < TMW; ++t) fa[t] = OA::frag(sA + par * C::STAGE, wm * TMW * 32, t, c, lane);
#pragma unroll
            for (int t = 0; t < TNW; ++t) fb[t] = OB::frag(sB + par * C::STAGE, wn * TNW * 32, t, c, lane);
            gt_unroll<c * NV / 4, (c + 1) * NV / 4>([&](auto i) { put(NEXT, i, NEXT); });
#pragma unroll
            for (int tn = 0; tn < TNW; ++tn)
#pragma unroll
                for (int tm = 0; tm < TMW; ++tm)
                    acc[tn][tm] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[tn], fa[tm], acc[tn][tm], 0, 0, 0);
        });
        load(NEXT, klen - (kt + 3) * BK);
        __syncthreads();
    };
    if (nk > 0) {
        load(I0, klen);
        load(I1, klen - BK);
        gt_unroll<0, NV>([&](auto i) { put(I0, i, 0); });
        load(I0, klen - 2 * BK);
        __syncthreads();
        for (int kt = 0; kt < nk; kt += 2) {
            step(I0, kt);
            if (kt + 1 >= nk) break;
            step(I1, kt + 1);
        }
    }
    __syncthreads();
    gt_write_back<bf16, C, false>(g, acc, smem, row0, col0, z, wave, lane);
}

template <typename C>
int gr_launch(const GemmArgs& g, int am, int bm, hipStream_t st) {
    const int64_t work = (int64_t)((g.n + C::TBM - 1) / C::TBM) * ((g.m + C::TBN - 1) / C::TBN) * g.splits;
    const dim3 grid((unsigned)work), block(C::THREADS);
#define GR_LAUNCH(AM, BMD) hipLaunchKernelGGL((gemm_ragged_kernel<AM, BMD, C>), grid, block, 0, st, g)
    switch (am * 3 + bm) {
        case 0: GR_LAUNCH(KMAJOR, KMAJOR); break;
        case 1: GR_LAUNCH(KMAJOR, MNMAJOR); break;
        case 3: GR_LAUNCH(MNMAJOR, KMAJOR); break;
        default: GR_LAUNCH(MNMAJOR, MNMAJOR); break;
    }
#undef GR_LAUNCH
    PTJ_CHECK_LAUNCH();
    return g.splits > 1 ? launch_splitk_reduce<bf16>(g, g.splits, st) : PTJ_OK;
}
