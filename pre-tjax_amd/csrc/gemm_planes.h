// fp32 GEMM on the bf16 matrix pipe whose operands are split ahead of the product.  Included by gemm_tile_launch.h inside its
// unnamed namespace; the split, its range and the fall-back are those of gemm_split.h.
//
// gemm_split_kernel converts an operand once for every tile that reads it, 24 or 32 times at the sizes of a trainer, with as
// many vector instructions as the matrix pipe takes clocks.  Here a pass over the operands (gs_planes_kernel) writes the three parts
// once, in the order in which a wavefront's lanes hold an MFMA operand: 32 rows x 16 contraction elements of one part are a
// fragment of 1024 contiguous bytes, lane l's sixteen at byte 16 l, and the fragments lie as [block of 32 rows][block of 16
// contraction elements][part].  Copies into LDS then move whole kilobytes, LDS reads are conflict-free without a swizzle, every
// layout of the operands costs the same, and the contraction is padded with zeros, so the product has one loop without borders.
//
// The product: 128x128 tile, four wavefronts of 64x64, two workgroups per CU.  Per 16 contraction elements a workgroup takes
// 768 clocks of MFMAs, 384 of LDS reads and 192 of arriving copies.  Three stages of 24 KB; one register set of
// fragments, each refilled for the next step right behind its last use: the step begins with the products of the middle
// parts, whose fragments were refilled first, and the barrier comes behind those four MFMAs.
//
// Measured, gemm_split_kernel / this with its pass: 4096x3072x768 118.6 / 103.8 us, 4096x2304x768 106 / 94, 4096x35374x768
// 1352 / 1074 (the pass: 11.6 us for 4096x3072x768, 4.7 TB/s); training step 8 x 512 22.65 / 22.10 ms.  Outputs 768 wide,
// which read every operand less often, are slower so (4096x768x768 34.7 / 42.6, 4096x768x3072 123 / 128) and stay there.
//
// The matrix pipe rounds its accumulator more coarsely than a vector add: the leading products (hh) of two steps are formed from
// zero and added by the vector ALU, as in gemm_split_kernel, and the five small terms have an accumulator of their own.
constexpr int GS_FRAG = 1024;                        // bytes of 32 rows x 16 contraction elements of one part
constexpr int64_t gs_kblocks(int64_t k) { return (k + 15) / 16; }
constexpr int64_t gs_plane_bytes(int64_t rows, int64_t k) { return (rows + 31) / 32 * gs_kblocks(k) * 3 * GS_FRAG; }

// One operand of gs_planes_kernel: element (row, k) = p[row * s_row + k * s_k]
struct GsSource {
    const float* p;
    char* planes;
    int64_t s_row, s_k;
    int rows, k, blocks_k;                           // blocks_k: workgroups along the contraction (64 elements each)
};

// One workgroup per 32 rows x 64 contraction elements; a thread splits eight consecutive contraction elements of a row.
__global__ __launch_bounds__(256) void gs_planes_kernel(const GsSource a, const GsSource b, int blocks_a) {
    const bool second = (int)blockIdx.x >= blocks_a;
    const GsSource s = second ? b : a;
    const int id = second ? (int)blockIdx.x - blocks_a : (int)blockIdx.x;
    const int rb = id / s.blocks_k, k0 = (id - rb * s.blocks_k) * 64, t = threadIdx.x;
    // lanes run along the operand's contiguous axis
    const bool along_k = s.s_k == 1;
    const int r = along_k ? t >> 3 : t & 31, kg = along_k ? t & 7 : t >> 5;
    const int row = rb * 32 + r, k = k0 + kg * 8;
    const int64_t kb = gs_kblocks(s.k);
    if (k / 16 >= kb) return;
    float x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) x[e] = 0.f;
    if (row < s.rows) {
        const float* p = s.p + (int64_t)row * s.s_row + (int64_t)k * s.s_k;
        if (along_k && k + 8 <= s.k) {
            const LoosePack<float, 8> v = *reinterpret_cast<const LoosePack<float, 8>*>(p);
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = v.v[e];
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (k + e < s.k) x[e] = p[(int64_t)e * s.s_k];
        }
    }
    gt_u32x4 part[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t h, m, l;
        gs_split2(x[2 * i], x[2 * i + 1], h, m, l);
        part[0][i] = h;
        part[1][i] = m;
        part[2][i] = l;
    }
    char* out = s.planes + ((int64_t)rb * kb + k / 16) * (3 * GS_FRAG) + ((kg & 1) * 32 + r) * 16;
#pragma unroll
    for (int i = 0; i < 3; ++i) *reinterpret_cast<gt_u32x4*>(out + i * GS_FRAG) = part[i];
}

struct GpCfg {
    static constexpr int TBM = 128, TBN = 128, WM = 2, WN = 2, KG = 1, NW = 4, THREADS = 256, TMW = 2, TNW = 2, STAGES = 3;
    static constexpr int CW = TNW * 32, OUT_PITCH = CW + 4, OUT_WAVE = 32 * OUT_PITCH * 4;
    static constexpr int STAGE = (TBM + TBN) / 32 * 3 * GS_FRAG, SMEM = STAGES * STAGE;
    static_assert(NW * OUT_WAVE <= SMEM && 2 * SMEM <= 163840, "two workgroups per CU");
};

template <bool MUL>
__global__ __launch_bounds__(GpCfg::THREADS, 2) void gemm_planes_kernel(const GemmArgs g) {
    typedef GpCfg C;
    constexpr int TMW = C::TMW, TNW = C::TNW;
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
    const int nk = (kend - kbeg + 15) / 16;

    // Copies: wavefronts 0 and 1 bring the fragments of A (two blocks of rows each), 2 and 3 those of B.  Blocks past the operand's
    // last one read as zero.
    const bool of_b = wave >= 2;
    const int64_t kb = gs_kblocks(g.k), block_bytes = kb * (3 * GS_FRAG);
    const int blocks = ((of_b ? g.m : g.n) + 31) / 32, first = (of_b ? col0 : row0) / 32 + (wave & 1) * 2;
    const int64_t src = (int64_t)(of_b ? g.planes_b : g.planes_a) + (int64_t)first * block_bytes + (int64_t)(kbeg / 16) * (3 * GS_FRAG);
    const char* base = (const char*)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(src >> 32)) << 32) |
                                     (uint32_t)__builtin_amdgcn_readfirstlane((int)src));
    const int have = __builtin_amdgcn_readfirstlane(blocks - first);     // blocks of rows from `first` on
    int left = nk;                                                        // steps not yet requested
    uint32_t slot_in = gt_lds_addr(smem) + wave * (6 * GS_FRAG);
    int in = 0;
    // copy I of the next stage: part I % 3 of block I / 3
    auto copy = [&](auto i) __attribute__((always_inline)) {
        constexpr int blk = i / 3, part = i % 3;
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(base + blk * block_bytes), 0,
                                                            left > 0 && blk < have ? 3 * GS_FRAG : 0, 0x00020000);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsrc, (__attribute__((address_space(3))) void*)(uintptr_t)(slot_in + in * C::STAGE + blk * (3 * GS_FRAG)), 16,
            lane * 16, 0, part * GS_FRAG, 0);
        if constexpr (i == 5) {
            base += 3 * GS_FRAG;
            --left;
            in = in + 1 == C::STAGES ? 0 : in + 1;
        }
    };

    gt_u32x4 fa[3][TMW], fb[3][TNW];                   // fragments of the three parts
    f32x16 acc[TNW][TMW], low[TNW][TMW], hh[TNW][TMW];
#pragma unroll
    for (int i = 0; i < TNW; ++i)
#pragma unroll
        for (int j = 0; j < TMW; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) { acc[i][j][e] = 0.f; low[i][j][e] = 0.f; }
    const uint32_t ra = gt_lds_addr(smem) + wm * (6 * GS_FRAG) + lane * 16;
    const uint32_t rb = gt_lds_addr(smem) + 12 * GS_FRAG + wn * (6 * GS_FRAG) + lane * 16;
    uint32_t addr_a = ra, addr_b = rb;                // of the stage that the refills read
    // The loop is a fixed sequence of volatile assembly: the compiler must neither move a product behind the refill of its operand
    // nor an operand to other registers while its refill is under way.  RD ties the fragment to its registers; a sum of leading
    // products is used behind three more products and GP_ADD's wait (19 wait states behind a 16-pass product).
#define GP_RD(F, ADDR, OFF) asm volatile("ds_read_b128 %0, %1 offset:%2" : "+v"(F) : "v"(ADDR), "n"((OFF) * GS_FRAG))
#define GP_RDA(P, T) GP_RD(fa[P][T], addr_a, (T) * 3 + (P))
#define GP_RDB(P, T) GP_RD(fb[P][T], addr_b, (T) * 3 + (P))
#define GP_LOW(PB, PA, TN, TM) \
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(low[TN][TM]) : "v"(fb[PB][TN]), "v"(fa[PA][TM]))
#define GP_HH(FIRST, TN, TM)                                                                                               \
    do {                                                                                                                   \
        if constexpr (FIRST) asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(hh[TN][TM]) : "v"(fb[0][TN]), "v"(fa[0][TM])); \
        else asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(hh[TN][TM]) : "v"(fb[0][TN]), "v"(fa[0][TM]));  \
    } while (0)
#define GP_ADD(FIRST, TN, TM)                                                               \
    do {                                                                                    \
        if constexpr (!FIRST) {                                                             \
            asm volatile("s_nop 7" : "+v"(hh[TN][TM]));                                     \
            _Pragma("unroll") for (int e = 0; e < 16; ++e) acc[TN][TM][e] += hh[TN][TM][e]; \
            __builtin_amdgcn_sched_barrier(0);                                              \
        }                                                                                   \
    } while (0)
#define GP_COPY(I) do { copy(std::integral_constant<int, I>{}); __builtin_amdgcn_sched_barrier(0); } while (0)

    if (kend - kbeg > GS_PLAIN_K) {
        gt_unroll<0, C::STAGES * 6>([&](auto i) __attribute__((always_inline)) { copy(std::integral_constant<int, i % 6>{}); });
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                fa[p][t] = gt_u32x4{0u, 0u, 0u, 0u};
                fb[p][t] = gt_u32x4{0u, 0u, 0u, 0u};
            }
        asm volatile("s_waitcnt vmcnt(12)\n\ts_barrier" ::: "memory");
        // in the order of the refills: the middle parts first
        GP_RDA(1, 0); GP_RDA(1, 1); GP_RDB(1, 0); GP_RDB(1, 1);
        GP_RDA(2, 0); GP_RDA(2, 1); GP_RDB(0, 0); GP_RDB(0, 1); GP_RDA(0, 0); GP_RDA(0, 1); GP_RDB(2, 0); GP_RDB(2, 1);
        int at = 0;                                   // stage of the step being multiplied
        // One step of 16 contraction elements.  `even`: the leading products start from zero; in the step behind it they are
        // added onto those, and the sums of both steps to acc.
        auto step = [&](auto even) __attribute__((always_inline)) {
            asm volatile("s_waitcnt lgkmcnt(8)" ::: "memory");
            GP_LOW(1, 1, 0, 0); GP_LOW(1, 1, 0, 1); GP_LOW(1, 1, 1, 0); GP_LOW(1, 1, 1, 1);
            at = at + 1 == C::STAGES ? 0 : at + 1;
            addr_a = ra + at * C::STAGE;
            addr_b = rb + at * C::STAGE;
            // this wavefront has read all of the stage, and its copies of the next one have landed; behind the barrier that
            // holds for every wavefront
            asm volatile("s_waitcnt vmcnt(6) lgkmcnt(0)\n\ts_barrier" ::: "memory");
            GP_LOW(0, 1, 0, 0); GP_COPY(0); GP_LOW(0, 1, 1, 0); GP_RDA(1, 0);
            GP_LOW(0, 1, 0, 1); GP_COPY(1); GP_LOW(0, 1, 1, 1); GP_RDA(1, 1);
            GP_LOW(1, 0, 0, 0); GP_COPY(2); GP_LOW(1, 0, 0, 1); GP_RDB(1, 0);
            GP_LOW(1, 0, 1, 0); GP_COPY(3); GP_LOW(1, 0, 1, 1); GP_RDB(1, 1);
            GP_HH(even, 0, 0); GP_COPY(4);
            GP_LOW(0, 2, 0, 0); GP_LOW(0, 2, 1, 0); GP_RDA(2, 0); GP_LOW(0, 2, 0, 1);
            GP_ADD(even, 0, 0);
            GP_HH(even, 0, 1); GP_COPY(5);
            GP_LOW(0, 2, 1, 1); GP_RDA(2, 1);
            GP_HH(even, 1, 0); GP_HH(even, 1, 1); GP_RDB(0, 0); GP_RDB(0, 1);
            GP_LOW(2, 0, 0, 0);
            GP_ADD(even, 0, 1);
            GP_LOW(2, 0, 1, 0); GP_RDA(0, 0);
            GP_ADD(even, 1, 0);
            GP_LOW(2, 0, 0, 1); GP_LOW(2, 0, 1, 1); GP_RDA(0, 1); GP_RDB(2, 0); GP_RDB(2, 1);
            GP_ADD(even, 1, 1);
        };
        constexpr std::bool_constant<true> EVEN{};
        constexpr std::bool_constant<false> ODD{};
        int kt = 0;
        for (; kt + 1 < nk; kt += 2) {
            step(EVEN);
            step(ODD);
        }
        if (kt < nk) {
            step(EVEN);
            asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");
            GP_ADD(false, 0, 0); GP_ADD(false, 0, 1); GP_ADD(false, 1, 0); GP_ADD(false, 1, 1);
        }
        asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");    // the last products, before the vector ALU reads their sums
    }
    // nothing may still be on its way into the stages when the output staging takes their place
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
#undef GP_RD
#undef GP_RDA
#undef GP_RDB
#undef GP_LOW
#undef GP_HH
#undef GP_ADD
#undef GP_COPY
    gs_finish<C, MUL>(g, acc, low, smem, row0, col0, z, kbeg, kend, wave, wm, wn, lane);
}

// the operands split into the workspace at `planes`, then the product
template <bool MUL>
int gp_launch(GemmArgs g, char* planes, hipStream_t st) {
    const int64_t bytes_a = gs_plane_bytes(g.n, g.k);
    g.planes_a = planes;
    g.planes_b = planes + bytes_a;
    const int kblocks = (int)((g.k + 63) / 64);
    const GsSource a = {(const float*)g.a, planes, g.a_row, g.a_k, g.n, g.k, kblocks};
    const GsSource b = {(const float*)g.b, planes + bytes_a, g.b_row, g.b_k, g.m, g.k, kblocks};
    const int64_t blocks_a = (int64_t)((g.n + 31) / 32) * kblocks, blocks_b = (int64_t)((g.m + 31) / 32) * kblocks;
    hipLaunchKernelGGL(gs_planes_kernel, dim3((unsigned)(blocks_a + blocks_b)), dim3(256), 0, st, a, b, (int)blocks_a);
    PTJ_CHECK_LAUNCH();
    const int64_t work = (int64_t)((g.n + GpCfg::TBM - 1) / GpCfg::TBM) * ((g.m + GpCfg::TBN - 1) / GpCfg::TBN) * g.splits;
    hipLaunchKernelGGL((gemm_planes_kernel<MUL>), dim3((unsigned)work), dim3(GpCfg::THREADS), 0, st, g);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}
