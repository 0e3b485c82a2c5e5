// fp32 GEMM on the bf16 matrix pipe.  Included by gemm_tile_launch.h inside its unnamed namespace.  Products whose operands are
// read by many tiles are split ahead of the product instead (gemm_planes.h, same arithmetic).
//
// The three-way split of Henry, Tang and Heinecke ("Leveraging the bfloat16 Artificial Intelligence Datatype For
// Higher-Precision Computations", 2019): every fp32 value is the exact sum of three bf16 values h + m + l (each the
// round-to-nearest of what is left: 8 + 8 + 8 significant bits and two signs cover the 24), so a product of two is the sum of
// nine products of bf16 values, all exact in the fp32 accumulator.  Six of them are formed (hh, hm, mh, hl, lh, mm).  Of the
// other three, |m| <= 2^-8 and |l| <= 2^-17 of the value's power of two bound ml and lm by 2^-25 |a b| each and ll by
// 2^-34: together at most the rounding (2^-24) that a multiply-add makes, 7e-9 rms.  Sixteen products enter the accumulator
// per rounding where the fp32 instructions round after every one.  Measured against fp64, relative to sum |a b|: rms 5.7e-9
// for N(0,1) operands and 7.2e-8 for positive ones at k = 768 (9.1e-9 and 4.7e-8 at k = 64, 3.0e-9 and 6.0e-8 at 4096),
// where the fp32 instructions leave 2.8e-8 in one chain and 1.4e-8 and 1.0e-7 in four (tests/test_gpu_gemm_split.py holds
// the order).  Six v_mfma_f32_32x32x16_bf16 take 192 clocks where eight v_mfma_f32_32x32x2_f32 take 512.
//
// Range.  Unscaled, the parts of values below 2^-110 would leave bf16's range: operands of 1e-37 would come out with 1e-4 of
// error.  Every fp32 number is a multiple of 2^-149 and every bf16 number one of 2^-133, so 2^16 times any fp32 value has its
// three parts exactly (the matrix instructions keep subnormal operands); both operands are split so and the 2^32 is taken
// out of the finished sums.  What that pushes out at the other end -- operands from 2^112, sums from 2^96, also infinities
// and NaN -- leaves an infinite or NaN sum: wavefronts that hold one form their tiles again with the fp32 instructions,
// unscaled (4096x3072x768 wholly so: 460 us).  Contractions of up to four elements go there as well: with so few roundings
// the products left out show (6e-8 -> 9e-8 at worst for a single product).  A scale from the largest value of a panel would
// lose tiny values beside large ones.  The multiplication costs 3 % (108 -> 111 us).
//
// 4096x3072x768: 111-121 us by box, 148-163 on the fp32 instructions.  Under it the chip runs at 1.75 GHz with the matrix
// pipe busy 53 % and LDS 35 % of the clocks: 1060 TFLOP/s of bf16 products, where the bf16 kernels of this size are too.
// The element-wise fetch of ragged steps lies in a loop of its own: a branch in every step around two kinds of loads made
// the register sets meet behind it, with waits and spills, and cost 119-126 us.  Reading the fragments of a chunk under the
// products of the one before it (twice the fragment registers, one barrier in the middle of a step) was slower, 147-156 us.
//
// Panels travel HBM -> registers as fp32, two steps ahead, are split once per workgroup and stored as three bf16 planes
// (the conversion costs 6.5 vector instructions per element, spread between the MFMAs), 32 contraction elements per
// step, double-buffered in LDS.  KMAJOR operands: [row][64 bytes], 16-byte chunks XOR-swizzled; MNMAJOR: [k][rows], read
// through ds_read_b64_tr_b16.  Rows may start at any element: a buffer load needs 4-byte alignment.  What
// lies past the operand's end reads as zero (buffer descriptors), and the last step, whose vectors may hold elements of
// the next row or cross that end, is fetched element by element.  Write-back is that of gemm_tile.h.
typedef float gs_f32x2 __attribute__((ext_vector_type(2)));
typedef short gs_i16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t gs_pk(float a, float b) {
    const gs_f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}
// Operands are split as 2^16 times their value, so accumulators hold 2^32 times the product.
constexpr int GS_PLAIN_K = 4;        // contractions up to this length are left to the fp32 instructions
constexpr float GS_SCALE = 65536.f, GS_UNSCALE = 1.f / (65536.f * 65536.f);

// two values -> the h, m and l parts of GS_SCALE times them, packed
__device__ __forceinline__ void gs_split2(float x0, float x1, uint32_t& h, uint32_t& m, uint32_t& l) {
    x0 *= GS_SCALE;
    x1 *= GS_SCALE;
    h = gs_pk(x0, x1);
    const float r0 = x0 - __uint_as_float(h << 16), r1 = x1 - __uint_as_float(h & 0xffff0000u);
    m = gs_pk(r0, r1);
    l = gs_pk(r0 - __uint_as_float(m << 16), r1 - __uint_as_float(m & 0xffff0000u));
}

template <int MODE, int ROWS, int NT, int NTHREADS>
struct GsOperand {
    static constexpr int BK = 32, VEC = 4;
    static constexpr int PLANE = ROWS * BK * 2;                 // bytes of one bf16 plane
    static constexpr int PER = ROWS * BK / VEC / NTHREADS;      // float4 loads per thread and step
    static constexpr int PITCH = ROWS * 2;                      // MNMAJOR: bytes per k-row of a plane
    static_assert(PER * NTHREADS * VEC == ROWS * BK, "loads divide evenly among the threads");
    uint32_t voff[PER];
    uint32_t loff[PER];                                         // LDS offset inside a plane
    const char* base;
    int64_t left, step;
    bool cut;                                                   // MNMAJOR: the tile ends inside a vector
    gt_u32x4 r[2][PER];                                         // two steps in flight

    __device__ __forceinline__ void init(const void* p, int64_t s_row, int64_t s_k, int row0, int nrows, int kbeg, int k, int tid) {
        const float* first = (const float*)p + (MODE == KMAJOR ? (int64_t)row0 * s_row + kbeg : (int64_t)kbeg * s_k + row0);
        base = (const char*)first;
        left = 4 * (MODE == KMAJOR ? (int64_t)(nrows - 1 - row0) * s_row + (k - kbeg)
                                   : (int64_t)(k - 1 - kbeg) * s_k + (nrows - row0));
        cut = nrows - row0 < ROWS && (nrows - row0) % 4 != 0;
        step = (MODE == KMAJOR ? (int64_t)1 : s_k) * BK * 4;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int v = i * NTHREADS + tid;
            if constexpr (MODE == KMAJOR) {
                const int row = v >> 3, g = v & 7;              // group of four k
                voff[i] = ((uint32_t)row * (uint32_t)s_row + (uint32_t)g * 4u) * 4u;
                loff[i] = row * 64 + (((g >> 1) ^ ((row >> 2) & 3)) << 4) + (g & 1) * 8;
            } else {
                constexpr int VPR = ROWS / 4;                   // vectors per k-row
                const int kk = v / VPR, rv = v - kk * VPR;
                voff[i] = ((uint32_t)kk * (uint32_t)s_k + (uint32_t)rv * 4u) * 4u;
                loff[i] = kk * PITCH + (((rv >> 1) ^ gt_mn_swz<ROWS>(kk)) << 4) + (rv & 1) * 8;
            }
        }
    }

    // Requests the next step's values into register set SET.  kleft: contraction elements from its first one to the end.
    // WHOLE: no vector of the operand crosses its end.
    template <int SET, bool WHOLE>
    __device__ __forceinline__ void load(int kleft, int tid) {
        const uint32_t records = kleft <= 0 ? 0u : (uint32_t)(left < 0xFFFFFF00ll ? left : 0xFFFFFF00ll);
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, records, 0x00020000);
        if (!WHOLE && (MODE == KMAJOR ? kleft > 0 && kleft < BK : cut && kleft > 0 && kleft <= BK)) {
            // (opaque copies: the offsets of these rare loads are formed here and hold no registers through the main loop)
            int lane_id = tid;
            asm volatile("" : "+v"(lane_id));
#pragma unroll
            for (int i = 0; i < PER; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    uint32_t v = voff[i];
                    asm volatile("" : "+v"(v));
                    v += 4 * e;
                    if constexpr (MODE == KMAJOR) v = ((i * NTHREADS + lane_id) & 7) * 4 + e < kleft ? v : 0xFFFFFFF0u;
                    r[SET][i][e] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, v, 0, 0);
                }
        } else {
#pragma unroll
            for (int i = 0; i < PER; ++i)
                r[SET][i] = __builtin_bit_cast(gt_u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, voff[i], 0, 0));
        }
        base += step;
        left -= step;
    }

    // Splits vector I of register set SET and stores its parts into the planes at `lds`.
    template <int SET, int I>
    __device__ __forceinline__ void split_store(char* __restrict__ lds) const {
        float x[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = __uint_as_float(r[SET][I][e]);
        gt_u32x2 h, m, l;
        uint32_t a, b, c;
        gs_split2(x[0], x[1], a, b, c);
        h[0] = a; m[0] = b; l[0] = c;
        gs_split2(x[2], x[3], a, b, c);
        h[1] = a; m[1] = b; l[1] = c;
        *reinterpret_cast<gt_u32x2*>(lds + loff[I]) = h;
        *reinterpret_cast<gt_u32x2*>(lds + PLANE + loff[I]) = m;
        *reinterpret_cast<gt_u32x2*>(lds + 2 * PLANE + loff[I]) = l;
    }

    // Part `plane` of the fragment of MFMA tile t (rows wrow + 32 t ...), contraction chunk c of the step
    __device__ __forceinline__ static bf16x8 frag(const char* __restrict__ lds, int plane, int wrow, int t, int c, int lane) {
        if constexpr (MODE == KMAJOR) {
            const int row = wrow + t * 32 + (lane & 31), ch = c * 2 + (lane >> 5);
            return *reinterpret_cast<const bf16x8*>(lds + plane * PLANE + row * 64 + ((ch ^ ((row >> 2) & 3)) << 4));
        } else {
            const int l16 = lane & 15, mhalf = (lane >> 4) & 1, lg = lane >> 5, kq = l16 >> 2;
            const int piece = (wrow >> 3) + t * 4 + 2 * mhalf + ((l16 & 3) >> 1);
            const char* p = lds + plane * PLANE + (16 * c + 8 * lg + kq) * PITCH + ((piece ^ gt_mn_swz<ROWS>(kq)) << 4) + 8 * (l16 & 1);
            const gs_i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) gs_i16x4*)(p));
            const gs_i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) gs_i16x4*)(p + 4 * PITCH));
            return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
};

template <int TBM_, int TBN_, int WM_, int WN_>
struct GsCfg {
    static constexpr int TBM = TBM_, TBN = TBN_, WM = WM_, WN = WN_, KG = 1;
    static constexpr int NW = WM * WN, THREADS = NW * 64;
    static constexpr int TMW = TBM / WM / 32, TNW = TBN / WN / 32;
    static_assert(TMW * WM * 32 == TBM && TNW * WN * 32 == TBN, "whole MFMA tiles per wavefront");
    static constexpr int CW = TNW * 32;
    static constexpr int STAGE = 3 * (TBM + TBN) * 64;               // planes of one step
    static constexpr int OUT_PITCH = CW + 4, OUT_WAVE = 32 * OUT_PITCH * 4;
    static constexpr int SMEM = 2 * STAGE > NW * OUT_WAVE ? 2 * STAGE : NW * OUT_WAVE;
    static constexpr int BLOCKS = SMEM > 81920 ? 1 : 2;
    static constexpr int WAVES_EU = (BLOCKS * NW + 3) / 4;
};

// acc = the wavefront's TMW x TNW MFMA tiles (from row `row0` of A, column `col0` of B) by the fp32 matrix instructions,
// operands straight from memory: for the rare tiles whose values the split does not take.  Every lane of the wavefront calls it.
// LONG, chain: as for gs_tile.
template <int TMW, int TNW, bool LONG>
__device__ __forceinline__ void gs_plain_product(const GemmArgs& g, f32x16 (&acc)[TNW][TMW], int row0, int col0, int kbeg, int kend,
                                                 int lane, int chain) {
    f32x16 total[TNW][TMW];
    const int lr = lane & 31, lg = lane >> 5;
    const float *pa[TMW], *pb[TNW];
#pragma unroll
    for (int t = 0; t < TMW; ++t) {
        const int row = row0 + t * 32 + lr;
        pa[t] = (const float*)g.a + (int64_t)(row < g.n ? row : g.n - 1) * g.a_row;
    }
#pragma unroll
    for (int t = 0; t < TNW; ++t) {
        const int col = col0 + t * 32 + lr;
        pb[t] = (const float*)g.b + (int64_t)(col < g.m ? col : g.m - 1) * g.b_row;
    }
#pragma unroll
    for (int i = 0; i < TNW; ++i)
#pragma unroll
        for (int j = 0; j < TMW; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = total[i][j][e] = 0.f;
#pragma unroll 1
    for (int64_t k0 = kbeg; k0 < kend; k0 += 16) {
        f32x4 fa[2][TMW], fb[2][TNW];
#pragma unroll
        for (int c = 0; c < 2; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int64_t k = k0 + c * 8 + lg * 4 + e;
#pragma unroll
                for (int t = 0; t < TMW; ++t) fa[c][t][e] = k < kend ? pa[t][k * g.a_k] : 0.f;
#pragma unroll
                for (int t = 0; t < TNW; ++t) fb[c][t][e] = k < kend ? pb[t][k * g.b_k] : 0.f;
            }
        // these instructions round after every product: a sum per 16 of them keeps the error of a long contraction low
#pragma unroll
        for (int i = 0; i < TNW; ++i)
#pragma unroll
            for (int j = 0; j < TMW; ++j) {
                f32x16 part;
#pragma unroll
                for (int e = 0; e < 16; ++e) part[e] = 0.f;
                mma_chunk(part, fb[0][i], fa[0][j]);
                mma_chunk(part, fb[1][i], fa[1][j]);
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] += part[e];
            }
        if constexpr (LONG) {
            if ((k0 - kbeg + 16) % (chain * 32) == 0)
#pragma unroll
                for (int i = 0; i < TNW; ++i)
#pragma unroll
                    for (int j = 0; j < TMW; ++j)
#pragma unroll
                        for (int e = 0; e < 16; ++e) {
                            total[i][j][e] += acc[i][j][e];
                            acc[i][j][e] = 0.f;
                        }
        }
    }
    if constexpr (LONG)
#pragma unroll
        for (int i = 0; i < TNW; ++i)
#pragma unroll
            for (int j = 0; j < TMW; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] += total[i][j][e];
}

// Both accumulators -> the tile of C: unscaled, formed again by the fp32 instructions where a sum is not finite, and written.
template <typename C, bool MUL, bool LONG = false>
__device__ __forceinline__ void gs_finish(const GemmArgs& g, f32x16 (&acc)[C::TNW][C::TMW], const f32x16 (&low)[C::TNW][C::TMW],
                                          char* __restrict__ smem, int row0, int col0, int z, int kbeg, int kend, int wave, int wm,
                                          int wn, int lane, int chain = 0) {
#pragma unroll
    for (int i = 0; i < C::TNW; ++i)
#pragma unroll
        for (int j = 0; j < C::TMW; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] += low[i][j][e];
    float nan = 0.f;          // one multiply-add per element: 0, or NaN if one is not finite
#pragma unroll
    for (int i = 0; i < C::TNW; ++i)
#pragma unroll
        for (int j = 0; j < C::TMW; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) {
                nan = fmaf(acc[i][j][e], 0.f, nan);
                acc[i][j][e] *= GS_UNSCALE;
            }
    if (__builtin_expect(__any(nan != nan) || kend - kbeg <= GS_PLAIN_K, 0))
        gs_plain_product<C::TMW, C::TNW, LONG>(g, acc, row0 + wm * C::TMW * 32, col0 + wn * C::TNW * 32, kbeg, kend, lane, chain);
    __syncthreads();
    gt_write_back<float, C, MUL>(g, acc, smem, row0, col0, z, wave, lane);
}

// LONG: a long contraction whose K split is left out.  One accumulator over all its steps would take a rounding of the whole sum's size
// in each, where a K split has short chains.  So the accumulators are added to totals every `chain` steps, and the rounding of that
// addition starts the next chain (Dekker's fast two-sum: exact where the total is the larger one, else no worse than a rounding).
// Chains are as long as the parts of the K split that the product would have by itself (gs_chain).  Weight gradients of N(0,1)
// operands, 2-norm of the error against fp64 relative to the result, single products / one chain / this: 768x768 over 4096
// elements 1.06e-7 / 2.1e-7 / 9.1e-8, 768x3072 1.33e-7 / 2.1e-7 / 1.28e-7, 768x768 over 1024 8.3e-8 / 1.14e-7 / 7.3e-8
// (tests/test_gpu_weight_groups_error.py).  The totals lie in LDS behind the planes, which the registers have no room for (238 of 256
// are taken).  Weight gradients of twelve blocks, 4096 elements: 4.03 ms in one chain, 4.22 so, 4.14 of it without a fold (the compiler
// orders the loop in another way).  A chain of 256, 384, 512 elements whatever the product: 4.27, 4.24, 4.21; the loads of a step wait for
// each other where the folds are a branch in the loop instead of a loop around it.
template <typename C> constexpr int gs_chain_smem = C::SMEM + C::TBM * C::TBN * 4;

// steps, an even number, for parts of so many elements of k (below 2^20); of one part: more than there are
inline int gs_chain(int part, int k) { return part < 64 || part >= k ? 1 << 20 : part / 64 * 2; }

template <int AMODE, int BMODE, typename C, bool MUL, bool LONG = false>
__device__ __forceinline__ void gs_tile(const GemmArgs& g, int tile_m, int tile_n, int z, char* smem, int chain = 0) {
    constexpr int BK = 32, TMW = C::TMW, TNW = C::TNW;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / C::WN, wn = wave - wm * C::WN;
    const int row0 = tile_m * C::TBM, col0 = tile_n * C::TBN;
    const int kbeg = z * g.k_per_split;
    const int kend = g.splits > 1 && kbeg + g.k_per_split < g.k ? kbeg + g.k_per_split : g.k;
    const int klen = kend - kbeg, nk = (klen + BK - 1) / BK;

    typedef GsOperand<AMODE, C::TBM, TMW, C::THREADS> OA;
    typedef GsOperand<BMODE, C::TBN, TNW, C::THREADS> OB;
    OA oa;
    OB ob;
    oa.init(g.a, g.a_row, g.a_k, row0, g.n, kbeg, g.k, tid);
    ob.init(g.b, g.b_row, g.b_k, col0, g.m, kbeg, g.k, tid);
    constexpr int NV = OA::PER + OB::PER;                            // vectors per thread and step
    char* const sA = smem;
    char* const sB = smem + 3 * OA::PLANE;                           // behind the A planes of the same stage

    // The matrix pipe rounds its accumulator once per instruction, more coarsely than a vector add: the products of the
    // leading parts are summed over one step (part) and added to acc by the vector ALU, and the five small terms are
    // kept out of the sum that is large (low).
    f32x16 acc[TNW][TMW], part[TNW][TMW], low[TNW][TMW];
#pragma unroll
    for (int i = 0; i < TNW; ++i)
#pragma unroll
        for (int j = 0; j < TMW; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) { acc[i][j][e] = 0.f; low[i][j][e] = 0.f; }

    // FIRST: the accumulators become the thread's totals; else they are added to them and the rounding of that is left in their place;
    // LAST: the totals there, the rounding in `low`
    enum { FIRST, MORE, LAST };
    f32x4* const total = (f32x4*)(smem + C::SMEM) + wave * (TNW * TMW * 4 * 64) + lane;
    auto fold = [&](auto which) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < TNW; ++i)
#pragma unroll
            for (int j = 0; j < TMW; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    f32x4& t = total[((i * TMW + j) * 4 + q) * 64];
                    f32x4 was{}, sum;
                    if constexpr (which != FIRST) was = t;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float a = acc[i][j][q * 4 + e], s = was[e] + a, rest = a - (s - was[e]);
                        sum[e] = which == FIRST ? a : s;
                        acc[i][j][q * 4 + e] = which == FIRST ? 0.f : which == LAST ? s : rest;
                        if constexpr (which == LAST) low[i][j][q * 4 + e] += rest;
                    }
                    if constexpr (which != LAST) t = sum;
                }
    };

    auto split_piece = [&](auto set, auto i, int buf) __attribute__((always_inline)) {
        if constexpr (i < OA::PER) oa.template split_store<set, i>(sA + buf * C::STAGE);
        else ob.template split_store<set, i - OA::PER>(sB + buf * C::STAGE);
    };
    // One contraction chunk (16 wide) of stage `buf`: six products per MFMA tile; with `split` the vectors [v0, v1) of
    // register set `set` are converted into the other stage between them.
    auto chunk = [&](auto c, auto buf, auto set, auto v0, auto v1) __attribute__((always_inline)) {
        bf16x8 fa[3][TMW], fb[3][TNW];
#pragma unroll
        for (int p = 0; p < 3; ++p) {
#pragma unroll
            for (int t = 0; t < TMW; ++t) fa[p][t] = OA::frag(sA + buf * C::STAGE, p, wm * TMW * 32, t, c, lane);
#pragma unroll
            for (int t = 0; t < TNW; ++t) fb[p][t] = OB::frag(sB + buf * C::STAGE, p, wn * TNW * 32, t, c, lane);
        }
        constexpr int PA[6] = {0, 2, 0, 1, 1, 0}, PB[6] = {0, 0, 2, 1, 0, 1};
        gt_unroll<0, 6>([&](auto term) __attribute__((always_inline)) {
#pragma unroll
            for (int tn = 0; tn < TNW; ++tn)
#pragma unroll
                for (int tm = 0; tm < TMW; ++tm) {
                    const bf16x8 b = fb[PB[term]][tn], a = fa[PA[term]][tm];
                    if constexpr (term == 0) {
                        f32x16 zero;
#pragma unroll
                        for (int e = 0; e < 16; ++e) zero[e] = 0.f;
                        part[tn][tm] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, c == 0 ? zero : part[tn][tm], 0, 0, 0);
                    } else {
                        low[tn][tm] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b, a, low[tn][tm], 0, 0, 0);
                    }
                    if constexpr (c == 1 && term == 4) {
#pragma unroll
                        for (int e = 0; e < 16; ++e) acc[tn][tm][e] += part[tn][tm][e];
                    }
                }
            constexpr int nv = v1 - v0;
            if constexpr (nv > 0)
                gt_unroll<v0 + term * nv / 6, v0 + (term + 1) * nv / 6>(
                    [&](auto i) __attribute__((always_inline)) { split_piece(set, i, 1 - buf); });
        });
    };
    auto load = [&](auto set, auto whole, int kleft) __attribute__((always_inline)) {
        oa.template load<set, whole>(kleft, tid);
        ob.template load<set, whole>(kleft, tid);
    };
    constexpr std::integral_constant<int, 0> I0{};
    constexpr std::integral_constant<int, 1> I1{};
    constexpr std::integral_constant<int, (NV + 1) / 2> IH{};
    constexpr std::integral_constant<int, NV> IN{};
    // Step kt (stage kt & 1) while the values of step kt + 1 (register set (kt + 1) & 1) are split into the other stage;
    // the set is then refilled with step kt + 3.
    auto step = [&](auto par, auto whole, int kt) __attribute__((always_inline)) {
        constexpr std::integral_constant<int, 1 - par> NEXT{};
        chunk(I0, par, NEXT, I0, IH);
        chunk(I1, par, NEXT, IH, IN);
        load(NEXT, whole, klen - (kt + 3) * BK);
        __syncthreads();
    };
    // no vector of either operand crosses a row's or the operand's end in any step
    const bool whole_vectors = ((AMODE != KMAJOR && BMODE != KMAJOR) || klen % BK == 0) && (AMODE == KMAJOR || !oa.cut) &&
                               (BMODE == KMAJOR || !ob.cut);
    if (klen > GS_PLAIN_K) {
        constexpr std::bool_constant<true> WHOLE{};
        constexpr std::bool_constant<false> ANY{};
        load(I0, ANY, klen);
        load(I1, ANY, klen - BK);
        gt_unroll<0, NV>([&](auto i) __attribute__((always_inline)) { split_piece(I0, i, 0); });
        load(I0, ANY, klen - 2 * BK);
        __syncthreads();
        auto all_steps = [&](auto whole) __attribute__((always_inline)) {
            int kt = 0;
            if constexpr (LONG) {
                for (int end = chain; end + 1 < nk; end += chain) {
                    for (; kt < end; kt += 2) {
                        step(I0, whole, kt);
                        step(I1, whole, kt + 1);
                    }
                    if (end == chain) fold(std::integral_constant<int, FIRST>{});
                    else fold(std::integral_constant<int, MORE>{});
                }
            }
            for (; kt + 1 < nk; kt += 2) {
                step(I0, whole, kt);
                step(I1, whole, kt + 1);
            }
            if (kt < nk) step(I0, whole, kt);
            if constexpr (LONG)
                if (chain + 1 < nk) fold(std::integral_constant<int, LAST>{});
        };
        if (whole_vectors) all_steps(WHOLE);
        else all_steps(ANY);
    }
    gs_finish<C, MUL, LONG>(g, acc, low, smem, row0, col0, z, kbeg, kend, wave, wm, wn, lane, chain);
}

template <int AMODE, int BMODE, typename C, bool MUL>
__global__ __launch_bounds__(C::THREADS, C::WAVES_EU) void gemm_split_kernel(const GemmArgs g) {
    __shared__ __attribute__((aligned(1024))) char smem[C::SMEM];
    int tile_m, tile_n, z;
    gt_item(g, blockIdx.x, (g.n + C::TBM - 1) / C::TBM, (g.m + C::TBN - 1) / C::TBN, tile_m, tile_n, z);
    gs_tile<AMODE, BMODE, C, MUL>(g, tile_m, tile_n, z, smem);
}

// A tile of a group of products
template <typename C>
__global__ __launch_bounds__(C::THREADS, C::WAVES_EU) void gemm_split_group_kernel(const ptj_gemm_detail::GemmGroup group) {
    __shared__ __attribute__((aligned(1024))) char smem[gs_chain_smem<C>];
    int kind, block, tile_m, tile_n;
    group_tile<false>(group, blockIdx.x, C::TBM, C::TBN, kind, block, tile_m, tile_n);
    GemmArgs g{};
    g.a = group.p.d[kind][block];
    g.b = group.p.x[kind][block];
    g.c = group.p.dw[kind][block];
    g.n = group.p.n[kind];
    g.m = group.p.m[kind];
    g.k = g.k_per_split = group.p.k;
    g.a_row = g.b_row = 1;
    g.a_k = g.n;
    g.b_k = g.c_rs = g.m;
    g.splits = g.tail_splits = g.vec_out = 1;
    gs_tile<MNMAJOR, MNMAJOR, C, false, true>(g, tile_m, tile_n, 0, smem, group.chain[kind]);
}
// parts[kind]: what the K split of a single product would be
template <typename C>
int gs_group_launch(const PtjGradGroup& p, const int (&parts)[PtjGradGroup::KINDS], hipStream_t st) {
    ptj_gemm_detail::GemmGroup g = group_of<C>(p);
    for (int i = 0; i < PtjGradGroup::KINDS; ++i) g.chain[i] = gs_chain(parts[i], p.k);
    hipLaunchKernelGGL((gemm_split_group_kernel<C>), dim3((unsigned)(g.first[PtjGradGroup::KINDS] * p.blocks)), dim3(C::THREADS), 0, st, g);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

template <typename C, bool MUL>
int gs_launch(const GemmArgs& g, int am, int bm, hipStream_t st) {
    const int64_t work = (int64_t)((g.n + C::TBM - 1) / C::TBM) * ((g.m + C::TBN - 1) / C::TBN) * g.splits;
    const dim3 grid((unsigned)work), block(C::THREADS);
#define GS_LAUNCH(AM, BMD) hipLaunchKernelGGL((gemm_split_kernel<AM, BMD, C, MUL>), grid, block, 0, st, g)
    switch (am * 3 + bm) {
        case 0: GS_LAUNCH(KMAJOR, KMAJOR); break;
        case 1: GS_LAUNCH(KMAJOR, MNMAJOR); break;
        case 3: GS_LAUNCH(MNMAJOR, KMAJOR); break;
        default: GS_LAUNCH(MNMAJOR, MNMAJOR); break;
    }
#undef GS_LAUNCH
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}
