// Persistent bf16 GEMM whose operand panels travel HBM -> LDS by asynchronous buffer copies into two rings,
// one per operand.  Included by gemm_core.h inside its unnamed namespace, after gemm_tile.h.
//
// What bounds it: the LDS and the matrix pipe together.  Per 64 contraction elements a 256x256 tile (eight wavefronts of
// 128x64) costs 2048 clocks of MFMAs, 1536 of fragment reads and 512 of arriving copies; a 256x192 tile
// (wavefronts of 64x96) 1536, 1280 and 448, so the wider tile gets more out of the matrix pipe and the narrower one is for
// outputs that it cuts into fuller rounds (gemm_plan.h).  The A ring has three stages and the B ring two: the chunks
// of a step are read into registers half a step ahead, so a stage is refilled halfway through the step that
// multiplies it, and the copies of A have a step more to arrive than those of B.  160 KB hold no third stage
// of B.  Reads and copies are spread over the MFMAs (bunched behind the barrier: 5 % slower).  What a step does besides is
// kept small and away from the barrier, where both wavefronts of a SIMD wait and the matrix pipe idles: 167
// instructions beside 32 MFMAs.
// 8192x8192x8192: 783 us, 1400 TFLOP/s (the loops with two stages of 56 KB before this one: 975 us); 4096^3 with both
// operands transposed 107 (147); 16384x768x3072 68 (74), with transposed B 67 (79).  Four wavefronts of 128x128 with one
// chunk per register set: 905 us for 8192^3.
//
// The output goes straight from the accumulators to memory: two lane swaps bring eight consecutive columns of a row
// into a lane and 64 bytes of each of sixteen rows into a store, without LDS, which the rings fill.  At k = 768 the
// output is a quarter of the time (16384x3072x768: 81 us, 60 without stores; 100 MB at 4.9 TB/s are 20).
// GELU and its derivative come from one exponential (130 -> 118 us for 16384x3072x768 with both outputs).
//
// The copies run ahead across the tiles of a workgroup, but a tile's start waits for them all the same: the accumulators start
// from bias registers that a vector path, an element path or zeros may have filled, and the compiler puts s_waitcnt vmcnt(0)
// in front of their use, with a bias or without.  That drains the stores of the tile before as well, and in the 256x256 kernels
// spilled registers (33-50 in all) are reloaded there.  Measured with this in place: stores kept in registers and sent between the MFMAs
// of the next tile 86 us instead of 81; non-temporal ones 75, and 8192x50257x768 with them 620 -> 690; waits that leave
// younger operations in flight the same.  None of it says what they would do without the drain.
//
// Rows and contraction indices past the operand's end read as zero (buffer descriptors).

// TBM x TBN tile of C by WM x WN wavefronts
template <int TBN_, int WM_, int WN_>
struct RingCfg {
    static constexpr int TBM = 256, TBN = TBN_, WM = WM_, WN = WN_, NA = 3, NB = 2;
    static constexpr int NW = WM * WN, THREADS = NW * 64, TMW = TBM / WM / 32, TNW = TBN / WN / 32;
    static_assert(TMW * WM * 32 == TBM && TNW * WN * 32 == TBN && NW == 8, "whole MFMA tiles, two wavefronts per SIMD");
    static constexpr int A_STAGE = TBM * BKB, B_STAGE = TBN * BKB, SMEM = NA * A_STAGE + NB * B_STAGE;
};
typedef RingCfg<256, 2, 4> RingFull;
typedef RingCfg<192, 4, 2> RingNarrow;

// A work item: a C tile, or one K slice of one.  part: dense partial tile of a K-split tile of the last round.
struct RingItem {
    int row0, col0, kbeg, klen, z;
    float* part;
};
template <typename C>
__device__ __forceinline__ RingItem ring_item(const GemmArgs& g, int item) {
    const int num_m = (g.n + C::TBM - 1) / C::TBM, num_n = (g.m + C::TBN - 1) / C::TBN;
    RingItem d;
    int tm, tn, kps = g.splits > 1 ? g.k_per_split : g.k;
    d.part = nullptr;
    if (g.tail_splits > 1 && item >= g.tail_first) {
        const int r = item - g.tail_first, t = r / g.tail_splits;
        gt_item(g, g.tail_first + t, num_m, num_n, tm, tn, d.z);
        d.z = r - t * g.tail_splits;
        kps = g.tail_kps;
        d.part = g.partial + (int64_t)r * (C::TBM * C::TBN);
    } else {
        gt_item(g, item, num_m, num_n, tm, tn, d.z);
    }
    d.row0 = tm * C::TBM;
    d.col0 = tn * C::TBN;
    d.kbeg = d.z * kps;
    d.klen = (d.kbeg + kps < g.k ? d.kbeg + kps : g.k) - d.kbeg;
    return d;
}

// A wave-uniform value into scalar registers (a descriptor that the compiler cannot tell to be uniform costs a loop per copy)
__device__ __forceinline__ int64_t ring_uniform(int64_t v) {
    return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
}

// One operand: the cursor of its copies, which runs ahead of the multiplications across work items, and the LDS addresses
// of this wavefront's fragments.  ROWS rows of the tile in a stage, NT MFMA tiles of 32 rows per wavefront.
template <int MODE, int ROWS, int NT, int STAGES>
struct RingOperand {
    static constexpr int NW = 8, PER = ROWS * BKB / 1024 / NW;           // copies per wavefront and stage
    static constexpr int PPR = ROWS / 8, PITCH = ROWS * 2;               // MNMAJOR: 16-byte pieces and bytes per k-row
    // the copies of a stage lie a whole number of swizzle periods apart: one address register for all of them
    static constexpr bool EVEN = MODE == KMAJOR || (NW * 64 % PPR == 0 && NW * 64 / PPR % 4 == 0);
    uint32_t voff[EVEN ? 1 : PER], istep;
    int kk;                                                              // KMAJOR: k of this lane's vector in a step
    uint32_t raddr[MODE == KMAJOR ? 1 : NT];
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t v0;
    const char* base;                                                    // the next stage's first element
    int64_t left, step;                                                  // bytes from there to the operand's end; per stage
    int item, kleft, slot;                                               // kleft: contraction elements of the item not yet requested

    __device__ __forceinline__ void init(int64_t s_row, int64_t s_k, uint32_t region, int wrow, int tid) {
        const int lane = tid & 63;
        if constexpr (MODE == KMAJOR) {
            const int r = tid >> 3, row = wrow + (lane & 31);
            kk = ((lane & 7) ^ sw(r)) * 8;
            voff[0] = ((uint32_t)r * (uint32_t)s_row + (uint32_t)kk) * 2u;
            istep = NW * 8 * (uint32_t)s_row * 2u;
            step = 128;
            raddr[0] = region + row * BKB + (((lane >> 5) ^ sw(row)) << 4);
        } else {
            const int l16 = lane & 15, mhalf = (lane >> 4) & 1, lg = lane >> 5, kq = l16 >> 2;
            kk = 0;
#pragma unroll
            for (int i = 0; i < (EVEN ? 1 : PER); ++i) {
                const int pc = i * NW * 64 + tid, k = pc / PPR, pos = pc - k * PPR;
                voff[i] = ((uint32_t)k * (uint32_t)s_k + (uint32_t)(pos ^ gt_mn_swz<ROWS>(k)) * 8u) * 2u;
            }
            istep = NW * 64 / PPR * (uint32_t)s_k * 2u;
            step = 128 * s_k;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int piece = (wrow >> 3) + t * 4 + 2 * mhalf + ((l16 & 3) >> 1);
                raddr[t] = region + (8 * lg + kq) * PITCH + ((piece ^ gt_mn_swz<ROWS>(kq)) << 4) + 8 * (l16 & 1);
            }
        }
        slot = 0;
    }
    __device__ __forceinline__ void start(const void* p, int64_t s_row, int64_t s_k, int row0, int nrows, int kbeg, int klen, int k) {
        const bf16* first = (const bf16*)p + (MODE == KMAJOR ? (int64_t)row0 * s_row + kbeg : (int64_t)kbeg * s_k + row0);
        base = (const char*)ring_uniform((int64_t)first);
        left = ring_uniform(2 * (MODE == KMAJOR ? (int64_t)(nrows - 1 - row0) * s_row + ((k - kbeg + 7) >> 3 << 3)
                                                : (int64_t)(k - 1 - kbeg) * s_k + ((nrows - row0 + 7) >> 3 << 3)));
        kleft = __builtin_amdgcn_readfirstlane(klen);
    }
    // The next stage: descriptor and address of its first copy.  Past the last item nothing is fetched and the stage fills with
    // zeros; lanes past the end of their row (the next row's data) point past the operand.
    __device__ __forceinline__ void begin_stage() {
        const uint32_t records = kleft <= 0 ? 0u : (uint32_t)(left < 0x80000000ll ? left : 0x80000000ll);
        rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, records, 0x00020000);
        v0 = voff[0];
        if constexpr (MODE == KMAJOR) {
            if (kleft < 64) v0 = kk < kleft ? v0 : 0x80000000u;
        }
    }
    template <int I>
    __device__ __forceinline__ void copy(uint32_t stage) const {
        uint32_t v = EVEN ? v0 : voff[EVEN ? 0 : I];
        if constexpr (EVEN && I > 0) asm volatile("v_add_u32 %0, %1, %2" : "=v"(v) : "s"(I * istep), "v"(v0));   // (not kept over the loop)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(uintptr_t)(stage + I * NW * 1024), 16, v, 0, 0, 0);
    }
    // LDS address of the fragments of chunk CH (KMAJOR: of every MFMA tile; MNMAJOR: of tile CH, every chunk) of the stage at
    // byte offset soff
    template <int CH>
    __device__ __forceinline__ uint32_t read_addr(uint32_t soff) const {
        uint32_t a;
        if constexpr (MODE != KMAJOR) a = raddr[CH] + soff;
        else if constexpr (CH < 3) asm volatile("v_xad_u32 %0, %1, %2, %3" : "=v"(a) : "v"(raddr[0]), "n"(CH << 5), "s"(soff));
        else asm volatile("v_xor_b32 %0, 0x60, %1\n\tv_add_u32 %0, %2, %0" : "=&v"(a) : "v"(raddr[0]), "s"(soff));
        return a;
    }
    // fragment of MFMA tile TI, chunk CH
    template <int CH, int TI>
    __device__ __forceinline__ static void read_one(GtFrag<bf16, MODE>& f, uint32_t addr) {
        if constexpr (MODE == KMAJOR) f.template read<TI * 32 * BKB>(addr);
        else f.template read<16 * CH * PITCH, PITCH>(addr);
    }
    // KMAJOR: clears the elements of every row of a stage from contraction index `tail` to the end of their vector
    __device__ __forceinline__ static void clear_tail(char* __restrict__ stage, int tail, int tid) {
        if constexpr (MODE == KMAJOR) {
            if (tail % 8 == 0 || tid >= ROWS) return;
            bf16* p = (bf16*)(stage + tid * BKB + (((tail / 8) ^ sw(tid)) << 4));
            for (int e = tail % 8; e < 8; ++e) p[e] = from_f32<bf16>(0.f);
        }
    }
};

// lanes 32-63 of a <-> lanes 0-31 of b;  in each half, lanes 16-31 of a <-> lanes 0-15 of b
__device__ __forceinline__ void ring_swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void ring_swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ uint32_t ring_pack2(float a, float b) {
    const f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}

// Write-back of a 32x32 accumulator tile.  acc[i] of lane (lr, lg) is row lr, column (i/4)*8 + lg*4 + i%4; d holds those values
// rounded, two a word.  Afterwards lane l has in out[h] the eight columns (l>>4 & 1)*16 + (l>>5)*8 ... of row h*16 + (l & 15).
__device__ __forceinline__ void ring_rows(uint32_t (&d)[8], gt_u32x4 (&out)[2]) {
    ring_swap32(d[0], d[2]);
    ring_swap32(d[1], d[3]);
    ring_swap32(d[4], d[6]);
    ring_swap32(d[5], d[7]);
#pragma unroll
    for (int i = 0; i < 4; ++i) ring_swap16(d[i], d[4 + i]);
    out[0] = gt_u32x4{d[0], d[1], d[2], d[3]};
    out[1] = gt_u32x4{d[4], d[5], d[6], d[7]};
}

// What becomes of an accumulator: RAW itself, GELU its GELU, BOTH the GELU's derivative as well (second output)
enum { RING_RAW, RING_GELU, RING_BOTH };
template <int ACT>
__device__ __forceinline__ void ring_pack_tile(const f32x16& acc, gt_u32x4 (&out)[2], gt_u32x4 (&aux)[2]) {
    uint32_t d[8], a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        float x = acc[2 * i], y = acc[2 * i + 1];
        if constexpr (ACT == RING_GELU) { x = gelu_f(x); y = gelu_f(y); }
        if constexpr (ACT == RING_BOTH) {
            float dx, dy;
            gelu_both_f(acc[2 * i], x, dx);
            gelu_both_f(acc[2 * i + 1], y, dy);
            a[i] = ring_pack2(dx, dy);
        }
        d[i] = ring_pack2(x, y);
    }
    ring_rows(d, out);
    if constexpr (ACT == RING_BOTH) ring_rows(a, aux);
}

// Memory behind a pointer that came through ring_args: the compiler cannot tell that it is global, and an access that might
// be to LDS counts where the waits for LDS reads look.
typedef __attribute__((address_space(1))) char ring_global;

// Wave-uniform addresses of the rows 0 and 16 of an MFMA tile, moved from one row of tiles to the next (opaque, or the compiler
// forms all of them ahead and spills scalar registers)
struct RingRows {
    ring_global *p0, *p1;
    int64_t bytes;                    // of 16 rows
    __device__ __forceinline__ RingRows(const void* base, int64_t rs, int elt) : p0((ring_global*)base), bytes(16 * rs * elt) {
        asm volatile("" : "+s"(p0), "+s"(bytes));
        p1 = p0 + bytes;
    }
    // T at byte `off` of the lane's part of row 16 h
    template <typename T, typename OFF> __device__ __forceinline__ __attribute__((address_space(1))) T* at(int h, int off, OFF voff) const {
        return (__attribute__((address_space(1))) T*)((h ? p1 : p0) + off + voff);
    }
    __device__ __forceinline__ void next() {
        p0 = p1 + bytes;
        asm volatile("" : "+s"(p0));
        p1 = p0 + bytes;
    }
};

// Pitches from which on the offset of a lane's row, up to 15 rows, leaves 32 bits: such blocks are written like those at the
// borders, whose offsets have 64 bits (ring_far).
constexpr int64_t RING_WIDE = 1ll << 27;
// bytes to the lane's part of its row, formed where they are used (opaque: only the borders hold registers for them)
__device__ __forceinline__ int64_t ring_far(int lrow, int lcol, int64_t rs) {
    asm volatile("" : "+v"(lrow));
    return ((int64_t)lrow * rs + lcol) * 2;
}

// half word e of a vector (borders of C: a loop, so that the kernels stay small)
__device__ __forceinline__ uint16_t ring_half(const gt_u32x4& v, int e) {
    const uint32_t w = e < 4 ? (e < 2 ? v[0] : v[1]) : (e < 6 ? v[2] : v[3]);
    return (uint16_t)(w >> (16 * (e & 1)));
}

// Eight columns of a row, of which `ne` are inside C
__device__ __forceinline__ void ring_store(__attribute__((address_space(1))) bf16* p, const gt_u32x4& v, int ne, bool aligned) {
    if (aligned && ne >= 8) {
        *(__attribute__((address_space(1))) gt_u32x4*)p = v;
    } else {
#pragma unroll 1
        for (int e = 0; e < (ne < 8 ? ne : 8); ++e) p[e] = __builtin_bit_cast(bf16, ring_half(v, e));
    }
}

// The wavefront's block at (row0, col0) as ACT of the accumulators, to c (and aux).  Addresses are a wave-uniform part and one
// offset per lane, 32 bits wide in whole blocks, formed here (fresh_tid) so that they hold no registers through the main loop.
template <typename C, int ACT>
__device__ __forceinline__ void ring_write(const GemmArgs& g, const f32x16 (&acc)[C::TNW][C::TMW], bf16* c, int64_t rs, bf16* aux,
                                           int64_t aux_rs, int row0, int col0) {
    const int lane = fresh_tid() & 63, lrow = lane & 15, lcol = ((lane >> 4) & 1) * 16 + (lane >> 5) * 8;
    RingRows cr(c + (int64_t)row0 * rs + col0, rs, 2), ar(aux + (int64_t)row0 * aux_rs + col0, aux_rs, 2);
    const uint32_t voff = ((uint32_t)lrow * (uint32_t)rs + (uint32_t)lcol) * 2u, aoff = ((uint32_t)lrow * (uint32_t)aux_rs + (uint32_t)lcol) * 2u;
    const bool aligned = g.vec_out, whole = aligned && rs < RING_WIDE && aux_rs < RING_WIDE && row0 + C::TMW * 32 <= g.n &&
                                            col0 + C::TNW * 32 <= g.m;   // wave-uniform
    const int rows = g.n - row0 - lrow, cols = g.m - col0 - lcol;
#pragma unroll
    for (int tm = 0; tm < C::TMW; ++tm) {
#pragma unroll
        for (int tn = 0; tn < C::TNW; ++tn) {
            gt_u32x4 v[2], w[2];
            ring_pack_tile<ACT>(acc[tn][tm], v, w);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                if (whole) {
                    *cr.at<gt_u32x4>(h, tn * 64, voff) = v[h];
                    if constexpr (ACT == RING_BOTH) *ar.at<gt_u32x4>(h, tn * 64, aoff) = w[h];
                } else {
                    int ne = cols;                        // (opaque: no lane masks kept from one store to the next)
                    asm volatile("" : "+v"(ne));
                    ne = tm * 32 + h * 16 < rows ? ne - tn * 32 : 0;
                    ring_store(cr.at<bf16>(h, tn * 64, ring_far(lrow, lcol, rs)), v[h], ne, aligned);
                    if constexpr (ACT == RING_BOTH) ring_store(ar.at<bf16>(h, tn * 64, ring_far(lrow, lcol, aux_rs)), w[h], ne, aligned);
                }
            }
        }
        cr.next();
        if constexpr (ACT == RING_BOTH) ar.next();
    }
}

// fp32 partial sums of the block at (row0, col0) of dst, rows of `rs` elements and 16-byte aligned where 4 divides rs; four
// columns of row h*16 + (l & 15) per lane and store.  (rs is a tile's width or that of an output of fewer than 2 num_cus
// tiles, the only ones that are K-split: 32-bit offsets.)
template <typename C>
__device__ __forceinline__ void ring_write_partial(const f32x16 (&acc)[C::TNW][C::TMW], float* __restrict__ dst, int64_t rs, int row0,
                                                   int col0, int nrows, int ncols) {
    const int lane = fresh_tid() & 63, lrow = lane & 15, lcol = ((lane >> 4) & 1) * 8 + (lane >> 5) * 4;
    RingRows pr(dst + (int64_t)row0 * rs + col0, rs, 4);
    const uint32_t voff = ((uint32_t)lrow * (uint32_t)rs + (uint32_t)lcol) * 4u;
    const bool whole = rs % 4 == 0 && row0 + C::TMW * 32 <= nrows && col0 + C::TNW * 32 <= ncols;
#pragma unroll
    for (int tm = 0; tm < C::TMW; ++tm) {
#pragma unroll
        for (int tn = 0; tn < C::TNW; ++tn)
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                uint32_t x[4], y[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x[e] = __float_as_uint(acc[tn][tm][q * 8 + e]);
                    y[e] = __float_as_uint(acc[tn][tm][q * 8 + 4 + e]);
                    ring_swap16(x[e], y[e]);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const uint32_t* s = h ? y : x;
                    if (whole) {
                        *pr.at<gt_u32x4>(h, (tn * 32 + q * 16) * 4, voff) = gt_u32x4{s[0], s[1], s[2], s[3]};
                    } else {
                        int ne = ncols - col0 - lcol;
                        asm volatile("" : "+v"(ne));
                        ne = row0 + tm * 32 + h * 16 + lrow < nrows ? ne - (tn * 32 + q * 16) : 0;
#pragma unroll 1
                        for (int e = 0; e < (ne < 4 ? ne : 4); ++e)
                            pr.at<float>(h, (tn * 32 + q * 16) * 4, voff)[e] = __uint_as_float(e < 2 ? (e < 1 ? s[0] : s[1]) : (e < 3 ? s[2] : s[3]));
                    }
                }
            }        pr.next();
    }
}

// C = round(acc) * mul and the column sums of what is stored over the wavefront's TMW * 32 rows (g.colpart).  The
// multipliers of a row of MFMA tiles are requested while the one before it is multiplied.
template <typename C>
__device__ __forceinline__ void ring_write_mul(const GemmArgs& g, const f32x16 (&acc)[C::TNW][C::TMW], int row0, int col0) {
    constexpr int TMW = C::TMW, TNW = C::TNW;
    const int lane = fresh_tid() & 63, lrow = lane & 15, lcol = ((lane >> 4) & 1) * 16 + (lane >> 5) * 8;
    const int64_t mul_rs = g.mul_rs, c_rs = g.c_rs;
    RingRows mr((bf16*)g.mul + (int64_t)row0 * mul_rs + col0, mul_rs, 2), cr((bf16*)g.c + (int64_t)row0 * c_rs + col0, c_rs, 2);
    const uint32_t moff = ((uint32_t)lrow * (uint32_t)mul_rs + (uint32_t)lcol) * 2u, coff = ((uint32_t)lrow * (uint32_t)c_rs + (uint32_t)lcol) * 2u;
    const bool aligned = g.vec_out, whole = aligned && mul_rs < RING_WIDE && c_rs < RING_WIDE && row0 + TMW * 32 <= g.n &&
                                            col0 + TNW * 32 <= g.m;   // wave-uniform
    const int rows = g.n - row0 - lrow, cols = g.m - col0 - lcol;
    float cs[TNW][8];
#pragma unroll
    for (int tn = 0; tn < TNW; ++tn)
#pragma unroll
        for (int e = 0; e < 8; ++e) cs[tn][e] = 0.f;
    gt_u32x4 mv[2][TNW][2];
    auto request = [&](auto tm) __attribute__((always_inline)) {
        if (whole) {
#pragma unroll
            for (int tn = 0; tn < TNW; ++tn)
#pragma unroll
                for (int h = 0; h < 2; ++h) mv[tm & 1][tn][h] = *mr.at<gt_u32x4>(h, tn * 64, moff);
        } else {
#pragma unroll
            for (int tn = 0; tn < TNW; ++tn)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    int ne = cols;
                    asm volatile("" : "+v"(ne));
                    ne = tm * 32 + h * 16 < rows ? ne - tn * 32 : 0;
                    uint32_t w[4] = {0u, 0u, 0u, 0u};
                    if (aligned && ne >= 8) {
                        const gt_u32x4 all = *mr.at<gt_u32x4>(h, tn * 64, ring_far(lrow, lcol, mul_rs));
#pragma unroll
                        for (int e = 0; e < 4; ++e) w[e] = all[e];
                    } else {
#pragma unroll 1
                        for (int e = 0; e < (ne < 8 ? ne : 8); ++e) {
                            const uint32_t x = (uint32_t)*(mr.at<uint16_t>(h, tn * 64, ring_far(lrow, lcol, mul_rs)) + e) << (16 * (e & 1));
#pragma unroll
                            for (int i = 0; i < 4; ++i) w[i] |= i == e >> 1 ? x : 0u;
                        }
                    }
                    mv[tm & 1][tn][h] = gt_u32x4{w[0], w[1], w[2], w[3]};
                }
        }
        mr.next();
    };
    request(std::integral_constant<int, 0>{});
    gt_unroll<0, TMW>([&](auto tm) __attribute__((always_inline)) {
        if constexpr (tm + 1 < TMW) request(std::integral_constant<int, tm + 1>{});
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int tn = 0; tn < TNW; ++tn) {
            gt_u32x4 v[2], none[2];
            ring_pack_tile<RING_RAW>(acc[tn][tm], v, none);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                Pack<bf16, 8> s = __builtin_bit_cast(Pack<bf16, 8>, v[h]);
                const Pack<bf16, 8> m = __builtin_bit_cast(Pack<bf16, 8>, mv[tm & 1][tn][h]);
#pragma unroll
                for (int e = 0; e < 8; ++e) s.v[e] = from_f32<bf16>(to_f32(s.v[e]) * to_f32(m.v[e]));
                if (whole) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) cs[tn][e] += to_f32(s.v[e]);
                    *cr.at<gt_u32x4>(h, tn * 64, coff) = __builtin_bit_cast(gt_u32x4, s);
                } else {
                    int ne = cols;
                    asm volatile("" : "+v"(ne));
                    ne = tm * 32 + h * 16 < rows ? ne - tn * 32 : 0;
                    if (aligned && ne >= 8) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) cs[tn][e] += to_f32(s.v[e]);
                        *cr.at<gt_u32x4>(h, tn * 64, ring_far(lrow, lcol, c_rs)) = __builtin_bit_cast(gt_u32x4, s);
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; ++e) cs[tn][e] += e < ne ? to_f32(s.v[e]) : 0.f;
                        ring_store(cr.at<bf16>(h, tn * 64, ring_far(lrow, lcol, c_rs)), __builtin_bit_cast(gt_u32x4, s), ne, false);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        cr.next();
        __builtin_amdgcn_sched_barrier(0);
    });
    // the lanes of a row of sixteen hold the same columns of different rows of C
    __attribute__((address_space(1))) float* const out =
        (__attribute__((address_space(1))) float*)g.colpart + (int64_t)(row0 / (TMW * 32)) * g.m;
#pragma unroll
    for (int tn = 0; tn < TNW; ++tn)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            float s = cs[tn][e];
            s += dpp_move<0xB1>(s);
            s += dpp_move<0x4E>(s);
            s += dpp_move<0x124>(s);
            s += dpp_move<0x128>(s);
            const int col = col0 + tn * 32 + lcol + e;
            if (lrow == 0 && row0 < g.n && col < g.m) out[col] = s;
        }
}

// The bias of the lane's columns in the layout of the accumulators (ring_pack_tile)
template <typename C>
__device__ __forceinline__ void ring_load_bias(const GemmArgs& g, Pack<bf16, 4> (&b)[C::TNW * 4], int col0) {
    const int lane = fresh_tid() & 63;
    const __attribute__((address_space(1))) bf16* bias = (const __attribute__((address_space(1))) bf16*)g.bias;
#pragma unroll
    for (int q = 0; q < C::TNW * 4; ++q) {
        const int c = col0 + q * 8 + (lane >> 5) * 4;
        if (g.vec_out && col0 + C::TNW * 32 <= g.m) {
            b[q] = __builtin_bit_cast(Pack<bf16, 4>, *(const __attribute__((address_space(1))) gt_u32x2*)(bias + c));
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) b[q].v[e] = bias[c + e < g.m ? c + e : g.m - 1];
        }
    }
}
// PTJ_EPI_ACCUMULATE: the accumulators start from the stored C; elements outside C start from zero, their results are never stored
template <typename C>
__device__ __forceinline__ void ring_load_c(const GemmArgs& g, f32x16 (&acc)[C::TNW][C::TMW], int row0, int col0) {
    const int lane = fresh_tid() & 63;
    const int r0 = row0 + (lane & 31), c0 = col0 + (lane >> 5) * 4;
#pragma unroll
    for (int tn = 0; tn < C::TNW; ++tn)
#pragma unroll
        for (int tm = 0; tm < C::TMW; ++tm)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int row = r0 + tm * 32, col = c0 + tn * 32 + q * 8;
                const auto* p = (const __attribute__((address_space(1))) bf16*)g.c + (int64_t)row * g.c_rs + col;
                Pack<bf16, 4> v;
#pragma unroll
                for (int e = 0; e < 4; ++e) v.v[e] = from_f32<bf16>(0.f);
                if (row < g.n && col + 4 <= g.m) {
                    v = __builtin_bit_cast(Pack<bf16, 4>, *(const __attribute__((address_space(1))) gt_u32x2*)p);
                } else if (row < g.n) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (col + e < g.m) v.v[e] = p[e];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[tn][tm][q * 4 + e] = to_f32(v.v[e]);
            }
}

// The kernel's arguments, read again from where the launch left them: what only the start and the end of a tile need holds
// no scalar registers through the main loop.  (One kernel for all epilogues had 60 to 90 of them spilled otherwise and took
// 100 us instead of 80 for 16384x3072x768.)
__device__ __forceinline__ const GemmArgs& ring_args() {
    auto p = (const __attribute__((address_space(4))) GemmArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const GemmArgs*)p;
}

constexpr int clip(int x, int most) { return x < most ? x : most; }

template <int AMODE, int BMODE, typename C, bool MUL>
__global__ __launch_bounds__(C::THREADS, 2) void gemm_ring_kernel(const GemmArgs) {
    constexpr int TMW = C::TMW, TNW = C::TNW, NA = C::NA, NB = C::NB;
    __shared__ __attribute__((aligned(1024))) char smem[C::SMEM];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / C::WN, wn = wave - wm * C::WN;
    int work, end_k;                                                     // work items; contraction length
    bool ragged;                                                         // a vector of the last step holds a row's end
    char* const ring_a = smem;
    char* const ring_b = smem + NA * C::A_STAGE;

    typedef RingOperand<AMODE, C::TBM, TMW, NA> OA;
    typedef RingOperand<BMODE, C::TBN, TNW, NB> OB;
    constexpr int PA = OA::PER, PB = OB::PER;
    OA oa;
    OB ob;
    auto start_a = [&](const GemmArgs& g, const RingItem& it) __attribute__((always_inline)) {
        oa.start(g.a, g.a_row, g.a_k, it.row0, g.n, it.kbeg, it.klen, g.k);
    };
    auto start_b = [&](const GemmArgs& g, const RingItem& it) __attribute__((always_inline)) {
        ob.start(g.b, g.b_row, g.b_k, it.col0, g.m, it.kbeg, it.klen, g.k);
    };
    int item = blockIdx.x;
    RingItem cur;
    {
        const GemmArgs& g = ring_args();
        const int total = ((g.n + C::TBM - 1) / C::TBM) * ((g.m + C::TBN - 1) / C::TBN);
        work = g.tail_splits > 1 ? g.tail_first + (total - g.tail_first) * g.tail_splits : total * g.splits;
        end_k = g.k;
        ragged = g.k % 8 != 0 && (AMODE == KMAJOR || BMODE == KMAJOR);
        cur = ring_item<C>(g, item);
        oa.init(g.a_row, g.a_k, gt_lds_addr(ring_a), wm * TMW * 32, tid);
        ob.init(g.b_row, g.b_k, gt_lds_addr(ring_b), wn * TNW * 32, tid);
        oa.item = ob.item = item;
        start_a(g, cur);
        start_b(g, cur);
    }
    const uint32_t copy_a0 = gt_lds_addr(ring_a) + wave * 1024, copy_b0 = gt_lds_addr(ring_b) + wave * 1024;
    // a copy; behind the last one of a stage the cursor moves on, to the next item behind the last stage of one
    auto copy_a = [&](auto i) __attribute__((always_inline)) {
        if constexpr (i == 0) oa.begin_stage();
        oa.template copy<i>(copy_a0 + oa.slot * C::A_STAGE);
        if constexpr (i == PA - 1) {
            oa.base += oa.step;
            oa.left -= oa.step;
            oa.kleft -= 64;
            oa.slot = oa.slot + 1 == NA ? 0 : oa.slot + 1;
            if (__builtin_expect(oa.kleft <= 0 && oa.item < work, 0)) {
                oa.item += (int)gridDim.x;
                if (oa.item < work) {
                    const GemmArgs& g = ring_args();
                    start_a(g, ring_item<C>(g, oa.item));
                }
            }
        }
    };
    auto copy_b = [&](auto i) __attribute__((always_inline)) {
        if constexpr (i == 0) ob.begin_stage();
        ob.template copy<i>(copy_b0 + ob.slot * C::B_STAGE);
        if constexpr (i == PB - 1) {
            ob.base += ob.step;
            ob.left -= ob.step;
            ob.kleft -= 64;
            ob.slot = ob.slot + 1 == NB ? 0 : ob.slot + 1;
            if (__builtin_expect(ob.kleft <= 0 && ob.item < work, 0)) {
                ob.item += (int)gridDim.x;
                if (ob.item < work) {
                    const GemmArgs& g = ring_args();
                    start_b(g, ring_item<C>(g, ob.item));
                }
            }
        }
    };

    // two register sets of two contraction chunks each
    GtFrag<bf16, AMODE> fa[2][2][TMW];
    GtFrag<bf16, BMODE> fb[2][2][TNW];
    f32x16 acc[TNW][TMW];
    constexpr int NR = 2 * (TMW + TNW), NM = 2 * TMW * TNW, NC = PA + PB;   // reads, MFMAs of a set; copies of a step
    // Reads end a little before the set's last MFMA, so that they have landed by then, and copies two MFMAs earlier, so that the
    // cursors' bookkeeping runs under the last ones and not beside the barrier (8192^3: 783 us, 824 without).
    constexpr int READ_SPAN = NM * 7 / 8, COPY_SPAN = NM - 2;
    uint32_t addr_a[AMODE == KMAJOR ? 2 : TMW], addr_b[BMODE == KMAJOR ? 2 : TNW];
    auto read_addresses = [&](auto first, uint32_t soff_a, uint32_t soff_b) __attribute__((always_inline)) {
        gt_unroll<0, (AMODE == KMAJOR ? 2 : TMW)>([&](auto i) __attribute__((always_inline)) {
            addr_a[i] = oa.template read_addr<(AMODE == KMAJOR ? first + i : i)>(soff_a);
        });
        gt_unroll<0, (BMODE == KMAJOR ? 2 : TNW)>([&](auto i) __attribute__((always_inline)) {
            addr_b[i] = ob.template read_addr<(BMODE == KMAJOR ? first + i : i)>(soff_b);
        });
    };
    auto read_piece = [&](auto set, auto first, auto i) __attribute__((always_inline)) {
        constexpr int c = i / (TMW + TNW), t = i % (TMW + TNW);
        if constexpr (t < TMW) OA::template read_one<first + c, t>(fa[set][c][t], addr_a[AMODE == KMAJOR ? c : t]);
        else OB::template read_one<first + c, t - TMW>(fb[set][c][t - TMW], addr_b[BMODE == KMAJOR ? c : t - TMW]);
    };
    auto landed = [&](auto set) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int t = 0; t < TMW; ++t) fa[set][c][t].landed();
#pragma unroll
            for (int t = 0; t < TNW; ++t) fb[set][c][t].landed();
        }
    };
    uint32_t sa = 0, sb = 0;                   // offsets of the stages that hold the step being multiplied
    // the MFMAs of register set `set`, with the reads of chunks first, first + 1 into the other one between them, and with
    // `copies` those of a stage of either operand
    auto phase = [&](auto set, auto first, auto copies, uint32_t soff_a, uint32_t soff_b) __attribute__((always_inline)) {
        constexpr std::integral_constant<int, 1 - set> OTHER{};
        read_addresses(first, soff_a, soff_b);
        gt_unroll<0, NM>([&](auto j) __attribute__((always_inline)) {
            constexpr int c = j / (TMW * TNW), tn = j / TMW % TNW, tm = j % TMW;
            mma_chunk(acc[tn][tm], fb[set][c][tn].get(), fa[set][c][tm].get());
            __builtin_amdgcn_sched_barrier(0);
            gt_unroll<clip(j * NR / READ_SPAN, NR), clip((j + 1) * NR / READ_SPAN, NR)>(
                [&](auto i) __attribute__((always_inline)) { read_piece(OTHER, first, i); });
            if constexpr (copies)
                gt_unroll<clip(j * NC / COPY_SPAN, NC), clip((j + 1) * NC / COPY_SPAN, NC)>([&](auto i) __attribute__((always_inline)) {
                    if constexpr (i < PB) copy_b(std::integral_constant<int, i>{});
                    else copy_a(std::integral_constant<int, i - PB>{});
                });
            if constexpr (!copies && j == 1) {     // the next stages, under an early MFMA
                sa = sa + C::A_STAGE == NA * C::A_STAGE ? 0 : sa + C::A_STAGE;
                sb = sb + C::B_STAGE == NB * C::B_STAGE ? 0 : sb + C::B_STAGE;
            }
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    constexpr std::integral_constant<int, 0> I0{};
    constexpr std::integral_constant<int, 1> I1{};
    constexpr std::integral_constant<int, 2> I2{};
    constexpr std::bool_constant<true> YES{};
    constexpr std::bool_constant<false> NO{};
    auto clear_tails = [&](int klen) __attribute__((always_inline)) {
        const int tail = klen - (klen - 1) / 64 * 64;
        OA::clear_tail(ring_a + sa, tail, tid);
        OB::clear_tail(ring_b + sb, tail, tid);
        __syncthreads();
    };

    // the accumulators of a tile start from the bias, requested before the write-back of the tile before it
    Pack<bf16, 4> bias[TNW * 4];
    auto load_bias = [&](const RingItem& it) __attribute__((always_inline)) {
        if constexpr (!MUL) {
            const GemmArgs& g = ring_args();
            if (g.bias != nullptr && g.epilogue != PTJ_EPI_NONE && g.splits == 1 && it.part == nullptr) {
                ring_load_bias<C>(g, bias, it.col0 + wn * TNW * 32);
                return;
            }
        }
#pragma unroll
        for (int q = 0; q < TNW * 4; ++q)
#pragma unroll
            for (int e = 0; e < 4; ++e) bias[q].v[e] = from_f32<bf16>(0.f);
    };
    load_bias(cur);

    gt_unroll<0, NA>([&](auto s) __attribute__((always_inline)) {
        gt_unroll<0, PA>([&](auto i) __attribute__((always_inline)) { copy_a(i); });
        if constexpr (s < NB) gt_unroll<0, PB>([&](auto i) __attribute__((always_inline)) { copy_b(i); });
    });
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((NA - 1) * PA + (NB - 1) * PB) : "memory");
    if (ragged && cur.klen <= 64) clear_tails(cur.klen);
    read_addresses(I0, 0u, 0u);
    gt_unroll<0, NR>([&](auto i) __attribute__((always_inline)) { read_piece(I0, I0, i); });
    for (;;) {
        const int nitem = item + (int)gridDim.x;
        const bool more = nitem < work;
#pragma unroll
        for (int i = 0; i < TNW; ++i)
#pragma unroll
            for (int j = 0; j < TMW; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) acc[i][j][e] = to_f32(bias[i * 4 + (e >> 2)].v[e & 3]);
        if constexpr (!MUL) {
            const GemmArgs& g = ring_args();
            if (g.epilogue == PTJ_EPI_ACCUMULATE) ring_load_c<C>(g, acc, cur.row0 + wm * TMW * 32, cur.col0 + wn * TNW * 32);
        }
        for (int kt = 0; kt < cur.klen; kt += 64) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            landed(I0);
            phase(I0, I2, NO, sa, sb);
            // This wavefront has read all of the stage and its copies of the next one have landed (younger: A's of the one
            // after it); after the barrier that holds for every wavefront, so the next stage may be read and this one refilled.
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NA - 2) * PA) : "memory");
            landed(I1);
            if (__builtin_expect(ragged, 0)) {
                // the next step ends the contraction: the last one of this item, or the only one of the next
                int end = kt + 128 >= cur.klen && kt + 64 < cur.klen && cur.kbeg + cur.klen == end_k ? cur.klen : 0;
                if (kt + 64 >= cur.klen && more) {
                    const RingItem n = ring_item<C>(ring_args(), nitem);
                    end = n.klen <= 64 && n.kbeg + n.klen == end_k ? n.klen : 0;
                }
                if (end > 0) clear_tails(end);
            }
            phase(I1, I0, YES, sa, sb);
        }
        const int row0 = cur.row0 + wm * TMW * 32, col0 = cur.col0 + wn * TNW * 32;
        const GemmArgs& g = ring_args();
        RingItem nxt = cur;
        if (more) {
            nxt = ring_item<C>(g, nitem);
            load_bias(nxt);
        }
        if constexpr (MUL) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the reads that they are read again for)
            landed(I0);
            ring_write_mul<C>(g, acc, row0, col0);
        } else if (cur.part != nullptr) {
            ring_write_partial<C>(acc, cur.part, C::TBN, wm * TMW * 32, wn * TNW * 32, C::TBM, C::TBN);
        } else if (g.splits > 1) {
            ring_write_partial<C>(acc, g.partial + (int64_t)cur.z * g.n * g.m, g.m, row0, col0, g.n, g.m);
        } else {
            bf16 *c = (bf16*)g.c, *aux = (bf16*)g.c_aux;
            if (g.epilogue == PTJ_EPI_BIAS_GELU_DERIV) {
                ring_write<C, RING_BOTH>(g, acc, c, g.c_rs, aux, g.c_aux_rs, row0, col0);
            } else {
                if (aux != nullptr) ring_write<C, RING_RAW>(g, acc, aux, g.c_aux_rs, nullptr, 0, row0, col0);
                if (g.epilogue == PTJ_EPI_BIAS_GELU) ring_write<C, RING_GELU>(g, acc, c, g.c_rs, nullptr, 0, row0, col0);
                else ring_write<C, RING_RAW>(g, acc, c, g.c_rs, nullptr, 0, row0, col0);
            }
        }
        if (!more) break;
        item = nitem;
        cur = nxt;
        // the multiplying write-back takes the registers of the next tile's first fragments, which are read again here
        if constexpr (MUL) {
            read_addresses(I0, sa, sb);
            gt_unroll<0, NR>([&](auto i) __attribute__((always_inline)) { read_piece(I0, I0, i); });
        }
    }
    // nothing of this workgroup may still be on its way into LDS when its wavefronts end
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

// Whether a launch can take these kernels: two vector layouts and 32-bit offsets inside a tile; where the contraction ends
// inside a step, also rows that do not overlap (what lies past an operand's end is told by its address).  All 64 contraction
// indices of a step have to fit, those past the end as well: an offset that wrapped would read something else than zero there.
// Rows past the end of an operand may read anything of it; their results are not stored.
inline bool ring_eligible(const GemmArgs& g, int am, int bm) {
    if (am == GENERIC || bm == GENERIC || g.k < 1) return false;
    auto fits = [&](int mode, int64_t row, int64_t kst, int64_t nrows) {
        const int64_t pitch = mode == KMAJOR ? row : kst, lines = mode == KMAJOR ? (nrows < 256 ? nrows : 256) : 64;
        const int64_t length = mode == KMAJOR ? g.k : nrows;
        return pitch >= 0 && pitch < (1ll << 31) && (lines * pitch + 256) * 2 < 0x80000000ll + 512 && (g.k % 64 == 0 || pitch >= length);
    };
    return fits(am, g.a_row, g.a_k, g.n) && fits(bm, g.b_row, g.b_k, g.m);
}

template <typename C, bool MUL>
int ring_launch(const GemmArgs& g, int am, int bm, hipStream_t st) {
    const int64_t total = (int64_t)((g.n + C::TBM - 1) / C::TBM) * ((g.m + C::TBN - 1) / C::TBN);
    const int64_t work = g.tail_splits > 1 ? g.tail_first + (total - g.tail_first) * g.tail_splits : total * g.splits;
    const int cus = num_cus();
    const dim3 grid((unsigned)(work < cus ? work : cus)), block(C::THREADS);
#define RING_LAUNCH(AM, BMD) hipLaunchKernelGGL((gemm_ring_kernel<AM, BMD, C, MUL>), grid, block, 0, st, g)
    switch (am * 3 + bm) {
        case 0: RING_LAUNCH(KMAJOR, KMAJOR); break;
        case 1: RING_LAUNCH(KMAJOR, MNMAJOR); break;
        case 3: RING_LAUNCH(MNMAJOR, KMAJOR); break;
        default: RING_LAUNCH(MNMAJOR, MNMAJOR); break;
    }
#undef RING_LAUNCH
    PTJ_CHECK_LAUNCH();
    if constexpr (!MUL) {
        if (g.splits > 1 && !g.leave_partials) return launch_splitk_reduce<bf16>(g, g.splits, st);
        if (g.tail_splits > 1) return launch_tail_reduce<bf16, C::TBN>(g, (int)total, st);
    }
    return PTJ_OK;
}
