// Persistent bf16 GEMM whose operand panels travel HBM -> LDS by asynchronous buffer copies into two rings,
// one per operand.  Included by gemm_core.h inside its unnamed namespace, after gemm_tile.h.
//
// What bounds it: at long contractions the clock, at K = 768 what a tile does before and behind its loop (below).  Under this load the
// part holds 1.5-1.9 GHz, whatever switches is paid for in clock, and the 16x16x32 instructions take less for the same products than
// the 32x32x16 ones (their accumulators move half as often).  Alone, with N(0,1) factors in registers and the matrix pipe 97-99 %
// busy, they run at 2.03 against 1.77 GHz, 1915 against 1665 TFLOP/s (with equal factors, where little switches, both at 2.35 GHz,
// 2440); 8192^3 reaches 78 % of that, 16384x3072x768 with bias 52 %.  Per 64 contraction elements a 256x256 tile (eight
// wavefronts of 128x64) costs 2048 clocks of MFMAs, 1536 of fragment reads and 512 of arriving copies; a 256x192 tile
// (wavefronts of 64x96) 1536, 1280 and 448, so the wider tile gets more out of the matrix pipe and the narrower one is for
// outputs that it cuts into fuller rounds (gemm_plan.h).  The A ring has three stages and the B ring two: the chunk
// of half a step is read into registers half a step ahead, so a stage is refilled halfway through the step that
// multiplies it, and the copies of A have a step more to arrive than those of B.  160 KB hold no third stage
// of B.  Reads are spread over the first 5/8 of the MFMAs that they run beside (7/8: 8192^3 763 us instead of 755), copies over all but
// the last ones (bunched behind the barrier: 5 % slower), and the wavefronts that are past the barrier go first (740).
// 32x32x16 instructions before / now, us on one box: 8192^3 812 / 740 (1486 TFLOP/s), 8192x50257x768 with bias 683 / 628, its
// two gradient products 511 / 497 and 535 / 515, 16384x3072x768 with bias 86.9 / 80.4, with GELU and its derivative 118.8 / 113.6
// (77.6 and 102.3 with the walk of gemm_core.h), 16384x768x3072 70.3 / 67.3, dX of it 68.9 / 66.4, dW of it 82.6 / 81.9.  (With 32x32x16 the four plain 256x256 kernels spilled 33-50
// registers as well.)  Four wavefronts of 128x128 with one chunk per register set: 905 us for 8192^3 where eight took 783.
//
// The output goes straight from the accumulators to memory: a lane swap brings eight consecutive columns of a row
// into a lane and 64 bytes of each of sixteen rows into a store, without LDS, which the rings fill.  At k = 768 a workgroup
// of 16384x3072x768 spends 4 us before its first products, 15.7-18.8 in a tile's loop, 3.7 in the write-back (9 with GELU and its
// derivative, which are vector work; 11 with a multiplier, which is memory) and 0.6 until the next loop.  That 0.6 is a wait for
// everything under way, the stores included: the accumulators start from bias registers that a vector path, an element path or
// zeros may have filled, and the compiler waits in front of their use.  Measured and not kept: non-temporal stores (alone up to
// 8 % faster, but what reads the output next takes longer: training step 16 x 1024 +0.7 %, feed-forward block of 3001 tokens +14 %),
// workgroups that start staggered so that their stores do not coincide (no gain).
//
// Rows and contraction indices past the operand's end read as zero (buffer descriptors).

// TBM x TBN tile of C by WM x WN wavefronts
template <int TBN_, int WM_, int WN_>
struct RingCfg {
    static constexpr int TBM = 256, TBN = TBN_, WM = WM_, WN = WN_, NA = 3, NB = 2;
    static constexpr int NW = WM * WN, THREADS = NW * 64, TMW = TBM / WM / 32, TNW = TBN / WN / 32;
    static constexpr int TM = 2 * TMW, TN = 2 * TNW;                     // MFMA tiles of 16 x 16 per wavefront
    static_assert(TMW * WM * 32 == TBM && TNW * WN * 32 == TBN && NW == 8, "whole pairs of MFMA tiles, two wavefronts per SIMD");
    static constexpr int A_STAGE = TBM * BKB, B_STAGE = TBN * BKB, SMEM = NA * A_STAGE + NB * B_STAGE;
};
typedef RingCfg<256, 2, 4> RingFull;
typedef RingCfg<192, 4, 2> RingNarrow;

// A work item: a C tile, or one K slice of one.  part: dense partial tile of a K-split tile of the last round.
struct RingItem {
    int row0, col0, kbeg, klen, z;
    float* part;
    int kind, block;      // GemmGroup
};
template <typename C>
__device__ __forceinline__ RingItem ring_item(const GemmArgs& g, int item) {
    const int num_m = (g.n + C::TBM - 1) / C::TBM, num_n = (g.m + C::TBN - 1) / C::TBN;
    RingItem d;
    int tm, tn, kps = g.splits > 1 ? g.k_per_split : g.k;
    d.part = nullptr;
    if (g.tail_splits > 1 && item >= g.tail_first) {
        const int r = item - g.tail_first, t = r / g.tail_splits;
        gt_item<true>(g, g.tail_first + t, num_m, num_n, tm, tn, d.z);
        d.z = r - t * g.tail_splits;
        kps = g.tail_kps;
        d.part = g.partial + (int64_t)r * (C::TBM * C::TBN);
    } else {
        gt_item<true>(g, item, num_m, num_n, tm, tn, d.z);
    }
    d.row0 = tm * C::TBM;
    d.col0 = tn * C::TBN;
    d.kbeg = d.z * kps;
    d.klen = (d.kbeg + kps < g.k ? d.kbeg + kps : g.k) - d.kbeg;
    return d;
}

// The same for a tile of a group of products, whole along the contraction
template <typename C>
__device__ __forceinline__ RingItem ring_item(const ptj_gemm_detail::GemmGroup& g, int item) {
    int tm, tn;
    RingItem d;
    group_tile<true>(g, item, C::TBM, C::TBN, d.kind, d.block, tm, tn);
    d.row0 = tm * C::TBM;
    d.col0 = tn * C::TBN;
    d.kbeg = d.z = 0;
    d.klen = g.p.k;
    d.part = nullptr;
    return d;
}

// A wave-uniform value into scalar registers (a descriptor that the compiler cannot tell to be uniform costs a loop per copy)
__device__ __forceinline__ int64_t ring_uniform(int64_t v) {
    return (int64_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32) |
                     (uint32_t)__builtin_amdgcn_readfirstlane((int)v));
}

// Order of the 16-byte pieces in LDS (XORed into a piece's index).  A fragment is 16 rows x 32 contraction elements.  KMAJOR: half
// a wavefront reads two pieces of each of its sixteen rows; the sixteen lanes that are served at once (0-3, 12-15, 20-27, and
// the others) find theirs in different banks.  MNMAJOR: half a wavefront reads two pieces of the k-rows 0-3 and 8-11, which the order
// puts into different banks (192 rows: their pitch does half of it, and the order stays inside eight pieces).
__device__ __forceinline__ int ring_sw(int row) { return row & 6; }
template <int ROWS> __device__ __forceinline__ int ring_mn_sw(int k) {
    if constexpr (ROWS == 192) return ((k >> 1) & 1) * 2 + ((k >> 3) & 1) * 4;
    else return (k & 3) * 2 + ((k >> 3) & 1) * 8;
}

// One operand: the cursor of its copies, which runs ahead of the multiplications across work items, and the LDS addresses
// of this wavefront's fragments.  ROWS rows of the tile in a stage, NT MFMA tiles of 16 rows per wavefront.
template <int MODE, int ROWS, int NT, int STAGES>
struct RingOperand {
    static constexpr int NW = 8, PER = ROWS * BKB / 1024 / NW;           // copies per wavefront and stage
    static constexpr int PPR = ROWS / 8, PITCH = ROWS * 2;               // MNMAJOR: 16-byte pieces and bytes per k-row
    // the copies of a stage lie a whole number of swizzle periods apart: one address register for all of them
    static constexpr bool EVEN = MODE == KMAJOR || (NW * 64 % PPR == 0 && NW * 64 / PPR % 16 == 0);
    static constexpr int NADDR = MODE == MNMAJOR && ROWS == 192 ? 4 : 1;   // address registers
    uint32_t voff[EVEN ? 1 : PER], istep;
    int kk;                                                              // KMAJOR: k of this lane's vector in a step
    uint32_t raddr[NADDR];
    __amdgpu_buffer_rsrc_t rsrc;
    uint32_t v0;
    const char* base;                                                    // the next stage's first element
    int64_t left, step;                                                  // bytes from there to the operand's end; per stage
    int item, kleft, slot;                                               // kleft: contraction elements of the item not yet requested

    // where the lane's copies come from, by the operand's strides
    __device__ __forceinline__ void source(int64_t s_row, int64_t s_k, int tid) {
        const int lane = tid & 63;
        if constexpr (MODE == KMAJOR) {
            const int r = tid >> 3;
            kk = ((lane & 7) ^ ring_sw(r)) * 8;
            voff[0] = ((uint32_t)r * (uint32_t)s_row + (uint32_t)kk) * 2u;
            istep = NW * 8 * (uint32_t)s_row * 2u;
            step = 128;
        } else {
            kk = 0;
#pragma unroll
            for (int i = 0; i < (EVEN ? 1 : PER); ++i) {
                const int pc = i * NW * 64 + tid, k = pc / PPR, pos = pc - k * PPR;
                voff[i] = ((uint32_t)k * (uint32_t)s_k + (uint32_t)(pos ^ ring_mn_sw<ROWS>(k)) * 8u) * 2u;
            }
            istep = NW * 64 / PPR * (uint32_t)s_k * 2u;
            step = 128 * s_k;
        }
    }
    __device__ __forceinline__ void init(int64_t s_row, int64_t s_k, uint32_t region, int wrow, int tid) {
        source(s_row, s_k, tid);
        const int lane = tid & 63;
        if constexpr (MODE == KMAJOR) {
            const int row = wrow + (lane & 15);
            raddr[0] = region + row * BKB + (((lane >> 4) ^ ring_sw(row)) << 4);
        } else {
            const int l16 = lane & 15, kf = 8 * (lane >> 4) + (l16 >> 2);
#pragma unroll
            for (int t = 0; t < NADDR; ++t) {
                const int piece = (wrow >> 3) + 2 * t + ((l16 & 3) >> 1);
                raddr[t] = region + kf * PITCH + ((piece ^ ring_mn_sw<ROWS>(kf)) << 4) + 8 * (l16 & 1);
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
    // LDS address of the fragments (KMAJOR: of chunk I, every MFMA tile; MNMAJOR: of tile I, every chunk) of the stage at byte
    // offset soff.  256 rows: the first piece of a wavefront has no bits where those of its tiles differ.
    template <int I>
    __device__ __forceinline__ uint32_t read_addr(uint32_t soff) const {
        uint32_t a;
        if constexpr (NADDR > 1) a = raddr[I % NADDR] + soff;
        else if constexpr (I == 0) a = raddr[0] + soff;
        else if constexpr ((I << (MODE == KMAJOR ? 6 : 5)) <= 64) asm volatile("v_xad_u32 %0, %1, %2, %3" : "=v"(a) : "v"(raddr[0]), "n"(I << (MODE == KMAJOR ? 6 : 5)), "s"(soff));
        else asm volatile("v_xor_b32 %0, %1, %2\n\tv_add_u32 %0, %3, %0" : "=&v"(a) : "n"(I << 5), "v"(raddr[0]), "s"(soff));
        return a;
    }
    // fragment of MFMA tile TI, chunk CH (of 32 contraction elements)
    template <int CH, int TI>
    __device__ __forceinline__ static void read_one(GtFrag<bf16, MODE>& f, uint32_t addr) {
        if constexpr (MODE == KMAJOR) f.template read<TI * 16 * BKB>(addr);
        else f.template read<32 * CH * PITCH + (NADDR > 1 ? TI / NADDR * 128 : 0), PITCH>(addr);
    }
    // KMAJOR: clears the elements of every row of a stage from contraction index `tail` to the end of their vector
    __device__ __forceinline__ static void clear_tail(char* __restrict__ stage, int tail, int tid) {
        if constexpr (MODE == KMAJOR) {
            if (tail % 8 == 0 || tid >= ROWS) return;
            bf16* p = (bf16*)(stage + tid * BKB + (((tail / 8) ^ ring_sw(tid)) << 4));
            for (int e = tail % 8; e < 8; ++e) p[e] = from_f32<bf16>(0.f);
        }
    }
};

// in each half of the wavefront, lanes 16-31 of a <-> lanes 0-15 of b
__device__ __forceinline__ void ring_swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ uint32_t ring_pack2(float a, float b) {
    const f32x2 f = {a, b};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
}

// Write-back of two accumulator tiles side by side.  x[i], y[i] of lane l are row l & 15, columns (l >> 4) * 4 + i and 16 more.
// Afterwards lane l has in `out` the eight columns (l>>4 & 1)*16 + (l>>5)*8 ... of that row, rounded.
__device__ __forceinline__ gt_u32x4 ring_rows(const f32x4& x, const f32x4& y) {
    uint32_t x0 = ring_pack2(x[0], x[1]), x1 = ring_pack2(x[2], x[3]), y0 = ring_pack2(y[0], y[1]), y1 = ring_pack2(y[2], y[3]);
    ring_swap16(x0, y0);
    ring_swap16(x1, y1);
    return gt_u32x4{x0, x1, y0, y1};
}

// What becomes of an accumulator: RAW itself, GELU its GELU, BOTH the GELU's derivative as well (second output)
enum { RING_RAW, RING_GELU, RING_BOTH };
template <int ACT>
__device__ __forceinline__ void ring_pack_tile(const f32x4& x, const f32x4& y, gt_u32x4& out, gt_u32x4& aux) {
    if constexpr (ACT == RING_RAW) {
        out = ring_rows(x, y);
    } else {
        f32x4 a[2] = {x, y}, d[2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float v = a[t][e];
                float g, dg;
                if constexpr (ACT == RING_GELU) g = gelu_f(v);
                else gelu_both_f(v, g, dg);
                a[t][e] = g;
                if constexpr (ACT == RING_BOTH) d[t][e] = dg;
            }
        out = ring_rows(a[0], a[1]);
        if constexpr (ACT == RING_BOTH) aux = ring_rows(d[0], d[1]);
    }
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
__device__ __forceinline__ void ring_write(const GemmArgs& g, const f32x4 (&acc)[C::TN][C::TM], bf16* c, int64_t rs, bf16* aux,
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
#pragma unroll
            for (int h = 0; h < 2; ++h) ring_pack_tile<ACT>(acc[2 * tn][2 * tm + h], acc[2 * tn + 1][2 * tm + h], v[h], w[h]);
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
__device__ __forceinline__ void ring_write_partial(const f32x4 (&acc)[C::TN][C::TM], float* __restrict__ dst, int64_t rs, int row0,
                                                   int col0, int nrows, int ncols) {
    const int lane = fresh_tid() & 63, lrow = lane & 15, lcol = (lane >> 4) * 4;
    RingRows pr(dst + (int64_t)row0 * rs + col0, rs, 4);
    const uint32_t voff = ((uint32_t)lrow * (uint32_t)rs + (uint32_t)lcol) * 4u;
    const bool whole = rs % 4 == 0 && row0 + C::TMW * 32 <= nrows && col0 + C::TNW * 32 <= ncols;
#pragma unroll
    for (int tm = 0; tm < C::TMW; ++tm) {
#pragma unroll
        for (int tn = 0; tn < C::TN; ++tn)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const f32x4& x = acc[tn][2 * tm + h];
                if (whole) {
                    *pr.at<f32x4>(h, tn * 64, voff) = x;
                } else {
                    int ne = ncols - col0 - lcol;
                    asm volatile("" : "+v"(ne));
                    ne = row0 + tm * 32 + h * 16 + lrow < nrows ? ne - tn * 16 : 0;
#pragma unroll 1
                    for (int e = 0; e < (ne < 4 ? ne : 4); ++e) pr.at<float>(h, tn * 64, voff)[e] = e < 2 ? (e < 1 ? x[0] : x[1]) : (e < 3 ? x[2] : x[3]);
                }
            }
        pr.next();
    }
}

// C = round(acc) * mul and the column sums of what is stored over the wavefront's TMW * 32 rows (g.colpart).  The multipliers of two
// rows of MFMA tiles are under way (three: 108.2 us instead of 107.6 for 16384x3072x768; four spill).
template <typename C>
__device__ __forceinline__ void ring_write_mul(const GemmArgs& g, const f32x4 (&acc)[C::TN][C::TM], int row0, int col0) {
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
    constexpr int AHEAD = 2;
    gt_u32x4 mv[AHEAD][TNW][2];
    auto request = [&](auto tm) __attribute__((always_inline)) {
        if (whole) {
#pragma unroll
            for (int tn = 0; tn < TNW; ++tn)
#pragma unroll
                for (int h = 0; h < 2; ++h) mv[tm % AHEAD][tn][h] = *mr.at<gt_u32x4>(h, tn * 64, moff);
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
                    mv[tm % AHEAD][tn][h] = gt_u32x4{w[0], w[1], w[2], w[3]};
                }
        }
        mr.next();
    };
    gt_unroll<0, AHEAD>([&](auto tm) __attribute__((always_inline)) { request(tm); });
    __builtin_amdgcn_sched_barrier(0);
    gt_unroll<0, TMW>([&](auto tm) __attribute__((always_inline)) {
#pragma unroll
        for (int tn = 0; tn < TNW; ++tn) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                Pack<bf16, 8> s = __builtin_bit_cast(Pack<bf16, 8>, ring_rows(acc[2 * tn][2 * tm + h], acc[2 * tn + 1][2 * tm + h]));
                const Pack<bf16, 8> m = __builtin_bit_cast(Pack<bf16, 8>, mv[tm % AHEAD][tn][h]);
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
        if constexpr (tm + AHEAD < TMW) request(std::integral_constant<int, tm + AHEAD>{});
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

// The bias of the lane's columns in the layout of the accumulators (ring_rows)
template <typename C>
__device__ __forceinline__ void ring_load_bias(const GemmArgs& g, Pack<bf16, 4> (&b)[C::TN], int col0) {
    const int lane = fresh_tid() & 63;
    const __attribute__((address_space(1))) bf16* bias = (const __attribute__((address_space(1))) bf16*)g.bias;
#pragma unroll
    for (int q = 0; q < C::TN; ++q) {
        const int c = col0 + q * 16 + (lane >> 4) * 4;
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
__device__ __forceinline__ void ring_load_c(const GemmArgs& g, f32x4 (&acc)[C::TN][C::TM], int row0, int col0) {
    const int lane = fresh_tid() & 63;
    const int r0 = row0 + (lane & 15), c0 = col0 + (lane >> 4) * 4;
#pragma unroll
    for (int tn = 0; tn < C::TN; ++tn)
#pragma unroll
        for (int tm = 0; tm < C::TM; ++tm) {
            const int row = r0 + tm * 16, col = c0 + tn * 16;
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
            for (int e = 0; e < 4; ++e) acc[tn][tm][e] = to_f32(v.v[e]);
        }
}

// The kernel's arguments, read again from where the launch left them: what only the start and the end of a tile need holds
// no scalar registers through the main loop.  (One kernel for all epilogues had 60 to 90 of them spilled otherwise and took
// 100 us instead of 80 for 16384x3072x768.)
template <typename ARGS = GemmArgs>
__device__ __forceinline__ const ARGS& ring_args() {
    auto p = (const __attribute__((address_space(4))) ARGS*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const ARGS*)p;
}

constexpr int clip(int x, int most) { return x < most ? x : most; }

// ARGS: GemmArgs, or GemmGroup (plain products of two MNMAJOR operands)
template <int AMODE, int BMODE, typename C, bool MUL, typename ARGS = GemmArgs>
__global__ __launch_bounds__(C::THREADS, 2) void gemm_ring_kernel(const ARGS) {
    constexpr bool GROUP = !std::is_same<ARGS, GemmArgs>::value;
    static_assert(!GROUP || (AMODE == MNMAJOR && BMODE == MNMAJOR && !MUL), "layouts of a group");
    constexpr int TMW = C::TMW, TNW = C::TNW, TM = C::TM, TN = C::TN, NA = C::NA, NB = C::NB;
    __shared__ __attribute__((aligned(1024))) char smem[C::SMEM];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / C::WN, wn = wave - wm * C::WN;
    int work, end_k;                                                     // work items; contraction length
    bool ragged;                                                         // a vector of the last step holds a row's end
    char* const ring_a = smem;
    char* const ring_b = smem + NA * C::A_STAGE;

    typedef RingOperand<AMODE, C::TBM, TM, NA> OA;
    typedef RingOperand<BMODE, C::TBN, TN, NB> OB;
    constexpr int PA = OA::PER, PB = OB::PER;
    OA oa;
    OB ob;
    auto start_a = [&](const ARGS& g, const RingItem& it) __attribute__((always_inline)) {
        if constexpr (GROUP) {
            const int n = g.p.n[it.kind];
            oa.source(1, n, fresh_tid());
            oa.start(g.p.d[it.kind][it.block], 1, n, it.row0, n, 0, it.klen, it.klen);
        } else {
            oa.start(g.a, g.a_row, g.a_k, it.row0, g.n, it.kbeg, it.klen, g.k);
        }
    };
    auto start_b = [&](const ARGS& g, const RingItem& it) __attribute__((always_inline)) {
        if constexpr (GROUP) {
            const int m = g.p.m[it.kind];
            ob.source(1, m, fresh_tid());
            ob.start(g.p.x[it.kind][it.block], 1, m, it.col0, m, 0, it.klen, it.klen);
        } else {
            ob.start(g.b, g.b_row, g.b_k, it.col0, g.m, it.kbeg, it.klen, g.k);
        }
    };
    int item = blockIdx.x;
    RingItem cur;
    {
        const ARGS& g = ring_args<ARGS>();
        cur = ring_item<C>(g, item);
        if constexpr (GROUP) {
            work = g.first[PtjGradGroup::KINDS] * g.p.blocks;
            end_k = g.p.k;
            ragged = false;
            oa.init(1, 0, gt_lds_addr(ring_a), wm * TMW * 32, tid);
            ob.init(1, 0, gt_lds_addr(ring_b), wn * TNW * 32, tid);
        } else {
            const int total = ((g.n + C::TBM - 1) / C::TBM) * ((g.m + C::TBN - 1) / C::TBN);
            work = g.tail_splits > 1 ? g.tail_first + (total - g.tail_first) * g.tail_splits : total * g.splits;
            end_k = g.k;
            ragged = g.k % 8 != 0 && (AMODE == KMAJOR || BMODE == KMAJOR);
            oa.init(g.a_row, g.a_k, gt_lds_addr(ring_a), wm * TMW * 32, tid);
            ob.init(g.b_row, g.b_k, gt_lds_addr(ring_b), wn * TNW * 32, tid);
        }
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
                    const ARGS& g = ring_args<ARGS>();
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
                    const ARGS& g = ring_args<ARGS>();
                    start_b(g, ring_item<C>(g, ob.item));
                }
            }
        }
    };

    // two register sets of one contraction chunk each
    GtFrag<bf16, AMODE> fa[2][TM];
    GtFrag<bf16, BMODE> fb[2][TN];
    f32x4 acc[TN][TM];
    constexpr int NR = TM + TN, NM = TM * TN, NC = PA + PB;   // reads, MFMAs of a set; copies of a step
    // Reads take the first 5/8 of the set's MFMAs, so that they have landed by its end, and copies all but the last four, so that
    // the cursors' bookkeeping runs under those and not beside the barrier (figures at the top).
    constexpr int READ_SPAN = NM * 5 / 8, COPY_SPAN = NM - 4;
    uint32_t addr_a, addr_b;                   // KMAJOR
    auto read_addresses = [&](auto ch, uint32_t soff_a, uint32_t soff_b) __attribute__((always_inline)) {
        if constexpr (AMODE == KMAJOR) addr_a = oa.template read_addr<ch>(soff_a);
        if constexpr (BMODE == KMAJOR) addr_b = ob.template read_addr<ch>(soff_b);
    };
    auto read_piece = [&](auto set, auto ch, auto i, uint32_t soff_a, uint32_t soff_b) __attribute__((always_inline)) {
        if constexpr (i < TM) {
            if constexpr (AMODE != KMAJOR) addr_a = oa.template read_addr<i>(soff_a);
            OA::template read_one<ch, i>(fa[set][i], addr_a);
        } else {
            if constexpr (BMODE != KMAJOR) addr_b = ob.template read_addr<i - TM>(soff_b);
            OB::template read_one<ch, i - TM>(fb[set][i - TM], addr_b);
        }
    };
    auto landed = [&](auto set) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TM; ++t) fa[set][t].landed();
#pragma unroll
        for (int t = 0; t < TN; ++t) fb[set][t].landed();
    };
    uint32_t sa = 0, sb = 0;                   // offsets of the stages that hold the step being multiplied
    // the MFMAs of register set `set`, with the reads of chunk `ch` into the other one between them, and with
    // `copies` those of a stage of either operand
    auto phase = [&](auto set, auto ch, auto copies, uint32_t soff_a, uint32_t soff_b) __attribute__((always_inline)) {
        constexpr std::integral_constant<int, 1 - set> OTHER{};
        read_addresses(ch, soff_a, soff_b);
        __builtin_amdgcn_s_setprio(set);
        gt_unroll<0, NM>([&](auto j) __attribute__((always_inline)) {
            constexpr int tn = j / TM, tm = j % TM;
            acc[tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[set][tn].get(), fa[set][tm].get(), acc[tn][tm], 0, 0, 0);
            gt_unroll<clip(j * NR / READ_SPAN, NR), clip((j + 1) * NR / READ_SPAN, NR)>(
                [&](auto i) __attribute__((always_inline)) { read_piece(OTHER, ch, i, soff_a, soff_b); });
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
    constexpr std::bool_constant<true> YES{};
    constexpr std::bool_constant<false> NO{};
    auto clear_tails = [&](int klen) __attribute__((always_inline)) {
        const int tail = klen - (klen - 1) / 64 * 64;
        OA::clear_tail(ring_a + sa, tail, tid);
        OB::clear_tail(ring_b + sb, tail, tid);
        __syncthreads();
    };

    // the accumulators of a tile start from the bias, requested before the write-back of the tile before it
    Pack<bf16, 4> bias[TN];
    auto load_bias = [&](const RingItem& it) __attribute__((always_inline)) {
        if constexpr (!MUL && !GROUP) {
            const GemmArgs& g = ring_args();
            if (g.bias != nullptr && g.epilogue != PTJ_EPI_NONE && g.splits == 1 && it.part == nullptr) {
                ring_load_bias<C>(g, bias, it.col0 + wn * TNW * 32);
                return;
            }
        }
#pragma unroll
        for (int q = 0; q < TN; ++q)
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
    gt_unroll<0, NR>([&](auto i) __attribute__((always_inline)) { read_piece(I0, I0, i, 0u, 0u); });
    for (;;) {
        const int nitem = item + (int)gridDim.x;
        const bool more = nitem < work;
#pragma unroll
        for (int i = 0; i < TN; ++i)
#pragma unroll
            for (int j = 0; j < TM; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][j][e] = to_f32(bias[i].v[e]);
        if constexpr (!MUL && !GROUP) {
            const GemmArgs& g = ring_args();
            if (g.epilogue == PTJ_EPI_ACCUMULATE) ring_load_c<C>(g, acc, cur.row0 + wm * TMW * 32, cur.col0 + wn * TNW * 32);
        }
        for (int kt = 0; kt < cur.klen; kt += 64) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            landed(I0);
            phase(I0, I1, NO, sa, sb);
            // This wavefront has read all of the stage and its copies of the next one have landed (younger: A's of the one
            // after it); after the barrier that holds for every wavefront, so the next stage may be read and this one refilled.
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NA - 2) * PA) : "memory");
            landed(I1);
            if (__builtin_expect(ragged, 0)) {
                // the next step ends the contraction: the last one of this item, or the only one of the next
                int end = kt + 128 >= cur.klen && kt + 64 < cur.klen && cur.kbeg + cur.klen == end_k ? cur.klen : 0;
                if (kt + 64 >= cur.klen && more) {
                    const RingItem n = ring_item<C>(ring_args<ARGS>(), nitem);
                    end = n.klen <= 64 && n.kbeg + n.klen == end_k ? n.klen : 0;
                }
                if (end > 0) clear_tails(end);
            }
            phase(I1, I0, YES, sa, sb);
        }
        const int row0 = cur.row0 + wm * TMW * 32, col0 = cur.col0 + wn * TNW * 32;
        const ARGS& g = ring_args<ARGS>();
        RingItem nxt = cur;
        if (more) {
            nxt = ring_item<C>(g, nitem);
            load_bias(nxt);
        }
        if constexpr (GROUP) {
            GemmArgs out{};
            out.n = g.p.n[cur.kind];
            out.m = g.p.m[cur.kind];
            out.vec_out = 1;
            ring_write<C, RING_RAW>(out, acc, (bf16*)g.p.dw[cur.kind][cur.block], out.m, nullptr, 0, row0, col0);
        } else if constexpr (MUL) {
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
            gt_unroll<0, NR>([&](auto i) __attribute__((always_inline)) { read_piece(I0, I0, i, sa, sb); });
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
        if (g.tail_splits > 1) return launch_tail_reduce<bf16, C::TBN, true>(g, (int)total, st);
    }
    return PTJ_OK;
}

// The products of a group, whole tiles of each
template <typename C>
int ring_group_launch(const PtjGradGroup& p, hipStream_t st) {
    const ptj_gemm_detail::GemmGroup g = group_of<C>(p);
    const int work = g.first[PtjGradGroup::KINDS] * p.blocks, cus = num_cus();
    hipLaunchKernelGGL((gemm_ring_kernel<MNMAJOR, MNMAJOR, C, false, ptj_gemm_detail::GemmGroup>), dim3((unsigned)(work < cus ? work : cus)),
                       dim3(C::THREADS), 0, st, g);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}
