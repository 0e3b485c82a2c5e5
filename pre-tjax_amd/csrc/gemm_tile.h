// MFMA GEMM for products that do not fill the chip with the 256x192 tiles of gemm_core.h: one
// workgroup per (C tile, K split), tile shape and wavefront arrangement as template parameters.
// Included by gemm_core.h inside its unnamed namespace.
//
// Panels travel HBM -> LDS by asynchronous buffer copies (16 bytes per lane) into a ring of S
// stages; a stage holds KG panels of 128 bytes of the contraction axis per row (64 bf16 / 32 fp32),
// and the wavefronts of K group g multiply panel g only, so a small C tile still keeps four
// wavefronts busy and the loop over K is KG times shorter.  The groups' accumulators are added in
// group order on the way out.  Buffer descriptors do the border handling: rows and contraction
// indices past the operand's end read as zero, so there is one code path for whole and ragged
// tiles, and a K-major operand whose length is no multiple of 16 bytes has the surplus elements of
// its last vector cleared in LDS.
//
// LDS layouts: KMAJOR as in mma_tile.h ([row][128 bytes], XOR-swizzled); MNMAJOR, 2-byte:
// [k][rows] as it lies in memory, read through ds_read_b64_tr_b16 (sixteen lanes fetch a 4 (k) x 16 (rows) block and each
// ends up with four consecutive k of one row; 4-byte: [k][rows] read by ds_read_b32,
// four contraction indices per fragment).
typedef uint32_t gt_u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t gt_u32x4 __attribute__((ext_vector_type(4)));

// XORed into the index of a 16-byte piece inside its k-row so that the four k-rows that a transposing
// read touches lie in different banks (pitches of 64 and 192 bytes spread them by themselves)
template <int ROWS> __device__ __forceinline__ int gt_mn_swz(int k) {
    if constexpr (ROWS == 64) return ((k >> 1) & 1) * 4;
    else if constexpr (ROWS == 128) return (10 * (k & 3)) & 15;
    else if constexpr (ROWS == 192) return 2 * (k & 3);
    else if constexpr (ROWS == 256) return 10 * (k & 3);
    else return 0;
}

__device__ __forceinline__ uint32_t gt_lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}

// One MFMA operand fragment (16 bytes of contraction per lane) and how it is read from a stage.
template <typename T, int MODE> struct GtFrag;
template <typename T> struct GtFrag<T, KMAJOR> {
    gt_u32x4 v;
    template <int OFF> __device__ __forceinline__ void read(uint32_t addr) {
        asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
    }
    __device__ __forceinline__ void landed() { asm volatile("" : "+v"(v)); }
    __device__ __forceinline__ typename Frag<T>::type get() const { return __builtin_bit_cast(typename Frag<T>::type, v); }
};
template <> struct GtFrag<bf16, MNMAJOR> {
    gt_u32x2 lo, hi;
    template <int OFF, int PITCH> __device__ __forceinline__ void read(uint32_t addr) {
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(lo) : "v"(addr), "n"(OFF));
        asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(hi) : "v"(addr), "n"(OFF + 4 * PITCH));
    }
    __device__ __forceinline__ void landed() { asm volatile("" : "+v"(lo), "+v"(hi)); }
    __device__ __forceinline__ bf16x8 get() const {
        const gt_u32x4 q = {lo[0], lo[1], hi[0], hi[1]};
        return __builtin_bit_cast(bf16x8, q);
    }
};
template <> struct GtFrag<float, MNMAJOR> {
    float f0, f1, f2, f3;
    template <int OFF, int PITCH> __device__ __forceinline__ void read(uint32_t addr) {
        asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(f0) : "v"(addr), "n"(OFF));
        asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(f1) : "v"(addr), "n"(OFF + PITCH));
        asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(f2) : "v"(addr), "n"(OFF + 2 * PITCH));
        asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(f3) : "v"(addr), "n"(OFF + 3 * PITCH));
    }
    __device__ __forceinline__ void landed() { asm volatile("" : "+v"(f0), "+v"(f1), "+v"(f2), "+v"(f3)); }
    __device__ __forceinline__ f32x4 get() const { return f32x4{f0, f1, f2, f3}; }
};

// Per-lane state of one operand: ROWS rows of the C tile, NT MFMA tiles of 32 rows per wavefront, KG panels per
// stage, NW wavefronts sharing the copies.
template <typename T, int MODE, int ROWS, int NT, int KG, int NW>
struct GtOperand {
    static constexpr int ELT = (int)sizeof(T), VEC = 16 / ELT, BK = BKB / ELT;
    static constexpr int PANEL = ROWS * BKB;               // bytes
    static constexpr int BYTES = KG * PANEL;               // one stage
    static constexpr int PER = BYTES / 1024 / NW;          // copies per wavefront and stage
    static constexpr int PITCH = ROWS * ELT;               // MNMAJOR: bytes per k-row
    static constexpr int NADDR = MODE == KMAJOR ? 4 : (ELT == 2 ? NT : 1);
    static_assert(PER * NW * 1024 == BYTES, "copies divide evenly among the wavefronts");
    uint32_t voff[PER];
    uint32_t raddr[NADDR];
    // operand bytes from the stage's first element on: the descriptor of the next copy
    const char* base;
    int64_t left;
    int64_t step;

    __device__ __forceinline__ void init(const void* p, int64_t s_row, int64_t s_k, int row0, int nrows, int kbeg, int k,
                                         uint32_t region, int wrow, int kg, int tid) {
        const int lane = tid & 63, wave = tid >> 6;
        const T* first = (const T*)p + (MODE == KMAJOR ? (int64_t)row0 * s_row + kbeg : (int64_t)kbeg * s_k + row0);
        base = (const char*)first;
        const int64_t elems = MODE == KMAJOR
            ? (int64_t)(nrows - 1 - row0) * s_row + ((k - kbeg + VEC - 1) / VEC) * VEC
            : (int64_t)(k - 1 - kbeg) * s_k + ((nrows - row0 + VEC - 1) / VEC) * VEC;
        left = elems * ELT;
        step = (MODE == KMAJOR ? (int64_t)1 : s_k) * (BK * KG) * ELT;
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int inst = wave * PER + i;
            if constexpr (MODE == KMAJOR) {
                const int panel = inst / (ROWS / 8);
                const int r = (inst - panel * (ROWS / 8)) * 8 + (lane >> 3);
                const int chunk = (lane & 7) ^ sw(r);
                voff[i] = ((uint32_t)r * (uint32_t)s_row + (uint32_t)(panel * BK + chunk * VEC)) * (uint32_t)ELT;
            } else {
                constexpr int PPR = ROWS / VEC;                // 16-byte pieces per k-row
                const int pc = inst * 64 + lane;
                const int kk = pc / PPR, pos = pc - kk * PPR;
                const int piece = ELT == 2 ? pos ^ gt_mn_swz<ROWS>(kk) : pos;
                voff[i] = ((uint32_t)kk * (uint32_t)s_k + (uint32_t)piece * VEC) * (uint32_t)ELT;
            }
        }
        const uint32_t reg = region + kg * PANEL;
        if constexpr (MODE == KMAJOR) {
            const int row = wrow + (lane & 31), lg = lane >> 5;
#pragma unroll
            for (int c = 0; c < 4; ++c) raddr[c] = reg + row * BKB + (((c * 2 + lg) ^ sw(row)) << 4);
        } else if constexpr (ELT == 2) {
            const int l16 = lane & 15, mhalf = (lane >> 4) & 1, lg = lane >> 5, kq = l16 >> 2;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int piece = (wrow >> 3) + t * 4 + 2 * mhalf + ((l16 & 3) >> 1);
                raddr[t] = reg + (8 * lg + kq) * PITCH + ((piece ^ gt_mn_swz<ROWS>(kq)) << 4) + 8 * (l16 & 1);
            }
        } else {
            raddr[0] = reg + (lane >> 5) * 4 * PITCH + (wrow + (lane & 31)) * 4;
        }
    }

    // Copy I of the next stage (wave-uniform LDS address `stage`).  kleft: contraction elements from the stage's first
    // one to the end (<= 0: past the end, everything reads as zero and nothing is fetched).
    template <int I>
    __device__ __forceinline__ void copy(char* __restrict__ stage, int kleft, int wave, int lane) const {
        const uint32_t records = kleft <= 0 ? 0u : (uint32_t)(left < 0xFFFFFF00ll ? left : 0xFFFFFF00ll);
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, records, 0x00020000);
        uint32_t v = voff[I];
        if constexpr (MODE == KMAJOR) {
            if (kleft < BK * KG) {                              // vectors past the end of their row: the next row's data
                const int inst = wave * PER + I;
                const int panel = inst / (ROWS / 8);
                const int r = (inst - panel * (ROWS / 8)) * 8 + (lane >> 3);
                const int kk = panel * BK + ((lane & 7) ^ sw(r)) * VEC;
                v = kk < kleft ? v : 0xFFFFFFF0u;
            }
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rsrc, (__attribute__((address_space(3))) void*)(stage + (wave * PER + I) * 1024), 16, v, 0, 0, 0);
    }
    __device__ __forceinline__ void advance() {
        base += step;
        left -= step;
    }

    // KMAJOR: clears the elements [kleft, next multiple of a vector) of every row of the stage
    __device__ __forceinline__ void clear_tail(char* __restrict__ stage, int kleft, int tid) const {
        if constexpr (MODE == KMAJOR) {
            const int e0 = kleft % VEC;
            if (e0 == 0 || tid >= ROWS) return;
            const int panel = kleft / BK, chunk = (kleft - panel * BK) / VEC;
            T* p = (T*)(stage + panel * PANEL + tid * BKB + ((chunk ^ sw(tid)) << 4));
            for (int e = e0; e < VEC; ++e) p[e] = from_f32<T>(0.f);
        }
    }

    // fragment of MFMA tile TI, contraction chunk C, of the stage at byte offset soff
    template <int C, int TI>
    __device__ __forceinline__ void read_one(GtFrag<T, MODE>& f, uint32_t soff) const {
        if constexpr (MODE == KMAJOR) f.template read<TI * 32 * BKB>(raddr[C] + soff);
        else if constexpr (ELT == 2) f.template read<16 * C * PITCH, PITCH>(raddr[TI] + soff);
        else f.template read<8 * C * PITCH + TI * 128, PITCH>(raddr[0] + soff);
    }
};

template <int I, int N, typename F>
__device__ __forceinline__ void gt_unroll(F&& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        gt_unroll<I + 1, N>(f);
    }
}

// Tile geometry: TBM x TBN tile of C, WM x WN wavefronts over it, KG K groups, S stages, CPS contraction chunks
// (of the four in a panel) per register set: a set is read from LDS while the MFMAs of the other one run.
template <int TBM_, int TBN_, int WM_, int WN_, int KG_, int S_, int CPS_>
struct GtCfg {
    static constexpr int TBM = TBM_, TBN = TBN_, WM = WM_, WN = WN_, KG = KG_, S = S_, CPS = CPS_;
    static constexpr int NW = WM * WN * KG, THREADS = NW * 64;
    static constexpr int TMW = TBM / WM / 32, TNW = TBN / WN / 32;   // MFMA tiles per wavefront
    static_assert(TMW * WM * 32 == TBM && TNW * WN * 32 == TBN, "whole MFMA tiles per wavefront");
    static constexpr int CW = TNW * 32;                              // columns per wavefront
    static constexpr int A_STAGE = KG * TBM * BKB, B_STAGE = KG * TBN * BKB;
    static constexpr int RING = S * (A_STAGE + B_STAGE);
    static constexpr int OUT_PITCH = CW + 4;                         // fp32 elements per staged row
    static constexpr int OUT_WAVE = 32 * OUT_PITCH * 4;              // bytes per wavefront: 32 rows
    static constexpr int SMEM = RING > NW * OUT_WAVE ? RING : NW * OUT_WAVE;
    static constexpr int BLOCKS = SMEM > 81920 ? 1 : 2;              // workgroups per CU that registers are budgeted for
    static constexpr int WAVES_EU = (BLOCKS * NW + 3) / 4;
};

// Work item of the grid -> tile and K split.  Without a K split as in gemm_core.h (tile_walk); with one each XCD works on a
// contiguous range as well, and the tiles along the smaller C dimension vary fastest, then the other ones, then the split.
template <bool RING = false>
__device__ __forceinline__ void gt_item(const GemmArgs& g, int pid, int num_m, int num_n, int& tile_m, int& tile_n, int& z) {
    const int total = num_m * num_n;
    z = 0;
    if (g.splits > 1) {
        const int idx = xcd_range<false>(pid, total * g.splits);
        if (g.n >= g.m) {
            tile_n = idx % num_n;
            const int pair = idx / num_n;
            tile_m = pair % num_m;
            z = pair / num_m;
        } else {
            tile_m = idx % num_m;
            const int pair = idx / num_m;
            tile_n = pair % num_n;
            z = pair / num_n;
        }
        return;
    }
    tile_walk<RING>(xcd_range<RING>(pid, total), num_m, num_n, tile_m, tile_n);
}

// Write-back of a finished tile: 32 rows at a time through an fp32 staging area per wavefront (the K groups'
// accumulators are added in group order on the way), then rows of 16-byte vectors with the epilogue applied.
// PTJ_EPI_ACCUMULATE is gemm_ring.h's alone.
// acc[tn][tm][i] of lane (lr, lg) is C[row0 + (wm * TMW + tm) * 32 + lr][col0 + wn * CW + tn * 32 + (i/4)*8 + lg*4 + i%4].
template <typename T, typename C, bool MUL>
__device__ __forceinline__ void gt_write_back(const GemmArgs& g, const f32x16 (&acc)[C::TNW][C::TMW], char* __restrict__ smem,
                                              int row0, int col0, int z, int wave, int lane) {
    constexpr int VEC = 16 / (int)sizeof(T), TMW = C::TMW, TNW = C::TNW, KG = C::KG;
    const int kg = wave / (C::WM * C::WN), wpos = wave - kg * (C::WM * C::WN);
    const int wm = wpos / C::WN, wn = wpos - wm * C::WN;
    float* const st = (float*)(smem + wave * C::OUT_WAVE);
    constexpr int GROUP_STEP = C::WM * C::WN * C::OUT_WAVE / 4;      // staging areas of the K groups of one position
    const float* const st0 = (const float*)(smem + wpos * C::OUT_WAVE);
    constexpr int LPR = C::CW / VEC;                                 // vectors per row
    constexpr int ROWS = 32 / KG;                                    // rows of a pass that this wavefront writes
    const int lr = lane & 31, lg = lane >> 5;
    const int gc0 = col0 + wn * C::CW;
    const bool partial = !MUL && g.splits > 1;
    float* const part = partial ? g.partial + (int64_t)z * g.n * (int64_t)g.m : nullptr;
    float csum[(C::CW + 63) / 64];
#pragma unroll
    for (int i = 0; i < (C::CW + 63) / 64; ++i) csum[i] = 0.f;
#pragma unroll
    for (int tm = 0; tm < TMW; ++tm) {
#pragma unroll
        for (int tn = 0; tn < TNW; ++tn)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4*>(st + lr * C::OUT_PITCH + tn * 32 + q * 8 + lg * 4) =
                    f32x4{acc[tn][tm][q * 4], acc[tn][tm][q * 4 + 1], acc[tn][tm][q * 4 + 2], acc[tn][tm][q * 4 + 3]};
        if constexpr (KG > 1) __syncthreads();
        else __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const int gr0 = row0 + (wm * TMW + tm) * 32;
        for (int idx = lane; idx < ROWS * LPR; idx += 64) {
            const int r = kg * ROWS + idx / LPR, c = (idx % LPR) * VEC;
            float v[VEC];
#pragma unroll
            for (int h = 0; h < VEC / 4; ++h) {
                f32x4 s = *reinterpret_cast<const f32x4*>(st0 + r * C::OUT_PITCH + c + h * 4);
#pragma unroll
                for (int k2 = 1; k2 < KG; ++k2)
                    s += *reinterpret_cast<const f32x4*>(st0 + k2 * GROUP_STEP + r * C::OUT_PITCH + c + h * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[h * 4 + e] = s[e];
            }
            const int row = gr0 + r, col = gc0 + c;
            const bool inside = row < g.n && col < g.m;
            const bool whole = col + VEC <= g.m;       // rows may start at any element
            const int ne = g.m - col < VEC ? g.m - col : VEC;
            if constexpr (MUL) {
                const T* mp = (const T*)g.mul + (int64_t)row * g.mul_rs + col;
                T* p = (T*)g.c + (int64_t)row * g.c_rs + col;
                float o[VEC];
#pragma unroll
                for (int e = 0; e < VEC; ++e) o[e] = 0.f;
                if (inside && whole) {
                    const LoosePack<T, VEC> mv = *reinterpret_cast<const LoosePack<T, VEC>*>(mp);
                    LoosePack<T, VEC> s;
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        s.v[e] = from_f32<T>(to_f32(from_f32<T>(v[e])) * to_f32(mv.v[e]));
                        o[e] = to_f32(s.v[e]);
                    }
                    *reinterpret_cast<LoosePack<T, VEC>*>(p) = s;
                } else if (inside) {
#pragma unroll
                    for (int e = 0; e < VEC; ++e)
                        if (e < ne) {
                            const T s = from_f32<T>(to_f32(from_f32<T>(v[e])) * to_f32(mp[e]));
                            p[e] = s;
                            o[e] = to_f32(s);
                        }
                }
                // the stored values take the place of the first group's, for the column sums
#pragma unroll
                for (int h = 0; h < VEC / 4; ++h)
                    *reinterpret_cast<f32x4*>(const_cast<float*>(st0) + r * C::OUT_PITCH + c + h * 4) =
                        f32x4{o[h * 4], o[h * 4 + 1], o[h * 4 + 2], o[h * 4 + 3]};
            } else if (inside) {
                if (partial) {
                    float* p = part + (int64_t)row * g.m + col;
                    if (whole) {
#pragma unroll
                        for (int h = 0; h < VEC / 4; ++h)
                            store_loose<float, 4>(p + h * 4, v + h * 4);
                    } else {
#pragma unroll
                        for (int e = 0; e < VEC; ++e)
                            if (e < ne) p[e] = v[e];
                    }
                } else {
                    const bool deriv = g.epilogue == PTJ_EPI_BIAS_GELU_DERIV;
                    const bool act = deriv || g.epilogue == PTJ_EPI_BIAS_GELU;
                    T* p = (T*)g.c + (int64_t)row * g.c_rs + col;
                    T* pa = g.c_aux != nullptr ? (T*)g.c_aux + (int64_t)row * g.c_aux_rs + col : nullptr;
                    const T* add = g.epilogue != PTJ_EPI_NONE ? (const T*)g.bias + col : nullptr;
                    if (whole) {
                        if (add != nullptr) {
                            const LoosePack<T, VEC> b = *reinterpret_cast<const LoosePack<T, VEC>*>(add);
#pragma unroll
                            for (int e = 0; e < VEC; ++e) v[e] += to_f32(b.v[e]);
                        }
                        if (pa != nullptr) {
                            float o[VEC];
#pragma unroll
                            for (int e = 0; e < VEC; ++e) o[e] = deriv ? gelu_grad_f(v[e]) : v[e];
                            store_loose<T, VEC>(pa, o);
                        }
                        if (act) {
#pragma unroll
                            for (int e = 0; e < VEC; ++e) v[e] = gelu_f(v[e]);
                        }
                        store_loose<T, VEC>(p, v);
                    } else {
#pragma unroll
                        for (int e = 0; e < VEC; ++e)
                            if (e < ne) {
                                float x = v[e];
                                if (add != nullptr) x += to_f32(add[e]);
                                if (pa != nullptr) pa[e] = from_f32<T>(deriv ? gelu_grad_f(x) : x);
                                p[e] = from_f32<T>(act ? gelu_f(x) : x);
                            }
                    }
                }
            }
        }
        if constexpr (MUL) {
            if constexpr (KG > 1) __syncthreads();
            else __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (kg == 0) {
#pragma unroll
                for (int i = 0; i < (C::CW + 63) / 64; ++i)
                    if (i * 64 + lane < C::CW)
                        for (int r = 0; r < 32; ++r) csum[i] += st0[r * C::OUT_PITCH + i * 64 + lane];
            }
        }
        if constexpr (KG > 1) __syncthreads();
        else __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    }
    if constexpr (MUL) {
        // one row of sums per wavefront's block of rows (TMW * 32 of them)
        const int gr = row0 + wm * TMW * 32;
        if (kg == 0 && gr < g.n) {
#pragma unroll
            for (int i = 0; i < (C::CW + 63) / 64; ++i) {
                const int c = i * 64 + lane;
                if (c < C::CW && gc0 + c < g.m) g.colpart[(int64_t)(gr / (TMW * 32)) * g.m + gc0 + c] = csum[i];
            }
        }
    }
}

template <typename T, int AMODE, int BMODE, typename C, bool MUL>
__device__ __forceinline__ void gt_tile(const GemmArgs& g, int pid, char* __restrict__ smem) {
    constexpr int ELT = (int)sizeof(T), VEC = 16 / ELT, BK = BKB / ELT, BKT = BK * C::KG;
    constexpr int TMW = C::TMW, TNW = C::TNW, S = C::S, KG = C::KG;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / (C::WM * C::WN), wpos = wave - kg * (C::WM * C::WN);
    const int wm = wpos / C::WN, wn = wpos - wm * C::WN;
    const int num_m = (g.n + C::TBM - 1) / C::TBM, num_n = (g.m + C::TBN - 1) / C::TBN;
    int tile_m, tile_n, z;
    gt_item(g, pid, num_m, num_n, tile_m, tile_n, z);
    const int row0 = tile_m * C::TBM, col0 = tile_n * C::TBN;
    const int kbeg = z * g.k_per_split;
    const int kend = g.splits > 1 && kbeg + g.k_per_split < g.k ? kbeg + g.k_per_split : g.k;
    const int nk = (kend - kbeg + BKT - 1) / BKT;

    GtOperand<T, AMODE, C::TBM, TMW, KG, C::NW> oa;
    GtOperand<T, BMODE, C::TBN, TNW, KG, C::NW> ob;
    constexpr int PT = oa.PER + ob.PER;
    char* const sA = smem;
    char* const sB = smem + S * C::A_STAGE;
    oa.init(g.a, g.a_row, g.a_k, row0, g.n, kbeg, g.k, gt_lds_addr(sA), wm * TMW * 32, kg, tid);
    ob.init(g.b, g.b_row, g.b_k, col0, g.m, kbeg, g.k, gt_lds_addr(sB), wn * TNW * 32, kg, tid);

    constexpr int CPS = C::CPS, NSET = 4 / CPS;
    static_assert(CPS == 2 || CPS == 4, "a panel is one or two register sets");
    GtFrag<T, AMODE> fa[2][CPS][TMW];
    GtFrag<T, BMODE> fb[2][CPS][TNW];
    f32x16 acc[TNW][TMW];
#pragma unroll
    for (int i = 0; i < TNW; ++i)
#pragma unroll
        for (int j = 0; j < TMW; ++j)
#pragma unroll
            for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

    int kleft = kend - kbeg;                 // contraction elements not yet requested
    const int ktail = (kend - kbeg) - (nk - 1) * BKT;   // those of the last stage
    const bool ragged = ktail % VEC != 0 && (AMODE == KMAJOR || BMODE == KMAJOR);
    // ---- pieces of the pipeline, all with compile-time indexes
    constexpr int NR = CPS * (TMW + TNW), NM = CPS * TMW * TNW;   // fragment reads and MFMA tiles of a register set
    auto read_piece = [&](auto set, auto first, auto i, uint32_t sa, uint32_t sb) {
        constexpr int c = i / (TMW + TNW), t = i % (TMW + TNW);
        if constexpr (t < TMW) oa.template read_one<first + c, t>(fa[set][c][t], sa);
        else ob.template read_one<first + c, t - TMW>(fb[set][c][t - TMW], sb);
    };
    auto copy_piece = [&](auto i, int slot) {
        if constexpr (i < oa.PER) oa.template copy<i>(sA + slot * C::A_STAGE, kleft, wave, lane);
        else ob.template copy<i - oa.PER>(sB + slot * C::B_STAGE, kleft, wave, lane);
        if constexpr (i == PT - 1) {
            oa.advance();
            ob.advance();
            kleft -= BKT;
        }
    };
    auto landed = [&](auto set) {
#pragma unroll
        for (int c = 0; c < CPS; ++c) {
#pragma unroll
            for (int t = 0; t < TMW; ++t) fa[set][c][t].landed();
#pragma unroll
            for (int t = 0; t < TNW; ++t) fb[set][c][t].landed();
        }
    };
    // The MFMAs of register set `set` with the reads of chunks [first, first + CPS) into the other set and copies
    // [c0, c1) of a stage spread between them: a wavefront that is alone on its SIMD then keeps the matrix pipe, the
    // LDS and the copy path busy side by side instead of one after the other.
    auto phase = [&](auto set, auto other, auto first, auto c0, auto c1, uint32_t sa, uint32_t sb, int slot) {
        gt_unroll<0, NM>([&](auto j) {
            constexpr int c = j / (TMW * TNW), tn = (j / TMW) % TNW, tm = j % TMW;
            mma_chunk(acc[tn][tm], fb[set][c][tn].get(), fa[set][c][tm].get());
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (first >= 0) gt_unroll<j * NR / NM, (j + 1) * NR / NM>([&](auto i) { read_piece(other, first, i, sa, sb); });
            constexpr int nc = c1 - c0;
            if constexpr (nc > 0) gt_unroll<c0 + j * nc / NM, c0 + (j + 1) * nc / NM>([&](auto i) { copy_piece(i, slot); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto clear_tail = [&](int slot) {
        oa.clear_tail(sA + slot * C::A_STAGE, ktail, tid);
        ob.clear_tail(sB + slot * C::B_STAGE, ktail, tid);
        __syncthreads();
    };
    constexpr std::integral_constant<int, 0> I0{};
    constexpr std::integral_constant<int, 1> I1{};
    constexpr std::integral_constant<int, -1> NONE{};
    constexpr std::integral_constant<int, PT> IPT{};
    constexpr std::integral_constant<int, 4 - CPS> ILAST{};
    if (nk > 0) {
#pragma unroll
        for (int s = 0; s < S - 1; ++s) gt_unroll<0, PT>([&](auto i) { copy_piece(i, s); });
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((S - 2) * PT) : "memory");
        if (ragged && nk == 1) clear_tail(0);
        gt_unroll<0, NR>([&](auto i) { read_piece(I0, I0, i, 0u, 0u); });
        gt_unroll<0, PT>([&](auto i) { copy_piece(i, S - 1); });
        int slot = 0;
        // The compiler takes a fragment to be there behind its read and may copy it to other registers where control flow joins
        // or leaves a loop, so no read is under way where a loop ends: its copies there came ahead of the wait in front of the
        // products.  Two register sets per panel: the wait is the body's last statement.  One: around its loop the compiler leaves
        // the fragments where they are and a wait behind the loop is enough (in the body: dW on 3001 tokens 21.6 -> 22.5 us; the
        // barrier at the end as well: 0.1 us a launch, and 3-5 % of the products of 1536 to 2560 tokens).  What the compiler
        // does is checked on the code that was built.
#define GT_READ(SET)                                                                                    \
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                              \
        landed(SET);
        // In front of a stage's last register set: the next stage has landed and this one has been read, by every wavefront
        // after the barrier, so the next stage may be read and this one refilled.
#define GT_TURN(SET)                                                                                    \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * PT) : "memory");     \
        landed(SET);
        if constexpr (NSET == 2) {
            GT_READ(I0)
            phase(I0, I1, ILAST, I0, I0, 0u, 0u, 0);
            GT_READ(I1)
            for (int kt = 0; kt + 1 < nk; ++kt) {
                const int next = slot + 1 == S ? 0 : slot + 1;
                GT_TURN(I1)
                if (ragged && kt + 2 == nk) clear_tail(next);
                phase(I1, I0, I0, I0, IPT, next * C::A_STAGE, next * C::B_STAGE, slot);
                GT_READ(I0)
                phase(I0, I1, ILAST, I0, I0, next * C::A_STAGE, next * C::B_STAGE, slot);
                GT_READ(I1)
                slot = next;
            }
            phase(I1, I0, NONE, I0, I0, 0u, 0u, 0);
        } else {
            int kt = 0;
            for (; kt + 2 < nk; ++kt) {
                {
                    const int next = slot + 1 == S ? 0 : slot + 1;
                    GT_TURN(I0)
                    phase(I0, I1, I0, I0, IPT, next * C::A_STAGE, next * C::B_STAGE, slot);
                    slot = next;
                }
                ++kt;
                {
                    const int next = slot + 1 == S ? 0 : slot + 1;
                    GT_TURN(I1)
                    if (ragged && kt + 2 == nk) clear_tail(next);
                    phase(I1, I0, I0, I0, IPT, next * C::A_STAGE, next * C::B_STAGE, slot);
                    slot = next;
                }
            }
            GT_READ(I0)
            if (kt + 1 < nk) {
                const int next = slot + 1 == S ? 0 : slot + 1;
                GT_TURN(I0)
                if (ragged) clear_tail(next);
                phase(I0, I1, I0, I0, IPT, next * C::A_STAGE, next * C::B_STAGE, slot);
                GT_READ(I1)
                phase(I1, I0, NONE, I0, I0, 0u, 0u, 0);
            } else {
                phase(I0, I1, NONE, I0, I0, 0u, 0u, 0);
            }
        }
#undef GT_TURN
#undef GT_READ
    }
    // Nothing may still be on its way into the ring when the output staging takes its place.  The wait states that the last
    // product's result needs are spelled out: where the write-back begins with a branch the compiler has left them out of the
    // shorter way (fp32, 32x32 tiles: 13 of 18).
    if constexpr (ELT == 2) asm volatile("s_nop 11" ::: "memory");
    else asm volatile("s_nop 15\n\ts_nop 1" ::: "memory");
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    gt_write_back<T, C, MUL>(g, acc, smem, row0, col0, z, wave, lane);
}

template <typename T, int AMODE, int BMODE, typename C, bool MUL>
__global__ __launch_bounds__(C::THREADS, C::WAVES_EU) void gemm_tile_kernel(const GemmArgs g) {
    __shared__ __attribute__((aligned(1024))) char smem[C::SMEM];
    gt_tile<T, AMODE, BMODE, C, MUL>(g, (int)blockIdx.x, smem);
}

// Whether a launch can take these kernels: operands with one unit stride (with the alignment of pick_mode, or for the
// kernels that take any: rows of at least one vector), non-overlapping rows, and 32-bit offsets inside a tile.
inline bool gt_eligible(const GemmArgs& g, int am, int bm, int64_t least_pitch = 1) {
    if (am == GENERIC || bm == GENERIC || g.k < 1) return false;
    const int64_t lim = 1 << 21;
    const int64_t a_pitch = am == KMAJOR ? g.a_row : g.a_k, b_pitch = bm == KMAJOR ? g.b_row : g.b_k;
    return a_pitch >= (am == KMAJOR ? g.k : g.n) && a_pitch >= least_pitch && a_pitch < lim &&
           b_pitch >= (bm == KMAJOR ? g.k : g.m) && b_pitch >= least_pitch && b_pitch < lim;
}

template <typename T, typename C, bool MUL>
int gt_launch(const GemmArgs& g, int am, int bm, hipStream_t st) {
    const int64_t work = (int64_t)((g.n + C::TBM - 1) / C::TBM) * ((g.m + C::TBN - 1) / C::TBN) * g.splits;
    const dim3 grid((unsigned)work), block(C::THREADS);
#define GT_LAUNCH(AM, BMD) hipLaunchKernelGGL((gemm_tile_kernel<T, AM, BMD, C, MUL>), grid, block, 0, st, g)
    switch (am * 3 + bm) {
        case 0: GT_LAUNCH(KMAJOR, KMAJOR); break;
        case 1: GT_LAUNCH(KMAJOR, MNMAJOR); break;
        case 3: GT_LAUNCH(MNMAJOR, KMAJOR); break;
        default: GT_LAUNCH(MNMAJOR, MNMAJOR); break;
    }
#undef GT_LAUNCH
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}
