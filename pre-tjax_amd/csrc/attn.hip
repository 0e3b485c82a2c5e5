// Causal flash attention for gfx950, head dimension 64: forward, and a backward that
// recomputes P from the saved row max / row sum-exp.  The kernels of 2-byte storage, what masks and dropout need, and the C entry
// points; 4-byte storage: attn_f32.hip.
//
// Layout trick shared by the three MFMA kernels: scores are produced TRANSPOSED.  With
// 32x32 MFMA tiles, D[m][n] of lane l sits at n = l & 31, m = 8*(i/4) + 4*(l>>5) + i%4
// (register i).  Forward and the dQ pass compute S^T = K Q^T, so a lane owns ONE query
// (n) and 16 keys per 32-key tile (m): row max / row sum / rescaling are per-lane
// scalars (one cross-lane exchange with lane^32), and the probabilities are already in
// MFMA B-operand position for O^T = V^T P^T (contraction over keys, which live in the
// lane's registers), so P never travels through LDS.  The dK/dV pass computes S = Q K^T
// with the same trick mirrored: a lane owns one key, dV^T = dO^T P and dK^T = Q^T dS.
// The operand that must be read "across" its memory layout (V^T, K^T, Q^T, dO^T: row
// index d, contraction along keys / queries) comes out of the same rows in LDS with transposing reads;
// the four wavefronts share it.
//
// Softmax is evaluated in base 2 (scores pre-multiplied by log2(e)/sqrt(dh)); the saved
// statistics `ms` are converted back to natural units.  Masked scores take the
// reference's fill value -1e9 (not -inf); the running maximum starts above it, so a masked
// element contributes exactly 0.  A row without any visible key therefore has sum-exp 0: its
// output row is 0, its saved statistics are (ms, ls) = (-1e9, 0), and the backward gives it
// (and takes from it) no gradient.
//
// An explicit mask arrives bit-packed in both orientations together with one class per 32x32
// tile of (mask AND causal): hidden everywhere / mixed / equal to the causal pattern.  Hidden
// tiles are skipped, tiles equal to the causal pattern run the index-masked code, and only
// mixed tiles read their mask words -- a plain lower-triangular tensor costs what mask = NULL
// costs, and packed documents cost what they attend to.
//
// Dropout on the probabilities: element (q, k) of batch-head g is kept iff
// philox(seed + g, q + k) passes the threshold -- the offset depends on q + k only, so
// one line of 2T keep bits per batch-head is generated once (attn_keepbits_kernel); the
// kernels read it through the scalar unit and turn it into 64-lane select masks.
//
// The backward is two passes without atomics: dQ over query tiles (it also forms
// delta = rowsum(dO * O) of its queries and stores it), then (dK, dV) over key tiles,
// which reads delta; both recompute S and dP.
#include "attn_common.h"

namespace {

constexpr int ATT_THREADS = 256;
constexpr int MAX_T = 8192;
constexpr int MAX_BITWORDS = 2 * MAX_T / 32 + 2;

typedef bf16x8 RowPieces[4];   // the MFMA operand pieces of one 64-element row (lane half lg)

__device__ __forceinline__ void load_row_frags(RowPieces& f, const bf16* __restrict__ row, int lg) {
#pragma unroll
    for (int c = 0; c < 4; ++c) f[c] = *reinterpret_cast<const bf16x8*>(reinterpret_cast<const char*>(row) + c * 32 + lg * 16);
}

// ---- tiles, copied straight into LDS ---------------------------------------------------------
// Tiles go from memory into LDS without registers, two tiles ahead of their use, and lie there once.  Before, they went
// through registers one tile ahead and lay in LDS a second time, transposed by vector permutes: dK/dV and dQ read Q, dO and
// K from memory twice, and a third of the vector instructions of a step were the loader's.  Batch 8 x 1024 x 12 heads,
// before / after (with the order of place()): forward 26.8 / 24.4 us, dQ 38.1 / 32.8, dK/dV 51.4 / 46.2; both in one launch,
// batch 8 x 512: 35.9 / 29.6.  What bounds them now: a step's matrix and vector instructions hardly overlap (forward: 512
// and 1000 clocks of 1670 per SIMD and step of 64 keys, batch 16 x 1024), and the chain of a step, LDS - product - softmax
// - product, with the two or three wavefronts per SIMD that the registers allow.  Four wavefronts per SIMD (two tiles in LDS,
// 128 registers) changed the forward and dQ by 1 %.
//
// A panel is 64 rows of 128 bytes as they lie in memory, its 16-byte pieces permuted inside each row by row_swizzle: the
// sixteen lanes that a 16-byte read serves at once (0-3, 12-15, 20-27 of the half wavefront, and the others) find their rows'
// pieces in different banks (RowFrags), and so do the four rows x 64 bytes that half a wavefront fetches with a transposing read
// (TpFrags), so ONE panel serves both directions.
constexpr int RING = 3;                   // tiles in LDS: one in use, two on their way
constexpr int WAVE_COPY = 64 * 16;        // bytes of one copy of a wavefront: eight rows
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)p;
}
// lane l's 16 (4) bytes at src land at lds + 16 l (4 l).  Inline assembly: the compiler would wait for every copy under way
// before any LDS read.  (m0 is reserved; nothing else in this file uses it.)
__device__ __forceinline__ void copy16_to_lds(const char* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(src) : "memory");
}
__device__ __forceinline__ void copy4_to_lds(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, off" ::"s"(lds), "v"(src) : "memory");
}
// One operand's tiles of 64 rows: wavefront w copies rows 8w .. 8w+7 and 32 + 8w .. of each.
struct PanelCopy {
    const char* src;     // the lane's piece of tile 0
    int64_t half;        // bytes from a row to the row 32 further on
    __device__ __forceinline__ void init(const bf16* __restrict__ p, int64_t row_stride, int tid) {
        const int r = tid >> 3;
        src = reinterpret_cast<const char*>(p + r * row_stride) + (((tid & 7) ^ row_swizzle(r)) << 4);
        half = row_stride * 64;
    }
    __device__ __forceinline__ void issue(int tile, uint32_t panel, int wave) const {
        const char* s = src + (int64_t)tile * 2 * half;
        copy16_to_lds(s, panel + wave * WAVE_COPY);
        copy16_to_lds(s + half, panel + 32 * 128 + wave * WAVE_COPY);
    }
};
// Waits for this wavefront's copies, all but the newest N of them (everything unless `more` follow).
template <int N> __device__ __forceinline__ void copies_landed(bool more) {
    if (more) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}
// The fragments are in their registers from here on (a compiler's wait inside the loop would wait for every copy as well).
template <typename F, int N> __device__ __forceinline__ void frags_landed(F (&f)[N]) {
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int c = 0; c < N; ++c) {
        u32x4_t v = __builtin_bit_cast(u32x4_t, f[c]);
        asm volatile("" : "+v"(v)::"memory");
        f[c] = __builtin_bit_cast(F, v);
    }
}
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ int next_slot(int slot) { return slot == RING - 1 ? 0 : slot + 1; }

// s += panel_rows(j*32 + lr) x register_rows : panel rows become MFMA rows (m), the
// lane's register row the MFMA column (n); contraction over the 64-element axis d.
// (NJ sub-tiles' fragments are read together ahead of the products)
template <int NJ> struct RowFrags {
    bf16x8 a[NJ][4];
    __device__ __forceinline__ void read(const char* __restrict__ panel, int j0, int lr, int lg) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int j = 0; j < NJ; ++j)
                a[j][c] = *reinterpret_cast<const bf16x8*>(panel + ((j0 + j) * 32 + lr) * BKB + (((c * 2 + lg) ^ row_swizzle(lr)) << 4));
    }
    __device__ __forceinline__ void mma(f32x16 (&s)[NJ], const RowPieces& f) const {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int j = 0; j < NJ; ++j) mma_chunk(s[j], a[j][c], f[c]);
    }
};

// Eight floats -> eight bf16, converted two at a time (one packed conversion per pair).
__device__ __forceinline__ bf16x8 pack8_bf16(const float* __restrict__ p) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
    u32x4_t w;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const f32x2_t f = {p[2 * e], p[2 * e + 1]};
        w[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
    }
    return __builtin_bit_cast(bf16x8, w);
}

// o[t] += transposed panel (row t*32 + lr of the transpose) x p : contraction over the 32 positions of
// sub-tile j whose values p[i] the lane holds in accumulator order
// (position = j*32 + 8*(i/4) + 4*lg + i%4).
// The panel's fragments are read ahead of the element-wise work that forms p (TpFrags::read), so that their way out of LDS is
// hidden behind it.
typedef short i16x4_t __attribute__((ext_vector_type(4)));
struct TpFrags {
    bf16x8 a[2][2];
    // transposing reads: sixteen lanes fetch four positions x 16 columns, each ends up with the four positions of its column;
    // two of them make the eight positions that a lane holds of p, in the same order
    __device__ __forceinline__ void read(const char* __restrict__ panel, int j, int lr, int lg) {
        const int x = 4 * lg + ((lr & 15) >> 2);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const int piece = t * 4 + 2 * (lr >> 4) + ((lr & 3) >> 1);
                const char* pp = panel + (j * 32 + h * 16 + x) * BKB + 8 * (lr & 1);
                const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(pp + ((piece ^ row_swizzle(x)) << 4)));
                const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(pp + 8 * BKB + ((piece ^ row_swizzle(x + 8)) << 4)));
                a[h][t] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            }
    }
    __device__ __forceinline__ void mma(f32x16 (&o)[2], const float (&p)[16]) const {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bf16x8 b = pack8_bf16(&p[8 * h]);
#pragma unroll
            for (int t = 0; t < 2; ++t) o[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[h][t], b, o[t], 0, 0, 0);
        }
    }
};

// ---- keep-bit line per batch-head ---------------------------------------------------
constexpr int KEEP_SEEDS = 64;   // attention calls per launch
struct KeepSeeds { uint64_t s[KEEP_SEEDS]; };
__global__ __launch_bounds__(256) void attn_keepbits_kernel(uint32_t* __restrict__ bits, int bitwords, const KeepSeeds seeds) {
    const int bh = blockIdx.y;
    bits += (int64_t)blockIdx.z * gridDim.y * bitwords;
    const int o = blockIdx.x * 256 + threadIdx.x;
    const uint64_t s = seeds.s[blockIdx.z] + (uint64_t)bh;
    const bool keep = philox_keep((uint32_t)o, (uint32_t)s, (uint32_t)(s >> 32));
    const uint64_t m = __ballot(keep);
    if ((threadIdx.x & 63) == 0) {
        const int w = o >> 5;
        uint32_t* dst = bits + (int64_t)bh * bitwords;
        if (w < bitwords) dst[w] = (uint32_t)m;
        if (w + 1 < bitwords) dst[w + 1] = (uint32_t)(m >> 32);
    }
}

// ---- attention mask, bit-packed in both orientations, and the class of every 32x32 tile ----
// out word (o, b, g, x), o = 0: bits r = mask[b, 32g + r, x] (a word per key x: 32 queries);
//                        o = 1: bits r = mask[b, x, 32g + r] (a word per query x: 32 keys).
// Class of a tile of (mask AND causal):
//   TILE_CAUSAL  the tile equals the causal pattern (also every tile above the diagonal, where
//                both are empty): index masking alone is exact
//   TILE_HIDDEN  no element visible
//   TILE_MIXED   anything else: the mask words are needed
// written twice: cq[(b, q/32, k/32)] and ck[(b, k/32, q/32)].
//
// A half wavefront takes a tile, a lane a row of it: 32 bytes in two loads make the word along the keys, the words along
// the queries are their transpose across the lanes, and the class comes from two ballots.  Bound by the launch and by the one
// read of the mask: a thread per word that collected its 32 bytes one by one, with the classes in a second launch, took 8.0 + 4.6 us
// for 8 x 1024 x 1024, this 5.0.
typedef uint32_t mask_u32x4 __attribute__((ext_vector_type(4), aligned(1)));   // the mask may start at any byte
constexpr int PACK_THREADS = 256;
// four bytes, each zero or not -> four bits
__device__ __forceinline__ uint32_t mask_nibble(uint32_t w) {
    w |= (w >> 4) & 0x0f0f0f0fu;
    w |= (w >> 2) & 0x03030303u;
    w |= (w >> 1) & 0x01010101u;
    return ((w & 0x01010101u) * 0x01020408u >> 24) & 15u;
}
__global__ __launch_bounds__(PACK_THREADS) void attn_pack_mask_kernel(const uint8_t* __restrict__ mask, uint32_t* __restrict__ out, int B,
                                                                      int T) {
    const int G = T >> 5;
    const int64_t tiles = (int64_t)B * G * G, per = (int64_t)B * G * T;
    const int r = threadIdx.x & 31, half = (threadIdx.x >> 5) & 1;
    // neighbouring tiles along the keys lie in one wavefront
    const int64_t step = (int64_t)gridDim.x * (PACK_THREADS / 32);
    for (int64_t id0 = ((int64_t)blockIdx.x * PACK_THREADS + threadIdx.x) / 64 * 2; id0 < tiles; id0 += step) {
        const int64_t id = id0 + half, tile = id < tiles ? id : tiles - 1;   // a half without a tile looks at the last one
        const int kg = (int)(tile % G), qg = (int)(tile / G % G);
        const int64_t b = tile / ((int64_t)G * G);
        const mask_u32x4* src = reinterpret_cast<const mask_u32x4*>(mask + (b * T + 32 * qg + r) * (int64_t)T + 32 * kg);
        const mask_u32x4 m0 = src[0], m1 = src[1];
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) w |= mask_nibble(m0[i]) << (4 * i) | mask_nibble(m1[i]) << (16 + 4 * i);
        // transpose of the 32 x 32 bits that the 32 lanes hold: blocks of n x n change places, from n = 16 down
        uint32_t t = w, low = 0x0000ffffu;
#pragma unroll
        for (int n = 16; n > 0; n >>= 1) {
            const uint32_t y = (uint32_t)__shfl_xor((int)t, n, 64);
            t = r & n ? (t & ~low) | ((y >> n) & low) : (t & low) | ((y & low) << n);
            low ^= low << (n >> 1);
        }
        // keys 32 kg + k of the lane's query are causally visible for k <= d
        const int d = 32 * (qg - kg) + r;
        const uint32_t causal = d < 0 ? 0u : (d >= 31 ? 0xffffffffu : (2u << d) - 1u), eff = w & causal;
        const uint32_t any = (uint32_t)(__ballot(eff != 0) >> (32 * half)), differ = (uint32_t)(__ballot(eff != causal) >> (32 * half));
        if (id < tiles) {
            out[(b * G + qg) * (int64_t)T + 32 * kg + r] = t;
            out[per + (b * G + kg) * (int64_t)T + 32 * qg + r] = w;
            if (r == 0) {
                const uint32_t cls = differ == 0 ? TILE_CAUSAL : (any != 0 ? TILE_MIXED : TILE_HIDDEN);
                uint32_t* const cq = out + 2 * per;
                cq[tile] = cls;
                cq[tiles + (b * G + kg) * (int64_t)G + qg] = cls;
            }
        }
    }
}
// classes of the 32-wide sub-tiles from number `g` on that a wavefront takes of a tile (wave-uniform)
struct TileClasses { uint32_t c0, c1; };
template <bool HALVES> __device__ __forceinline__ TileClasses load_classes(const uint32_t* __restrict__ row, int g) {
    const uniform_words p = as_uniform(row + g);
    return {p[0], HALVES ? (uint32_t)TILE_HIDDEN : p[1]};
}
template <bool HALVES> __device__ __forceinline__ KeepWords load_keep(const uint32_t* __restrict__ line, int base) {
    if constexpr (HALVES) return load_keep_half(line, base);
    else return load_keep_words(line, base);
}

// Which tile and batch-head a workgroup of a grid (B*H, tiles) takes.  In dispatch order tiles go from long to short; the
// second layer of 256 workgroups (one per CU) runs backwards, so that the CU with the longest of the first gets the shortest of
// the next instead of the longest again.  Only a whole layer is turned, and a workgroup keeps its number modulo 8, hence its
// XCD and the K and V in that one's L2.  Batch 8 x 1024 x 12 heads (three layers): forward 25.9 -> 24.6 us, dQ 35.2 -> 33.3.
// Two or three layers are there at once; later ones go to the CUs that are free first, the longest first: turned as well, the
// last workgroups to start were not the shortest ones, and 16 x 1024 (six layers) took 43.9 us forward, now 41.9 (50.6 -> 48.0
// with dropout).
struct Place { int tile, bh; };
__device__ __forceinline__ Place place() {
    const uint32_t total = gridDim.x * gridDim.y;
    uint32_t id = blockIdx.y * gridDim.x + blockIdx.x;
    if (id >> 8 == 1 && (id | 255) < total) id ^= 31 << 3;
    return {(int)(id / gridDim.x), (int)(id % gridDim.x)};
}

// ---- forward -------------------------------------------------------------------------
// grid (B*H, ceil(T/128)), see place(); wave w owns queries q0 + 32w .. +31; K/V tiles of 64 keys.
// (three workgroups per CU = three wavefronts per SIMD, 168 registers each)
template <bool HAS_MASK, bool TRAIN>
__global__ __launch_bounds__(ATT_THREADS, 3) void attn_fwd_kernel(const AttnArgs a) {
    constexpr int STAGE = 2 * PANEL;          // K, V
    __shared__ __attribute__((aligned(16))) char smem[RING * STAGE];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int lr = lane & 31, lg = lane >> 5;
    // grid (B*H, T/128): the batch-head index is the fast dispatch dimension and the query
    // tiles go from the longest (last) to the shortest, so the workgroups that start last
    // are the cheapest ones (causal work per tile grows with the query position).
    const Place pl = place();
    const int bh = pl.bh, bidx = bh / a.H, hidx = bh % a.H;
    const int q0 = (gridDim.y - 1 - pl.tile) * 128;
    const int qw0 = q0 + wave * 32;
    const int query = qw0 + lr;
    const int qrow = query < a.T ? query : a.T - 1;

    const bf16* Qb = (const bf16*)a.q + bidx * a.q_bs + hidx * a.q_hs;
    const bf16* Kb = (const bf16*)a.k + bidx * a.k_bs + hidx * a.k_hs;
    const bf16* Vb = (const bf16*)a.v + bidx * a.v_bs + hidx * a.v_hs;

    RowPieces qf;
    load_row_frags(qf, Qb + (int64_t)qrow * a.q_rs, lg);

    int nkt = (q0 + 128) / 64;
    if (nkt > a.T / 64) nkt = a.T / 64;

    const int wave_u = __builtin_amdgcn_readfirstlane(wave);
    const uint32_t lds0 = lds_addr(smem);
    PanelCopy ck, cv;
#define FWD_COPY(KT, SLOT)                                                             \
    {                                                                                  \
        ck.issue(KT, lds0 + (SLOT) * STAGE, wave_u);                                   \
        cv.issue(KT, lds0 + (SLOT) * STAGE + PANEL, wave_u);                           \
    }
    ck.init(Kb, a.k_rs, tid);
    cv.init(Vb, a.v_rs, tid);
    FWD_COPY(0, 0)
    frags_landed(qf);
    if (nkt > 1) FWD_COPY(1, 1)
    // keep-bit line of this batch-head and the wave's first query as scalars
    const uint32_t* __restrict__ kline = a.keepbits + (int64_t)bh * a.bitwords;
    const int qw0u = lookup_row(q0 + wave_u * 32, a.T);
    copies_landed<4>(nkt > 1);
    lds_barrier();

    const float sc = a.scale * LOG2E;
    float m_run = M_START, m_true = M_START, l_run = 0.f;
    f32x16 o[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;

    KeepWords kw_next;
    if constexpr (TRAIN) kw_next = load_keep_words(kline, qw0u);
    // tile classes of the wave's 32 queries against every 32-key group (explicit mask only)
    const uint32_t* __restrict__ crow = nullptr;
    TileClasses tc_next = {TILE_CAUSAL, TILE_CAUSAL};
    if constexpr (HAS_MASK) {
        const int G = a.T >> 5;
        crow = a.mask + 2 * (int64_t)a.B * G * a.T + ((int64_t)bidx * G + (qw0u >> 5)) * G;
        tc_next = load_classes<false>(crow, 0);
    }
    int st = 0;   // this tile's place in LDS
    for (int kt = 0; kt < nkt; ++kt) {
        if (kt + 2 < nkt) FWD_COPY(kt + 2, next_slot(next_slot(st)))
        // keep bits and classes of this tile were requested one step ago; request the next tile's now
        const KeepWords kw = kw_next;
        if constexpr (TRAIN) kw_next = load_keep_words(kline, qw0u + (kt + 1) * 64);
        const TileClasses tc = tc_next;
        if constexpr (HAS_MASK) tc_next = load_classes<false>(crow, 2 * (kt + 1 < nkt ? kt + 1 : kt));
        __builtin_amdgcn_sched_barrier(0);
        const int key0 = kt * 64;
        // some key of this tile is visible to some query of the wave
        if (key0 <= qw0 + 31 && (!HAS_MASK || (tc.c0 | tc.c1) != TILE_HIDDEN)) {
            const char* kp = smem + st * STAGE;
            const char* vp = kp + PANEL;
            RowFrags<2> ka;
            ka.read(kp, 0, lr, lg);
            __builtin_amdgcn_sched_barrier(0);
            f32x16 s[2];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int e = 0; e < 16; ++e) s[j][e] = 0.f;
            ka.mma(s, qf);
            TpFrags va[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) va[j].read(vp, j, lr, lg);
            __builtin_amdgcn_sched_barrier(0);

            if (key0 + 63 > qw0) {   // tile touches the diagonal for this wave
#pragma unroll
                for (int j = 0; j < 2; ++j) apply_causal<true>(s[j], query - key0 - j * 32 - lg * 4);
            }
            if constexpr (HAS_MASK) {
                // one word per key: the mask bits of the wave's 32 queries (wave-uniform loads), read
                // only for a half whose tile is not already described by the causal pattern
                const uniform_words mw = as_uniform(a.mask + ((int64_t)bidx * (a.T >> 5) + (qw0u >> 5)) * a.T + key0);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if ((j == 0 ? tc.c0 : tc.c1) == TILE_CAUSAL) continue;
                    uint32_t w[32];
#pragma unroll
                    for (int t = 0; t < 32; ++t) w[t] = mw[j * 32 + t];
#pragma unroll
                    for (int i = 0; i < 16; ++i) s[j][i] = mask_select(s[j][i], NEG_RAW, mask_lanes(w, i));
                }
            }
            float tmax = s[0][0];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 16; ++i) tmax = fmaxf(tmax, s[j][i]);
            tmax = max_xor32(tmax) * sc;
            m_true = fmaxf(m_true, tmax);
            // The exponentials are taken relative to m_run, which follows the true row maximum
            // only when some row of the wavefront has outgrown it by more than 2^RESCALE_SLACK:
            // softmax does not depend on the reference point, p stays below 2^RESCALE_SLACK, and
            // the 32 rescaling multiplies of the accumulators are skipped on most tiles.  The
            // saved statistics are converted to the true maximum at the end.
            if (__builtin_amdgcn_ballot_w64(tmax > m_run + RESCALE_SLACK) != 0) {
                const float m_new = fmaxf(m_run, tmax);
                const float alpha = fast_exp2(m_run - m_new);
                l_run *= alpha;
                m_run = m_new;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
            }
            float p[2][16];
            float lsum = 0.f;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float e = fast_exp2(fmaf(s[j][i], sc, -m_run));
                    p[j][i] = e;
                    lsum += e;
                }
            l_run += sum_xor32(lsum);
            if constexpr (TRAIN) {
                keep_apply<0>(p[0], kw);
                keep_apply<1>(p[1], kw);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) va[j].mma(o, p[j]);
        }
        __builtin_amdgcn_sched_barrier(0);
        copies_landed<4>(kt + 2 < nkt);
        lds_barrier();
        st = next_slot(st);
    }
#undef FWD_COPY

    if (query < a.T) {
        // l_run = 0: no key of the row is visible (a row with a visible key has l_run >= 1)
        const bool empty = l_run == 0.f;
        const float f = empty ? 0.f : (TRAIN ? 1.0f : 0.9f) / l_run;
        store_rows<bf16>((bf16*)a.out0 + bidx * a.out0_bs + hidx * a.out0_hs + (int64_t)query * a.out0_rs, o, f, lg);
        if (lg == 0) {
            // statistics relative to the true row maximum: sum exp(s - m_true) = l_run 2^(m_run - m_true)
            a.ms[(int64_t)bh * a.T + query] = empty ? NEG_NAT : m_true * LN2;
            a.ls[(int64_t)bh * a.T + query] = empty ? 0.f : l_run * fast_exp2(m_run - m_true);
        }
    }
}

// How the four wavefronts of a workgroup share the backward's work on its tiles of 64 rows.  Whole: four blocks of 32 rows of their own,
// each against every tile.  Halves: two blocks, and of every tile one half for each wavefront of a block; the two results are put
// together at the end.
template <bool HALVES> struct Share {
    static constexpr int BLOCKS = HALVES ? 2 : 4, ROWS = 32 * BLOCKS, NJ = HALVES ? 1 : 2;
    int block, half;     // the wavefront's block; first sub-tile of 32 rows that it takes of a tile
    __device__ __forceinline__ Share(int wave) : block(wave % BLOCKS), half(wave / BLOCKS) {}
};

// ---- backward: dK, dV -------------------------------------------------------------------
// One workgroup per (batch-head, 128 keys): wave w owns keys key0 + 32w .. +31 (lane = key); query tiles of 64.
// OWN_DELTA: delta = rowsum(dO * O) is formed here, from the dO rows on their way into LDS and the O rows beside
// them, instead of being read from what the dQ pass stored.
typedef float StatTile[3][64];            // m2, 1/l, delta of a query tile
// delta of row (tid >> 3) + 32 i from the 16-byte pieces x of dO and y of O: eight neighbouring lanes hold a row
template <typename F>
__device__ __forceinline__ float piece_dot(const F& x, const F& y) {
    float part = 0.f;
#pragma unroll
    for (int e = 0; e < (int)(sizeof(F) / sizeof(x[0])); ++e) part += (float)x[e] * (float)y[e];
    return part;
}
__device__ __forceinline__ void store_delta(float* __restrict__ delta, int i, float part, int tid) {
    part += __shfl_xor(part, 1, 64);
    part += __shfl_xor(part, 2, 64);
    part += __shfl_xor(part, 4, 64);
    if ((tid & 7) == 0) delta[(tid >> 3) + 32 * i] = part;
}
constexpr int RAW_STATS = 3 * 64 * 4;     // bytes of a query tile's saved maxima, sums and delta
constexpr int dkdv_stage(bool own_delta) { return (own_delta ? 3 : 2) * PANEL + RAW_STATS; }   // Q, dO (, O), statistics
template <bool OWN_DELTA> constexpr int dkdv_lds() { return RING * dkdv_stage(OWN_DELTA); }
template <bool HAS_MASK, bool TRAIN, bool OWN_DELTA, bool HALVES>
__device__ __forceinline__ void attn_bwd_dkdv(const AttnArgs& a, const int bh, const int key_tile, char* smem, StatTile* sstat) {
    constexpr int STAGE = dkdv_stage(OWN_DELTA);

    const int tid = threadIdx.x, lane = tid & 63, wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Share<HALVES> share(wave_u);
    const int lr = lane & 31, lg = lane >> 5;
    const int bidx = bh / a.H, hidx = bh % a.H;
    const int key0 = key_tile * Share<HALVES>::ROWS;
    const int kw0 = key0 + share.block * 32;
    const int key = kw0 + lr;
    const int krow = key < a.T ? key : a.T - 1;

    const bf16* Qb = (const bf16*)a.q + bidx * a.q_bs + hidx * a.q_hs;
    const bf16* Kb = (const bf16*)a.k + bidx * a.k_bs + hidx * a.k_hs;
    const bf16* Vb = (const bf16*)a.v + bidx * a.v_bs + hidx * a.v_hs;
    const bf16* dOb = (const bf16*)a.d_o + bidx * a.do_bs + hidx * a.do_hs;
    const bf16* Ob = (const bf16*)a.o + bidx * a.o_bs + hidx * a.o_hs;

    RowPieces kf, vf;
    load_row_frags(kf, Kb + (int64_t)krow * a.k_rs, lg);
    load_row_frags(vf, Vb + (int64_t)krow * a.v_rs, lg);

    const int qt0 = key0 / 64, nqt = a.T / 64;

    // 1/l goes into the exponent (p = 2^(s - m - log2 l)), one multiplication less
    // per element.  A row without a visible key (saved l = 0) gets m = 0 and no log2 l instead: all
    // of its scores are masked (-1.44e9 in the exponent), so its p is exactly 0.
    const int64_t stat0 = (int64_t)bh * a.T + (tid & 63);

    f32x16 dk[2], dv[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) dk[t][e] = dv[t][e] = 0.f;

    const uint32_t lds0 = lds_addr(smem);
    PanelCopy cq, cd, co;
    // The statistics come with the tile; the first wavefront copies them, converts them once they have landed
    // and leaves them in sstat for the workgroup.  Each wavefront waits for its own copies only: the rows of
    // dO and O that it multiplies for delta are those that it copied itself.
    constexpr int RAW = (OWN_DELTA ? 3 : 2) * PANEL, COPIES = OWN_DELTA ? 6 : 4, STAT_COPIES = OWN_DELTA ? 2 : 3;
#define KV_COPY(QT, SLOT)                                                              \
    {                                                                                  \
        const uint32_t to__ = lds0 + (SLOT) * STAGE;                                   \
        cq.issue(QT, to__, wave_u);                                                    \
        cd.issue(QT, to__ + PANEL, wave_u);                                            \
        if constexpr (OWN_DELTA) co.issue(QT, to__ + 2 * PANEL, wave_u);               \
        if (wave_u == 0) {                                                             \
            copy4_to_lds(a.ms + stat0 + (QT) * 64, to__ + RAW);                        \
            copy4_to_lds(a.ls + stat0 + (QT) * 64, to__ + RAW + 256);                  \
            if constexpr (!OWN_DELTA) copy4_to_lds(a.delta + stat0 + (QT) * 64, to__ + RAW + 512); \
        }                                                                              \
    }
#define KV_LAND(SLOT, PAR, MORE)                                                       \
    {                                                                                  \
        const char* in__ = smem + (SLOT) * STAGE;                                      \
        if (wave_u == 0) {                                                             \
            copies_landed<COPIES + STAT_COPIES>(MORE);                                 \
            const float* raw__ = reinterpret_cast<const float*>(in__ + RAW);           \
            const float m__ = raw__[lane], l__ = raw__[64 + lane];                     \
            const bool none__ = l__ == 0.f;                                            \
            sstat[PAR][0][lane] = none__ ? 0.f : fmaf(m__, LOG2E, __builtin_amdgcn_logf(l__)); \
            if constexpr (!OWN_DELTA) sstat[PAR][2][lane] = raw__[128 + lane];         \
        } else copies_landed<COPIES>(MORE);                                            \
        if constexpr (OWN_DELTA)                                                       \
            _Pragma("unroll") for (int i = 0; i < 2; ++i) {                            \
                const char* x__ = in__ + PANEL + i * 32 * BKB + tid * 16;              \
                store_delta(sstat[PAR][2], i, piece_dot(*reinterpret_cast<const bf16x8*>(x__),  \
                            *reinterpret_cast<const bf16x8*>(x__ + PANEL)), tid);      \
            }                                                                          \
        lds_barrier();                                                                 \
    }
    cq.init(Qb, a.q_rs, tid);
    cd.init(dOb, a.do_rs, tid);
    if constexpr (OWN_DELTA) co.init(Ob, a.o_rs, tid);
    KV_COPY(qt0, 0)
    frags_landed(kf);
    frags_landed(vf);
    if (qt0 + 1 < nqt) KV_COPY(qt0 + 1, 1)
    KV_LAND(0, 0, qt0 + 1 < nqt)

    const float sc = a.scale * LOG2E;
    // keep-bit line of this batch-head and the wave's first key as scalars
    const uint32_t* __restrict__ kline = a.keepbits + (int64_t)bh * a.bitwords;
    const int kw0u = lookup_row(kw0, a.T);
    KeepWords kw_next;
    if constexpr (TRAIN) kw_next = load_keep<HALVES>(kline, kw0u + share.half * 32 + qt0 * 64);
    // tile classes of the wave's 32 keys against every 32-query group (explicit mask only)
    const uint32_t* __restrict__ crow = nullptr;
    TileClasses tc_next = {TILE_CAUSAL, TILE_CAUSAL};
    if constexpr (HAS_MASK) {
        const int G = a.T >> 5;
        crow = a.mask + 2 * (int64_t)a.B * G * a.T + (int64_t)a.B * G * G + ((int64_t)bidx * G + (kw0u >> 5)) * G;
        tc_next = load_classes<HALVES>(crow, 2 * qt0 + share.half);
    }
    int slot = 0;   // this tile's place in LDS
    for (int qt = qt0; qt < nqt; ++qt) {
        const int st = (qt - qt0) & 1;
        if (qt + 2 < nqt) KV_COPY(qt + 2, next_slot(next_slot(slot)))
        const KeepWords kw = kw_next;   // requested one step ago
        const int ahead = qt + 1 < nqt ? qt + 1 : qt;
        if constexpr (TRAIN) kw_next = load_keep<HALVES>(kline, kw0u + share.half * 32 + ahead * 64);
        const TileClasses tc = tc_next;
        if constexpr (HAS_MASK) tc_next = load_classes<HALVES>(crow, 2 * ahead + share.half);
        __builtin_amdgcn_sched_barrier(0);
        const int q0 = qt * 64;
        if (q0 + 63 >= kw0) {   // some query of the tile sees some key of the wave
            const char* base = smem + slot * STAGE;
            // The two 32-query halves are processed one after the other: half the live
            // accumulators, which keeps two wavefronts per SIMD resident.
#pragma unroll
            for (int jj = 0; jj < Share<HALVES>::NJ; ++jj) {
                const int j = HALVES ? share.half : jj;
                if (q0 + j * 32 + 31 < kw0) continue;   // every query of this half precedes the wave's keys
                const uint32_t cls = jj == 0 ? tc.c0 : tc.c1;
                if (HAS_MASK && cls == TILE_HIDDEN) continue;
                RowFrags<1> qa, da;
                qa.read(base, j, lr, lg);
                da.read(base + PANEL, j, lr, lg);
                __builtin_amdgcn_sched_barrier(0);
                f32x16 s1[1], dp1[1];
#pragma unroll
                for (int e = 0; e < 16; ++e) s1[0][e] = dp1[0][e] = 0.f;
                qa.mma(s1, kf);      // S  [query][key]
                da.mma(dp1, vf);     // dP [query][key]
                f32x16 &s = s1[0], &dp = dp1[0];
                TpFrags dot, qtr;
                dot.read(base + PANEL, j, lr, lg);
                qtr.read(base, j, lr, lg);
                __builtin_amdgcn_sched_barrier(0);

                const bool diag = q0 + j * 32 < kw0 + 31;
                if (diag) apply_causal<false>(s, key - q0 - j * 32 - lg * 4);
                if (HAS_MASK && cls != TILE_CAUSAL) {
                    // one word per query: the mask bits of the wave's 32 keys (wave-uniform loads)
                    const uniform_words mw = as_uniform(a.mask + (int64_t)a.B * (a.T >> 5) * a.T +
                                         ((int64_t)bidx * (a.T >> 5) + (kw0u >> 5)) * a.T + q0 + j * 32);
                    uint32_t mwords[32];
#pragma unroll
                    for (int t = 0; t < 32; ++t) mwords[t] = mw[t];
#pragma unroll
                    for (int i = 0; i < 16; ++i) s[i] = mask_select(s[i], NEG_RAW, mask_lanes(mwords, i));
                }
                float pd[16], ds[16];
#pragma unroll
                for (int g4 = 0; g4 < 4; ++g4) {
                    const int qi = j * 32 + g4 * 8 + lg * 4;  // first of 4 consecutive queries (tile-relative)
                    const f32x4 m4 = *reinterpret_cast<const f32x4*>(&sstat[st][0][qi]);
                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(&sstat[st][2][qi]);
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const int i = g4 * 4 + b;
                        const float p = fast_exp2(fmaf(s[i], sc, -m4[b]));
                        if constexpr (TRAIN) {
                            // dS = P (keep ? dP : 0) - P delta = (keep ? P : 0) dP - P delta: the dropped
                            // probability is needed anyway, so one select serves both products
                            const uint64_t km = keep_lane_mask_at(kw, jj * 32 + g4 * 8 + b);
                            pd[i] = keep_select(p, km);
                            ds[i] = fmaf(pd[i], dp[i], -(p * d4[b]));
                        } else {
                            pd[i] = 0.9f * p;
                            ds[i] = p * fmaf(dp[i], 0.9f, -d4[b]);
                        }
                    }
                }
                // Hidden elements (causal or masked) need no separate dS masking: their score is the
                // fill value and the row's reference point is a real maximum (or 0 for a row without
                // visible keys), so p, hence dS, is exactly 0 there.
                dot.mma(dv, pd);   // dV^T += dO^T P
                qtr.mma(dk, ds);    // dK^T += Q^T dS
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        slot = next_slot(slot);
        if (qt + 1 < nqt) KV_LAND(slot, st ^ 1, qt + 2 < nqt)
    }
#undef KV_COPY
#undef KV_LAND

    if constexpr (HALVES) {
        // both halves of the queries together: the wavefronts of the first half finish dK, those of the second dV
        lds_barrier();
        float give[32], take[32];
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) give[16 * t + e] = share.half ? dk[t][e] : dv[t][e];
        exchange(give, take, smem, wave_u, wave_u ^ 2, lane);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) dk[t][e] = (share.half ? dv[t][e] : dk[t][e]) + take[16 * t + e];
        store_rows<bf16>(share.half ? (bf16*)a.out1 + bidx * a.out1_bs + hidx * a.out1_hs + (int64_t)key * a.out1_rs
                                    : (bf16*)a.out0 + bidx * a.out0_bs + hidx * a.out0_hs + (int64_t)key * a.out0_rs,
                         dk, share.half ? 1.0f : a.scale, lg);
    } else if (key < a.T) {
        store_rows<bf16>((bf16*)a.out0 + bidx * a.out0_bs + hidx * a.out0_hs + (int64_t)key * a.out0_rs, dk, a.scale, lg);
        store_rows<bf16>((bf16*)a.out1 + bidx * a.out1_bs + hidx * a.out1_hs + (int64_t)key * a.out1_rs, dv, 1.0f, lg);
    }
}

// ---- backward: dQ -----------------------------------------------------------------------
// Same geometry as the forward (lane = query, key tiles of 64).
constexpr int DQ_LDS = RING * 2 * PANEL;
template <bool HAS_MASK, bool TRAIN, bool STORE_DELTA, bool HALVES>
__device__ __forceinline__ void attn_bwd_dq(const AttnArgs& a, const int bh, const int query_tile, char* smem) {
    constexpr int STAGE = 2 * PANEL;          // K, V

    const int tid = threadIdx.x, lane = tid & 63, wave_u = __builtin_amdgcn_readfirstlane(tid >> 6);
    const Share<HALVES> share(wave_u);
    const int lr = lane & 31, lg = lane >> 5;
    const int bidx = bh / a.H, hidx = bh % a.H;
    const int q0 = query_tile * Share<HALVES>::ROWS;
    const int qw0 = q0 + share.block * 32;
    const int query = qw0 + lr;
    const int qrow = query < a.T ? query : a.T - 1;

    const bf16* Qb = (const bf16*)a.q + bidx * a.q_bs + hidx * a.q_hs;
    const bf16* Kb = (const bf16*)a.k + bidx * a.k_bs + hidx * a.k_hs;
    const bf16* Vb = (const bf16*)a.v + bidx * a.v_bs + hidx * a.v_hs;
    const bf16* dOb = (const bf16*)a.d_o + bidx * a.do_bs + hidx * a.do_hs;

    RowPieces qf, dof;
    load_row_frags(qf, Qb + (int64_t)qrow * a.q_rs, lg);
    load_row_frags(dof, dOb + (int64_t)qrow * a.do_rs, lg);
    const int64_t si = (int64_t)bh * a.T + qrow;
    // as in the dK/dV pass: 1/l folded into the exponent, and a row without a visible key (saved l = 0) takes m = 0
    const float lsum = a.ls[si];
    const bool none = lsum == 0.f;
    // delta = rowsum(dO * O) of the lane's query: each lane of the pair (lr, lg) holds one half
    // of the dO row already.
    float delta;
    {
        RowPieces of;
        load_row_frags(of, (const bf16*)a.o + bidx * a.o_bs + hidx * a.o_hs + (int64_t)qrow * a.o_rs, lg);
        float part = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int e = 0; e < 8; ++e) part += (float)dof[c][e] * (float)of[c][e];
        delta = part + xor32(part);
        if (STORE_DELTA && lg == 0 && query < a.T) a.delta[si] = delta;
    }
    const float m2 = none ? 0.f : fmaf(a.ms[si], LOG2E, __builtin_amdgcn_logf(lsum));

    int nkt = (q0 + Share<HALVES>::ROWS) / 64;
    if (nkt > a.T / 64) nkt = a.T / 64;

    const uint32_t lds0 = lds_addr(smem);
    PanelCopy ck, cv;
#define DQ_COPY(KT, SLOT)                                                              \
    {                                                                                  \
        ck.issue(KT, lds0 + (SLOT) * STAGE, wave_u);                                   \
        cv.issue(KT, lds0 + (SLOT) * STAGE + PANEL, wave_u);                           \
    }
    ck.init(Kb, a.k_rs, tid);
    cv.init(Vb, a.v_rs, tid);
    DQ_COPY(0, 0)
    frags_landed(qf);
    frags_landed(dof);
    if (nkt > 1) DQ_COPY(1, 1)
    copies_landed<4>(nkt > 1);
    lds_barrier();

    const float sc = a.scale * LOG2E;
    f32x16 dq[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) dq[t][e] = 0.f;

    const uint32_t* __restrict__ kline = a.keepbits + (int64_t)bh * a.bitwords;
    const int qw0u = lookup_row(qw0, a.T);
    KeepWords kw_next;
    if constexpr (TRAIN) kw_next = load_keep<HALVES>(kline, qw0u + share.half * 32);
    const uint32_t* __restrict__ crow = nullptr;
    TileClasses tc_next = {TILE_CAUSAL, TILE_CAUSAL};
    if constexpr (HAS_MASK) {
        const int G = a.T >> 5;
        crow = a.mask + 2 * (int64_t)a.B * G * a.T + ((int64_t)bidx * G + (qw0u >> 5)) * G;
        tc_next = load_classes<HALVES>(crow, share.half);
    }
    int st = 0;   // this tile's place in LDS
    for (int kt = 0; kt < nkt; ++kt) {
        if (kt + 2 < nkt) DQ_COPY(kt + 2, next_slot(next_slot(st)))
        const KeepWords kw = kw_next;   // requested one step ago
        const int ahead = kt + 1 < nkt ? kt + 1 : kt;
        if constexpr (TRAIN) kw_next = load_keep<HALVES>(kline, qw0u + share.half * 32 + ahead * 64);
        const TileClasses tc = tc_next;
        if constexpr (HAS_MASK) tc_next = load_classes<HALVES>(crow, 2 * ahead + share.half);
        __builtin_amdgcn_sched_barrier(0);
        const int key0 = kt * 64;
        if (key0 <= qw0 + 31) {
            const char* base = smem + st * STAGE;
            // The two 32-key halves one after the other: half the live accumulators, and a half
            // whose keys all follow the wave's queries is skipped.
#pragma unroll
            for (int jj = 0; jj < Share<HALVES>::NJ; ++jj) {
                const int j = HALVES ? share.half : jj;
                const int kh0 = key0 + j * 32;
                if (kh0 > qw0 + 31) continue;
                const uint32_t cls = jj == 0 ? tc.c0 : tc.c1;
                if (HAS_MASK && cls == TILE_HIDDEN) continue;
                RowFrags<1> ka, va;
                ka.read(base, j, lr, lg);
                va.read(base + PANEL, j, lr, lg);
                __builtin_amdgcn_sched_barrier(0);
                f32x16 s1[1], dp1[1];
#pragma unroll
                for (int e = 0; e < 16; ++e) s1[0][e] = dp1[0][e] = 0.f;
                ka.mma(s1, qf);      // S^T  [key][query]
                va.mma(dp1, dof);    // dP^T [key][query]
                f32x16 &s = s1[0], &dp = dp1[0];
                TpFrags ktr;
                ktr.read(base, j, lr, lg);
                __builtin_amdgcn_sched_barrier(0);

                const bool masked = kh0 + 31 > qw0;
                if (masked) apply_causal<true>(s, query - kh0 - lg * 4);
                if (HAS_MASK && cls != TILE_CAUSAL) {
                    // one word per key: the mask bits of the wave's 32 queries (wave-uniform loads)
                    const uniform_words mw = as_uniform(a.mask + ((int64_t)bidx * (a.T >> 5) + (qw0u >> 5)) * a.T + kh0);
                    uint32_t mwords[32];
#pragma unroll
                    for (int t = 0; t < 32; ++t) mwords[t] = mw[t];
#pragma unroll
                    for (int i = 0; i < 16; ++i) s[i] = mask_select(s[i], NEG_RAW, mask_lanes(mwords, i));
                }
                float ds[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const float p = fast_exp2(fmaf(s[i], sc, -m2));
                    if constexpr (TRAIN)
                        ds[i] = p * (keep_select(dp[i], keep_lane_mask_at(kw, jj * 32 + (i >> 2) * 8 + (i & 3))) - delta);
                    else
                        ds[i] = p * fmaf(dp[i], 0.9f, -delta);
                }
                // as in the dK/dV pass: p, hence dS, is exactly 0 on hidden elements
                ktr.mma(dq, ds);   // dQ^T += K^T dS^T
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        copies_landed<4>(kt + 2 < nkt);
        lds_barrier();
        st = next_slot(st);
    }
#undef DQ_COPY

    if constexpr (HALVES) {
        float give[16], take[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) give[e] = share.half ? dq[0][e] : dq[1][e];
        exchange(give, take, smem, wave_u, wave_u ^ 2, lane);
#pragma unroll
        for (int e = 0; e < 16; ++e) take[e] += share.half ? dq[1][e] : dq[0][e];
        store_half_row<bf16>((bf16*)a.out2 + bidx * a.out2_bs + hidx * a.out2_hs + (int64_t)query * a.out2_rs + share.half * 32, take, a.scale, lg);
    } else if (query < a.T)
        store_rows<bf16>((bf16*)a.out2 + bidx * a.out2_bs + hidx * a.out2_hs + (int64_t)query * a.out2_rs, dq, a.scale, lg);
}

// The backward as two launches, grid (B*H, ceil(T/128)) each: dQ, which stores delta, then dK/dV.  The tiles with the
// longest way go first in every grid: the last query tiles, the first key tiles.
// (without an explicit mask it fits three wavefronts per SIMD; the bound keeps it there)
template <bool HAS_MASK, bool TRAIN>
__global__ __launch_bounds__(ATT_THREADS, 3) void attn_bwd_dq_kernel(const AttnArgs a) {
    __shared__ __attribute__((aligned(16))) char smem[DQ_LDS];
    const Place pl = place();
    attn_bwd_dq<HAS_MASK, TRAIN, true, false>(a, pl.bh, gridDim.y - 1 - pl.tile, smem);
}
template <bool HAS_MASK, bool TRAIN>
__global__ __launch_bounds__(ATT_THREADS, 2) void attn_bwd_dkdv_kernel(const AttnArgs a) {
    __shared__ __attribute__((aligned(16))) char smem[dkdv_lds<false>()];
    __shared__ __attribute__((aligned(16))) StatTile sstat[2];
    const Place pl = place();
    attn_bwd_dkdv<HAS_MASK, TRAIN, false, false>(a, pl.bh, pl.tile, smem, sstat);
}
// Both in one launch, grid (B*H, 2 ceil(T/ROWS)).
template <bool HAS_MASK, bool TRAIN, bool HALVES>
__global__ __launch_bounds__(ATT_THREADS, 2) void attn_bwd_kernel(const AttnArgs a) {
    __shared__ __attribute__((aligned(16))) char smem[dkdv_lds<true>()];
    __shared__ __attribute__((aligned(16))) StatTile sstat[2];
    const int tile = blockIdx.y >> 1;
    if (blockIdx.y & 1) attn_bwd_dq<HAS_MASK, TRAIN, false, HALVES>(a, blockIdx.x, (gridDim.y >> 1) - 1 - tile, smem);
    else attn_bwd_dkdv<HAS_MASK, TRAIN, true, HALVES>(a, blockIdx.x, tile, smem, sstat);
}

// Launch one of the (mask, train) specialisations; further template arguments behind them.
#define ATTN_LAUNCH(KERNEL, grid, st, args, ...)                                                                              \
    do {                                                                                                                      \
        const bool hm__ = (args).mask != nullptr, tr__ = (args).train != 0;                                                   \
        if (hm__ && tr__) hipLaunchKernelGGL((KERNEL<true, true __VA_ARGS__>), grid, dim3(ATT_THREADS), 0, st, args);         \
        else if (hm__) hipLaunchKernelGGL((KERNEL<true, false __VA_ARGS__>), grid, dim3(ATT_THREADS), 0, st, args);           \
        else if (tr__) hipLaunchKernelGGL((KERNEL<false, true __VA_ARGS__>), grid, dim3(ATT_THREADS), 0, st, args);           \
        else hipLaunchKernelGGL((KERNEL<false, false __VA_ARGS__>), grid, dim3(ATT_THREADS), 0, st, args);                    \
    } while (0)
#define ATT_COMMA ,

// ---- host side ----------------------------------------------------------------------------
inline size_t bits_bytes(int64_t BH, int64_t T) { return (size_t)BH * ptj_attn_bitwords(T) * sizeof(uint32_t); }
inline size_t delta_bytes(int64_t BH, int64_t T) { return (size_t)BH * T * sizeof(float); }

int check_common(const char* what, int64_t B, int64_t H, int64_t T, int64_t dh, int dtype,
                 std::initializer_list<const void*> ptrs, std::initializer_list<int64_t> strides) {
    if (B < 1 || H < 1) return ptj_set_error(PTJ_ERR_INVALID, "%s: B and H must be positive", what);
    if (dh != DH) return ptj_set_error(PTJ_ERR_INVALID, "%s: head dimension %lld unsupported (64 only)", what, (long long)dh);
    if (T < 64 || T % 64 != 0 || T > MAX_T)
        return ptj_set_error(PTJ_ERR_INVALID, "%s: T=%lld must be a multiple of 64 in [64, %d]", what, (long long)T, MAX_T);
    if (dtype != PTJ_F32 && dtype != PTJ_BF16) return ptj_set_error(PTJ_ERR_INVALID, "%s: unknown dtype %d", what, dtype);
    const int vec = dtype == PTJ_BF16 ? 8 : 4;
    for (const void* p : ptrs)
        if (!p || !ptj_aligned16(p)) return ptj_set_error(PTJ_ERR_INVALID, "%s: null or not 16-byte aligned pointer", what);
    for (int64_t s : strides)
        if (s % vec != 0 || s < 0) return ptj_set_error(PTJ_ERR_INVALID, "%s: strides must be multiples of 16 bytes", what);
    return PTJ_OK;
}

int launch_keepbits(uint32_t* bits, int64_t count, const int64_t* seeds, int64_t stride, int64_t BH, int bitwords,
                    hipStream_t st) {
    for (int64_t c = 0; c < count; c += KEEP_SEEDS) {
        const int64_t n = count - c < KEEP_SEEDS ? count - c : KEEP_SEEDS;
        KeepSeeds ks = {};
        for (int64_t i = 0; i < n; ++i) ks.s[i] = (uint64_t)seeds[(c + i) * stride];
        hipLaunchKernelGGL(attn_keepbits_kernel, dim3((bitwords * 32 + 255) / 256, (unsigned)BH, (unsigned)n), dim3(256), 0, st,
                           bits + c * BH * bitwords, bitwords, ks);
        PTJ_CHECK_LAUNCH();
    }
    return PTJ_OK;
}

void launch_fwd(const AttnArgs& a, int dtype, hipStream_t st) {
    const dim3 grid((unsigned)(a.B * a.H), (unsigned)((a.T + 127) / 128));
    if (dtype == PTJ_F32) ptj_attn_detail::launch_fwd_f32(a, st);
    else ATTN_LAUNCH(attn_fwd_kernel, grid, st, a, );
}

// Halves (Share) where the grid leaves CUs idle: twice the workgroups and half the work per wavefront and tile, against a second
// look at every tile and the exchange at the end.  Up to three workgroups of 64 rows per CU from T = 512 on, where the short ones
// fill in behind the long ones, and fewer below, where they are more alike.  One tile has nothing to share.  us, whole / halves, 12
// heads with dropout: 2 x 128 11.5 / 10.7, 8 x 128 12.5 / 13.0, 2 x 192 14.1 / 12.3, 8 x 192 16.1 / 18.4, 2 x 256 16.5 / 13.9, 4 x 448
// 24.7 / 21.5, 7 x 448 29.2 / 31.6, 2 x 1024 43.0 / 34.8, 4 x 1024 46.3 / 57.1.  (The forward would gain as well, 2 x 256 11.0 / 9.2, but its
// bits are the same for a row in every batch.)
bool bwd_in_halves(int64_t bh, int64_t T) { return T > 64 && bh * 2 * ((T > 512 ? T : 512) / 64) <= 3 * (int64_t)ptj_num_cus(); }

// One launch while the two passes' workgroups make no more than four rounds of one per CU, two launches beyond.  The passes
// then fill each other's idle CUs and a launch is saved, against an O tile read again per query tile of dK/dV (delta) and
// the dQ tiles at the dK/dV kernel's occupancy.  From the first kernel's start to the last one's end, two launches / one, bf16
// and 12 heads (workgroups): 2 x 256 (96) 29.6 / 14.1 us, 7 x 448 (672) 37.9 / 26.8, 8 x 512 (768) 40.5 / 31.1, 4 x 1024 (768)
// 61.8 / 47.6, 8 x 1024 (1536) 79.1 / 77.1, 16 x 1024 (3072) 138.9 / 148.1.
void launch_bwd(const AttnArgs& a, int dtype, hipStream_t st) {
    if (dtype == PTJ_F32) return ptj_attn_detail::launch_bwd_f32(a, st);
    const int64_t nt = (a.T + 127) / 128;
    const unsigned bh = (unsigned)(a.B * a.H);
    if (bwd_in_halves(bh, a.T)) {
        ATTN_LAUNCH(attn_bwd_kernel, dim3(bh, (unsigned)(2 * (a.T / 64))), st, a, ATT_COMMA true);
    } else if ((int64_t)bh * nt * 2 <= (int64_t)4 * ptj_num_cus()) {
        ATTN_LAUNCH(attn_bwd_kernel, dim3(bh, (unsigned)(2 * nt)), st, a, ATT_COMMA false);
    } else {
        ATTN_LAUNCH(attn_bwd_dq_kernel, dim3(bh, (unsigned)nt), st, a, );
        ATTN_LAUNCH(attn_bwd_dkdv_kernel, dim3(bh, (unsigned)nt), st, a, );
    }
}

// Q, K, V as the column slices of one [B*T, H*3*64] buffer, O as [B*T, H*64].
AttnArgs packed_args(const void* qkv, const uint32_t* mask, float* ms, float* ls, const uint32_t* bits, int64_t B, int64_t H,
                     int64_t T, int train, int dtype) {
    AttnArgs a = {};
    const int64_t e = dtype == PTJ_BF16 ? 2 : 4, row = H * 3 * DH;
    a.q = qkv;
    a.k = (const char*)qkv + DH * e;
    a.v = (const char*)qkv + 2 * DH * e;
    a.mask = mask; a.ms = ms; a.ls = ls; a.keepbits = bits;
    a.B = (int)B; a.H = (int)H; a.T = (int)T; a.bitwords = (int)ptj_attn_bitwords(T);
    a.q_bs = a.k_bs = a.v_bs = T * row;
    a.q_hs = a.k_hs = a.v_hs = 3 * DH;
    a.q_rs = a.k_rs = a.v_rs = row;
    a.train = train != 0;
    a.scale = 0.125f;
    return a;
}

}  // namespace

int ptj_attn_keepbits_many(uint32_t* bits, int64_t count, const int64_t* seeds, int64_t stride, int64_t BH, int64_t T,
                           hipStream_t st) {
    return launch_keepbits(bits, count, seeds, stride, BH, (int)ptj_attn_bitwords(T), st);
}

int ptj_attn_fwd_packed(const void* qkv, const uint32_t* mask, void* o, float* ms, float* ls, const uint32_t* bits, int64_t B,
                        int64_t H, int64_t T, int train, int dtype, hipStream_t st) {
    const int rc = check_common("attn_fwd", B, H, T, DH, dtype, {qkv, o}, {});
    if (rc) return rc;
    AttnArgs a = packed_args(qkv, mask, ms, ls, bits, B, H, T, train, dtype);
    a.out0 = o;
    a.out0_bs = T * H * DH; a.out0_hs = DH; a.out0_rs = H * DH;
    launch_fwd(a, dtype, st);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

int ptj_attn_bwd_packed(const void* d_o, const void* qkv, const void* o, const float* ms, const float* ls,
                        const uint32_t* mask, void* dqkv, float* delta, const uint32_t* bits, int64_t B, int64_t H, int64_t T,
                        int train, int dtype, hipStream_t st) {
    const int rc = check_common("attn_bwd", B, H, T, DH, dtype, {d_o, qkv, o, dqkv}, {});
    if (rc) return rc;
    AttnArgs a = packed_args(qkv, mask, const_cast<float*>(ms), const_cast<float*>(ls), bits, B, H, T, train, dtype);
    a.o = o; a.d_o = d_o; a.delta = delta;
    a.o_bs = a.do_bs = T * H * DH;
    a.o_hs = a.do_hs = DH;
    a.o_rs = a.do_rs = H * DH;
    const int64_t e = dtype == PTJ_BF16 ? 2 : 4;
    a.out0 = (char*)dqkv + DH * e;
    a.out1 = (char*)dqkv + 2 * DH * e;
    a.out2 = dqkv;
    a.out0_bs = a.out1_bs = a.out2_bs = a.q_bs;
    a.out0_hs = a.out1_hs = a.out2_hs = a.q_hs;
    a.out0_rs = a.out1_rs = a.out2_rs = a.q_rs;
    launch_bwd(a, dtype, st);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

extern "C" {

size_t ptj_attn_workspace_bytes(int64_t B, int64_t H, int64_t T) {
    if (B < 1 || H < 1 || T < 1) return 0;
    return bits_bytes(B * H, T) + delta_bytes(B * H, T);
}

size_t ptj_attn_packed_mask_bytes(int64_t B, int64_t T) {
    if (B < 1 || T < 32 || T % 32) return 0;
    // the mask words in both orientations, then the tile classes in both index orders
    return ((size_t)2 * B * (T / 32) * T + (size_t)2 * B * (T / 32) * (T / 32)) * sizeof(uint32_t);
}

int ptj_attn_pack_mask(const uint8_t* mask, uint32_t* packed, int64_t B, int64_t T, void* stream) {
    PTJ_CHECK_ARG(mask && packed, "attn_pack_mask: null pointer");
    PTJ_CHECK_ARG(B >= 1 && T >= 32 && T % 32 == 0 && T < (1 << 24), "attn_pack_mask: need B >= 1 and T a multiple of 32");
    const int64_t tiles = B * (T / 32) * (T / 32), most = (int64_t)ptj_num_cus() * 64;
    int64_t blocks = (tiles * 32 + PACK_THREADS - 1) / PACK_THREADS;
    if (blocks > most) blocks = most;
    hipLaunchKernelGGL(attn_pack_mask_kernel, dim3((unsigned)blocks), dim3(PACK_THREADS), 0, (hipStream_t)stream, mask, packed, (int)B,
                       (int)T);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

int ptj_attn_fwd(const void* q, const void* k, const void* v, const uint32_t* mask, void* o, float* ms, float* ls,
                 void* workspace, size_t workspace_bytes, int64_t B, int64_t H, int64_t T, int64_t dh,
                 int64_t q_bs, int64_t q_hs, int64_t q_rs, int64_t k_bs, int64_t k_hs, int64_t k_rs,
                 int64_t v_bs, int64_t v_hs, int64_t v_rs, int64_t o_bs, int64_t o_hs, int64_t o_rs,
                 int train, int64_t seed, int dtype, void* stream) {
    int rc = check_common("attn_fwd", B, H, T, dh, dtype, {q, k, v, o},
                          {q_bs, q_hs, q_rs, k_bs, k_hs, k_rs, v_bs, v_hs, v_rs, o_bs, o_hs, o_rs});
    if (rc) return rc;
    PTJ_CHECK_ARG(ms && ls, "attn_fwd: null statistics pointer");
    PTJ_CHECK_ARG(!mask || (reinterpret_cast<uintptr_t>(mask) & 3) == 0, "attn_fwd: mask must be 4-byte aligned");
    const int64_t BH = B * H;
    hipStream_t st = (hipStream_t)stream;
    AttnArgs a = {};
    a.q = q; a.k = k; a.v = v; a.out0 = o; a.mask = mask; a.ms = ms; a.ls = ls;
    a.B = (int)B; a.H = (int)H; a.T = (int)T; a.bitwords = (int)ptj_attn_bitwords(T);
    a.q_bs = q_bs; a.q_hs = q_hs; a.q_rs = q_rs; a.k_bs = k_bs; a.k_hs = k_hs; a.k_rs = k_rs;
    a.v_bs = v_bs; a.v_hs = v_hs; a.v_rs = v_rs;
    a.out0_bs = o_bs; a.out0_hs = o_hs; a.out0_rs = o_rs;
    a.train = train != 0; a.scale = 0.125f;
    if (a.train) {
        if (!workspace || workspace_bytes < bits_bytes(BH, T))
            return ptj_set_error(PTJ_ERR_WORKSPACE, "attn_fwd: workspace %zu < %zu bytes", workspace_bytes, bits_bytes(BH, T));
        a.keepbits = (const uint32_t*)workspace;
        rc = launch_keepbits((uint32_t*)workspace, 1, &seed, 1, BH, a.bitwords, st);
        if (rc) return rc;
    }
    launch_fwd(a, dtype, st);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

int ptj_attn_bwd(const void* d_o, const void* q, const void* k, const void* v, const void* o, const float* ms,
                 const float* ls, const uint32_t* mask, void* dq, void* dk, void* dv, void* workspace,
                 size_t workspace_bytes, int64_t B, int64_t H, int64_t T, int64_t dh,
                 int64_t do_bs, int64_t do_hs, int64_t do_rs, int64_t q_bs, int64_t q_hs, int64_t q_rs,
                 int64_t k_bs, int64_t k_hs, int64_t k_rs, int64_t v_bs, int64_t v_hs, int64_t v_rs,
                 int64_t o_bs, int64_t o_hs, int64_t o_rs, int64_t dq_bs, int64_t dq_hs, int64_t dq_rs,
                 int64_t dk_bs, int64_t dk_hs, int64_t dk_rs, int64_t dv_bs, int64_t dv_hs, int64_t dv_rs,
                 int train, int64_t seed, int dtype, void* stream) {
    int rc = check_common("attn_bwd", B, H, T, dh, dtype, {d_o, q, k, v, o, dq, dk, dv},
                          {do_bs, do_hs, do_rs, q_bs, q_hs, q_rs, k_bs, k_hs, k_rs, v_bs, v_hs, v_rs, o_bs, o_hs, o_rs,
                           dq_bs, dq_hs, dq_rs, dk_bs, dk_hs, dk_rs, dv_bs, dv_hs, dv_rs});
    if (rc) return rc;
    PTJ_CHECK_ARG(ms && ls, "attn_bwd: null statistics pointer");
    PTJ_CHECK_ARG(!mask || (reinterpret_cast<uintptr_t>(mask) & 3) == 0, "attn_bwd: mask must be 4-byte aligned");
    const int64_t BH = B * H;
    if (!workspace || workspace_bytes < ptj_attn_workspace_bytes(B, H, T))
        return ptj_set_error(PTJ_ERR_WORKSPACE, "attn_bwd: workspace %zu < %zu bytes", workspace_bytes,
                             ptj_attn_workspace_bytes(B, H, T));
    hipStream_t st = (hipStream_t)stream;
    uint32_t* bits = (uint32_t*)workspace;
    float* delta = (float*)((char*)workspace + bits_bytes(BH, T));
    AttnArgs a = {};
    a.q = q; a.k = k; a.v = v; a.o = o; a.d_o = d_o; a.mask = mask;
    a.ms = const_cast<float*>(ms); a.ls = const_cast<float*>(ls); a.delta = delta; a.keepbits = bits;
    a.B = (int)B; a.H = (int)H; a.T = (int)T; a.bitwords = (int)ptj_attn_bitwords(T);
    a.q_bs = q_bs; a.q_hs = q_hs; a.q_rs = q_rs; a.k_bs = k_bs; a.k_hs = k_hs; a.k_rs = k_rs;
    a.v_bs = v_bs; a.v_hs = v_hs; a.v_rs = v_rs; a.o_bs = o_bs; a.o_hs = o_hs; a.o_rs = o_rs;
    a.do_bs = do_bs; a.do_hs = do_hs; a.do_rs = do_rs;
    a.train = train != 0; a.scale = 0.125f;
    if (a.train) {
        rc = launch_keepbits(bits, 1, &seed, 1, BH, a.bitwords, st);
        if (rc) return rc;
    }
    a.out0 = dk; a.out0_bs = dk_bs; a.out0_hs = dk_hs; a.out0_rs = dk_rs;
    a.out1 = dv; a.out1_bs = dv_bs; a.out1_hs = dv_hs; a.out1_rs = dv_rs;
    a.out2 = dq; a.out2_bs = dq_bs; a.out2_hs = dq_hs; a.out2_rs = dq_rs;
    launch_bwd(a, dtype, st);
    PTJ_CHECK_LAUNCH();
    return PTJ_OK;
}

}  // extern "C"
