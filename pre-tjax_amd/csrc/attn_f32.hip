// Causal flash attention of 4-byte storage: the algorithm, layouts, masks and statistics of attn.hip, multiplied on the bf16
// matrix pipe.
//
// Every factor is the exact sum of three bf16 values (Split8), and six products of the parts stand for one, as in gemm_split.h, which
// names the method and bounds the other three by 2^-25 |a b| and less: 192 clocks per 32x32x16 where the fp32 instructions take
// 512.  Q, K, V and dO are split once per workgroup on their way into registers or LDS, P and dS where they are formed.  The
// parts lie in LDS as bf16 panels, which transposing reads serve in both directions, so no transposed copies exist.
// What bounds it: the waits of two wavefronts per SIMD (the registers and, in the backward, 149 KB of LDS allow no third) for LDS,
// memory and each other, 35 to 48 % of their time.  Forward / backward, matrix pipe and vector ALU busy: batch 8 x 1024 x 12 heads
// 39 / 45 % and 47 / 39 %, 8 x 512 27 / 33 % and 38 / 35 %, 8 x 512 with padding and dropout 17 / 21 % and 32 / 30 %.  8 x 1024 multiplies at
// 940 and 1075 TFLOP/s of bf16 products, where this repository's fp32 GEMMs reach 1000 to 1290.
// Eight wavefronts share a 64-row tile: four blocks of 32 rows x the two halves of the tile, so that two wavefronts per SIMD
// overlap matrix and vector work, every conversion serves 128 rows, and the way through a row's keys is half as long; the
// halves' results are added at the end.  The wavefronts of the second half convert the next tile before their products, those of
// the first half behind them (8 x 1024: backward 283 -> 277 us, forward 94 -> 89).
// fp32 instructions / this file, us, 12 heads, causal mask: 8 x 512 forward 58 / 34, backward 149 / 93; 8 x 1024 136 / 93 and 481 / 281;
// 2 x 256 24 / 16 and 46 / 25; padded documents with dropout 8 x 512 66 / 39 and 152 / 97, 8 x 1024 133 / 91 and 469 / 257.
// Error against fp64 (2-norm, 8 x 512): O 2.8e-7 / 1.5e-7, dQ 3.6e-7 / 1.9e-7, dK 5.7e-7 / 3.1e-7, dV 5.6e-7 / 3.1e-7.  Rows by the
// number of their terms (visible keys of a query, queries of a key; T = 64 to 448, scores of N(0, 1) and three times that), as a share of what
// the fp32 instructions leave: one term 0.7 to 1.1 (above 1 in O alone: a product is rounded once either way), two to 64 terms 0.3 to 0.97.
#include "attn_common.h"

namespace {

constexpr int THREADS = 512;
constexpr int TILE = 3 * PANEL;           // 64 x 64 elements as three panels

// Range, as in gemm_split.h: unscaled, the parts of factors below 2^-109 would leave bf16's range.  Q, K, V, dO and P are split as
// 2^16 times their value, of which every fp32 number has its three parts exactly; scores, dP and the gradient of V are formed 2^32
// times their value, dS 2^48 and the gradients of Q and K 2^64, and the powers are taken out where the sums are used.
constexpr float UP = 0x1p16f, UP2 = 0x1p32f, DOWN = 0x1p-16f, DOWN2 = 0x1p-32f, DOWN4 = 0x1p-64f;
constexpr float HIDDEN = NEG_RAW * UP2;

// Eight fp32 values as three times eight bf16 values whose sum they are, exactly if none is below 2^-109.
struct Split8 { bf16x8 p[3]; };
__device__ __forceinline__ Split8 split8(const float (&x)[8]) {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    u32x4 w[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float lo = x[2 * e], hi = x[2 * e + 1];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const f32x2_t f = {lo, hi};
            w[i][e] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2));
            lo -= __uint_as_float(w[i][e] << 16);
            hi -= __uint_as_float(w[i][e] & 0xffff0000u);
        }
    }
    Split8 s;
#pragma unroll
    for (int i = 0; i < 3; ++i) s.p[i] = __builtin_bit_cast(bf16x8, w[i]);
    return s;
}
// Values of the caller, the largest of which is noted: a workgroup that meets one of SPLIT_MOST or more, and a wavefront whose results
// are not finite, forms them again by the fp32 instructions (plain_fwd, plain_dkdv, plain_dq; 4 times the time).  The parts of an
// infinity or of what rounds to one are not numbers.  Below SPLIT_MOST no score and no product of dO and V overflows, and what
// overflows later is seen in the results.  The parts are those of UP times the values.
constexpr float SPLIT_MOST = 0x1p32f;
__device__ __forceinline__ Split8 split8_noted(const float (&x)[8], float& most) {
#pragma unroll
    for (int e = 0; e < 8; ++e) most = fmaxf(most, fabsf(x[e]));
    float up[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) up[e] = x[e] * UP;
    return split8(up);
}
// one multiply-add per value: NaN if one of them is not finite
template <int N> __device__ __forceinline__ bool finite(const float (&x)[N]) {
    float nan = 0.f;
#pragma unroll
    for (int e = 0; e < N; ++e) nan = fmaf(x[e], 0.f, nan);
    return nan == 0.f;
}
__device__ __forceinline__ Split8 split_row_piece(const float* __restrict__ p, float& most) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
    const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
    return split8_noted(x, most);
}
// The MFMA operand pieces of one 64-element row (lane half lg) in registers
__device__ __forceinline__ void load_row_splits(Split8 (&f)[4], const float* __restrict__ row, int lg, float& most) {
#pragma unroll
    for (int c = 0; c < 4; ++c) f[c] = split_row_piece(row + c * 16 + lg * 8, most);
}

__device__ __forceinline__ void mma(f32x16& acc, const bf16x8& a, const bf16x8& b) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
}
// MFMA operand pieces of rows 32 j .. of a tile, contraction chunk c
__device__ __forceinline__ Split8 row_split(const char* __restrict__ tile, int j, int c, int lr, int lg) {
    const char* p = tile + (j * 32 + lr) * BKB + (((c * 2 + lg) ^ row_swizzle(lr)) << 4);
    Split8 a;
#pragma unroll
    for (int i = 0; i < 3; ++i) a.p[i] = *reinterpret_cast<const bf16x8*>(p + i * PANEL);
    return a;
}
// The leading part alone
__device__ __forceinline__ bf16x8 row_first(const char* __restrict__ tile, int j, int c, int lr, int lg) {
    return *reinterpret_cast<const bf16x8*>(tile + (j * 32 + lr) * BKB + (((c * 2 + lg) ^ row_swizzle(lr)) << 4));
}
// The parts of two factors in the order of their products: the lower ones first.  Scores are sums of one chain, with the products of
// leading parts behind all others: the matrix pipe rounds its accumulator with every instruction, here four times at its full
// size and twenty times at 2^-8 of it.  (All six of a chunk after one another: twice the error against fp64 in every result.)
// P is formed again in the backward against the forward's row maximum and sum, which only cancels what error the scores have if they are
// the same bits: all three kernels keep to this order of (K, Q).
constexpr int FIRST[6] = {2, 0, 1, 1, 0, 0}, SECOND[6] = {0, 2, 1, 0, 1, 0};
__device__ __forceinline__ void mma_low(f32x16& s, const Split8& a, const Split8& b) {
#pragma unroll
    for (int i = 0; i < 5; ++i) mma(s, a.p[FIRST[i]], b.p[SECOND[i]]);
}
// Two chains side by side.  SWAPPED: the second factor's parts in the order of the first's
template <int N = 6, bool SWAPPED = false>
__device__ __forceinline__ void mma_two(f32x16& s0, const Split8& a0, const Split8& b0, f32x16& s1, const Split8& a1, const Split8& b1) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int x = SWAPPED ? SECOND[i] : FIRST[i], y = SWAPPED ? FIRST[i] : SECOND[i];
        mma(s0, a0.p[x], b0.p[y]);
        mma(s1, a1.p[x], b1.p[y]);
    }
}
// The leading parts are read again behind the lower products (kept in registers, the backward spills)
__device__ __forceinline__ void forget_rows() { asm volatile("" ::: "memory"); }

// o[t] += (columns 32 t .. of the tile, transposed) x p: contraction over the tile's rows 32 j + 16 h .. + 15, of which the lane
// holds p[e] for row 32 j + 16 h + 8 (e / 4) + 4 lg + e % 4
typedef short i16x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void columns_x_regs(f32x16 (&o)[2], const char* __restrict__ tile, const Split8& p, int j, int h, int lr, int lg) {
    const int x = 4 * lg + ((lr & 15) >> 2);
    Split8 a[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int piece = t * 4 + 2 * (lr >> 4) + ((lr & 3) >> 1);
        const char* pp = tile + (j * 32 + h * 16 + x) * BKB + 8 * (lr & 1);
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(pp + i * PANEL + ((piece ^ row_swizzle(x)) << 4)));
            const i16x4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4_t*)(pp + i * PANEL + 8 * BKB + ((piece ^ row_swizzle(x + 8)) << 4)));
            a[t].p[i] = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        }
    }
    mma_two(o[0], a[0], p, o[1], a[1], p);
}

// A 64 x 64 tile on its way from memory to LDS: every thread has eight elements of a row
struct TileCopy {
    const float* src;        // the thread's piece of tile 0
    int64_t step;            // elements from a tile to the next
    f32x4 r[2];
    __device__ __forceinline__ void init(const float* __restrict__ p, int64_t row_stride, int tid) {
        src = p + (int64_t)(tid >> 3) * row_stride + (tid & 7) * 8;
        step = 64 * row_stride;
    }
    __device__ __forceinline__ void fetch(int tile) {
        const float* s = src + tile * step;
        r[0] = *reinterpret_cast<const f32x4*>(s);
        r[1] = *reinterpret_cast<const f32x4*>(s + 4);
    }
    __device__ __forceinline__ void store(char* __restrict__ tile, int tid, float& most) const {
        const float x[8] = {r[0][0], r[0][1], r[0][2], r[0][3], r[1][0], r[1][1], r[1][2], r[1][3]};
        const Split8 s = split8_noted(x, most);
        char* to = tile + (tid >> 3) * BKB + (((tid & 7) ^ row_swizzle(tid >> 3)) << 4);
#pragma unroll
        for (int i = 0; i < 3; ++i) *reinterpret_cast<bf16x8*>(to + i * PANEL) = s.p[i];
    }
};

__device__ __forceinline__ uint64_t keep_mask(const KeepWords& w, int i) { return keep_lane_mask_at(w, (i >> 2) * 8 + (i & 3)); }

// The mask words of a mixed tile: hidden elements become `hidden`
__device__ __forceinline__ void apply_mask(f32x16& s, const uint32_t* __restrict__ words, float hidden) {
    const uniform_words mw = as_uniform(words);
    uint32_t w[32];
#pragma unroll
    for (int t = 0; t < 32; ++t) w[t] = mw[t];
#pragma unroll
    for (int i = 0; i < 16; ++i) s[i] = mask_select(s[i], hidden, mask_lanes(w, i));
}

struct RowStats { float m_run, m_true, l; };      // reference point of the exponentials, true maximum (both base 2), sum
// The reference point follows the row maximum only when it has been outgrown by 2^RESCALE_SLACK, see attn.hip
__device__ __forceinline__ void follow_maximum(const f32x16& s, float sc, RowStats& r, f32x16 (&o)[2]) {
    float tmax = s[0];
#pragma unroll
    for (int i = 1; i < 16; ++i) tmax = fmaxf(tmax, s[i]);
    tmax = max_xor32(tmax) * sc;
    r.m_true = fmaxf(r.m_true, tmax);
    if (__builtin_amdgcn_ballot_w64(tmax > r.m_run + RESCALE_SLACK) != 0) {
        const float m_new = fmaxf(r.m_run, tmax), alpha = fast_exp2(r.m_run - m_new);
        r.l *= alpha;
        r.m_run = m_new;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) o[t][e] *= alpha;
    }
}
__device__ __forceinline__ void store_stats(const AttnArgs& a, int64_t at, const RowStats& r) {
    const bool empty = r.l == 0.f;
    a.ms[at] = empty ? NEG_NAT : r.m_true * LN2;
    a.ls[at] = empty ? 0.f : r.l * fast_exp2(r.m_run - r.m_true);
}
// l = 0: no key of the row is visible (a row with a visible key has l >= 1)
template <bool TRAIN> __device__ __forceinline__ float row_factor(float l) { return l == 0.f ? 0.f : (TRAIN ? 1.0f : 0.9f) / l; }

// The forward's results of both wavefronts: the columns of its own half are finished here.
__device__ __forceinline__ RowStats merge_halves(float (&out)[16], const f32x16 (&o)[2], RowStats mine, int half, char* __restrict__ smem, int wave,
                                                 int partner, int lane) {
    float give[19], take[19];
#pragma unroll
    for (int e = 0; e < 16; ++e) give[e] = half ? o[0][e] : o[1][e];
    give[16] = mine.m_run;
    give[17] = mine.m_true;
    give[18] = mine.l;
    exchange(give, take, smem, wave, partner, lane);
    const float m_run = fmaxf(mine.m_run, take[16]), f0 = fast_exp2(mine.m_run - m_run), f1 = fast_exp2(take[16] - m_run);
#pragma unroll
    for (int e = 0; e < 16; ++e) out[e] = (half ? o[1][e] : o[0][e]) * f0 + take[e] * f1;
    return {m_run, fmaxf(mine.m_true, take[17]), half ? fmaf(take[18], f1, mine.l * f0) : fmaf(mine.l, f0, take[18] * f1)};
}

// ---- the same by the fp32 instructions, operands straight from memory: for workgroups whose values the split does not take ----
// Each function: one wavefront, 32 rows (all of them exist) against every tile of 32; of the results what `half` finishes.
// s += (32 rows, the lane's at x) x (32 rows, the lane's at y), contraction over their 64 columns.  (Rolled: nothing is kept in
// registers that the main loops need.)
__device__ __forceinline__ void plain_rows(f32x16& s, const float* __restrict__ x, const float* __restrict__ y, int lg) {
#pragma unroll 1
    for (int c = 0; c < 8; ++c)
        mma_chunk(s, *reinterpret_cast<const f32x4*>(x + c * 8 + lg * 4), *reinterpret_cast<const f32x4*>(y + c * 8 + lg * 4));
}
// o[t] += (columns 32 t .. of 32 rows, transposed) x p, contraction over the rows
__device__ __forceinline__ void plain_columns(f32x16 (&o)[2], const float* __restrict__ rows, int64_t rs, const float (&p)[16], int lr, int lg) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f32x4 x, y;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[e] = rows[(c * 8 + lg * 4 + e) * rs + t * 32 + lr];
                y[e] = p[4 * c + e];
            }
            mma_chunk(o[t], x, y);
        }
        __builtin_amdgcn_sched_barrier(0);
    }
}
__device__ __forceinline__ float plain_delta(const float* __restrict__ d_o, const float* __restrict__ o, int lg) {
    float sum = 0.f;
#pragma unroll 1
    for (int c = 0; c < 8; ++c) {
        const f32x4 x = *reinterpret_cast<const f32x4*>(d_o + c * 8 + lg * 4), y = *reinterpret_cast<const f32x4*>(o + c * 8 + lg * 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) sum += x[e] * y[e];
    }
    return sum + xor32(sum);
}
// Mask words and tile classes of the 32 rows from row0 on (AttnArgs::mask)
struct PlainMask { const uint32_t *words, *classes; };
template <bool LANE_IS_QUERY> __device__ __forceinline__ PlainMask plain_mask(const AttnArgs& a, int bidx, int row0) {
    const int64_t G = a.T >> 5, block = bidx * G + (row0 >> 5), all = (int64_t)a.B * G;
    return {a.mask + (LANE_IS_QUERY ? 0 : all * a.T) + block * a.T, a.mask + 2 * all * a.T + (LANE_IS_QUERY ? 0 : all * G) + block * G};
}

template <bool HAS_MASK, bool TRAIN>
__device__ __forceinline__ void plain_fwd(const AttnArgs& a, int bh, int qw0, int half) {
    const int lane = threadIdx.x & 63, lr = lane & 31, lg = lane >> 5, bidx = bh / a.H, hidx = bh % a.H, query = qw0 + lr;
    const float* const k = (const float*)a.k + bidx * a.k_bs + hidx * a.k_hs;
    const float* const v = (const float*)a.v + bidx * a.v_bs + hidx * a.v_hs;
    const float* const q_row = (const float*)a.q + bidx * a.q_bs + hidx * a.q_hs + query * a.q_rs;
    const float sc = a.scale * LOG2E;
    RowStats row = {M_START, M_START, 0.f};
    f32x16 o[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;
#pragma unroll 1
    for (int key0 = 0; key0 <= qw0; key0 += 32) {
        uint32_t cls = TILE_CAUSAL;
        if constexpr (HAS_MASK) cls = as_uniform(plain_mask<true>(a, bidx, qw0).classes)[key0 >> 5];
        if (cls == TILE_HIDDEN) continue;
        f32x16 s;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = 0.f;
        plain_rows(s, k + (key0 + lr) * a.k_rs, q_row, lg);
        if (key0 == qw0) apply_causal<true>(s, query - key0 - lg * 4);
        if (HAS_MASK && cls != TILE_CAUSAL) apply_mask(s, plain_mask<true>(a, bidx, qw0).words + key0, NEG_RAW);
        follow_maximum(s, sc, row, o);
        KeepWords kw;
        if constexpr (TRAIN) kw = load_keep_half(a.keepbits + (int64_t)bh * a.bitwords, qw0 + key0);
        float p[16], lsum = 0.f;
#pragma unroll
        for (int e = 0; e < 16; ++e) {
            p[e] = fast_exp2(fmaf(s[e], sc, -row.m_run));
            lsum += p[e];
            if constexpr (TRAIN) p[e] = keep_select(p[e], keep_mask(kw, e));
        }
        plain_columns(o, v + key0 * a.v_rs, a.v_rs, p, lr, lg);
        row.l += sum_xor32(lsum);
    }
    float out[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) out[e] = half ? o[1][e] : o[0][e];
    store_half_row<float>((float*)a.out0 + bidx * a.out0_bs + hidx * a.out0_hs + query * a.out0_rs + half * 32, out, row_factor<TRAIN>(row.l), lg);
    if (lg == 0 && half == 0) store_stats(a, (int64_t)bh * a.T + query, row);
}

template <bool HAS_MASK, bool TRAIN>
__device__ __forceinline__ void plain_dkdv(const AttnArgs& a, int bh, int kw0, int half) {
    const int lane = threadIdx.x & 63, lr = lane & 31, lg = lane >> 5, bidx = bh / a.H, hidx = bh % a.H, key = kw0 + lr;
    const float* const q = (const float*)a.q + bidx * a.q_bs + hidx * a.q_hs;
    const float* const d_o = (const float*)a.d_o + bidx * a.do_bs + hidx * a.do_hs;
    const float* const o = (const float*)a.o + bidx * a.o_bs + hidx * a.o_hs;
    const float* const k_row = (const float*)a.k + bidx * a.k_bs + hidx * a.k_hs + key * a.k_rs;
    const float* const v_row = (const float*)a.v + bidx * a.v_bs + hidx * a.v_hs + key * a.v_rs;
    const float sc = a.scale * LOG2E;
    f32x16 dk[2], dv[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) dk[t][e] = dv[t][e] = 0.f;
#pragma unroll 1
    for (int q0 = kw0; q0 < a.T; q0 += 32) {
        uint32_t cls = TILE_CAUSAL;
        if constexpr (HAS_MASK) cls = as_uniform(plain_mask<false>(a, bidx, kw0).classes)[q0 >> 5];
        if (cls == TILE_HIDDEN) continue;
        f32x16 s, dp;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = dp[e] = 0.f;
        plain_rows(s, q + (q0 + lr) * a.q_rs, k_row, lg);
        plain_rows(dp, d_o + (q0 + lr) * a.do_rs, v_row, lg);
        if (q0 == kw0) apply_causal<false>(s, key - q0 - lg * 4);
        if (HAS_MASK && cls != TILE_CAUSAL) apply_mask(s, plain_mask<false>(a, bidx, kw0).words + q0, NEG_RAW);
        KeepWords kw;
        if constexpr (TRAIN) kw = load_keep_half(a.keepbits + (int64_t)bh * a.bitwords, kw0 + q0);
        // the statistics of query q0 + lr, passed to the lanes that hold elements of its row
        const float delta = plain_delta(d_o + (q0 + lr) * a.do_rs, o + (q0 + lr) * a.o_rs, lg);
        const int64_t si = (int64_t)bh * a.T + q0 + lr;
        const float l = a.ls[si];
        const bool none = l == 0.f;
        const float linv = none ? 0.f : 1.0f / l, m2 = none ? 0.f : a.ms[si] * LOG2E;
        float pd[16], ds[16];
        int first = 4 * lg;
        asm volatile("" : "+v"(first));          // (sixteen lane numbers are not kept over the loop)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const int qi = first + 8 * (i >> 2) + (i & 3);
            const float d = __shfl(delta, qi, 64), p = fast_exp2(fmaf(s[i], sc, -__shfl(m2, qi, 64))) * __shfl(linv, qi, 64);
            if constexpr (TRAIN) {
                pd[i] = keep_select(p, keep_mask(kw, i));
                ds[i] = fmaf(pd[i], dp[i], -(p * d));
            } else {
                pd[i] = 0.9f * p;
                ds[i] = p * fmaf(dp[i], 0.9f, -d);
            }
        }
        plain_columns(dv, d_o + q0 * a.do_rs, a.do_rs, pd, lr, lg);
        plain_columns(dk, q + q0 * a.q_rs, a.q_rs, ds, lr, lg);
    }
    if (half) store_rows<float>((float*)a.out1 + bidx * a.out1_bs + hidx * a.out1_hs + key * a.out1_rs, dv, 1.0f, lg);
    else store_rows<float>((float*)a.out0 + bidx * a.out0_bs + hidx * a.out0_hs + key * a.out0_rs, dk, a.scale, lg);
}

template <bool HAS_MASK, bool TRAIN>
__device__ __forceinline__ void plain_dq(const AttnArgs& a, int bh, int qw0, int half) {
    const int lane = threadIdx.x & 63, lr = lane & 31, lg = lane >> 5, bidx = bh / a.H, hidx = bh % a.H, query = qw0 + lr;
    const float* const k = (const float*)a.k + bidx * a.k_bs + hidx * a.k_hs;
    const float* const v = (const float*)a.v + bidx * a.v_bs + hidx * a.v_hs;
    const float* const q_row = (const float*)a.q + bidx * a.q_bs + hidx * a.q_hs + query * a.q_rs;
    const float* const do_row = (const float*)a.d_o + bidx * a.do_bs + hidx * a.do_hs + query * a.do_rs;
    const float delta = plain_delta(do_row, (const float*)a.o + bidx * a.o_bs + hidx * a.o_hs + query * a.o_rs, lg);
    const int64_t si = (int64_t)bh * a.T + query;
    const float l = a.ls[si], sc = a.scale * LOG2E;
    const bool none = l == 0.f;
    const float linv = none ? 0.f : 1.0f / l, m2 = none ? 0.f : a.ms[si] * LOG2E;
    f32x16 dq[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) dq[t][e] = 0.f;
#pragma unroll 1
    for (int key0 = 0; key0 <= qw0; key0 += 32) {
        uint32_t cls = TILE_CAUSAL;
        if constexpr (HAS_MASK) cls = as_uniform(plain_mask<true>(a, bidx, qw0).classes)[key0 >> 5];
        if (cls == TILE_HIDDEN) continue;
        f32x16 s, dp;
#pragma unroll
        for (int e = 0; e < 16; ++e) s[e] = dp[e] = 0.f;
        plain_rows(s, k + (key0 + lr) * a.k_rs, q_row, lg);
        plain_rows(dp, v + (key0 + lr) * a.v_rs, do_row, lg);
        if (key0 == qw0) apply_causal<true>(s, query - key0 - lg * 4);
        if (HAS_MASK && cls != TILE_CAUSAL) apply_mask(s, plain_mask<true>(a, bidx, qw0).words + key0, NEG_RAW);
        KeepWords kw;
        if constexpr (TRAIN) kw = load_keep_half(a.keepbits + (int64_t)bh * a.bitwords, qw0 + key0);
        float ds[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            const float p = fast_exp2(fmaf(s[i], sc, -m2)) * linv;
            if constexpr (TRAIN) ds[i] = p * (keep_select(dp[i], keep_mask(kw, i)) - delta);
            else ds[i] = p * fmaf(dp[i], 0.9f, -delta);
        }
        plain_columns(dq, k + key0 * a.k_rs, a.k_rs, ds, lr, lg);
    }
    float out[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) out[e] = half ? dq[1][e] : dq[0][e];
    store_half_row<float>((float*)a.out2 + bidx * a.out2_bs + hidx * a.out2_hs + query * a.out2_rs + half * 32, out, a.scale, lg);
}

// ---- forward -------------------------------------------------------------------------
// grid (B*H, ceil(T/128)): wavefront (half, block) owns queries q0 + 32 block .. +31 against the keys of its half of each tile
template <bool HAS_MASK, bool TRAIN>
__global__ __launch_bounds__(THREADS, 2) void attn_fwd_f32_kernel(const AttnArgs a) {
    __shared__ __attribute__((aligned(16))) char smem[2][2 * TILE];      // K, V
    __shared__ int big;
    if (threadIdx.x == 0) big = 0;

    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lg = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2;
    const int bh = blockIdx.x, bidx = bh / a.H, hidx = bh % a.H;
    const int q0 = (gridDim.y - 1 - blockIdx.y) * 128;
    const int qw0 = q0 + (wave & 3) * 32;
    const int query = qw0 + lr;
    const int qrow = query < a.T ? query : a.T - 1;

    TileCopy ck, cv;
    ck.init((const float*)a.k + bidx * a.k_bs + hidx * a.k_hs, a.k_rs, tid);
    cv.init((const float*)a.v + bidx * a.v_bs + hidx * a.v_hs, a.v_rs, tid);
    ck.fetch(0);
    cv.fetch(0);
    float most = 0.f;
    Split8 qf[4];
    load_row_splits(qf, (const float*)a.q + bidx * a.q_bs + hidx * a.q_hs + (int64_t)qrow * a.q_rs, lg, most);
    ck.store(smem[0], tid, most);
    cv.store(smem[0] + TILE, tid, most);
    __syncthreads();

    int nkt = (q0 + 128) / 64;
    if (nkt > a.T / 64) nkt = a.T / 64;
    const float sc = a.scale * LOG2E * DOWN2;
    RowStats row = {M_START, M_START, 0.f};
    f32x16 o[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) o[t][e] = 0.f;

    // keep bits and tile class of a step are requested one step ahead
    const uint32_t* __restrict__ kline = a.keepbits + (int64_t)bh * a.bitwords;
    const int lookup = lookup_row(qw0, a.T);
    KeepWords kw_next;
    if constexpr (TRAIN) kw_next = load_keep_half(kline, lookup + half * 32);
    const uint32_t* __restrict__ crow = nullptr;
    uint32_t cls_next = TILE_CAUSAL;
    if constexpr (HAS_MASK) {
        const int G = a.T >> 5;
        crow = a.mask + 2 * (int64_t)a.B * G * a.T + ((int64_t)bidx * G + (lookup >> 5)) * G + half;
        cls_next = as_uniform(crow)[0];
    }
    auto fetch = [&](int tile) __attribute__((always_inline)) {
        ck.fetch(tile);
        cv.fetch(tile);
    };
    auto store = [&](int tile) __attribute__((always_inline)) {
        ck.store(smem[tile & 1], tid, most);
        cv.store(smem[tile & 1] + TILE, tid, most);
    };
    if (half && nkt > 1) fetch(1);
    for (int kt = 0; kt < nkt; ++kt) {
        const bool more = kt + 1 < nkt;
        const int ahead = more ? kt + 1 : kt;
        if (half == 0) {
            if (more) fetch(kt + 1);
        } else {
            if (more) store(kt + 1);
            if (kt + 2 < nkt) fetch(kt + 2);
        }
        const KeepWords kw = kw_next;
        if constexpr (TRAIN) kw_next = load_keep_half(kline, lookup + half * 32 + ahead * 64);
        const uint32_t cls = cls_next;
        if constexpr (HAS_MASK) cls_next = as_uniform(crow)[2 * ahead];
        const int key0 = kt * 64 + half * 32;
        if (key0 <= qw0 + 31 && (!HAS_MASK || cls != TILE_HIDDEN)) {
            const char* kp = smem[kt & 1];
            f32x16 s;
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c) mma_low(s, row_split(kp, half, c, lr, lg), qf[c]);       // S^T [key][query]
            forget_rows();
#pragma unroll
            for (int c = 0; c < 4; ++c) mma(s, row_first(kp, half, c, lr, lg), qf[c].p[0]);
            if (key0 + 31 > qw0) apply_causal<true>(s, query - key0 - lg * 4, HIDDEN);
            if (HAS_MASK && cls != TILE_CAUSAL) apply_mask(s, a.mask + ((int64_t)bidx * (a.T >> 5) + (lookup >> 5)) * a.T + key0, HIDDEN);
            follow_maximum(s, sc, row, o);
            float lsum = 0.f;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float p[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    p[e] = fast_exp2(fmaf(s[8 * h + e], sc, -row.m_run)) * UP;
                    lsum += p[e];
                    if constexpr (TRAIN) p[e] = keep_select(p[e], keep_mask(kw, 8 * h + e));
                }
                columns_x_regs(o, kp + TILE, split8(p), half, h, lr, lg);
            }
            row.l += sum_xor32(lsum);         // (UP times the sum)
        }
        if (half == 0 && more) store(kt + 1);
        __syncthreads();
    }

    // Both halves of the keys together; each wavefront finishes the columns of its own half.
    float out[16];
    if (most >= SPLIT_MOST) big = 1;
    RowStats r = merge_halves(out, o, row, half, &smem[0][0], wave, wave ^ 4, lane);
    if (qw0 >= a.T) return;
    if (__builtin_expect(big || __any(!finite(out)), 0)) {
        plain_fwd<HAS_MASK, TRAIN>(a, bh, qw0, half);
    } else {
        r.l *= DOWN;
        store_half_row<float>((float*)a.out0 + bidx * a.out0_bs + hidx * a.out0_hs + (int64_t)query * a.out0_rs + half * 32, out, row_factor<TRAIN>(r.l) * DOWN2, lg);
        if (lg == 0 && half == 0) store_stats(a, (int64_t)bh * a.T + query, r);
    }
}

// ---- backward: dK, dV -------------------------------------------------------------------
// One workgroup per (batch-head, 128 keys): wavefront (half, block) owns keys key0 + 32 block .. +31 (lane = key) against the
// queries of its half of each tile.  delta = rowsum(dO * O) is formed on the rows' way into LDS.  The keys' rows of K wait in
// registers, those of V in LDS: both in registers spill (8 x 512: 122 us instead of 93).
typedef float StatTile[3][64];            // m2, UP / l, UP2 delta of a query tile
template <bool HAS_MASK, bool TRAIN>
__device__ __forceinline__ void bwd_dkdv(const AttnArgs& a, const int bh, const int key_tile, char (*smem)[2 * TILE], char (*vrows)[TILE], StatTile* sstat, int& big) {
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lg = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2;
    const int bidx = bh / a.H, hidx = bh % a.H;
    const int kw0 = key_tile * 128 + (wave & 3) * 32;
    const int key = kw0 + lr;
    const int krow = key < a.T ? key : a.T - 1;
    const int qt0 = key_tile * 2, nqt = a.T / 64;

    TileCopy cq, cd, co;
    cq.init((const float*)a.q + bidx * a.q_bs + hidx * a.q_hs, a.q_rs, tid);
    cd.init((const float*)a.d_o + bidx * a.do_bs + hidx * a.do_hs, a.do_rs, tid);
    co.init((const float*)a.o + bidx * a.o_bs + hidx * a.o_hs, a.o_rs, tid);
    const int64_t stat0 = (int64_t)bh * a.T + (tid & 63);
    float st_m = 0.f, st_l = 0.f, most = 0.f;
    auto fetch = [&](int qt) __attribute__((always_inline)) {
        cq.fetch(qt);
        cd.fetch(qt);
        co.fetch(qt);
        st_m = a.ms[stat0 + qt * 64];
        st_l = a.ls[stat0 + qt * 64];
    };
    auto store = [&](int b) __attribute__((always_inline)) {
        float part = 0.f;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) part += cd.r[i][e] * co.r[i][e];
        part += __shfl_xor(part, 1, 64);
        part += __shfl_xor(part, 2, 64);
        part += __shfl_xor(part, 4, 64);
        if ((tid & 7) == 0) sstat[b][2][tid >> 3] = part * UP2;
        if (tid < 64) {
            // a row without a visible key (saved l = 0) takes m = 0 and 1/l = 0, which makes its p exactly 0
            const bool none = st_l == 0.f;
            sstat[b][0][tid] = none ? 0.f : st_m * LOG2E;
            sstat[b][1][tid] = none ? 0.f : UP / st_l;
        }
        cq.store(smem[b], tid, most);
        cd.store(smem[b] + TILE, tid, most);
    };
    fetch(qt0);
    {
        // the workgroup's rows of V (the last tile's second half may lie past the end: repeated, not used)
        TileCopy cv;
        cv.init((const float*)a.v + bidx * a.v_bs + hidx * a.v_hs, a.v_rs, tid);
        cv.fetch(key_tile * 2);
        cv.store(vrows[0], tid, most);
        cv.fetch(key_tile * 2 + 1 < nqt ? key_tile * 2 + 1 : nqt - 1);
        cv.store(vrows[1], tid, most);
    }
    Split8 kf[4];
    load_row_splits(kf, (const float*)a.k + bidx * a.k_bs + hidx * a.k_hs + (int64_t)krow * a.k_rs, lg, most);
    store(0);
    __syncthreads();

    const float sc = a.scale * LOG2E * DOWN2;
    f32x16 dk[2], dv[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) dk[t][e] = dv[t][e] = 0.f;

    const uint32_t* __restrict__ kline = a.keepbits + (int64_t)bh * a.bitwords;
    const int lookup = lookup_row(kw0, a.T);
    KeepWords kw_next;
    if constexpr (TRAIN) kw_next = load_keep_half(kline, lookup + qt0 * 64 + half * 32);
    const uint32_t* __restrict__ crow = nullptr;
    uint32_t cls_next = TILE_CAUSAL;
    if constexpr (HAS_MASK) {
        const int G = a.T >> 5;
        crow = a.mask + 2 * (int64_t)a.B * G * a.T + (int64_t)a.B * G * G + ((int64_t)bidx * G + (lookup >> 5)) * G + half;
        cls_next = as_uniform(crow)[2 * qt0];
    }
    if (half && qt0 + 1 < nqt) fetch(qt0 + 1);
    for (int qt = qt0; qt < nqt; ++qt) {
        const int b = (qt - qt0) & 1;
        const bool more = qt + 1 < nqt;
        const int ahead = more ? qt + 1 : qt;
        const KeepWords kw = kw_next;
        if constexpr (TRAIN) kw_next = load_keep_half(kline, lookup + half * 32 + ahead * 64);
        const uint32_t cls = cls_next;
        if constexpr (HAS_MASK) cls_next = as_uniform(crow)[2 * ahead];
        const int q0 = qt * 64 + half * 32;
        const bool live = q0 + 31 >= kw0 && (!HAS_MASK || cls != TILE_HIDDEN);
        const char *qp = smem[b], *dp_ = smem[b] + TILE;
        f32x16 s, dp;
        if (half == 0) {
            if (more) fetch(qt + 1);
        } else {
            if (more) store(b ^ 1);
            if (qt + 2 < nqt) fetch(qt + 2);
        }
        if (live) {
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = dp[e] = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c)       // S and dP [query][key]
                mma_two<5, true>(s, row_split(qp, half, c, lr, lg), kf[c], dp, row_split(dp_, half, c, lr, lg), row_split(vrows[(wave & 3) >> 1], wave & 1, c, lr, lg));
            forget_rows();
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                mma(s, row_first(qp, half, c, lr, lg), kf[c].p[0]);
                mma(dp, row_first(dp_, half, c, lr, lg), row_first(vrows[(wave & 3) >> 1], wave & 1, c, lr, lg));
            }
        }
        if (live) {
            if (q0 < kw0 + 31) apply_causal<false>(s, key - q0 - lg * 4, HIDDEN);
            if (HAS_MASK && cls != TILE_CAUSAL)
                apply_mask(s, a.mask + (int64_t)a.B * (a.T >> 5) * a.T + ((int64_t)bidx * (a.T >> 5) + (lookup >> 5)) * a.T + q0, HIDDEN);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float pd[8], ds[8];
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    const int qi = half * 32 + (2 * h + g) * 8 + lg * 4;   // first of 4 consecutive queries (tile-relative)
                    const f32x4 m4 = *reinterpret_cast<const f32x4*>(&sstat[b][0][qi]);
                    const f32x4 l4 = *reinterpret_cast<const f32x4*>(&sstat[b][1][qi]);
                    const f32x4 d4 = *reinterpret_cast<const f32x4*>(&sstat[b][2][qi]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int i = 8 * h + 4 * g + e;
                        const float p = fast_exp2(fmaf(s[i], sc, -m4[e])) * l4[e];
                        if constexpr (TRAIN) {
                            // dS = P (keep ? dP : 0) - P delta = (keep ? P : 0) dP - P delta
                            pd[4 * g + e] = keep_select(p, keep_mask(kw, i));
                            ds[4 * g + e] = fmaf(pd[4 * g + e], dp[i], -(p * d4[e]));
                        } else {
                            pd[4 * g + e] = 0.9f * p;
                            ds[4 * g + e] = p * fmaf(dp[i], 0.9f, -d4[e]);
                        }
                    }
                }
                // p, hence dS, is exactly 0 on hidden elements, see attn.hip
                columns_x_regs(dv, dp_, split8(pd), half, h, lr, lg);   // dV^T += dO^T P
                columns_x_regs(dk, qp, split8(ds), half, h, lr, lg);    // dK^T += Q^T dS
            }
        }
        if (half == 0 && more) store(b ^ 1);
        __syncthreads();
    }

    // Both halves of the queries together: the wavefronts of the first half finish dK, those of the second dV.
    float give[32], take[32];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) give[16 * t + e] = half ? dk[t][e] : dv[t][e];
    if (most >= SPLIT_MOST) big = 1;
    exchange(give, take, &smem[0][0], wave, wave ^ 4, lane);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) take[16 * t + e] += half ? dv[t][e] : dk[t][e];
    if (kw0 >= a.T) return;
    if (__builtin_expect(big || __any(!finite(take)), 0)) {
        plain_dkdv<HAS_MASK, TRAIN>(a, bh, kw0, half);
    } else {
        float* const row = half ? (float*)a.out1 + bidx * a.out1_bs + hidx * a.out1_hs + (int64_t)key * a.out1_rs
                                : (float*)a.out0 + bidx * a.out0_bs + hidx * a.out0_hs + (int64_t)key * a.out0_rs;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int e = 0; e < 16; ++e) dk[t][e] = take[16 * t + e];
        store_rows<float>(row, dk, half ? DOWN2 : a.scale * DOWN4, lg);
    }
}

// ---- backward: dQ -----------------------------------------------------------------------
// Same geometry as the forward.
template <bool HAS_MASK, bool TRAIN>
__device__ __forceinline__ void bwd_dq(const AttnArgs& a, const int bh, const int query_tile, char (*smem)[2 * TILE], int& big) {
    const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lg = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), half = wave >> 2;
    const int bidx = bh / a.H, hidx = bh % a.H;
    const int q0 = query_tile * 128;
    const int qw0 = q0 + (wave & 3) * 32;
    const int query = qw0 + lr;
    const int qrow = query < a.T ? query : a.T - 1;

    TileCopy ck, cv;
    ck.init((const float*)a.k + bidx * a.k_bs + hidx * a.k_hs, a.k_rs, tid);
    cv.init((const float*)a.v + bidx * a.v_bs + hidx * a.v_hs, a.v_rs, tid);
    ck.fetch(0);
    cv.fetch(0);
    const float* const do_row = (const float*)a.d_o + bidx * a.do_bs + hidx * a.do_hs + (int64_t)qrow * a.do_rs;
    const float* const o_row = (const float*)a.o + bidx * a.o_bs + hidx * a.o_hs + (int64_t)qrow * a.o_rs;
    // delta = rowsum(dO * O): each lane of the pair (lr, lg) has one half of the row
    float delta = 0.f;
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int at = (c >> 1) * 16 + lg * 8 + (c & 1) * 4;
        const f32x4 x = *reinterpret_cast<const f32x4*>(do_row + at), y = *reinterpret_cast<const f32x4*>(o_row + at);
#pragma unroll
        for (int e = 0; e < 4; ++e) delta += x[e] * y[e];
    }
    delta = (delta + xor32(delta)) * UP2;
    const int64_t si = (int64_t)bh * a.T + qrow;
    // as in dK/dV: a row without a visible key takes m = 0 and 1/l = 0
    const float lsum = a.ls[si];
    const bool none = lsum == 0.f;
    const float linv = none ? 0.f : UP / lsum, m2 = none ? 0.f : a.ms[si] * LOG2E;
    float most = 0.f;
    Split8 qf[4], dof[4];
    load_row_splits(qf, (const float*)a.q + bidx * a.q_bs + hidx * a.q_hs + (int64_t)qrow * a.q_rs, lg, most);
    load_row_splits(dof, do_row, lg, most);
    ck.store(smem[0], tid, most);
    cv.store(smem[0] + TILE, tid, most);
    __syncthreads();

    int nkt = (q0 + 128) / 64;
    if (nkt > a.T / 64) nkt = a.T / 64;
    const float sc = a.scale * LOG2E * DOWN2;
    f32x16 dq[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) dq[t][e] = 0.f;

    const uint32_t* __restrict__ kline = a.keepbits + (int64_t)bh * a.bitwords;
    const int lookup = lookup_row(qw0, a.T);
    KeepWords kw_next;
    if constexpr (TRAIN) kw_next = load_keep_half(kline, lookup + half * 32);
    const uint32_t* __restrict__ crow = nullptr;
    uint32_t cls_next = TILE_CAUSAL;
    if constexpr (HAS_MASK) {
        const int G = a.T >> 5;
        crow = a.mask + 2 * (int64_t)a.B * G * a.T + ((int64_t)bidx * G + (lookup >> 5)) * G + half;
        cls_next = as_uniform(crow)[0];
    }
    auto fetch = [&](int tile) __attribute__((always_inline)) {
        ck.fetch(tile);
        cv.fetch(tile);
    };
    auto store = [&](int tile) __attribute__((always_inline)) {
        ck.store(smem[tile & 1], tid, most);
        cv.store(smem[tile & 1] + TILE, tid, most);
    };
    if (half && nkt > 1) fetch(1);
    for (int kt = 0; kt < nkt; ++kt) {
        const bool more = kt + 1 < nkt;
        const int ahead = more ? kt + 1 : kt;
        if (half == 0) {
            if (more) fetch(kt + 1);
        } else {
            if (more) store(kt + 1);
            if (kt + 2 < nkt) fetch(kt + 2);
        }
        const KeepWords kw = kw_next;
        if constexpr (TRAIN) kw_next = load_keep_half(kline, lookup + half * 32 + ahead * 64);
        const uint32_t cls = cls_next;
        if constexpr (HAS_MASK) cls_next = as_uniform(crow)[2 * ahead];
        const int key0 = kt * 64 + half * 32;
        if (key0 <= qw0 + 31 && (!HAS_MASK || cls != TILE_HIDDEN)) {
            const char* kp = smem[kt & 1];
            f32x16 s, dp;
#pragma unroll
            for (int e = 0; e < 16; ++e) s[e] = dp[e] = 0.f;
#pragma unroll
            for (int c = 0; c < 4; ++c)       // S^T and dP^T [key][query]
                mma_two<5>(s, row_split(kp, half, c, lr, lg), qf[c], dp, row_split(kp + TILE, half, c, lr, lg), dof[c]);
            forget_rows();
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                mma(s, row_first(kp, half, c, lr, lg), qf[c].p[0]);
                mma(dp, row_first(kp + TILE, half, c, lr, lg), dof[c].p[0]);
            }
            if (key0 + 31 > qw0) apply_causal<true>(s, query - key0 - lg * 4, HIDDEN);
            if (HAS_MASK && cls != TILE_CAUSAL) apply_mask(s, a.mask + ((int64_t)bidx * (a.T >> 5) + (lookup >> 5)) * a.T + key0, HIDDEN);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                float ds[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int i = 8 * h + e;
                    const float p = fast_exp2(fmaf(s[i], sc, -m2)) * linv;
                    if constexpr (TRAIN) ds[e] = p * (keep_select(dp[i], keep_mask(kw, i)) - delta);
                    else ds[e] = p * fmaf(dp[i], 0.9f, -delta);
                }
                columns_x_regs(dq, kp, split8(ds), half, h, lr, lg);   // dQ^T += K^T dS^T
            }
        }
        if (half == 0 && more) store(kt + 1);
        __syncthreads();
    }

    float give[16], take[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) give[e] = half ? dq[0][e] : dq[1][e];
    if (most >= SPLIT_MOST) big = 1;
    exchange(give, take, &smem[0][0], wave, wave ^ 4, lane);
#pragma unroll
    for (int e = 0; e < 16; ++e) take[e] += half ? dq[1][e] : dq[0][e];
    if (qw0 >= a.T) return;
    if (__builtin_expect(big || __any(!finite(take)), 0)) plain_dq<HAS_MASK, TRAIN>(a, bh, qw0, half);
    else
        store_half_row<float>((float*)a.out2 + bidx * a.out2_bs + hidx * a.out2_hs + (int64_t)query * a.out2_rs + half * 32, take, a.scale * DOWN4, lg);
}

// grid (B*H, 2 ceil(T/128)): both passes in one launch, the tiles with the longest way first
template <bool HAS_MASK, bool TRAIN>
__global__ __launch_bounds__(THREADS, 2) void attn_bwd_f32_kernel(const AttnArgs a) {
    __shared__ __attribute__((aligned(16))) char smem[2][2 * TILE];
    __shared__ __attribute__((aligned(16))) char vrows[2][TILE];
    __shared__ __attribute__((aligned(16))) StatTile sstat[2];
    __shared__ int big;
    if (threadIdx.x == 0) big = 0;
    const int tile = blockIdx.y >> 1;
    if (blockIdx.y & 1) bwd_dq<HAS_MASK, TRAIN>(a, blockIdx.x, (gridDim.y >> 1) - 1 - tile, smem, big);
    else bwd_dkdv<HAS_MASK, TRAIN>(a, blockIdx.x, tile, smem, vrows, sstat, big);
}

}  // namespace

#define F32_LAUNCH(KERNEL, grid)                                                                                     \
    do {                                                                                                             \
        if (a.mask && a.train) hipLaunchKernelGGL((KERNEL<true, true>), grid, dim3(THREADS), 0, st, a);              \
        else if (a.mask) hipLaunchKernelGGL((KERNEL<true, false>), grid, dim3(THREADS), 0, st, a);                   \
        else if (a.train) hipLaunchKernelGGL((KERNEL<false, true>), grid, dim3(THREADS), 0, st, a);                  \
        else hipLaunchKernelGGL((KERNEL<false, false>), grid, dim3(THREADS), 0, st, a);                              \
    } while (0)

namespace ptj_attn_detail {
void launch_fwd_f32(const AttnArgs& a, hipStream_t st) {
    F32_LAUNCH(attn_fwd_f32_kernel, dim3((unsigned)(a.B * a.H), (unsigned)((a.T + 127) / 128)));
}
void launch_bwd_f32(const AttnArgs& a, hipStream_t st) {
    F32_LAUNCH(attn_bwd_f32_kernel, dim3((unsigned)(a.B * a.H), (unsigned)(2 * ((a.T + 127) / 128))));
}
}  // namespace ptj_attn_detail
