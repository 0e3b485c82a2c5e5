// What the attention kernels of 2-byte (attn.hip) and 4-byte storage (attn_f32.hip) share: arguments, keep bits, masks, LDS panels.
#pragma once
#include "common.h"
#include "internal.h"
#include "mma_tile.h"

namespace ptj_attn_detail {
struct AttnArgs {
    const void *q, *k, *v, *o, *d_o;
    void *out0, *out1, *out2;     // forward: out0 = O.  Backward: dK, dV, dQ
    // nullptr = causal by index; else the mask bit-packed in both orientations (ptj_attn_pack_mask):
    //   words [0, B*T/32*T):   word (b, q/32, k) holds M[b, 32*(q/32) + r, k] in bit r   (lane = query)
    //   then the same amount:  word (b, k/32, q) holds M[b, q, 32*(k/32) + r] in bit r   (lane = key)
    //   then B*(T/32)^2 words:  class of tile (b, q/32, k/32), then the same indexed (b, k/32, q/32)
    const uint32_t* mask;
    float *ms, *ls;               // [BH, T]
    float* delta;                 // [BH, T] rowsum(dO * O)  (2-byte storage in two launches: dQ writes it, dK/dV reads it)
    const uint32_t* keepbits;     // [BH, bitwords]  (train)
    int B, H, T, bitwords;
    // element strides: batch, head, row (the head dimension itself has unit stride)
    int64_t q_bs, q_hs, q_rs, k_bs, k_hs, k_rs, v_bs, v_hs, v_rs, o_bs, o_hs, o_rs, do_bs, do_hs, do_rs;
    int64_t out0_bs, out0_hs, out0_rs, out1_bs, out1_hs, out1_rs, out2_bs, out2_hs, out2_rs;
    int train;
    float scale;                  // 1/sqrt(dh)
};
// attn_f32.hip
void launch_fwd_f32(const AttnArgs& a, hipStream_t st);
void launch_bwd_f32(const AttnArgs& a, hipStream_t st);
}  // namespace ptj_attn_detail

namespace {

using ptj_attn_detail::AttnArgs;

constexpr int DH = 64;
constexpr int PANEL = 64 * BKB;  // bytes of one 64-row LDS panel of 2-byte elements
constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;
constexpr float NEG_NAT = -1e9f;

// ---- small device helpers -----------------------------------------------------------
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float xor32(float v) { return __shfl_xor(v, 32, 64); }
// max / sum of a value with its partner in the other half of the wavefront (lane ^ 32), the same
// in both lanes: v_permlane32_swap exchanges the upper half of one register with the lower half
// of another inside the vector ALU (no LDS round trip); with both registers holding v the two
// results are {lo, lo} and {hi, hi}.
__device__ __forceinline__ float max_xor32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ __forceinline__ float sum_xor32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Permutation of the 16-byte pieces inside row `row` of a panel (64 rows of 128 bytes): the sixteen lanes that a 16-byte read
// serves at once (0-3, 12-15, 20-27 of the half wavefront, and the others) find their rows' pieces in different banks, and so
// do the four rows x 64 bytes that half a wavefront fetches with a transposing read, so ONE panel serves both directions.
__device__ __forceinline__ int row_swizzle(int row) { return ((row & 2) << 1) | ((row >> 2) & 3); }

// Keep bits of one wavefront tile as wave-uniform (scalar) words.  Element (q, k) is kept
// iff bit q + k of the batch-head's line is set.  In the kernels whose lanes are queries
// (keys), the element in accumulator register i of sub-tile j sits at
//   q + k = base + C + (lane & 31) + 4 * (lane >> 5),   C = 32 j + 8 (i / 4) + i % 4,
// with base = (wave's first query) + (tile's first key), a multiple of 32.  So the keep
// decision of ONE register across the 64 lanes is two 32-bit windows of the line at the
// constant offsets C and C + 4: a lane mask that the scalar unit extracts with two
// shifts and that a single v_cndmask applies -- no per-lane bit arithmetic at all.
// Words that no kernel here writes, at wave-uniform addresses: scalar loads, also between the inline assembly's memory clobbers.
typedef __attribute__((address_space(4))) const uint32_t* uniform_words;
__device__ __forceinline__ uniform_words as_uniform(const uint32_t* p) { return (uniform_words)(uintptr_t)p; }
// First row of a wavefront where it looks up such words.  With T an odd multiple of 64 the last workgroup's upper two
// wavefronts have no rows; theirs would be words past the end of the lines and of the mask, so they read those of the lower two.
__device__ __forceinline__ int lookup_row(int row0, int T) { return row0 - (row0 < T ? 0 : 64); }
struct KeepWords { uint32_t d0, d1, d2; };
__device__ __forceinline__ KeepWords load_keep_words(const uint32_t* __restrict__ line, int base) {
    const uniform_words p = as_uniform(line + (base >> 5));
    KeepWords w;
    w.d0 = p[0];
    w.d1 = p[1];
    w.d2 = p[2];
    return w;
}
// The same for 32 x 32 elements (offsets below 32 look at two words)
__device__ __forceinline__ KeepWords load_keep_half(const uint32_t* __restrict__ line, int base) {
    const uniform_words p = as_uniform(line + (base >> 5));
    return {p[0], p[1], 0u};
}
template <int C> __device__ __forceinline__ uint32_t keep_win32(const KeepWords& w) {
    static_assert(C >= 0 && C < 64, "window offset");
    const uint64_t v = C < 32 ? (((uint64_t)w.d1 << 32) | w.d0) : (((uint64_t)w.d2 << 32) | w.d1);
    return (uint32_t)(v >> (C & 31));
}
template <int C> __device__ __forceinline__ uint64_t keep_lane_mask(const KeepWords& w) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    const u32x2_t halves = {keep_win32<C>(w), keep_win32<C + 4>(w)};
    return __builtin_bit_cast(uint64_t, halves);
}
// The same for an offset that is a constant only after loop unrolling.
__device__ __forceinline__ uint64_t keep_lane_mask_at(const KeepWords& w, int c) {
    typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
    const uint64_t lo_pair = ((uint64_t)w.d1 << 32) | w.d0, hi_pair = ((uint64_t)w.d2 << 32) | w.d1;
    const int c4 = c + 4;
    const u32x2_t halves = {(uint32_t)((c < 32 ? lo_pair : hi_pair) >> (c & 31)),
                            (uint32_t)((c4 < 32 ? lo_pair : hi_pair) >> (c4 & 31))};
    return __builtin_bit_cast(uint64_t, halves);
}
// v where the lane's bit of `mask` is set, else 0.  The builtin turns a wave-uniform 64-bit
// mask into a per-lane condition, i.e. one v_cndmask with the mask in scalar registers
// (left to the compiler rather than inline assembly so that its hazard handling --
// e.g. the wait state after a transcendental -- still applies).
__device__ __forceinline__ float keep_select(float v, uint64_t mask) {
    return __builtin_amdgcn_inverse_ballot_w64(mask) ? v : 0.f;
}
// Attention-mask words -> lane mask of accumulator register i of a 32x32 sub-tile: the
// register holds column c = (i/4)*8 + i%4 for lanes 0..31 and column c + 4 for lanes 32..63,
// and word w[c] carries the mask bits of the 32 lanes' rows for column c.
__device__ __forceinline__ uint64_t mask_lanes(const uint32_t (&w)[32], int i) {
    const int c = (i >> 2) * 8 + (i & 3);
    return (uint64_t)w[c] | ((uint64_t)w[c + 4] << 32);
}
__device__ __forceinline__ float mask_select(float v, float other, uint64_t mask) {
    return __builtin_amdgcn_inverse_ballot_w64(mask) ? v : other;
}
// p[i] = keep ? p[i] : 0 for the 16 registers of sub-tile J
template <int J, int I = 0>
__device__ __forceinline__ void keep_apply(float (&p)[16], const KeepWords& w) {
    if constexpr (I < 16) {
        p[I] = keep_select(p[I], keep_lane_mask<J * 32 + (I >> 2) * 8 + (I & 3)>(w));
        keep_apply<J, I + 1>(p, w);
    }
}

// Store the transposed accumulators acc[t][i] (row = the lane's position `pos`, column
// d = t*32 + 8*(i/4) + 4*lg + i%4) scaled by `f` as rows of a [.., 64] tensor.
template <typename T>
__device__ __forceinline__ void store_rows(T* __restrict__ row, const f32x16 (&acc)[2], float f, int lg) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
            float v[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) v[b] = acc[t][4 * a + b] * f;
            store_vec<T, 4>(row + t * 32 + a * 8 + lg * 4, v);
        }
}

// Where two wavefronts share a block of rows, each against one half of every tile: `give` goes to the partner, what the partner
// gives comes.  Everything in `smem` has been read.
template <int N>
__device__ __forceinline__ void exchange(const float (&give)[N], float (&take)[N], char* __restrict__ smem, int wave, int partner, int lane) {
    float* const f = reinterpret_cast<float*>(smem);
#pragma unroll
    for (int i = 0; i < N; ++i) f[(wave * N + i) * 64 + lane] = give[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) take[i] = f[(partner * N + i) * 64 + lane];
}
// 32 columns of a row: element e of lane half lg is column 8 (e / 4) + 4 lg + e % 4
template <typename T>
__device__ __forceinline__ void store_half_row(T* __restrict__ row, const float (&x)[16], float f, int lg) {
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const float v[4] = {x[4 * a] * f, x[4 * a + 1] * f, x[4 * a + 2] * f, x[4 * a + 3] * f};
        store_vec<T, 4>(row + a * 8 + lg * 4, v);
    }
}
// Class of a 32x32 tile of (mask AND causal), see attn_pack_mask_kernel
enum { TILE_HIDDEN = 0, TILE_MIXED = 1, TILE_CAUSAL = 2 };
// ---- element-wise pieces (VALU budget: a wave64 VALU op costs 4 cycles, v_exp 16, and one
//      K tile gives each lane 32 score elements against 16 MFMAs = 512 cycles; every
//      instruction per element counts, so masks and dropout are compiled in only where used)
constexpr float NEG_RAW = -8e9f;          // masked raw score: NEG_RAW * (1/sqrt(64)) = -1e9
constexpr float RESCALE_SLACK = 8.0f;     // forward: the reference point of the exponentials may lag the row maximum by 2^8
constexpr float M_START = -1e8f;          // log2-domain start of the running maximum: above every masked score
                                          // (-1.44e9), below every real one, so exp2(masked - m) is exactly 0

// Causal visibility of the lane's 16 elements of a sub-tile written into the raw scores
// (invisible -> `hidden`).
//   pos0 = (lane's own index) - (first index of the sub-tile along registers) - 4*lg
//   element i = 4a+b sits at register offset 8a+b: visible iff 8a+b <= pos0 (causal part).
template <bool LANE_IS_QUERY>
__device__ __forceinline__ void apply_causal(f32x16& s, int pos0, float hidden = NEG_RAW) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int off = (i >> 2) * 8 + (i & 3);
        // lane = query: key offset must be <= query;  lane = key: query offset must be >= key
        const bool ok = LANE_IS_QUERY ? (off <= pos0) : (off >= pos0);
        s[i] = ok ? s[i] : hidden;
    }
}


}  // namespace
