// Entry points that the library's own composites use besides the C ABI of include/ptj.h.
#pragma once
#include "common.h"

// Words per batch-head of the attention dropout's keep-bit line.
inline int64_t ptj_attn_bitwords(int64_t T) { return 2 * T / 32 + 2; }

// The keep-bit lines of `count` attention calls (seed seeds[i * stride]) in one launch: bits[i][B*H][bitwords].
int ptj_attn_keepbits_many(uint32_t* bits, int64_t count, const int64_t* seeds, int64_t stride, int64_t BH, int64_t T,
                           hipStream_t st);

// ptj_attn_fwd / ptj_attn_bwd on keep bits that are there already (nullptr: generated into the workspace).  Q, K, V
// (dQ, dK, dV) are the column slices of [B*T, H*3*64], O (dO) is [B*T, H*64].
int ptj_attn_fwd_packed(const void* qkv, const uint32_t* mask, void* o, float* ms, float* ls, const uint32_t* bits, int64_t B,
                        int64_t H, int64_t T, int train, int dtype, hipStream_t st);
int ptj_attn_bwd_packed(const void* d_o, const void* qkv, const void* o, const float* ms, const float* ls,
                        const uint32_t* mask, void* dqkv, float* delta, const uint32_t* bits, int64_t B, int64_t H, int64_t T,
                        int train, int dtype, hipStream_t st);
