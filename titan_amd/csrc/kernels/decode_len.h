// decode_len.h -- live lengths and splits of the fixed-split decode, shared by
// its split kernels and their merge.
#pragma once
#include <stdint.h>

struct len_src {
    const uint32_t* ptr;  // device lengths or position
    uint32_t mode;        // 0: host scalars, 1: *ptr is the query position, 2: ptr[b] = tokens
    uint32_t seq_tokens, query_pos, causal;
};

__device__ __forceinline__ uint32_t live_tokens(const len_src& L, uint32_t b) {
    if (L.mode == 2) return L.ptr[b];
    if (L.mode == 1) return L.ptr[0] + 1u;  // paged_attention.cu:21-24
    uint32_t n = L.seq_tokens;
    if (L.causal && L.query_pos + 1u < n) n = L.query_pos + 1u;
    return n;
}

// Tokens per split of n live tokens.  Under a device position the host knows
// only the table's capacity, and tps covers that in max_splits; a context below
// `shorter` tokens (max_splits * (tps - round) + 1; 0: none) is cut into at most
// as many splits of fewer whole rounds (2^round_log2 tokens, one pass of a
// workgroup's waves), which the grid and the workspace hold.  The test spares the
// others the divisions: 0.3 us of a 7 us step.
__device__ __forceinline__ uint32_t live_tps(uint32_t n, uint32_t tps, uint32_t max_splits, uint32_t round_log2,
                                             uint32_t shorter) {
    if (n >= shorter) return tps;
    const uint32_t rounds = ((n + max_splits - 1u) / max_splits + (1u << round_log2) - 1u) >> round_log2;
    return (rounds ? rounds : 1u) << round_log2;
}

// Splits covering n tokens, capped by the launched grid.  Callers size the
// grid so that n <= max_splits * tps; the cap only keeps a violating length
// inside the workspace.
__device__ __forceinline__ uint32_t split_count(uint32_t n, uint32_t tps, uint32_t max_splits) {
    const uint32_t s = n / tps + (n % tps != 0u);
    return s < max_splits ? s : max_splits;
}
