// Launch parameters of the attention kernels, shared by the C ABI wrapper and the model driver.
#pragma once
#include "agpu_internal.h"

struct AttnParams {
    const float *q;  // element (b, h, i, e) at q[b*q_batch_stride + h*q_head_stride + i*q_row_stride + e]
    const float *k;  // [batch*n_heads, kv_stride, 64]
    const float *v;
    float *o;        // element (b, h, i, e) at o[b*o_batch_stride + h*o_head_stride + i*o_row_stride + e]
    int n_heads, batch, q_len, kv_len, q_offset, kv_stride, causal;
    long long q_batch_stride, q_head_stride, q_row_stride;
    long long o_batch_stride, o_head_stride, o_row_stride;
    // When non-null the kernels read the number of positions already cached from here and use
    // kv_len = *pos_dev + q_len, q_offset = *pos_dev (lets one captured launch serve every step).
    const int *pos_dev;
    // Decode kernel: fetch the first pass of K/V rows before the context length is known (hides one memory
    // round trip; reads up to 32 * waves rows whatever the length).  Set by the launcher for small launches.
    int speculate;
    // Prefill kernel: a workgroup takes query block nb-1-x and then block x (set by the launcher).
    int pair_blocks;
    // Decode kernel with the keys split over gridDim.z workgroups (set by the launcher): keys per workgroup, where
    // the partial results go, and the tickets (one per query row and head, left at zero).
    int kv_chunk;
    float *kv_partial;
    unsigned int *counters;
    int strict;  // the context's strict_sync
    // Decode kernel, q_len == 1 and batch <= 16 only: the outputs once more as the bf16 pieces of the next Linear's
    // input (row = sequence, k = head * 64 + e; layout in linear_common.h), or null.
    uint4 *px_pieces;
    // Prefill kernels (q_len > 8): instead of o, the outputs times a power of two as the pairs of the next Linear's input (row = sequence *
    // q_len + i, k = head * 64 + e; gemm_pairs.h), or null.
    char *pairs;
    uint8_t *pair_marks;         // (PairMarks)
    uint32_t *pair_tiles, epoch;
    float pairs_up;
    // The same: all of the cache's K times 2^k_exp and V times 2^v_exp is known to stay below 2^15.
    int kv_known, k_exp, v_exp;
};

// max_kv_len bounds kv_len for launches that read it from pos_dev (sizes the key split).
int32_t agpu_attention_launch(agpu_ctx *ctx, const AttnParams &p, int max_kv_len);

// K and V as f16 operand fragments: [batch * n_heads][tiles_cap tiles of 32 keys][512 fragments of 16 bytes] each, in the layout that
// attention.hip describes, times powers of two that leave them below 2^15.
struct AttFrags {
    const uint4 *k, *v;
    // The tiles' exponents of K and V, and which dimensions of V are not all zeros, [batch * n_heads][tiles_cap] (split_kv_kernel), or null: k_exp
    // and v_exp for all.
    const int4 *exps;
    int k_exp, v_exp;
    int tiles_cap;
    // with k_exp and v_exp: heads that have `epoch` here are not fit for them (KvScatter)
    const uint32_t *v_small = nullptr;
    uint32_t epoch = 0;
};
// Tiles' exponents do not go beyond these, for tiles of (almost) nothing: they and their differences have to stay powers of two that fp32 has.
constexpr int kMaxFragExpK = 100, kMaxFragExpV = 78;

// Causal prefill attention of queries 0 .. q_len - 1 over keys 0 .. kv_len - 1 (kv_len >= q_len >= 256, host values; p.k and
// p.v, the same as rows, are read where the fragments do not do); agpu_attention_fragment_bytes sizes one array of fragments.
size_t agpu_attention_fragment_bytes(int heads, int kv_len);
int32_t agpu_attention_fragments_launch(agpu_ctx *ctx, const AttnParams &p, const AttFrags &fr);
