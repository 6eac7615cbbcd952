// Pieces shared by the int4 Linear kernels: epilogue, nibble unpack, GEMV launch arguments.
#pragma once
#include "agpu_internal.h"
#include "elementwise.h"

// bias -> GELU -> residual, applied to one output element.
__device__ __forceinline__ float epilogue(float v, int m, int n, int N, const float *bias, const float *residual,
                                          uint32_t flags) {
    if (bias) v += bias[n];
    if (flags & AGPU_EPI_GELU_TANH) v = gelu_tanh_dev(v);
    else if (flags & AGPU_EPI_GELU_QUICK) v = gelu_quick_dev(v);
    if (residual) v += residual[(size_t)m * N + n];
    return v;
}

// The 8 nibbles of a word as unsigned floats, nf[i] = nibble i (v_cvt_f32_ubyteN on masked words).
__device__ __forceinline__ void unpack_u8(uint32_t w, float (&nf)[8]) {
    const uint32_t lo = w & 0x0F0F0F0Fu;         // nibbles 0,2,4,6 in bytes 0..3
    const uint32_t hi = (w >> 4) & 0x0F0F0F0Fu;  // nibbles 1,3,5,7
    nf[0] = (float)(lo & 0xFFu);
    nf[1] = (float)(hi & 0xFFu);
    nf[2] = (float)((lo >> 8) & 0xFFu);
    nf[3] = (float)((hi >> 8) & 0xFFu);
    nf[4] = (float)((lo >> 16) & 0xFFu);
    nf[5] = (float)((hi >> 16) & 0xFFu);
    nf[6] = (float)(lo >> 24);
    nf[7] = (float)(hi >> 24);
}

// Arguments of the decode GEMV (M <= 16 rows).
struct GemvArgs {
    const float *x;         // [M, K]
    const uint32_t *packed; // [K/8, N]
    const float *scales;    // [ceil(K/group), N]
    const float *bias;      // [N] or null
    const float *residual;  // [M, N] or null (may alias y)
    float *y;               // [M, N]
    const float *ln_gamma;  // non-null: LayerNorm over K applied to the rows of x first
    const float *ln_beta;
    float ln_eps;
    int M, N, K, group;
    uint32_t flags;         // AGPU_EPI_GELU_*
    // Optional K/V scatter for a fused QKV projection with N = 3*d_model over rows b * new_len + s (new_len 0: one new position per row, b = row):
    // columns [d, 2d) also go to kcache[(b*n_heads + h), *pos_dev + s, e], columns [2d, 3d) to vcache.
    float *kcache;
    float *vcache;
    const int *pos_dev;
    int n_heads, n_positions, new_len;
    // Optional arg-max of output row 0 over columns [0, am_cols), computed by the same launch (greedy decoding on
    // the LM head; N may be padded beyond am_cols).  Ties: the smaller index wins, or the larger one with am_last;
    // NaN never wins.  am_adv (optional) is the token feed of the arg-max kernel.  M must be 1.
    uint32_t *am_idx_out;
    int am_cols, am_last;
    ArgmaxAdvance am_adv;
};

// Epilogue for one output element, plus the optional K/V scatter of a fused QKV projection.
__device__ __forceinline__ float finish_output(const GemvArgs &a, float v, float bias, float resid, int m, int n) {
    v += bias;
    if (a.flags & AGPU_EPI_GELU_TANH) v = gelu_tanh_dev(v);
    else if (a.flags & AGPU_EPI_GELU_QUICK) v = gelu_quick_dev(v);
    v += resid;
    a.y[(size_t)m * a.N + n] = v;
    if (a.kcache) {
        const int d_model = a.N / 3;
        if (n >= d_model) {
            const int j = n - d_model;
            const bool is_v = j >= d_model;
            const int jj = is_v ? j - d_model : j;
            const int h = jj >> 6, e = jj & 63;
            float *dst = is_v ? a.vcache : a.kcache;
            const int b = a.new_len > 1 ? (int)(((float)m + 0.5f) * __builtin_amdgcn_rcpf((float)a.new_len)) : m, s = a.new_len > 1 ? m - b * a.new_len : 0;  // m < 16: exact
            dst[((size_t)(b * a.n_heads + h) * a.n_positions + *a.pos_dev + s) * 64 + e] = v;
        }
    }
    return v;
}

// Order-preserving key of a float (NaN lowest, both zeros equal) with the column behind it: the larger 64-bit word wins.
__device__ __forceinline__ unsigned long long argmax_word(float v, int n, int last) {
    if (v != v) return 0ull;
    const uint32_t u = v == 0.0f ? 0u : __float_as_uint(v);
    const uint32_t key = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((unsigned long long)key << 32) | (uint32_t)(last ? n : ~n);
}

// Largest word over the workgroup (scratch: 2 x 16 uint32); every thread of wave 0 gets the result.
__device__ __forceinline__ unsigned long long block_max_word(unsigned long long w, uint32_t *scratch, int lane, int wave, int W) {
    uint32_t hi = (uint32_t)(w >> 32), lo = (uint32_t)w;
    const uint32_t mh = wave_minmax_u32<true>(hi);
    const uint32_t ml = wave_minmax_u32<true>(hi == mh ? lo : 0u);
    if (lane == 0) {
        scratch[wave] = mh;
        scratch[16 + wave] = ml;
    }
    __syncthreads();
    hi = (lane & 15) < W ? scratch[lane & 15] : 0u;
    lo = (lane & 15) < W ? scratch[16 + (lane & 15)] : 0u;
    const uint32_t gh = row16_minmax_u32<true>(hi);
    const uint32_t gl = row16_minmax_u32<true>(hi == gh ? lo : 0u);
    return ((unsigned long long)gh << 32) | gl;
}

// Arg-max over a launch whose workgroups each hold a candidate: the candidates go out past the L2, the last workgroup to
// take a ticket picks the winner and feeds it back (the token feed of the arg-max kernel).
struct ArgmaxShare {
    unsigned long long *partial;  // one word per workgroup
    unsigned int *counter;        // left at zero
    uint32_t *idx_out;
    int last, strict;
    ArgmaxAdvance adv;
};
// Called by all W waves of every workgroup, with `best` = the thread's own candidate (0: none); scratch: 2 x 16 uint32.
__device__ __forceinline__ void argmax_finish(const ArgmaxShare &s, unsigned long long best, uint32_t *scratch, int &s_last, int tid, int W) {
    const int lane = tid & 63, wave = tid >> 6;
    best = block_max_word(best, scratch, lane, wave, W);
    if (tid == 0) {
        __hip_atomic_store(&s.partial[blockIdx.x], best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        partials_published(s.strict);
        const unsigned int t = take_ticket(s.counter, s.strict);
        s_last = (t == gridDim.x - 1);
        if (s_last) __hip_atomic_store(s.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    best = 0ull;
    for (int i = tid; i < (int)gridDim.x; i += 64 * W) {
        const unsigned long long w = __hip_atomic_load(&s.partial[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        best = w > best ? w : best;
    }
    __syncthreads();
    best = block_max_word(best, scratch, lane, wave, W);
    if (tid == 0) {
        const uint32_t lo = (uint32_t)best;
        const uint32_t win = (best >> 32) == 0ull ? 0u : (s.last ? lo : ~lo);  // nothing comparable: index 0
        s.idx_out[0] = win;
        const ArgmaxAdvance &adv = s.adv;
        if (adv.cur_tok) {
            const int st = *adv.step_dev;
            adv.cur_tok[0] = win;
            if (st < adv.out_capacity) adv.out_tok[st] = win;
            if (adv.bump_counters) {
                *adv.pos_dev += adv.delta;
                *adv.step_dev = st + 1;
            }
        }
    }
}

// The same for up to sixteen rows at once, by workgroups of any number of candidates each.
struct HeadFeed {
    unsigned long long *partial;  // [workgroups, at most one a CU][16]
    unsigned int *counter;        // left at zero
    uint32_t *idx_out;            // null: no arg-max
    int last, strict;
    ArgmaxAdvance adv;            // cur_tok null: no feed; bump_counters: always
};
inline bool feed_rows_fits(const agpu_ctx *ctx) { return (size_t)ctx->num_cus * 16 * sizeof(unsigned long long) <= ctx->ws_bytes / 2; }
inline HeadFeed feed_of(agpu_ctx *ctx, uint32_t *idx_out, int last, const ArgmaxAdvance &adv) {
    return HeadFeed{reinterpret_cast<unsigned long long *>(ctx->workspace), ctx->counters + (ctx->n_counters - 1), idx_out, last, ctx->strict_sync, adv};
}
inline size_t feed_rows_lds(int slots, int threads) { return (size_t)(slots + threads / 16) * 16 * sizeof(unsigned long long); }
// Called by all T threads of every workgroup with best[slots][row] in LDS, T / 16 more of them behind it (feed_rows_lds): over the slots, then the workgroups; the
// last one feeds the winners back.
__device__ __forceinline__ void feed_rows(const HeadFeed &feed, int rows, unsigned long long (*s_best)[16], int slots, int tid, int T) {
    __shared__ int s_last;
    unsigned long long (*s_all)[16] = s_best + slots;
    __syncthreads();
    if (tid < rows) {
        unsigned long long b = 0ull;
        for (int i = 0; i < slots; ++i) b = s_best[i][tid] > b ? s_best[i][tid] : b;
        __hip_atomic_store(&feed.partial[(size_t)blockIdx.x * 16 + tid], b, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    partials_published(feed.strict);
    __syncthreads();
    if (tid == 0) {
        const unsigned int t = take_ticket(feed.counter, feed.strict);
        s_last = (t == gridDim.x - 1);
        if (s_last) __hip_atomic_store(feed.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!s_last) return;
    const int row = tid & 15;
    unsigned long long b = 0ull;
    const int lanes = T / 16;
    constexpr int ROUNDS = 4;  // loads on their way at once
    for (int i0 = tid >> 4; i0 < (int)gridDim.x; i0 += lanes * ROUNDS) {
        unsigned long long c[ROUNDS];
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i)
            c[i] = row < rows && i0 + i * lanes < (int)gridDim.x ? __hip_atomic_load(&feed.partial[(size_t)(i0 + i * lanes) * 16 + row], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
#pragma unroll
        for (int i = 0; i < ROUNDS; ++i) b = c[i] > b ? c[i] : b;
    }
    s_all[tid >> 4][row] = b;
    __syncthreads();
    const ArgmaxAdvance &adv = feed.adv;
    const int step = adv.cur_tok ? *adv.step_dev : 0;
    if (tid < rows) {
        for (int i = 0; i < lanes; ++i) b = s_all[i][tid] > b ? s_all[i][tid] : b;
        const uint32_t lo = (uint32_t)b, win = (b >> 32) == 0ull ? 0u : (feed.last ? lo : ~lo);  // nothing comparable: index 0
        feed.idx_out[tid] = win;
        if (adv.cur_tok) {
            adv.cur_tok[tid] = win;
            if (step < adv.out_capacity) adv.out_tok[(size_t)step * rows + tid] = win;
        }
    }
    __syncthreads();  // everybody has read the step
    if (tid == 0 && adv.cur_tok) {
        *adv.pos_dev += adv.delta;
        *adv.step_dev = step + 1;
    }
}

int32_t agpu_int4_gemv_launch(agpu_ctx *ctx, const GemvArgs &a);
// int8-MFMA variant for M <= 2 (needs group % 32 == 0, K % 64 == 0, N % 4 == 0, 16-byte aligned weights).
bool agpu_int4_gemv_i8_supported(const GemvArgs &a);
int32_t agpu_int4_gemv_i8_launch(agpu_ctx *ctx, const GemvArgs &a, int max_trips_per_split, int max_wgs);
// K/V scatter of a fused QKV projection over rows (sequence b = m / new_len, step s = m % new_len), N = 3*d_model:
// columns [d, 2d) also go to kcache[(b*n_heads + h), *pos_dev + s, e], columns [2d, 3d) to vcache.
struct KvScatter {
    float *kcache;
    float *vcache;
    const int *pos_dev;
    int n_heads, n_positions, new_len;
    // Optional (sequences written from position 0; with more than one sequence new_len % 32 == 0): K and V also as the
    // f16 operand fragments of the prefill attention, [sequence * n_heads + head][tiles_cap tiles of 32 keys][512
    // fragments of 16 bytes] each, times these powers of two (which leave them below 2^15).
    uint4 *kfrag = nullptr, *vfrag = nullptr;
    int tiles_cap = 0;
    float k_up = 0.0f, v_up = 0.0f;
    // [sequence * n_heads + head]: `epoch` is left there where V does not fill its fragments (v_is_small); it has to be another one for every launch
    uint32_t *v_small = nullptr, epoch = 0;
};
// bf16-MFMA GEMM for M > 16 with x split into three bf16 pieces (needs group / 32 a power of two, K % 32 == 0,
// 16-byte aligned x).  kv (optional): the K/V scatter above, done by the same launch.
bool agpu_int4_gemm_bf16_supported(const void *x, int M, int N, int K, int group);
// Whether the launch for this shape also writes kv->kfrag / kv->vfrag.
bool agpu_int4_gemm_bf16_writes_kv_frags(const agpu_ctx *ctx, int M, int N, int K);
int32_t agpu_int4_gemm_bf16_launch(agpu_ctx *ctx, const float *x, const uint32_t *packed, const float *scales, const float *bias,
                                   const float *residual, float *y, int M, int N, int K, int group, uint32_t flags,
                                   const KvScatter *kv = nullptr);
// The same for problems too small for it (few rows): csrc/int4_gemm_rows.hip.
bool agpu_int4_gemm_rows_wanted(const agpu_ctx *ctx, int M, int N, int K);
// The same for what no other kernel than those on fp32 operands takes: K a multiple of 8 only, any number of tiles, three rows and more.
bool agpu_int4_gemm_rows_any_supported(const void *x, int M, int N, int K, int group);
int32_t agpu_int4_gemm_rows_any_launch(agpu_ctx *ctx, const float *x, const uint32_t *packed, const float *scales, const float *bias, const float *residual, float *y, int M, int N,
                                        int K, int group, uint32_t flags);
bool agpu_int4_gemm_rows_can_norm(const agpu_ctx *ctx, int M, int N, int K);
// LayerNorm of its rows without a launch: statistics [columns / 32][rows, rounded up to 32] of (mean, sum of squared distances) by 32 columns, read with gamma and
// beta where the rows are to be normalised (in: agpu_int4_gemm_rows_can_norm), left of the outputs (out: N a multiple of 32).
struct RowsLn {
    static constexpr int kMaxK = 2048;
    const float2 *in;
    const float *gamma, *beta;
    float eps;
    float2 *out;
};
// Sum over each half wave, the same bits in all its lanes; the statistics of 32 columns, one a lane.
__device__ __forceinline__ float half_wave_sum(float v) {
    v = row16_sum(v);
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(s[0]) + __uint_as_float(s[1]);
}
__device__ __forceinline__ float2 stats_of_32(float v) {  // lane = column of its half wave
    const float mean = half_wave_sum(v) * (1.0f / 32.0f), dv = v - mean;
    return make_float2(mean, half_wave_sum(dv * dv));
}
inline size_t agpu_row_stats_bytes(int M, int N) { return (size_t)(N / 32) * ((M + 31) / 32 * 32) * sizeof(float2); }
int32_t agpu_int4_gemm_rows_launch(agpu_ctx *ctx, const float *x, const uint32_t *packed, const float *scales, const float *bias,
                                   const float *residual, float *y, int M, int N, int K, int group, uint32_t flags, const KvScatter *kv, const RowsLn *ln = nullptr);
// LayerNorm (optional) + Linear like agpu_ln_int4_linear; *kv_done tells whether the launch did the K/V scatter.
int32_t agpu_ln_int4_linear_kv(agpu_ctx *ctx, const float *x, const float *gamma, const float *beta, float eps,
                               const uint32_t *packed, const float *scales, const float *bias, const float *residual, float *y,
                               int32_t M, int32_t N, int32_t K, int32_t group, uint32_t flags, const KvScatter *kv, bool *kv_done);
// MFMA variant for 2 < M <= 16 (needs group % 32 == 0, K % 32 == 0, N % 4 == 0, 16-byte aligned weights).
// With a.ln_gamma the kernel normalises the rows itself; agpu_int4_skinny_can_fuse_ln says for which shapes.
bool agpu_int4_skinny_supported(const GemvArgs &a);
bool agpu_int4_skinny_can_fuse_ln(int M, int N, int K, int group);
int32_t agpu_int4_skinny_launch(agpu_ctx *ctx, const GemvArgs &a);
// The rows of the two embeddings that row `row` of a prompt or step is the sum of.  known_pos: the number of cached positions where the host knows it (the launch sets the
// counter to it), or -1: in *pos_dev.  Ids and positions are checked on the host wherever the host knows them; a bad one on the device reads the last
// row instead of faulting.
// A workgroup has its row's addresses from scalars; with a division by d an element, and the counter set by a launch of its own in front, us a pass: four layers, four
// chunks of 5 rows of 256 613, now 600; 30 rows of 512 205, 201; 900 rows of 1280 729, 723.
struct Embedded {
    const float *token, *position;
    __device__ __forceinline__ Embedded(const uint32_t *tokens, const float *wte, const float *wpe, int row, int new_len, int d, const int *pos_dev, int known_pos, int vocab,
                                        int n_positions) {
        const int pos = min((known_pos >= 0 ? known_pos : *pos_dev) + row % new_len, n_positions - 1);
        const uint32_t tok = min(tokens[row], (uint32_t)(vocab - 1));
        token = wte + (size_t)tok * d;
        position = wpe + (size_t)pos * d;
    }
};

// The same Linear inside a decode step, on inputs its producer has already split into bf16 pieces (layout and
// arithmetic: csrc/int4_skinny.hip).  PxIn: the pieces of x [K/32][3][64] x 16 bytes; with stats (per row and 32
// or 16 columns, `tiles` = K / 32 or K / 16 <= 64 of them) the LayerNorm in front of the Linear is applied through fold_a / fold_b.
// PxOut (all optional): the pieces of this Linear's outputs for the next one, times `gamma` where given, and their
// statistics.  Needs N % 32 == 0 to write pieces.
struct PxIn {
    const uint4 *pieces;
    const float2 *stats;
    int tiles;
    const float *fold_a, *fold_b;
};
struct PxOut {
    uint4 *pieces;
    const float *gamma;
    float2 *stats;
    int half;  // the statistics are of 16 columns, not 32
};
// the leading 16 bits of two floats as one register: a in the low half
__device__ __forceinline__ uint32_t sk_pack_top(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}
__device__ __forceinline__ float sk_top_bits(float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); }
// 8 consecutive k (from k0, a multiple of 8) of row `row` -> the lane's 16 bytes of the three piece planes of its trip:
// x = hi + mid + lo exactly, each piece the leading 8 bits of what the ones before it left; k order (0,4,1,5,2,6,3,7).
__device__ __forceinline__ void px_store_pieces(uint4 *pieces, int k0, int row, const float (&v)[8]) {
    float r1[8], r2[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        r1[e] = v[e] - sk_top_bits(v[e]);
        r2[e] = r1[e] - sk_top_bits(r1[e]);
    }
    uint4 *dst = pieces + (size_t)(k0 >> 5) * 192 + 16 * ((k0 & 31) >> 3) + row;
    dst[0] = make_uint4(sk_pack_top(r2[0], r2[4]), sk_pack_top(r2[1], r2[5]), sk_pack_top(r2[2], r2[6]), sk_pack_top(r2[3], r2[7]));
    dst[64] = make_uint4(sk_pack_top(r1[0], r1[4]), sk_pack_top(r1[1], r1[5]), sk_pack_top(r1[2], r1[6]), sk_pack_top(r1[3], r1[7]));
    dst[128] = make_uint4(sk_pack_top(v[0], v[4]), sk_pack_top(v[1], v[5]), sk_pack_top(v[2], v[6]), sk_pack_top(v[3], v[7]));
}
bool agpu_int4_skinny_px_supported(const GemvArgs &a, const PxIn &in, const PxOut &out);
int32_t agpu_int4_skinny_px_launch(agpu_ctx *ctx, const GemvArgs &a, const PxIn &in, const PxOut &out);
// fp32 rows [M <= 16, K] -> pieces (+ statistics), for values the Linear kernels do not produce themselves.
int32_t agpu_px_split_rows_launch(agpu_ctx *ctx, const float *x, int M, int K, const PxOut &out);
// The embedding rows of a step's tokens (one a sequence) -> x, and out as px_split_rows leaves it.
int32_t agpu_px_embed_launch(agpu_ctx *ctx, const uint32_t *tokens, const float *wte, const float *wpe, float *x, int M, int K, int *pos_dev, int known_pos,
                             int vocab, int n_positions, const PxOut &out);
// A_n = sum_k gamma_k W_kn and B_n = sum_k beta_k W_kn (+ bias_n where given) of an int4 Linear [K, N], rows `stride` apart.
int32_t agpu_px_fold_launch(agpu_ctx *ctx, const uint32_t *packed, const float *scales, int K, int N, int stride, int group, const float *gamma,
                            const float *beta, const float *bias, float *A, float *B);
// Whether the GEMV can apply LayerNorm itself for this shape (otherwise normalise first).
bool agpu_int4_gemv_can_fuse_ln(int M, int K);

// Dense fp32 GEMV, C[M,N] = A[M,K] B[K,N], M <= 16.
int32_t agpu_f32_gemv_launch(agpu_ctx *ctx, const float *a, const float *b, float *c, int M, int N, int K);
// The same for one row, with the arg-max over its N outputs and the token feed in the launch.
int32_t agpu_f32_gemv_argmax_launch(agpu_ctx *ctx, const float *a, const float *b, float *c, int N, int K, uint32_t *idx_out, int last,
                                    const ArgmaxAdvance &adv);
// The same two on a matrix stored row by row, w [N, K] (M <= 16, K a multiple of four, 256 to 2048, a and w on 16 bytes).
bool agpu_f32_gemv_rows_supported(const float *a, const float *w, int M, int N, int K);
int32_t agpu_f32_gemv_rows_launch(agpu_ctx *ctx, const float *a, const float *w, float *y, int M, int N, int K);
int32_t agpu_f32_gemv_rows_argmax_launch(agpu_ctx *ctx, const float *a, const float *w, float *y, int M, int N, int K, uint32_t *idx_out, int last, const ArgmaxAdvance &adv);
