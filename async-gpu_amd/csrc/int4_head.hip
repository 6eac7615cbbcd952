// The int4 LM head of two to sixteen rows (sequences of a decode step, the last rows of prompts): the final LayerNorm in front and the arg-max and the token feed
// of all rows behind it in one launch.
//
// Such a launch streams the matrix (32 MB at 50257 x 1024) past a few rows.  One workgroup a CU turns the rows into operands in LDS once, as three exact
// bf16 pieces an element (8 bits of the mantissa each); its sixteen waves then take tiles of 16 columns over all of K, each for itself: the words of eight
// scale groups on their way while one is worked on, no sums that meet between waves, no barrier.  Nibbles become bf16 numbers, products are exact, the pieces
// of a group's sum are added smallest first, then acc += scale * sum in fp32, every fourth group in a sum of its own (one chain over 50 groups: errors against
// float64 1.2e-7 of the logits in rms at 8 x 1600, four 0.8e-7; the kernels that this one has taken over from 0.9e-7).  The rows of v_mfma_f32_16x16x32_bf16 are
// (sequence, piece) for up to four sequences a set, so that a word costs one matrix instruction a set; for more than eight they are the sequences, and a word
// costs three, chained.
//
// What bounds it, us by its parts at 3 x 1024: nothing but a launch 4.6, rows staged 1, tiles 5 (6.4 TB/s), arg-max over workgroups and feed 5 (store,
// ticket, load: each a round trip through memory); 16.1 in all, in place of 21.4 + 8.2 + 4.7 of three launches (head, arg-max, counters).  At 2 x 768 13.5, 2 x
// 1600 20.3, 8 x 1024 18, 16 x 1600 27.  Tiles of 32 columns for eight waves: 17.5 at 3 x 1024 (a CU's 6 tiles leave waves idle); 16 groups ahead: no gain.
// ms per decode step before and after: 12 layers x 768, 2 sequences 0.1618 and 0.1570; 24 x 1024, 3 sequences 0.4446 and 0.4296, 8 sequences 0.780 and 0.766;
// 48 x 1600, 2 sequences 1.390 and 1.388, 16 sequences 2.014 and 2.009.
#include "int4_head.h"
#include "int4_head_layout.h"

#include <atomic>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int W = 16;           // waves of a workgroup
constexpr int CHAINS = 4;       // sums of a result: every fourth group's
constexpr int HR_MAX_K = 2048;  // a lane's share of a row in registers
constexpr float HR_UNIT = 16.0f;  // what nibbles_in_order divides by

struct HeadRowsParams {
    const float *x, *gamma, *beta;  // [rows][K]; gamma null: normalised already
    float eps;
    const uint32_t *packed;
    const float *scales;
    float *y;
    int rows, N, K, chunk_shift;
    int cols;  // the arg-max looks at
    HeadFeed feed;
};

__device__ __forceinline__ uint32_t top_halves(float a, float b) { return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u); }
__device__ __forceinline__ float top_half(float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); }

// Eight nibbles -> the bf16 numbers (n - 8) / 16 in their order: with its top bit flipped a nibble is the signed number n - 8.
#define AGPU_CVT_I4(dst, src, byte) \
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_" #byte : "=v"(dst) : "v"(src))
__device__ __forceinline__ bf16x8 nibbles_in_order(uint32_t w) {
    const uint32_t even = w ^ 0x88888888u, odd = even >> 4;
    float f[8];
    AGPU_CVT_I4(f[0], even, 0);
    AGPU_CVT_I4(f[1], odd, 0);
    AGPU_CVT_I4(f[2], even, 1);
    AGPU_CVT_I4(f[3], odd, 1);
    AGPU_CVT_I4(f[4], even, 2);
    AGPU_CVT_I4(f[5], odd, 2);
    AGPU_CVT_I4(f[6], even, 3);
    AGPU_CVT_I4(f[7], odd, 3);
    return __builtin_bit_cast(bf16x8, make_uint4(top_halves(f[0], f[1]), top_halves(f[2], f[3]), top_halves(f[4], f[5]), top_halves(f[6], f[7])));
}
#undef AGPU_CVT_I4

template <int SETS, bool LN>
__global__ __launch_bounds__(64 * W) void int4_head_rows_kernel(const HeadRowsParams p) {
    extern __shared__ __align__(16) unsigned char hr_smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, kq = lane >> 4;
    const int groups = p.K >> 5, batches = hr_batches(groups);
    const int tiles = p.N / 16, tile_end = (int)((long long)(blockIdx.x + 1) * tiles / gridDim.x);
    int tile = (int)((long long)blockIdx.x * tiles / gridDim.x) + wave;
    const uint32_t row_bytes = (uint32_t)p.N * 4u;

    // ---- words and scales of a tile's groups: one stream through the wave's tiles, every place of the ring refilled as soon as it has been worked on; always a
    // request, so that the wait for a place is counted by what stands behind it.  Groups beyond K's last one repeat it (they are not added), behind the last
    // tile its first groups come once more. ----
    const auto words = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(p.packed), 0, (uint32_t)(p.K >> 3) * row_bytes, 0x00020000);
    const auto factors = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.scales), 0, (uint32_t)(((groups - 1) >> p.chunk_shift) + 1) * row_bytes, 0x00020000);
    uint32_t w[HR_AHEAD];
    float sc[HR_AHEAD];
    const uint32_t lane_w = (uint32_t)kq * row_bytes + 4u * c16, lane_s = 4u * c16;
    auto request = [&](uint32_t at_w, uint32_t at_s, int g, int u) {  // of a tile's columns: what a lane adds; g: uniform
        const int gc = min(g, groups - 1);
        const uint32_t row_w = (uint32_t)(4 * gc) * row_bytes, row_s = (uint32_t)(gc >> p.chunk_shift) * row_bytes;
        w[u] = __builtin_amdgcn_raw_buffer_load_b32(words, at_w, row_w, 0);
        sc[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(factors, at_s, row_s, 0));
    };
    if (tile < tile_end)
#pragma unroll
        for (int u = 0; u < HR_AHEAD; ++u) request(lane_w + 64 * tile, lane_s + 64 * tile, u, u);

    // ---- the rows: wave w stages row w, normalised as the LayerNorm kernels do it (two passes over the registers) ----
    constexpr int QUADS = HR_MAX_K / 256;
    const int quads = p.K >> 2;
    if (const int row = wave; row < p.rows) {
        float4 x[QUADS];
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < QUADS; ++i) {
            x[i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            if (lane + 64 * i < quads) x[i] = *reinterpret_cast<const float4 *>(p.x + (size_t)row * p.K + 4 * (lane + 64 * i));
            if (LN) s += (x[i].x + x[i].y) + (x[i].z + x[i].w);
        }
        if constexpr (LN) {
            const float mean = wave_sum(s) / (float)p.K;
            float q = 0.0f;
#pragma unroll
            for (int i = 0; i < QUADS; ++i)
                if (lane + 64 * i < quads) {
                    const float d0 = x[i].x - mean, d1 = x[i].y - mean, d2 = x[i].z - mean, d3 = x[i].w - mean;
                    q += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
                }
            const float rstd = inverse_sqrt(quotient(wave_sum(q), (float)p.K) + p.eps);
#pragma unroll
            for (int i = 0; i < QUADS; ++i)
                if (lane + 64 * i < quads) {
                    const float4 g = *reinterpret_cast<const float4 *>(p.gamma + 4 * (lane + 64 * i)), b = *reinterpret_cast<const float4 *>(p.beta + 4 * (lane + 64 * i));
                    x[i].x = (x[i].x - mean) * rstd * g.x + b.x;
                    x[i].y = (x[i].y - mean) * rstd * g.y + b.y;
                    x[i].z = (x[i].z - mean) * rstd * g.z + b.z;
                    x[i].w = (x[i].w - mean) * rstd * g.w + b.w;
                }
        }
#pragma unroll
        for (int i = 0; i < QUADS; ++i) {
            const int quad = lane + 64 * i;
            if (quad >= quads) continue;
            const float v[4] = {x[i].x, x[i].y, x[i].z, x[i].w};
            float r1[4], r2[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {  // exact: what the leading 8 bits leave, and what the next 8 leave of that
                r1[e] = v[e] - top_half(v[e]);
                r2[e] = r1[e] - top_half(r1[e]);
            }
            unsigned char *dst = hr_smem + 8 * (quad & 1);
            *reinterpret_cast<uint2 *>(dst + hr_piece_at<SETS>(groups, quad >> 1, row, 0)) = make_uint2(top_halves(r2[0], r2[1]), top_halves(r2[2], r2[3]));
            *reinterpret_cast<uint2 *>(dst + hr_piece_at<SETS>(groups, quad >> 1, row, 1)) = make_uint2(top_halves(r1[0], r1[1]), top_halves(r1[2], r1[3]));
            *reinterpret_cast<uint2 *>(dst + hr_piece_at<SETS>(groups, quad >> 1, row, 2)) = make_uint2(top_halves(v[0], v[1]), top_halves(v[2], v[3]));
        }
    }
    __syncthreads();

    // ---- tiles ----
    constexpr int S = SETS > 0 ? SETS : 1, PIECES = SETS > 0 ? 1 : 3, OUT = SETS > 0 ? 1 : 4;  // OUT: results of a lane per set and column
    const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    unsigned long long best[S * OUT];
#pragma unroll
    for (int i = 0; i < S * OUT; ++i) best[i] = 0ull;
    float acc[CHAINS][S][OUT];
    bf16x8 a[2][S][PIECES];
    auto rows_of = [&](int g, int u, bf16x8 (&to)[S][PIECES]) {  // group g + u, g a multiple of HR_AHEAD
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < PIECES; ++i)
                to[s][i] = *reinterpret_cast<const bf16x8 *>(hr_smem + hr_operand_at<SETS>(groups, g, u, s, i, kq, c16));
    };
    floatx4 d[S];
    auto multiply = [&](int u) {
        const bf16x8 n = nibbles_in_order(w[u]);
#pragma unroll
        for (int s = 0; s < S; ++s) {
            d[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u & 1][s][0], n, zero, 0, 0, 0);
#pragma unroll
            for (int i = 1; i < PIECES; ++i) d[s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u & 1][s][i], n, d[s], 0, 0, 0);
        }
    };
    auto add = [&](int u) {
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < OUT; ++i) {
                const float sum = SETS > 0 ? (d[s][0] + d[s][1]) + d[s][2] : d[s][i];
                acc[u % CHAINS][s][i] = fmaf(sc[u], sum, acc[u % CHAINS][s][i]);
            }
    };
    auto finish = [&] {
        const int n = 16 * tile + c16;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int i = 0; i < OUT; ++i) {
                const int row = SETS > 0 ? 4 * s + kq : 4 * kq + i;
                const float v = HR_UNIT * ((acc[0][s][i] + acc[1][s][i]) + (acc[2][s][i] + acc[3][s][i]));
                if (row < p.rows) {
                    p.y[(size_t)row * p.N + n] = v;
                    const unsigned long long word = n < p.cols ? argmax_word(v, n, p.feed.last) : 0ull;
                    best[s * OUT + i] = word > best[s * OUT + i] ? word : best[s * OUT + i];
                }
            }
    };
    while (tile < tile_end) {
#pragma unroll
        for (int c = 0; c < CHAINS; ++c)
#pragma unroll
            for (int s = 0; s < S; ++s)
#pragma unroll
                for (int i = 0; i < OUT; ++i) acc[c][s][i] = 0.0f;
        rows_of(0, 0, a[0]);
        for (int b = 0; b < batches; ++b) {
            const bool end = b + 1 == batches;
            const int ahead_t = end && tile + W < tile_end ? tile + W : tile, g0 = b * HR_AHEAD, ahead_g = end ? 0 : g0 + HR_AHEAD;
            const uint32_t at_w = lane_w + 64 * ahead_t, at_s = lane_s + 64 * ahead_t;
#pragma unroll
            for (int u = 0; u < HR_AHEAD; ++u) {
                if (u + 1 < HR_AHEAD) rows_of(g0, u + 1, a[(u + 1) & 1]);
                else rows_of(ahead_g, 0, a[0]);
                if (g0 + u < groups) {
                    multiply(u);
                    add(u);
                }
                request(at_w, at_s, ahead_g + u, u);
                __builtin_amdgcn_sched_barrier(0);  // or all of a batch's words are waited for at once, and asked for at once
            }
        }
        finish();
        tile += W;
    }
    if (!p.feed.idx_out) return;  // uniform
    unsigned long long (*s_best)[16] = reinterpret_cast<unsigned long long (*)[16]>(hr_smem);  // in place of the rows
    __syncthreads();

    // ---- arg-max of every row: over the lanes of a row, the waves, the workgroups; the last workgroup feeds the winners back ----
#pragma unroll
    for (int i = 0; i < S * OUT; ++i) {
        const uint32_t hi = (uint32_t)(best[i] >> 32), lo = (uint32_t)best[i];
        const uint32_t mh = row16_minmax_u32<true>(hi), ml = row16_minmax_u32<true>(hi == mh ? lo : 0u);
        const int row = SETS > 0 ? 4 * i + kq : 4 * kq + i;
        if (c16 == 0) s_best[wave][row] = ((unsigned long long)mh << 32) | ml;
    }
    feed_rows(p.feed, p.rows, s_best, W, tid, 64 * W);
}

size_t rows_lds(int rows, int K) { return std::max(hr_rows_bytes(rows, K), feed_rows_lds(W, 64 * W)); }  // at least the arg-max's words

template <int SETS, bool LN>
int32_t head_go(agpu_ctx *ctx, const HeadRowsParams &p, int grid, size_t lds) {
    static std::atomic<unsigned long long> lds_raised{0};  // one bit per device
    const unsigned long long bit = 1ull << (ctx->device & 63);
    if (!(lds_raised.load(std::memory_order_relaxed) & bit)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(int4_head_rows_kernel<SETS, LN>), hipFuncAttributeMaxDynamicSharedMemorySize, kHeadRowsLds);
        if (e != hipSuccess) return agpu_hip(ctx, e, "hipFuncSetAttribute");
        lds_raised.fetch_or(bit, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL((int4_head_rows_kernel<SETS, LN>), dim3(grid), dim3(64 * W), lds, ctx->stream, p);
    return AGPU_LAUNCH_CHECK(ctx, "int4_head_rows_kernel");
}

}  // namespace

bool agpu_int4_head_rows_supported(const agpu_ctx *ctx, const float *x, int rows, int N, int K, int group) {
    return rows >= 2 && rows <= 16 && N >= 32 && N % 32 == 0 && K % 32 == 0 && K <= HR_MAX_K && group % 32 == 0 && ((group / 32) & (group / 32 - 1)) == 0 && ((uintptr_t)x & 15) == 0 &&
           rows_lds(rows, K) <= (size_t)kHeadRowsLds && (size_t)(K / 8) * N * 4 < (size_t(1) << 32) && feed_rows_fits(ctx);
}

int32_t agpu_int4_head_rows_launch(agpu_ctx *ctx, const float *x, const float *gamma, const float *beta, float eps, const uint32_t *packed, const float *scales, float *y, int rows,
                                   int N, int K, int group, int cols, uint32_t *idx_out, int last, const ArgmaxAdvance &adv) {
    HeadRowsParams p{};
    p.x = x; p.gamma = gamma; p.beta = beta; p.eps = eps;
    p.packed = packed; p.scales = scales; p.y = y;
    p.rows = rows; p.N = N; p.K = K; p.chunk_shift = __builtin_ctz((unsigned)(group / 32)); p.cols = cols;
    p.feed = feed_of(ctx, idx_out, last, adv);
    const int grid = std::min(ctx->num_cus, ceil_div(N, 32));
    const size_t lds = rows_lds(rows, K);
    switch (hr_sets(rows)) {
        case 1: return gamma ? head_go<1, true>(ctx, p, grid, lds) : head_go<1, false>(ctx, p, grid, lds);
        case 2: return gamma ? head_go<2, true>(ctx, p, grid, lds) : head_go<2, false>(ctx, p, grid, lds);
        default: return gamma ? head_go<0, true>(ctx, p, grid, lds) : head_go<0, false>(ctx, p, grid, lds);
    }
}
