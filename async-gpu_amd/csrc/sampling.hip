// Top-k sampling: the step after the logits when decoding is not greedy
// (top_k_sample, SimpleRng, generate_cached_sampling: nn/models/gpt2.rs:931-1058).
//
// The reference downloads the whole logit row and sorts it on the CPU.  Here the device picks the k
// candidates, the host gets k (index, value) pairs and does the k-element softmax and the draw with the
// reference's own arithmetic, so for the same logits the sampled token is the same.
//
// top_k_rows_kernel, one workgroup of 1024 threads per row (n <= 65536):
//   scaled = logit / max(temperature, 1e-8); key = order-preserving uint32 of scaled (NaN lowest).
//   1. Every thread takes the largest key of its elements, 13 runs of four of them on their way at a time.  The k-th largest of these 1024 maxima is a
//      lower bound of the row's k-th largest key, since the maxima are elements of the row; its upper 20 bits are built bit by bit by the first wave,
//      which holds all maxima, without a barrier.
//   2. Only threads whose maximum reaches the bound have elements that do, for k well below 1024 and values in no particular order hardly
//      more than k of them: their elements are read again by all threads, and what reaches the bound is gathered in LDS.
//   3. The k largest of the gathered ones are put in order (key descending, index ascending: the reference's sort is
//      stable) by counting, for each, how many come before it.
//   Where more than 1024 elements reach the bound (k close to 1024, or many large values in one thread's share), counting
//   rounds over the gathered elements, or over the row where LDS cannot hold them, find the exact k-th largest key and
//   how many of its equals are needed first.  All counts are exact, so the result is the same every run.
// What bounds it: a read of 200 KB by one CU, a chain of LDS and vector steps, and the code itself, which comes cold from memory (loops are not unrolled where they
// need not be: with the row kept in registers and 52 places that gather, 25 us).  50257 logits, k = 40: 12.4 us a launch; 18.9 with a
// barrier a bit for the bound and all of the row read twice.
#include "agpu_internal.h"

#include <cmath>
#include <cstring>
#include <vector>

namespace {

constexpr int TK_THREADS = 1024, TK_WAVES = TK_THREADS / 64, TK_MAX_N = 65536, TK_MAX_K = 1024;
constexpr int TK_CAND = 8192;  // gathered elements LDS has room for (64 KB)
constexpr int TK_UNROLL = 16;  // elements of the row a thread has on their way at a time, where it is read again
constexpr int TK_RUNS = 13;     // runs of four elements a thread has on their way at a time

__device__ __forceinline__ uint32_t order_key(float x) {
    if (x != x) return 0u;
    const uint32_t u = x == 0.0f ? 0u : __float_as_uint(x);  // -0.0 and 0.0 are one value
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

__device__ __forceinline__ float key_value(uint32_t key) {
    return __uint_as_float((key & 0x80000000u) ? (key & 0x7fffffffu) : ~key);
}

// Sum of one wave-uniform count per wave over the workgroup; buffers alternate so one barrier per call is enough.
__device__ __forceinline__ int block_count(int wave_count, int (*scratch)[TK_WAVES], int &phase, int lane, int wave) {
    if (lane == 0) scratch[phase][wave] = wave_count;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int w = 0; w < TK_WAVES; ++w) t += scratch[phase][w];
    phase ^= 1;
    return t;
}

// ALIGNED: rows begin at 16 bytes.
template <bool ALIGNED>
__global__ __launch_bounds__(TK_THREADS) void top_k_rows_kernel(const float *logits, int n, int stride, int k, float temperature,
                                                                uint32_t *idx_out, float *val_out) {
    // composites (key << 32 | ~index): unique, and in descending order exactly the candidates' order
    __shared__ unsigned long long s_cand[TK_CAND];
    __shared__ unsigned long long s_sel[TK_MAX_K];
    __shared__ __align__(16) uint32_t s_top[TK_THREADS];
    __shared__ int s_hot[TK_THREADS];
    __shared__ int s_cnt[2][TK_WAVES];
    __shared__ int s_fill, s_hots;
    __shared__ uint32_t s_bound;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const float *row = logits + (size_t)blockIdx.x * stride;
    const float temp = temperature < 1e-8f ? 1e-8f : temperature;
    if (tid == 0) s_fill = s_hots = 0;

    // visit(i, logit) for every element of the row, whole waves at a time (an index beyond n comes with the last logit)
    auto for_row = [&](auto &&visit) {
        for (int i0 = 0; i0 < n; i0 += TK_UNROLL * TK_THREADS) {
            float v[TK_UNROLL];
#pragma unroll
            for (int u = 0; u < TK_UNROLL; ++u) v[u] = row[min(i0 + u * TK_THREADS + tid, n - 1)];
#pragma unroll
            for (int u = 0; u < TK_UNROLL; ++u) visit(i0 + u * TK_THREADS + tid, v[u]);
        }
    };
    auto scaled_key = [&](float logit) { return order_key(logit / temp); };
    auto composite = [](uint32_t key, int i) { return ((unsigned long long)key << 32) | (0xffffffffu - (uint32_t)i); };
    // what `take` says of (i, key) for the lanes of a wave goes to consecutive places of dst; beyond cap it is only counted
    auto gather = [&](bool take, unsigned long long c, unsigned long long *dst, int cap) {
        const unsigned long long who = __ballot(take);
        if (who == 0ull) return;  // wave-uniform
        int base = 0;
        if (lane == 0) base = atomicAdd(&s_fill, __popcll(who));
        base = __builtin_amdgcn_readfirstlane(base);
        const int at = base + __popcll(who & ((1ull << lane) - 1ull));
        if (take && at < cap) dst[at] = c;
    };

    // dividing by a positive number keeps the order, so the largest logit has the largest key: one division per thread
    const int runs = (n + 4 * TK_THREADS - 1) / (4 * TK_THREADS);  // run t of a thread: elements 4 (1024 t + tid) ..
    float top = __builtin_nanf("");  // fmaxf takes the number of a number and a NaN
#pragma unroll 1
    for (int t0 = 0; t0 < runs; t0 += TK_RUNS) {
        float v[TK_RUNS][4];
#pragma unroll
        for (int t = 0; t < TK_RUNS; ++t) {
            const int i = 4 * ((t0 + t) * TK_THREADS + tid);
            if (ALIGNED) {
                const float4 x = *reinterpret_cast<const float4 *>(row + min(i, (n - 1) & ~3));
                v[t][0] = x.x; v[t][1] = x.y; v[t][2] = x.z; v[t][3] = x.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) v[t][e] = row[min(i + e, n - 1)];
            }
        }
#pragma unroll
        for (int t = 0; t < TK_RUNS; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) top = 4 * ((t0 + t) * TK_THREADS + tid) + e < n ? fmaxf(top, v[t][e]) : top;
    }
    const uint32_t my_top = scaled_key(top);
    s_top[tid] = my_top;
    __syncthreads();
    // The upper 20 bits of the k-th largest maximum (at least k threads have an element, or all of the row's have), by the first wave, from the first bit on that
    // not all maxima share.
    if (wave == 0) {
        uint32_t mine[TK_WAVES], most = 0u, least = 0xffffffffu;
#pragma unroll
        for (int i = 0; i < TK_WAVES / 4; ++i) {
            const uint4 q = *reinterpret_cast<const uint4 *>(s_top + 4 * (64 * i + lane));
            mine[4 * i] = q.x; mine[4 * i + 1] = q.y; mine[4 * i + 2] = q.z; mine[4 * i + 3] = q.w;
        }
#pragma unroll
        for (int i = 0; i < TK_WAVES; ++i) {
            most = max(most, mine[i]);
            least = min(least, mine[i]);
        }
        most = wave_minmax_u32<true>(most);
        least = wave_minmax_u32<false>(least);
        const int first = 31 - __builtin_clz((most ^ least) | 1u);
        uint32_t b = first >= 31 ? 0u : most & ~((2u << first) - 1u);
#pragma unroll 1
        for (int bit = first; bit >= 12; --bit) {
            const uint32_t cand = b | (1u << bit);
            int c = 0;
#pragma unroll
            for (int i = 0; i < TK_WAVES; ++i) c += __popcll(__ballot(mine[i] >= cand));
            if (c >= k) b = cand;
        }
        if (lane == 0) s_bound = b & 0xfffff000u;
    }
    __syncthreads();
    const uint32_t bound = s_bound;
    int phase = 0;
    // Logits that cannot reach the bound are told apart without a division: a hair below bound * temp (the division and
    // this product round by 2^-24 each); where the product or the bound is no ordinary number every element is divided.
    const float edge = key_value(bound) * temp;
    const float floor_logit = fabsf(edge) < 1e30f && fabsf(edge) > 1e-30f && fabsf(key_value(bound)) < 1e30f ? edge - fabsf(edge) * 1e-6f : -__builtin_inff();
    // Only threads whose largest element reaches the bound have any that do, hardly more than k of them: all threads read theirs again.
    if (my_top >= bound) s_hot[atomicAdd(&s_hots, 1)] = tid;  // (in any order: the places of the candidates are found by counting)
    __syncthreads();
    const int items = s_hots * 64;
#pragma unroll 1
    for (int item = tid; item < items; item += TK_THREADS) {  // whole waves: a wave is a thread's runs, at most sixteen
        const int i = 4 * ((lane >> 2) * TK_THREADS + s_hot[item >> 6]) + (lane & 3);
        const float x = row[min(i, n - 1)];
        const bool maybe = i < n && !(x < floor_logit);
        if (__ballot(maybe) == 0ull) continue;  // wave-uniform
        const uint32_t key = scaled_key(x);
        gather(maybe && key >= bound, composite(key, i), s_cand, TK_CAND);
    }
    __syncthreads();
    int count = s_fill;
    const unsigned long long *sel = s_cand;
    if (count > TK_MAX_K) {  // workgroup-uniform
        const bool in_lds = count <= TK_CAND;
        auto for_all = [&](auto &&visit) {  // (i, key) of everything that reaches the bound, whole waves at a time
            if (in_lds) {
                for (int c0 = 0; c0 < count; c0 += TK_THREADS) {
                    const bool have = c0 + tid < count;
                    const unsigned long long c = have ? s_cand[c0 + tid] : 0ull;
                    visit(have ? (int)(0xffffffffu - (uint32_t)c) : n, (uint32_t)(c >> 32));
                }
            } else {
                for_row([&](int i, float x) { visit(i, scaled_key(x)); });
            }
        };
        auto count_all = [&](auto &&pred) {
            int c = 0;
            for_all([&](int i, uint32_t key) { c += __popcll(__ballot(i < n && pred(i, key))); });
            return block_count(c, s_cnt, phase, lane, wave);
        };
        // the k-th largest key, from the top bit down: T = max { t : #(key >= t) >= k }
        uint32_t T = 0u;
        for (int bit = 31; bit >= 0; --bit) {
            const uint32_t cand = T | (1u << bit);
            if (count_all([&](int, uint32_t key) { return key >= cand; }) >= k) T = cand;
        }
        const int need = k - count_all([&](int, uint32_t key) { return key > T; });  // >= 1 elements equal to T, lowest indices first
        // J = index of the need-th element equal to T: the largest J with #(key == T, index < J) < need
        int J = 0;
        for (int bit = 16; bit >= 0; --bit) {
            const int cand = J | (1 << bit);
            if (count_all([&](int i, uint32_t key) { return key == T && i < cand; }) < need) J = cand;
        }
        if (tid == 0) s_fill = 0;  // the last count's barrier lies behind every read of it
        __syncthreads();
        // exactly k elements qualify
        for_all([&](int i, uint32_t key) { gather(i < n && (key > T || (key == T && i <= J)), composite(key, i), s_sel, TK_MAX_K); });
        __syncthreads();
        count = k;
        sel = s_sel;
    }
    // the place of an element is the number of elements before it
    if (tid < count) {
        const unsigned long long mine = sel[tid];
        int before = 0;
        for (int c = 0; c < count; ++c) before += sel[c] > mine ? 1 : 0;
        if (before < k) {
            idx_out[(size_t)blockIdx.x * k + before] = 0xffffffffu - (uint32_t)mine;
            val_out[(size_t)blockIdx.x * k + before] = key_value((uint32_t)(mine >> 32));
        }
    }
}

}  // namespace

int32_t agpu_top_k_launch(agpu_ctx *ctx, const float *logits, int rows, int n, int stride, int k, float temperature,
                          uint32_t *idx_out, float *val_out) {
    if (rows <= 0 || n <= 0 || k <= 0 || stride < n)
        return agpu_fail(ctx, AGPU_ERR_SHAPE_MISMATCH, "top_k: bad dims rows=%d n=%d k=%d stride=%d", rows, n, k, stride);
    if (n > TK_MAX_N) return agpu_fail(ctx, AGPU_ERR_UNSUPPORTED, "top_k: n = %d exceeds %d", n, TK_MAX_N);
    if (k > n) k = n;
    if (k > TK_MAX_K) return agpu_fail(ctx, AGPU_ERR_UNSUPPORTED, "top_k: k = %d exceeds %d", k, TK_MAX_K);
    const bool aligned = (uintptr_t)logits % 16 == 0 && stride % 4 == 0;  // (a run may reach beyond n, not beyond the row)
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(rows), dim3(TK_THREADS), 0, ctx->stream, logits, n, stride, k, temperature, idx_out, val_out); };
    aligned ? go(top_k_rows_kernel<true>) : go(top_k_rows_kernel<false>);
    return AGPU_LAUNCH_CHECK(ctx, "top_k_rows_kernel");
}

AGPU_EXPORT int32_t agpu_top_k(agpu_ctx *ctx, const float *logits, int32_t rows, int32_t n, int32_t k, float temperature,
                               uint32_t *idx_out, float *val_out) {
    AGPU_REQUIRE_CTX(ctx);
    if (!logits || !idx_out || !val_out) return agpu_fail(ctx, AGPU_ERR_NULL_POINTER, "top_k: null pointer");
    return agpu_top_k_launch(ctx, logits, rows, n, n, k, temperature, idx_out, val_out);
}

AGPU_EXPORT uint64_t agpu_simple_rng_new(uint64_t seed) { return seed == 0 ? 0xDEADBEEFCAFE1234ull : seed; }

AGPU_EXPORT float agpu_simple_rng_next_f32(uint64_t *state) {
    uint64_t x = *state;
    x ^= x << 13;
    x ^= x >> 7;
    x ^= x << 17;
    *state = x;
    return (float)(x >> 40) / (float)(1ull << 24);
}

AGPU_EXPORT uint32_t agpu_top_k_draw_host(const float *ranked_vals, const uint32_t *ranked_idx, int32_t k, float r) {
    if (!ranked_vals || !ranked_idx || k <= 0) return 0;
    std::vector<float> e((size_t)k);
    float sum = 0.0f;
    for (int j = 0; j < k; ++j) {
        e[j] = std::exp(ranked_vals[j] - ranked_vals[0]);
        sum += e[j];
    }
    float cum = 0.0f;
    for (int j = 0; j < k; ++j) {
        cum += e[j] / sum;
        if (r < cum) return ranked_idx[j];
    }
    return ranked_idx[k - 1];
}

AGPU_EXPORT int32_t agpu_top_k_sample(agpu_ctx *ctx, const float *logits, int32_t n, int32_t k, float temperature,
                                      uint64_t *rng_state, uint32_t *token_out_host) {
    AGPU_REQUIRE_CTX(ctx);
    if (!logits || !rng_state || !token_out_host) return agpu_fail(ctx, AGPU_ERR_NULL_POINTER, "top_k_sample: null pointer");
    if (k > n) k = n;
    if (k <= 0 || k > TK_MAX_K) return agpu_fail(ctx, AGPU_ERR_UNSUPPORTED, "top_k_sample: k = %d outside 1..%d", k, TK_MAX_K);
    // indices, then values right behind them: one copy brings both
    uint32_t *idx_dev = reinterpret_cast<uint32_t *>(ctx->workspace + ctx->ws_bytes - 2 * TK_MAX_K * 4);
    float *val_dev = reinterpret_cast<float *>(idx_dev + k);
    int32_t rc = agpu_top_k_launch(ctx, logits, 1, n, n, k, temperature, idx_dev, val_dev);
    if (rc != AGPU_OK) return rc;
    uint32_t pairs[2 * TK_MAX_K];
    if ((rc = agpu_memcpy_d2h(ctx, pairs, idx_dev, (size_t)k * 8)) != AGPU_OK) return rc;
    const uint32_t *idx = pairs;
    float val[TK_MAX_K];
    std::memcpy(val, pairs + k, (size_t)k * 4);
    *token_out_host = agpu_top_k_draw_host(val, idx, k, agpu_simple_rng_next_f32(rng_state));
    return AGPU_OK;
}
