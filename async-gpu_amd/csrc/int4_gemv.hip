// Decode GEMV of the int4 weight-only Linear, M <= 16 rows, for gfx950.
//
// grid (col_blocks, ksplit).  A workgroup owns 16*CPL adjacent columns (64 with CPL = 4) and one
// contiguous slice of K.  Inside a wave the 64 lanes form 4 row slots x 16 column groups: one
// load instruction fetches 4 consecutive packed rows, 4*CPL bytes per lane, i.e. four contiguous
// 64*CPL-byte pieces of the reference layout [K/8, N] (no repacking).  The W waves of the
// workgroup interleave over the rows, so one trip of the workgroup reads 4*W consecutive rows.
//
// The code is deliberately a short loop: the instruction cache starts cold at every launch and
// straight-line code costs about 0.4 us per KiB to fetch, which for decode-sized launches is
// more than the memory traffic.  Memory-level parallelism comes from the waves (up to 16 per
// workgroup, two row groups in flight each), not from unrolling.
//
// x (the workgroup's K slice; the whole row first when LayerNorm is fused) is staged in LDS once
// by all threads, with the sum of every 8 values.  Per packed row a lane computes
// s = sum_k x[k]*nibble[k] - 8*sum_k x[k] with the nibble as an unsigned float
// (v_cvt_f32_ubyteN on the masked word) and accumulates scale * s.
//
// Reductions are in a fixed order, so results are bit-identical from run to run: row slots by
// two lane exchanges, waves through LDS in wave order; with ksplit > 1 every workgroup publishes
// its partial sums and the last one to arrive (a ticket counter) adds them in split order and
// applies the epilogue.  Publishing uses agent-scope relaxed atomic stores and loads, which
// write through and read past the per-XCD L2, plus a wait for outstanding memory operations
// before the ticket; a full agent-scope fence would write back the whole L2 once per
// workgroup, which on this part costs more than the GEMV itself.
#include "linear_common.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

struct GemvParams {
    GemvArgs a;
    int strict;          // the context's strict_sync
    int rows_per_split;  // packed rows per workgroup (grid.y slices of K)
    int col_blocks;      // column tiles of 16*CPL columns; a workgroup strides over them
    float *partial;      // [ksplit, M, N], only with ksplit > 1
    unsigned int *counters;  // [col_blocks] tickets, zero on entry and on exit
};

template <int CPL>
struct WordVec;
template <>
struct WordVec<1> {
    using U = uint32_t;
    using F = float;
};
template <>
struct WordVec<4> {
    using U = uint4;
    using F = float4;
};

template <int CPL>
__device__ __forceinline__ void load_words(const uint32_t *p, uint32_t (&w)[CPL]) {
    using U = typename WordVec<CPL>::U;
    const U v = *reinterpret_cast<const U *>(p);
    if constexpr (CPL == 1) w[0] = v;
    if constexpr (CPL == 4) { w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w; }
}

template <int CPL>
__device__ __forceinline__ void load_floats(const float *p, float (&f)[CPL]) {
    using F = typename WordVec<CPL>::F;
    const F v = *reinterpret_cast<const F *>(p);
    if constexpr (CPL == 1) f[0] = v;
    if constexpr (CPL == 4) { f[0] = v.x; f[1] = v.y; f[2] = v.z; f[3] = v.w; }
}

// Sum over the workgroup, result in every thread.  scratch: 16 floats of LDS.
__device__ __forceinline__ float block_sum(float v, float *scratch, int lane, int wave, int W) {
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) scratch[wave] = v;
    __syncthreads();
    float t = 0.0f;
    for (int w = 0; w < W; ++w) t += scratch[w];
    return t;
}

// LDS layout (floats): xs[MT][xs_len] | xsum[MT][rows_per_split] | red[W][MT][COLS].
// xs_len = K when LayerNorm is fused (whole rows), else the K slice.
// A workgroup handles the column tiles blockIdx.x, blockIdx.x + gridDim.x, ...: x is staged once
// and the loads of the next tile's first two row trips are issued before the current tile is reduced.
template <int MT, int CPL, bool LN>
__global__ __launch_bounds__(MT == 1 ? 1024 : 512) void int4_gemv_kernel(const GemvParams p) {
    extern __shared__ __align__(16) float smem[];
    __shared__ float s_scratch[16];
    __shared__ int s_last;
    const GemvArgs &a = p.a;
    constexpr int COLS = 16 * CPL;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = blockDim.x >> 6, T = blockDim.x;
    const int rs = lane >> 4, cg = lane & 15;
    const int ksplit = gridDim.y, split = blockIdx.y;
    const int kp_total = a.K / 8;
    const int r0 = split * p.rows_per_split;
    const int r1 = min(kp_total, r0 + p.rows_per_split);
    const int k0 = r0 * 8, kslice = (r1 - r0) * 8;
    const int xs_len = LN ? a.K : p.rows_per_split * 8;
    float *xs = smem;
    float *xsum = smem + MT * xs_len;
    float *red = xsum + MT * p.rows_per_split;  // [W][MT][COLS]
    const int n_out = MT * COLS;
    const int row_a = r0 + 4 * wave + rs, row_b = row_a + 4 * W;

    // the first two row trips of a tile, for this lane
    uint32_t wa[CPL], wb[CPL];
    float sa[CPL], sb[CPL];
    auto preload = [&](int tile) {
        const int c0 = tile * COLS + cg * CPL;
        const bool ok = tile < p.col_blocks && c0 < a.N;  // N % CPL == 0 is guaranteed by the launcher
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            wa[c] = wb[c] = 0x88888888u;
            sa[c] = sb[c] = 0.0f;
        }
        if (ok && row_a < r1) {
            load_words<CPL>(a.packed + (size_t)row_a * a.N + c0, wa);
            load_floats<CPL>(a.scales + (size_t)((row_a * 8) / a.group) * a.N + c0, sa);
        }
        if (ok && row_b < r1) {
            load_words<CPL>(a.packed + (size_t)row_b * a.N + c0, wb);
            load_floats<CPL>(a.scales + (size_t)((row_b * 8) / a.group) * a.N + c0, sb);
        }
    };
    preload(blockIdx.x);  // these loads go out before anything else

    // ---- stage x once ----
    if constexpr (LN) {
        // whole rows into LDS, two-pass statistics over the workgroup, normalise the slice in place
        for (int i = tid; i < MT * a.K; i += T) {
            const int m = i / a.K, k = i - m * a.K;
            xs[i] = (m < a.M) ? a.x[(size_t)m * a.K + k] : 0.0f;
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float s = 0.0f;
            for (int k = tid; k < a.K; k += T) s += xs[m * a.K + k];
            const float mean = block_sum(s, s_scratch, lane, wave, W) / (float)a.K;
            float v = 0.0f;
            for (int k = tid; k < a.K; k += T) {
                const float d = xs[m * a.K + k] - mean;
                v += d * d;
            }
            const float rstd = 1.0f / sqrtf(block_sum(v, s_scratch, lane, wave, W) / (float)a.K + a.ln_eps);
            for (int kk = tid; kk < kslice; kk += T) {
                const int k = k0 + kk;
                xs[m * a.K + k] = (xs[m * a.K + k] - mean) * rstd * a.ln_gamma[k] + a.ln_beta[k];
            }
        }
        __syncthreads();
    } else {
        for (int i = tid; i < MT * kslice; i += T) {
            const int m = i / kslice, kk = i - m * kslice;
            xs[m * xs_len + kk] = (m < a.M) ? a.x[(size_t)m * a.K + k0 + kk] : 0.0f;
        }
        __syncthreads();
    }
    const float *xbase = LN ? xs + k0 : xs;  // xbase[m*xs_len + 8*(row - r0) + j]
    for (int i = tid; i < MT * (r1 - r0); i += T) {
        const int m = i / (r1 - r0), r = i - m * (r1 - r0);
        const float4 xa = *reinterpret_cast<const float4 *>(xbase + m * xs_len + r * 8);
        const float4 xb = *reinterpret_cast<const float4 *>(xbase + m * xs_len + r * 8 + 4);
        xsum[m * p.rows_per_split + r] = 8.0f * (((xa.x + xa.y) + (xa.z + xa.w)) + ((xb.x + xb.y) + (xb.z + xb.w)));
    }
    __syncthreads();

    float acc[MT][CPL];
    auto consume = [&](const uint32_t (&w)[CPL], const float (&sc)[CPL], int row) {
        const int r = row - r0;
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float4 xa = *reinterpret_cast<const float4 *>(xbase + m * xs_len + r * 8);
            const float4 xb = *reinterpret_cast<const float4 *>(xbase + m * xs_len + r * 8 + 4);
            const float xsum8 = xsum[m * p.rows_per_split + r];
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                float nf[8];
                unpack_u8(w[c], nf);
                float s = -xsum8;
                s = fmaf(xa.x, nf[0], s);
                s = fmaf(xa.y, nf[1], s);
                s = fmaf(xa.z, nf[2], s);
                s = fmaf(xa.w, nf[3], s);
                s = fmaf(xb.x, nf[4], s);
                s = fmaf(xb.y, nf[5], s);
                s = fmaf(xb.z, nf[6], s);
                s = fmaf(xb.w, nf[7], s);
                acc[m][c] = fmaf(sc[c], s, acc[m][c]);
            }
        }
    };

    for (int tile = blockIdx.x; tile < p.col_blocks; tile += gridDim.x) {
        const int c0 = tile * COLS + cg * CPL;
        const bool col_ok = c0 < a.N;
        // epilogue operands of this thread's output element, fetched early
        float e_bias = 0.0f, e_res = 0.0f;
        {
            const int m = tid / COLS, n = tile * COLS + (tid - m * COLS);
            if (tid < n_out && m < a.M && n < a.N) {
                if (a.bias) e_bias = a.bias[n];
                if (a.residual) e_res = a.residual[(size_t)m * a.N + n];
            }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < CPL; ++c) acc[m][c] = 0.0f;
        // rows r0 + 4*wave + rs + 4*W*i; trips 0 and 1 are already in registers
        for (int row = row_a; row < r1; row += 8 * W) {
            uint32_t wn0[CPL], wn1[CPL];
            float sn0[CPL], sn1[CPL];
            const int rn0 = row + 8 * W, rn1 = row + 12 * W;
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                wn0[c] = wn1[c] = 0x88888888u;
                sn0[c] = sn1[c] = 0.0f;
            }
            if (col_ok && rn0 < r1) {
                load_words<CPL>(a.packed + (size_t)rn0 * a.N + c0, wn0);
                load_floats<CPL>(a.scales + (size_t)((rn0 * 8) / a.group) * a.N + c0, sn0);
            }
            if (col_ok && rn1 < r1) {
                load_words<CPL>(a.packed + (size_t)rn1 * a.N + c0, wn1);
                load_floats<CPL>(a.scales + (size_t)((rn1 * 8) / a.group) * a.N + c0, sn1);
            }
            consume(wa, sa, row);
            if (row + 4 * W < r1) consume(wb, sb, row + 4 * W);
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                wa[c] = wn0[c]; sa[c] = sn0[c];
                wb[c] = wn1[c]; sb[c] = sn1[c];
            }
        }
        preload(tile + gridDim.x);  // next tile's loads fly during the reduction below
        // row slots -> lanes 0..15 (fixed order), then waves through LDS
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                float v = acc[m][c];
                v += __shfl_xor(v, 16, kWave);
                v += __shfl_xor(v, 32, kWave);
                acc[m][c] = v;
            }
        __syncthreads();  // the previous tile's readers of red are done
        if (rs == 0) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
                for (int c = 0; c < CPL; ++c) red[(wave * MT + m) * COLS + cg * CPL + c] = acc[m][c];
        }
        __syncthreads();
        if (ksplit == 1) {
            for (int i = tid; i < n_out; i += T) {
                const int m = i / COLS, n = tile * COLS + (i - m * COLS);
                if (m < a.M && n < a.N) {
                    float v = 0.0f;
                    for (int w = 0; w < W; ++w) v += red[w * n_out + i];
                    if (i != tid) {
                        e_bias = a.bias ? a.bias[n] : 0.0f;
                        e_res = a.residual ? a.residual[(size_t)m * a.N + n] : 0.0f;
                    }
                    finish_output(a, v, e_bias, e_res, m, n);
                }
            }
            continue;
        }
        // publish this workgroup's partial sums past the L2, then take a ticket
        for (int i = tid; i < n_out; i += T) {
            const int m = i / COLS, n = tile * COLS + (i - m * COLS);
            if (m < a.M && n < a.N) {
                float v = 0.0f;
                for (int w = 0; w < W; ++w) v += red[w * n_out + i];
                __hip_atomic_store(&p.partial[((size_t)split * a.M + m) * a.N + n], v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        partials_published(p.strict);
        __syncthreads();
        if (tid == 0) {
            const unsigned int t = take_ticket(&p.counters[tile], p.strict);
            s_last = (t == (unsigned int)(ksplit - 1));
        }
        __syncthreads();
        if (!s_last) continue;  // uniform over the workgroup
        for (int i = tid; i < n_out; i += T) {
            const int m = i / COLS, n = tile * COLS + (i - m * COLS);
            if (m < a.M && n < a.N) {
                const float *src = p.partial + (size_t)m * a.N + n;
                const size_t stride = (size_t)a.M * a.N;
                float t = 0.0f;
                for (int sp0 = 0; sp0 < ksplit; sp0 += 8) {  // 8 loads in flight, summed in split order
                    float part[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        part[u] = sp0 + u < ksplit
                                      ? __hip_atomic_load(src + (size_t)(sp0 + u) * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
                                      : 0.0f;
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (sp0 + u < ksplit) t += part[u];
                }
                if (i != tid) {
                    e_bias = a.bias ? a.bias[n] : 0.0f;
                    e_res = a.residual ? a.residual[(size_t)m * a.N + n] : 0.0f;
                }
                finish_output(a, t, e_bias, e_res, m, n);
            }
        }
        if (tid == 0) __hip_atomic_store(&p.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// Dense fp32 GEMV: lane = column, the W waves of a workgroup split K, reduced in wave order.  A stream of K N words: what
// bounds it is how many requests are on their way, sixteen per wave here (the 50257 x 768 head, one row: 40 us with
// four, 37 now).  AM (one row): the arg-max over the outputs and the token feed as well.
constexpr int GF_AHEAD = 16;
template <int MT, bool AM>
__global__ __launch_bounds__(1024) void gemv_f32_kernel(const float *__restrict__ x, const float *__restrict__ b,
                                                         float *y, int M, int N, int K, const ArgmaxShare am) {
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = blockDim.x >> 6;
    const int n = blockIdx.x * 64 + lane;
    const int kpw = (K + W - 1) / W;
    const int ka = __builtin_amdgcn_readfirstlane(wave * kpw), kb = min(K, ka + kpw);
    float acc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m] = 0.0f;
    const float *col = b + min(n, N - 1);  // a column beyond the last repeats it and is not stored
    int k = ka;
    for (; k + GF_AHEAD <= kb; k += GF_AHEAD) {
        float w[GF_AHEAD];
#pragma unroll
        for (int u = 0; u < GF_AHEAD; ++u) w[u] = col[(size_t)(k + u) * N];
#pragma unroll
        for (int u = 0; u < GF_AHEAD; ++u)
#pragma unroll
            for (int m = 0; m < MT; ++m)
                if (m < M) acc[m] = fmaf(x[(size_t)m * K + k + u], w[u], acc[m]);
    }
    for (; k < kb; ++k) {
        const float w = col[(size_t)k * N];
#pragma unroll
        for (int m = 0; m < MT; ++m)
            if (m < M) acc[m] = fmaf(x[(size_t)m * K + k], w, acc[m]);
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) smem[(wave * MT + m) * 64 + lane] = acc[m];
    __syncthreads();
    unsigned long long best = 0ull;
    for (int i = tid; i < MT * 64; i += blockDim.x) {
        const int m = i / 64, nn = blockIdx.x * 64 + (i & 63);
        if (m < M && nn < N) {
            float v = smem[i];
            for (int w = 1; w < W; ++w) v += smem[w * MT * 64 + i];
            y[(size_t)m * N + nn] = v;
            if (AM) best = argmax_word(v, nn, am.last);
        }
    }
    if constexpr (AM) {
        __shared__ uint32_t s_scratch[32];
        __shared__ int s_last;
        argmax_finish(am, best, s_scratch, s_last, tid, W);
    }
}

// The same with the matrix stored row by row, w [N, K] (the f32 LM head on the embedding table as it is).  A wave takes R rows of w at a time, 16 bytes a
// lane and contiguous, the next R already on their way; a row of x stays in registers, several in LDS.  A stream again, of N K words: eight waves a
// CU with 12 KB requested each.  50257 x 768, one row, us per launch: 26.0 (5.9 TB/s; the kernel above 37.4), with two workgroups of eight waves a CU 26.7, four 31.8.
// Sums of R rows over the 64 lanes: halves and rows of lanes change places, so that a register holds all of them before the last four steps.
template <int R>
__device__ __forceinline__ float sum_rows(const float (&v)[R], int lane, int &which) {  // lanes 16 i ..: the sum of v[which]
    static_assert(R == 2 || R == 4, "");
    auto swap32 = [](float a, float b) {
        const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(s[0]) + __uint_as_float(s[1]);  // lower half: a's two halves, upper: b's
    };
    auto swap16 = [](float a, float b) {
        const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
        return __uint_as_float(s[0]) + __uint_as_float(s[1]);  // even rows: a's, odd: b's
    };
    const float u = swap32(v[0], v[1]);
    which = lane >> 5;
    if constexpr (R == 2) return row16_sum(swap16(u, u));
    else {
        which += 2 * ((lane >> 4) & 1);
        return row16_sum(swap16(u, swap32(v[2], v[3])));
    }
}

// AM: the arg-max and the token feed of all rows in the launch, from one row's ArgmaxShare or several's HeadFeed.
template <int MT, int ITERS, int R, bool AM>
__global__ __launch_bounds__(512) void gemv_f32_rows_kernel(const float *__restrict__ x, const float *__restrict__ w, float *y, int M, int N, int K,
                                                            const std::conditional_t<MT == 1, ArgmaxShare, HeadFeed> am) {
    extern __shared__ __align__(16) float smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), W = blockDim.x >> 6;
    const int first = (int)((long long)blockIdx.x * N / gridDim.x), end = (int)((long long)(blockIdx.x + 1) * N / gridDim.x);
    const bool tail = 4 * lane + 256 * (ITERS - 1) < K;  // K is a multiple of four, more than 256 (ITERS - 1)
    float4 h[ITERS];
    const float4 *xs = reinterpret_cast<const float4 *>(smem) + lane;  // [MT][ITERS][64]
    if constexpr (MT == 1) {
#pragma unroll
        for (int i = 0; i < ITERS; ++i) h[i] = i < ITERS - 1 || tail ? *reinterpret_cast<const float4 *>(x + 4 * lane + 256 * i) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    } else {
        for (int i = tid; i < MT * ITERS * 64; i += blockDim.x) {
            const int m = i / (ITERS * 64), k = 4 * (i - m * (ITERS * 64));
            reinterpret_cast<float4 *>(smem)[i] = m < M && k < K ? *reinterpret_cast<const float4 *>(x + (size_t)m * K + k) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    }
    float4 v[2][R][ITERS];
    auto request = [&](int row, float4 (&b)[R][ITERS]) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float *src = w + (size_t)min(row + r, N - 1) * K + 4 * lane;
#pragma unroll
            for (int i = 0; i < ITERS; ++i) {
                b[r][i] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                if (i < ITERS - 1 || tail) b[r][i] = *reinterpret_cast<const float4 *>(src + 256 * i);
            }
        }
    };
    // A lane's rows of w come in ascending order: the largest so far and its row, of equal ones the first or the last.
    float most[MT];
    int at[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        most[m] = -INFINITY;
        at[m] = 0;
    }
    auto finish = [&](int row, const float4 (&b)[R][ITERS]) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            if (MT > 1 && m >= M) break;  // uniform
            float4 s[R];
#pragma unroll
            for (int r = 0; r < R; ++r) s[r] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
            for (int i = 0; i < ITERS; ++i) {
                const float4 hi = MT == 1 ? h[i] : xs[(m * ITERS + i) * 64];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    s[r].x = fmaf(hi.x, b[r][i].x, s[r].x);
                    s[r].y = fmaf(hi.y, b[r][i].y, s[r].y);
                    s[r].z = fmaf(hi.z, b[r][i].z, s[r].z);
                    s[r].w = fmaf(hi.w, b[r][i].w, s[r].w);
                }
            }
            float t[R];
#pragma unroll
            for (int r = 0; r < R; ++r) t[r] = (s[r].x + s[r].y) + (s[r].z + s[r].w);
            int which;
            const float sum = sum_rows<R>(t, lane, which);
            const int n = row + which;
            if ((lane & (R == 2 ? 31 : 15)) == 0 && n < end) {
                y[(size_t)m * N + n] = sum;
                if (AM) {
                    const bool more = sum > most[m] || (am.last && sum == most[m]);
                    most[m] = more ? sum : most[m];
                    at[m] = more ? n : at[m];
                }
            }
        }
    };
    const int step = W * R;
    int row = first + wave * R;
    if (row < end) request(row, v[0]);
    if constexpr (MT > 1) __syncthreads();
    for (; row < end; row += 2 * step) {
        if (row + step < end) request(row + step, v[1]);
        finish(row, v[0]);
        if (row + 2 * step < end) request(row + 2 * step, v[0]);
        if (row + step < end) finish(row + step, v[1]);
    }
    if constexpr (AM) {
        const bool leads = (lane & (R == 2 ? 31 : 15)) == 0;
        auto word = [&](int m) {
            unsigned long long best = 0ull;
            if (leads && most[m] > -INFINITY) best = argmax_word(most[m], at[m], am.last);
            else if (leads && m < M)  // nothing above -infinity, or nothing at all: NaN is told from it
                for (int r = first + wave * R + (R == 2 ? lane >> 5 : (lane >> 5) + 2 * ((lane >> 4) & 1)); r < end; r += step) {
                    const unsigned long long c = argmax_word(y[(size_t)m * N + r], r, am.last);
                    best = c > best ? c : best;
                }
            return best;
        };
        if constexpr (MT == 1) {
            __shared__ uint32_t s_scratch[32];
            __shared__ int s_last;
            argmax_finish(am, word(0), s_scratch, s_last, tid, W);
        } else {
            unsigned long long (*s_best)[16] = reinterpret_cast<unsigned long long (*)[16]>(smem);  // in place of the rows
            __syncthreads();
            if ((lane & 15) == 0)
#pragma unroll
                for (int m = 0; m < MT; ++m) s_best[4 * wave + (lane >> 4)][m] = word(m);
            feed_rows(am, M, s_best, 4 * W, tid, 64 * W);
        }
    }
}

template <int MT, int CPL>
int32_t launch_t(agpu_ctx *ctx, const GemvParams &p, dim3 grid, int W, size_t lds) {
    if constexpr (MT <= 2) {
        if (p.a.ln_gamma) {
            hipLaunchKernelGGL((int4_gemv_kernel<MT, CPL, true>), grid, dim3(64 * W), lds, ctx->stream, p);
            return AGPU_LAUNCH_CHECK(ctx, "int4_gemv_kernel");
        }
    }
    hipLaunchKernelGGL((int4_gemv_kernel<MT, CPL, false>), grid, dim3(64 * W), lds, ctx->stream, p);
    return AGPU_LAUNCH_CHECK(ctx, "int4_gemv_kernel");
}

template <int CPL>
int32_t launch_m(agpu_ctx *ctx, const GemvParams &p, int MT, dim3 grid, int W, size_t lds) {
    switch (MT) {
        case 1: return launch_t<1, CPL>(ctx, p, grid, W, lds);
        case 2: return launch_t<2, CPL>(ctx, p, grid, W, lds);
        case 4: return launch_t<4, CPL>(ctx, p, grid, W, lds);
        case 8: return launch_t<8, CPL>(ctx, p, grid, W, lds);
        default: return launch_t<16, CPL>(ctx, p, grid, W, lds);
    }
}

}  // namespace

bool agpu_int4_gemv_can_fuse_ln(int M, int K) { return M <= 2 && (size_t)M * K * sizeof(float) <= 32 * 1024; }

AGPU_EXPORT int32_t agpu_int4_gemv_tune(agpu_ctx *ctx, int32_t max_wgs, int32_t max_rows_per_wg, int32_t max_waves) {
    AGPU_REQUIRE_CTX(ctx);
    ctx->tune_max_waves = max_waves > 0 ? max_waves : 0;
    ctx->tune_target_wgs = max_wgs > 0 ? max_wgs : 0;
    ctx->tune_rows_per_split = max_rows_per_wg > 0 ? max_rows_per_wg : 256;
    return AGPU_OK;
}

int32_t agpu_int4_gemv_launch(agpu_ctx *ctx, const GemvArgs &a) {
    GemvParams p{};
    p.a = a;
    p.strict = ctx->strict_sync;
    if (a.ln_gamma && !agpu_int4_gemv_can_fuse_ln(a.M, a.K))
        return agpu_fail(ctx, AGPU_ERR_UNSUPPORTED, "int4_gemv: fused LayerNorm needs M <= 2 and M*K <= 8192");
    if (!(a.flags & AGPU_EPI_FORCE_FP32_GEMV) && agpu_int4_gemv_i8_supported(a))
        return agpu_int4_gemv_i8_launch(ctx, a, ctx->tune_rows_per_split / 8, ctx->tune_target_wgs);
    const int kp_total = a.K / 8;
    const int MT = a.M <= 1 ? 1 : a.M <= 2 ? 2 : a.M <= 4 ? 4 : a.M <= 8 ? 8 : 16;
    const bool aligned16 = (a.N % 4 == 0) && (((uintptr_t)a.packed | (uintptr_t)a.scales) % 16 == 0);
    const int cpl = aligned16 ? 4 : 1;
    const int col_blocks = ceil_div(a.N, 16 * cpl);
    if (col_blocks > ctx->n_counters) return agpu_fail(ctx, AGPU_ERR_WORKSPACE, "int4_gemv: N=%d too large", a.N);

    // K split over workgroups: a workgroup of 16 waves covers 64 packed rows per trip and keeps two
    // trips in flight, so up to 4 trips (256 rows) per workgroup cost two memory round trips.
    int ksplit = ceil_div(kp_total, ctx->tune_rows_per_split);
    while (ksplit > 1 && (size_t)ksplit * a.M * a.N * sizeof(float) > ctx->ws_bytes / 2) --ksplit;
    auto stage_floats = [&](int ks) {
        const int rps = ceil_div(kp_total, ks);
        const size_t xs_len = a.ln_gamma ? (size_t)a.K : (size_t)rps * 8;
        return (size_t)MT * xs_len + (size_t)MT * rps;
    };
    constexpr size_t kLdsBudget = 40 * 1024;
    while (stage_floats(ksplit) * sizeof(float) > kLdsBudget && ksplit < kp_total) ++ksplit;
    p.rows_per_split = ceil_div(kp_total, ksplit);
    ksplit = ceil_div(kp_total, p.rows_per_split);
    if (stage_floats(ksplit) * sizeof(float) > kLdsBudget)
        return agpu_fail(ctx, AGPU_ERR_UNSUPPORTED, "int4_gemv: staged x does not fit in LDS (M=%d K=%d)", a.M, a.K);
    if ((size_t)ksplit * a.M * a.N * sizeof(float) > ctx->ws_bytes / 2)
        return agpu_fail(ctx, AGPU_ERR_WORKSPACE, "int4_gemv: split-K partials exceed the workspace (M=%d N=%d K=%d)", a.M, a.N, a.K);
    // waves: one per 8 packed rows of the slice, bounded by the launch bound of the
    // instantiation and by the LDS the cross-wave reduction needs
    int max_w = MT == 1 ? 16 : 8;
    if (ctx->tune_max_waves > 0 && ctx->tune_max_waves < max_w) max_w = ctx->tune_max_waves;
    int W = ceil_div(p.rows_per_split, 8);  // two trips of 4 rows per wave
    W = W < 1 ? 1 : (W > max_w ? max_w : W);
    while (W > 1 && ((size_t)W * MT * 16 * cpl + stage_floats(ksplit)) * sizeof(float) > 64 * 1024) --W;
    const size_t red_floats = (size_t)W * MT * 16 * cpl;
    const size_t lds = sizeof(float) * (stage_floats(ksplit) + red_floats);
    p.partial = reinterpret_cast<float *>(ctx->workspace);
    p.counters = ctx->counters;
    p.col_blocks = col_blocks;
    // at most one workgroup per CU (measured best for the LM head); each strides over the column tiles
    int gx = col_blocks;
    const int cap = ctx->tune_target_wgs > 0 ? ctx->tune_target_wgs : ctx->num_cus;
    if (gx * ksplit > cap) gx = cap / ksplit > 0 ? cap / ksplit : 1;
    const dim3 grid(gx, ksplit);
    return cpl == 4 ? launch_m<4>(ctx, p, MT, grid, W, lds) : launch_m<1>(ctx, p, MT, grid, W, lds);
}

static int f32_gemv_waves(int K) { return std::max(1, std::min(16, K / 16)); }

int32_t agpu_f32_gemv_launch(agpu_ctx *ctx, const float *a, const float *b, float *c, int M, int N, int K) {
    const int MT = M <= 1 ? 1 : M <= 2 ? 2 : M <= 4 ? 4 : M <= 8 ? 8 : 16;
    const int W = f32_gemv_waves(K);
    const size_t lds = sizeof(float) * W * MT * 64;
    const dim3 grid(ceil_div(N, 64)), block(64 * W);
#define AGPU_GEMV_F32(MTV) hipLaunchKernelGGL((gemv_f32_kernel<MTV, false>), grid, block, lds, ctx->stream, a, b, c, M, N, K, ArgmaxShare{})
    switch (MT) {
        case 1: AGPU_GEMV_F32(1); break;
        case 2: AGPU_GEMV_F32(2); break;
        case 4: AGPU_GEMV_F32(4); break;
        case 8: AGPU_GEMV_F32(8); break;
        default: AGPU_GEMV_F32(16); break;
    }
#undef AGPU_GEMV_F32
    return AGPU_LAUNCH_CHECK(ctx, "gemv_f32_kernel");
}

bool agpu_f32_gemv_rows_supported(const float *a, const float *w, int M, int N, int K) {
    return M >= 1 && M <= 16 && N >= 1 && K % 4 == 0 && K >= 256 && K <= 2048 && (((uintptr_t)a | (uintptr_t)w) & 15u) == 0;
}

template <int MT, int ITERS, bool AM, class Feed>
static int32_t f32_rows_go(agpu_ctx *ctx, const float *a, const float *w, float *y, int M, int N, int K, const Feed &am) {
    constexpr int R = ITERS <= 4 ? 4 : 2;
    const size_t lds = MT == 1 ? 0 : std::max((size_t)MT * ITERS * 1024, feed_rows_lds(32, 512));
    static std::atomic<unsigned long long> lds_raised{0};  // one bit per device
    const unsigned long long bit = 1ull << (ctx->device & 63);
    if (lds > 64 * 1024 && !(lds_raised.load(std::memory_order_relaxed) & bit)) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(gemv_f32_rows_kernel<MT, ITERS, R, AM>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return agpu_hip(ctx, e, "hipFuncSetAttribute");
        lds_raised.fetch_or(bit, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL((gemv_f32_rows_kernel<MT, ITERS, R, AM>), dim3((unsigned)std::min(N, ctx->num_cus)), dim3(512), lds, ctx->stream, a, w, y, M, N, K, am);
    return AGPU_LAUNCH_CHECK(ctx, "gemv_f32_rows_kernel");
}
template <int MT, bool AM, class Feed>
static int32_t f32_rows_iters(agpu_ctx *ctx, const float *a, const float *w, float *y, int M, int N, int K, const Feed &am) {
    switch (ceil_div(K, 256)) {
        case 1: return f32_rows_go<MT, 1, AM>(ctx, a, w, y, M, N, K, am);
        case 2: return f32_rows_go<MT, 2, AM>(ctx, a, w, y, M, N, K, am);
        case 3: return f32_rows_go<MT, 3, AM>(ctx, a, w, y, M, N, K, am);
        case 4: return f32_rows_go<MT, 4, AM>(ctx, a, w, y, M, N, K, am);
        case 5: return f32_rows_go<MT, 5, AM>(ctx, a, w, y, M, N, K, am);
        case 6: return f32_rows_go<MT, 6, AM>(ctx, a, w, y, M, N, K, am);
        case 7: return f32_rows_go<MT, 7, AM>(ctx, a, w, y, M, N, K, am);
        default: return f32_rows_go<MT, 8, AM>(ctx, a, w, y, M, N, K, am);
    }
}

int32_t agpu_f32_gemv_rows_launch(agpu_ctx *ctx, const float *a, const float *w, float *y, int M, int N, int K) {
    if (M == 1) return f32_rows_iters<1, false>(ctx, a, w, y, M, N, K, ArgmaxShare{});
    if (M <= 4) return f32_rows_iters<4, false>(ctx, a, w, y, M, N, K, HeadFeed{});
    return f32_rows_iters<16, false>(ctx, a, w, y, M, N, K, HeadFeed{});
}

int32_t agpu_f32_gemv_rows_argmax_launch(agpu_ctx *ctx, const float *a, const float *w, float *y, int M, int N, int K, uint32_t *idx_out, int last, const ArgmaxAdvance &adv) {
    if (!feed_rows_fits(ctx)) return agpu_fail(ctx, AGPU_ERR_WORKSPACE, "gemv_f32_rows: the arg-max candidates exceed the workspace");
    if (M > 1) {
        const HeadFeed feed = feed_of(ctx, idx_out, last, adv);
        return M <= 4 ? f32_rows_iters<4, true>(ctx, a, w, y, M, N, K, feed) : f32_rows_iters<16, true>(ctx, a, w, y, M, N, K, feed);
    }
    const ArgmaxShare am{reinterpret_cast<unsigned long long *>(ctx->workspace), ctx->counters + (ctx->n_counters - 1), idx_out, last, ctx->strict_sync, adv};
    return f32_rows_iters<1, true>(ctx, a, w, y, 1, N, K, am);
}

int32_t agpu_f32_gemv_argmax_launch(agpu_ctx *ctx, const float *a, const float *b, float *c, int N, int K, uint32_t *idx_out, int last,
                                    const ArgmaxAdvance &adv) {
    const int W = f32_gemv_waves(K);
    const unsigned gx = (unsigned)ceil_div(N, 64);
    if ((size_t)gx * sizeof(unsigned long long) > ctx->ws_bytes / 2)
        return agpu_fail(ctx, AGPU_ERR_WORKSPACE, "gemv_f32: the arg-max candidates of %d columns exceed the workspace", N);
    const ArgmaxShare am{reinterpret_cast<unsigned long long *>(ctx->workspace), ctx->counters + (ctx->n_counters - 1), idx_out, last, ctx->strict_sync, adv};
    hipLaunchKernelGGL((gemv_f32_kernel<1, true>), dim3(gx), dim3(64 * W), sizeof(float) * W * 64, ctx->stream, a, b, c, 1, N, K, am);
    return AGPU_LAUNCH_CHECK(ctx, "gemv_f32_kernel");
}
