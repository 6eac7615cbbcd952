// GEMM of the int4 weight-only Linear for prompts that do not fill the chip with large tiles (more than 16 rows, but few), and from three rows on
// for shapes that no other matrix-core kernel takes (agpu_int4_gemm_rows_any_supported: K a multiple of 8 only, any N): the arithmetic of int4_gemm_bf16.hip (x as three exact bf16 pieces, the nibbles as (q - 8) / 16, one sum per
// 32 k of a scale group, then acc += scale * u in fp32), another split of the work.
//
// What bounds such a launch is not matrix or vector work but the chain of a workgroup: with K walked block by block
// through LDS a tile of 32 x 128 takes 8 - 12 us for K = 768 .. 3072 whatever M is, most of it waiting for the next block
// behind a barrier.  Here a workgroup owns a tile of 32 x 64 or 96 (32 x 32) outputs and its 8 (16) waves take the 32-k chunks of
// K in turn: every wave reads its own rows of x and its own weight words straight into registers, with AHEAD
// chunks on their way, splits and converts them itself and issues its MFMAs; no barrier until the waves' sums meet at the
// end.  x is split anew for every column tile, which costs 88 vector instructions per chunk beside the
// MFMAs' time of 12; the rule below lies where that begins to count.
//   M = 17, K = 768, N = 2304: 9.1 us before, 5.1 now; M = 150, K = 1024, N = 3072: 11.8, 7.4; M = 333, K = 768, N = 768:
//   10.8, 6.2.  A step (one chunk per wave, two waves per SIMD) takes 0.9 us with 64 columns: 190 vector instructions and
//   12 MFMAs per wave.  Tiles of 32 x 128 with the same split were no faster than the other kernel at any size.
#include "gemm_bf16.h"

#include <type_traits>

namespace {

struct RowsParams {
    const float *x;
    const uint32_t *packed;
    const float *scales;
    const float *bias;
    const float *residual;
    float *y;
    int M, N, K, chunk_shift;
    uint32_t flags;
    int row_tiles, col_tiles;
    int slices;              // of K, a workgroup each (SPLIT)
    float *partial;          // [slice][tile][wave][register][lane]
    unsigned int *counters;  // one ticket per tile, left at zero
    int strict;
    KvScatter kv;  // kcache == nullptr: none
    // LayerNorm of the rows on their way in (RowsLn)
    const float2 *stats_in;
    const float *gamma, *beta;
    float eps, inv_k, inv_chunks;
    float2 *stats_out;  // of the outputs, or null
};

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kMaxSlices = 8;

// LN_PIECES: statistics of a lane for the LayerNorm inside (0: none); STATS: statistics of the outputs; SPLIT: K in slices, the last workgroup of a
// tile adds them up; TAIL: K a multiple of 8, not of 32 (zeros for the rest of x's last chunk).
template <int CB, int NW, int AHEAD, int LN_PIECES, bool STATS, bool SPLIT, bool TAIL>
__global__ __launch_bounds__(64 * NW) void int4_gemm_rows_kernel(const RowsParams p) {
    constexpr bool NORM = LN_PIECES > 0;
    constexpr int COLS = 32 * CB, T = 64 * NW;
    constexpr int PER = CB * 16 / NW;  // registers (outputs) a lane finishes
    static_assert(PER >= 1 && CB * 16 % NW == 0, "every register of a tile is finished once");
    __shared__ __align__(16) float red[NW][CB * 16][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, hh = lane >> 5;
    // Workgroup b runs on XCD b % 8.  Every XCD takes an eighth of the tiles, numbered column by column, so that the weights
    // of a column tile come through one L2 (the rows of x, few here, through all of them).
    const int slices = SPLIT ? p.slices : 1, tiles = p.row_tiles * p.col_tiles, items = tiles * slices;
    const int t = (int)(blockIdx.x & 7) * ((items + 7) / 8) + (int)(blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= (items + 7) / 8 || t >= items) return;  // workgroup-uniform
    const int col_slice = t / p.row_tiles, tile_row = t - col_slice * p.row_tiles;
    const int tile_col = SPLIT ? col_slice / slices : col_slice, slice = col_slice - tile_col * slices;
    const int m0 = tile_row * 32, n0 = tile_col * COLS;
    const int all_chunks = TAIL ? (p.K + 31) / 32 : p.K / 32, chunk0 = SPLIT ? slice * all_chunks / slices : 0, chunks = SPLIT ? (slice + 1) * all_chunks / slices : all_chunks;  // the last one and one
    // fp32 rows are read by whole lines (eight lanes a row's 128 bytes, eight rows a request) and turned into operand
    // order through a part of LDS of the wave's own: read row by lane they cost 32 lines a request
    constexpr int NX = 4;
    // (32 rows of eight 16-byte units, unit u of row r at u ^ (r & 7): neither the lines written nor the operands read meet
    // in a bank)
    float *xs = &red[wave][0][0];
    static_assert(sizeof(red[0]) >= 32 * 128, "a wave's sums leave room for its rows of a chunk");
    auto unit = [&](int row, int u) { return xs + row * 32 + ((u ^ (row & 7)) << 2); };
    // a request's addresses: a base that depends on the chunk only (scalar) and an offset of the lane's own
    uint32_t xoff[NX], coff[CB];
#pragma unroll
    for (int i = 0; i < NX; ++i)  // rows beyond the last repeat it
        xoff[i] = ((uint32_t)(min(m0 + 8 * i + (lane >> 3), p.M - 1) - m0) * (uint32_t)p.K + 4u * (lane & 7)) * 4u;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) coff[cb] = (uint32_t)min(n0 + 32 * cb + j, p.N - 1) * 4u;  // columns beyond the last repeat it
    const char *xbase = reinterpret_cast<const char *>(p.x + (size_t)m0 * p.K);
    const uint32_t row_bytes = (uint32_t)p.N * 4u, hoff = (uint32_t)hh * row_bytes;
    u32x4 xv[AHEAD][NX], gv[NORM ? AHEAD : 1][2];  // (gv: gains and offsets)
    // native vectors: loop-carried uint4 structs come apart into registers that are moved, and waited for, on arrival
    uint32_t bw[AHEAD][CB][2];
    float bs[AHEAD][CB];
    auto request = [&](int c, int u) {  // c: scalar
        const char *src = xbase + (size_t)c * 128;
#pragma unroll
        for (int i = 0; i < NX; ++i) xv[u][i] = *reinterpret_cast<const u32x4 *>(src + (TAIL && 32 * c + 4 * (lane & 7) >= p.K ? xoff[i] - 16u * (lane & 7) : xoff[i]));
        if constexpr (NORM) {
            gv[u][0] = *reinterpret_cast<const u32x4 *>(p.gamma + 32 * c + 4 * (lane & 7));
            gv[u][1] = *reinterpret_cast<const u32x4 *>(p.beta + 32 * c + 4 * (lane & 7));
        }
        const char *wp = reinterpret_cast<const char *>(p.packed) + (size_t)(4 * c) * row_bytes;
        const char *sp = reinterpret_cast<const char *>(p.scales) + (size_t)(c >> p.chunk_shift) * row_bytes;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            if constexpr (TAIL) {  // words beyond K repeat the last row's
                const int rows = (p.K >> 3) - 4 * c;
                bw[u][cb][0] = *reinterpret_cast<const uint32_t *>(wp + ((uint32_t)min(hh, rows - 1) * row_bytes + coff[cb]));
                bw[u][cb][1] = *reinterpret_cast<const uint32_t *>(wp + ((uint32_t)min(2 + hh, rows - 1) * row_bytes + coff[cb]));
            } else {
                bw[u][cb][0] = *reinterpret_cast<const uint32_t *>(wp + (hoff + coff[cb]));
                bw[u][cb][1] = *reinterpret_cast<const uint32_t *>(wp + 2 * (size_t)row_bytes + (hoff + coff[cb]));
            }
            bs[u][cb] = *reinterpret_cast<const float *>(sp + coff[cb]);
        }
    };
    floatx16 acc[CB];
    const floatx16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) acc[cb] = zero;
    // No branch in the loop: with one, loaded registers are moved and waited for where they arrive.  Steps beyond a wave's
    // last chunk repeat that chunk with scales of zero.
    const int last = chunks - 1;
    // Mean and 1 / sqrt(variance + eps) of the rows this lane loads from (8 i + lane / 8) out of the statistics of their pieces of 32.  Every wave for itself
    // (lane: row j, every second piece): a barrier here would keep the waves in step for good, and all of a SIMD's vector instructions, then all of its
    // matrix instructions, would stand in a row.  They travel ahead of the first rows and weights, and no loop is around them (the wait for a loop's would be
    // one for the rows and weights too: 7.15 ms in place of 6.97 below).
    float mean[NORM ? NX : 1], rstd[NORM ? NX : 1];
    float2 st_in[NORM ? LN_PIECES : 1];
    if constexpr (NORM) {
#pragma unroll
        for (int i = 0; i < LN_PIECES; ++i) st_in[i] = (p.stats_in + m0 + j)[(size_t)min(2 * i + hh, chunks - 1) * (32 * p.row_tiles)];
    }
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) request(min(chunk0 + wave + u * NW, last), u);
    if constexpr (NORM) {
        auto both = [](float v) {
            const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
            return __uint_as_float(s[0]) + __uint_as_float(s[1]);
        };
        float sum = 0.0f, q = 0.0f;
#pragma unroll
        for (int i = 0; i < LN_PIECES; ++i) sum += 2 * i + hh < chunks ? st_in[i].x : 0.0f;
        const float row_mean = both(sum) * p.inv_chunks;
#pragma unroll
        for (int i = 0; i < LN_PIECES; ++i) {  // squared distances from the mean: the pieces' own, and 32 of each piece's mean
            const float dm = st_in[i].x - row_mean;
            q += 2 * i + hh < chunks ? fmaf(32.0f * dm, dm, st_in[i].y) : 0.0f;
        }
        const float row_rstd = inverse_sqrt(fmaf(both(q), p.inv_k, p.eps));
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            mean[i] = __shfl(row_mean, 8 * i + (lane >> 3), kWave);
            rstd[i] = __shfl(row_rstd, 8 * i + (lane >> 3), kWave);
        }
    }
    for (int c0 = chunk0 + wave; c0 < chunks; c0 += AHEAD * NW) {
#pragma unroll
        for (int u = 0; u < AHEAD; ++u) {
            const int c = c0 + u * NW;
            bf16x8 a[2][3], b[CB][2];  // [step][piece]
            float sc[CB];
            // LDS operations of a wave complete in order
#pragma unroll
            for (int i = 0; i < NX; ++i) {
                u32x4 x = xv[u][i];
                if constexpr (NORM) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        x[e] = __float_as_uint(fmaf((__uint_as_float(x[e]) - mean[i]) * rstd[i], __uint_as_float(gv[u][0][e]), __uint_as_float(gv[u][1][e])));
                }
                if constexpr (TAIL) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[e] = 32 * c + 4 * (lane & 7) < p.K ? x[e] : 0u;
                }
                *reinterpret_cast<u32x4 *>(unit(8 * i + (lane >> 3), lane & 7)) = x;
            }
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                const float4 lo4 = *reinterpret_cast<const float4 *>(unit(j, 4 * st + 2 * hh));
                const float4 hi4 = *reinterpret_cast<const float4 *>(unit(j, 4 * st + 2 * hh + 1));
                const float v[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
                split_pieces(v, a[st]);
            }
#pragma unroll
            for (int cb = 0; cb < CB; ++cb) {
#pragma unroll
                for (int st = 0; st < 2; ++st) b[cb][st] = nibbles_to_bf16(bw[u][cb][st]);
                sc[cb] = c < chunks ? bs[u][cb] * GB_NIBBLE_UNIT : 0.0f;
            }
            request(min(c + AHEAD * NW, last), u);  // into the registers just read
            floatx16 gs[CB];
#pragma unroll
            for (int piece = 0; piece < 3; ++piece)  // smallest piece first
#pragma unroll
                for (int st = 0; st < 2; ++st)
#pragma unroll
                    for (int cb = 0; cb < CB; ++cb)
                        gs[cb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[st][piece], b[cb][st], piece == 0 && st == 0 ? zero : gs[cb], 0, 0, 0);
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[cb][r] = fmaf(sc[cb], gs[cb][r], acc[cb][r]);
        }
    }
    // ---- the waves' sums meet in LDS, in wave order; wave w finishes the registers w PER .. of every lane ----
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
        for (int r = 0; r < 16; ++r) red[wave][cb * 16 + r][lane] = acc[cb][r];
    const int reg0 = wave * PER;
    auto row_of = [&](int i) { const int r = (reg0 + i) & 15; return 8 * (r >> 2) + 4 * hh + (r & 3); };  // of the wave's register i
    auto col_of = [&](int i) { return 32 * ((16 % PER ? reg0 + i : reg0) >> 4) + j; };
    float res[PER], bias[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int n = min(n0 + col_of(i), p.N - 1);
        bias[i] = p.bias ? p.bias[n] : 0.0f;
        res[i] = p.residual ? p.residual[(size_t)min(m0 + row_of(i), p.M - 1) * p.N + n] : 0.0f;
    }
    const int kv_pos = p.kv.kcache ? *p.kv.pos_dev : 0;
    __syncthreads();
    float vals[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v += red[w][reg0 + i][lane];
        vals[i] = v;
    }
    if constexpr (SPLIT) {
        const int tile = tile_col * p.row_tiles + tile_row;
        float *mine = p.partial + (((size_t)slice * tiles + tile) * NW + wave) * PER * 64 + lane;
#pragma unroll
        for (int i = 0; i < PER; ++i) __hip_atomic_store(mine + 64 * i, vals[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        partials_published(p.strict);
        __syncthreads();
        __shared__ int s_last;
        if (tid == 0) {
            const unsigned int tk = take_ticket(&p.counters[tile], p.strict);
            s_last = tk == (unsigned int)(slices - 1);
            if (s_last) __hip_atomic_store(&p.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!s_last) return;
        const float *first = mine - (size_t)slice * tiles * NW * PER * 64;
        float part[kMaxSlices][PER];
#pragma unroll
        for (int sp = 0; sp < kMaxSlices; ++sp) {
            if (sp >= slices) break;
#pragma unroll
            for (int i = 0; i < PER; ++i) part[sp][i] = __hip_atomic_load(first + (size_t)sp * tiles * NW * PER * 64 + 64 * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) vals[i] = 0.0f;
#pragma unroll
        for (int sp = 0; sp < kMaxSlices; ++sp) {  // slice order: the same sum every run
            if (sp >= slices) break;
#pragma unroll
            for (int i = 0; i < PER; ++i) vals[i] += part[sp][i];
        }
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        float v = vals[i] + bias[i];
        if (p.flags & AGPU_EPI_GELU_TANH) v = gelu_tanh_dev(v);
        else if (p.flags & AGPU_EPI_GELU_QUICK) v = gelu_quick_dev(v);
        vals[i] = v;
        const int m = m0 + row_of(i), n = n0 + col_of(i);
        if constexpr (STATS) {  // (N is a multiple of 32: a block of columns is whole, or none of it is there)
            const float2 st = stats_of_32(v + res[i]);
            if (j == 0 && n < p.N) p.stats_out[(size_t)(n >> 5) * (32 * p.row_tiles) + m] = st;
        }
        if (n < p.N && m < p.M) {
            v += res[i];
            p.y[(size_t)m * p.N + n] = v;
            if (p.kv.kcache && n >= p.N / 3) {
                const int dm = p.N / 3, jj = n - dm, in_v = jj >= dm ? 1 : 0, e = jj - in_v * dm;
                const int b = m / p.kv.new_len, s = m - b * p.kv.new_len;
                float *dst = in_v ? p.kv.vcache : p.kv.kcache;
                dst[((size_t)(b * p.kv.n_heads + (e >> 6)) * p.kv.n_positions + kv_pos + s) * 64 + (e & 63)] = v;
            }
        }
    }
    // ---- K and V once more as the prefill attention's operand fragments (layout: attention.hip), through LDS: the tile is
    // 32 keys of one sequence x CB times 32 dimensions, each 32 of one head's K or V ----
    if (p.kv.kfrag && n0 + COLS > p.N / 3) {  // workgroup-uniform
        constexpr int FIN_LD = COLS + 4;  // floats between rows of the finished tile
        __syncthreads();  // the sums have been read
        float *fin = &red[0][0][0];
#pragma unroll
        for (int i = 0; i < PER; ++i) fin[row_of(i) * FIN_LD + col_of(i)] = vals[i];
        __syncthreads();
        const int dm = p.N / 3, seq = m0 / p.kv.new_len, tile = (m0 - seq * p.kv.new_len) >> 5;
        for (int i = tid; i < COLS * 4; i += T) {  // per 32 columns: 4 x 32 (K) or 32 x 4 (V) runs of eight values
            const int cb = i >> 7, r = i & 127, n = n0 + 32 * cb;
            if (n < dm || n >= p.N) continue;
            const int in_v = n >= 2 * dm ? 1 : 0, c0 = n - dm - in_v * dm;
            const size_t base = ((size_t)(seq * p.kv.n_heads + (c0 >> 6)) * p.kv.tiles_cap + tile) * kKvFragsPerTile;
            float a[8];
            if (in_v) {
                const int d = r & 31, s = (r >> 5) & 1, h2 = r >> 6, dd = (c0 & 63) + d;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int row = 16 * s + 8 * (e >> 2) + 4 * h2 + (e & 3);
                    a[e] = m0 + row < p.M ? fin[row * FIN_LD + 32 * cb + d] : 0.0f;
                }
                if (v_is_small(a, p.kv.v_up, m0 + 32 <= p.M)) p.kv.v_small[seq * p.kv.n_heads + (c0 >> 6)] = p.kv.epoch;
                store_kv_frags(p.kv.vfrag + base + (size_t)(((dd >> 5) * 4 + s) * 2 + h2) * 32 + (dd & 31), 2 * 2 * 32, a, p.kv.v_up);
            } else {
                const int key = r & 31, d = 8 * (r >> 5), dd = (c0 & 63) + d;  // 8 dimensions from dd: step dd / 16, half
                const float4 lo = *reinterpret_cast<const float4 *>(fin + key * FIN_LD + 32 * cb + d);
                const float4 hi = *reinterpret_cast<const float4 *>(fin + key * FIN_LD + 32 * cb + d + 4);
                a[0] = lo.x; a[1] = lo.y; a[2] = lo.z; a[3] = lo.w; a[4] = hi.x; a[5] = hi.y; a[6] = hi.z; a[7] = hi.w;
                store_kv_frags(p.kv.kfrag + base + (size_t)((dd >> 4) * 4 + ((dd >> 3) & 1)) * 32 + key, 2 * 32, a, p.kv.k_up);
            }
        }
    }
}

template <int CB, int NW, int AHEAD, int LN_PIECES, bool STATS, bool SPLIT = false, bool TAIL = false>
int32_t rows_launch(agpu_ctx *ctx, RowsParams &p) {
    p.row_tiles = ceil_div(p.M, 32);
    p.col_tiles = ceil_div(p.N, 32 * CB);
    const dim3 grid(8u * (unsigned)ceil_div(p.row_tiles * p.col_tiles * (SPLIT ? p.slices : 1), 8));
    hipLaunchKernelGGL((int4_gemm_rows_kernel<CB, NW, AHEAD, LN_PIECES, STATS, SPLIT, TAIL>), grid, dim3(64 * NW), 0, ctx->stream, p);
    return AGPU_LAUNCH_CHECK(ctx, "int4_gemm_rows_kernel");
}
template <int CB, int NW, int AHEAD>
int32_t rows_go(agpu_ctx *ctx, RowsParams &p) {
    if constexpr (CB > 1) {
        if (p.stats_in) return p.K <= 1024 ? rows_launch<CB, NW, AHEAD, 16, false>(ctx, p) : rows_launch<CB, NW, AHEAD, 32, false>(ctx, p);
    }
    return p.stats_out ? rows_launch<CB, NW, AHEAD, 0, true>(ctx, p) : rows_launch<CB, NW, AHEAD, 0, false>(ctx, p);
}

int32_t rows_split_go(agpu_ctx *ctx, RowsParams &p) {
    const int steps = ceil_div(ceil_div(p.K / 32, p.slices), 8);
    const bool three = ceil_div(steps, 3) * 3 < ceil_div(steps, 2) * 2;
    if (p.stats_out) return three ? rows_launch<2, 8, 3, 0, true, true>(ctx, p) : rows_launch<2, 8, 2, 0, true, true>(ctx, p);
    return three ? rows_launch<2, 8, 3, 0, false, true>(ctx, p) : rows_launch<2, 8, 2, 0, false, true>(ctx, p);
}

}  // namespace

// Tiles of this kernel while each has a CU of its own and K is not so long that few waves per tile set the time (then the
// other kernel slices K over workgroups).  us per launch, that kernel against this: 32-column tiles, 16 waves: 17 rows
// 768 -> 2304 9.0 / 5.1, 3072 -> 768 11.2 / 9.4, 5120 -> 1280 13.3 / 14.9 (not taken;
// 150 rows 17.4 / 15.2), 6400 -> 1600 15.3 / 18.3 (not taken); 64-column tiles, 8 waves: 150 rows
// 768 -> 2304 10.7 / 6.5, 1024 -> 3072 12.0 / 8.0, 512 rows 3072 -> 768 17.6 / 16.4, 150 rows 6400 -> 1600 23.4 / 28
// (not taken); but with more tiles than CUs 333 rows 768 -> 2304 11.6 / 11.9, 150 rows 1600 -> 6400 18.9 / 26.
// 96-column tiles, which reach further up in M and N (a step takes 1.4 us with them, so only where the narrower ones do not
// fit): 150 rows 1024 -> 4096 12.8 / 9.8, 1280 -> 3840 17.4 / 12.7, 3072 -> 4608 27.7 / 21.0, 250 rows 768 -> 2304
// 12.3 / 9.8, 333 rows 1600 -> 1600 16.6 / 13.3, 300 rows 3328 -> 2000 22.7 / 23.5 (not taken).
namespace {
enum class RowsTile { None, Cols32, Cols64, Cols96 };

// Slices of K, a workgroup each, where K is long and the tiles of 64 columns leave half of the CUs or more without one; 1: none.  As many as there are CUs for, and
// of those the fewest that leave a wave as few steps as it gets (us, none / this: 33 x 3072 x 768 12.2 / 10.0, 128 x 3072 x 768 13.8 / 12.4, 200 x 3072 x 768
// 15.2 / 14.1; 40 x 4096 x 1024 15.0 / 11.4, 150 x 4096 x 1024 17.3 / 15.8, two slices 250 x 4096 x 1024 19.8 / 18.9; 60 x 5120 x 1280 17.8 / 12.9;
// 40 x 6400 x 1600 19.1 / 14.5, 160 x 6400 x 1600 27.9 / 23.3).  The last workgroup of a tile waits for two round trips through memory, so that shorter K gains
// nothing (60 x 2048 x 512 10.3 / 9.9, 300 x 2048 x 512 12.6 / 14.0, 64 x 1024 x 1024 7.5 / 9.1), nor do two slices of 3072 (200 rows x 768: 15.2 / 15.5).
// Not where calls share the scratch, nor where the sums of all slices do not fit into half of it.
int rows_slices(const agpu_ctx *ctx, int M, int N, int K) {
    const long long tiles = (long long)ceil_div(M, 32) * ceil_div(N, 64);
    if (ctx->shared_scratch || K < 3072 || K % 32 != 0 || 2 * tiles > ctx->num_cus || tiles > ctx->n_counters) return 1;
    auto steps = [&](int slices) { return ceil_div(ceil_div(K / 32, slices), 8); };
    int best = 2;
    for (int s = 3; s <= kMaxSlices && s * tiles <= ctx->num_cus; ++s)
        if (steps(s) < steps(best)) best = s;
    if (best == 2 && K < 4096) return 1;
    return best * tiles * (32 * 64 * sizeof(float)) <= ctx->ws_bytes / 2 ? best : 1;
}
RowsTile rows_tile(const agpu_ctx *ctx, int M, int N, int K) {
    const long long rt = ceil_div(M, 32);
    if (rows_slices(ctx, M, N, K) > 1) return RowsTile::Cols64;
    if (rt * ceil_div(N, 32) <= ctx->num_cus && (K <= 4096 || (K <= 5120 && rt >= 3))) return RowsTile::Cols32;
    if (rt * ceil_div(N, 64) <= ctx->num_cus && K <= 3328) return RowsTile::Cols64;
    if (rt * ceil_div(N, 96) <= ctx->num_cus && K <= 3072) return RowsTile::Cols96;
    return RowsTile::None;
}
}  // namespace

bool agpu_int4_gemm_rows_wanted(const agpu_ctx *ctx, int M, int N, int K) { return rows_tile(ctx, M, N, K) != RowsTile::None; }

// The LayerNorm of the rows inside, not a launch of its own in front (ms a pass, launch / this: 24 layers, five chunks of 150 rows of 1024 7.36 / 6.97; 12 layers,
// 128 rows of 768 1.097 / 1.072; 6 layers, 120 rows of 1280 0.486 / 0.476).  Tiles of 32 columns have eight waves then (12 layers: 49 rows of 128 0.450 / 0.403,
// 30 of 512 0.510 / 0.464, 60 of 640 0.581 / 0.558, 90 of 768 0.601 / 0.587, 64 of 1024 0.578 / 0.574; with sixteen 60 of 640 0.577), which are too few
// beyond K of 1024 (64 of 1280 0.663 / 0.691; sixteen 0.666).
bool agpu_int4_gemm_rows_can_norm(const agpu_ctx *ctx, int M, int N, int K) {
    const RowsTile tile = rows_tile(ctx, M, N, K);
    return tile == RowsTile::Cols32 ? K <= 1024 : tile != RowsTile::None && K <= RowsLn::kMaxK;
}

// Linears that neither the kernels of many rows nor those of up to sixteen take: K a multiple of 8 only, or few rows and columns no multiple of four.  us a launch (with a
// copy of x in front), before (fp32 operands, or a wave a column) / this: 39 x 1672 x 375 98 / 10.6, 201 x 2200 x 156 128 / 13.6, 1000 x 1672 x 1500 151 / 39, 2000 x 2200 x
// 5000 733 / 250, 17 x 72 x 64 10.7 / 9.2, 600 x 72 x 500 13.5 / 8.7; 16 x 1672 x 375 17.7 / 10.7, 5 13.2 / 10.6, 3 12.6 / 10.2, but 2 10.8 / 10.5 and 1 9.3 /
// 10.4; 4 x 840 x 3000 11.5 / 9.6, 10 x 1024 x 375 14.9 / 9.6, 16 x 5000 x 6000 74 / 20, 5 x 5000 x 800 18.9 / 18.6, but 5 x 6400 x 33 14.7 / 20.0 (one workgroup has
// all of a long K).  Errors a fifth of those on fp32 operands (6.2e-8 of the result for 3.4e-7).  The narrowest tiles that find a CU each.
bool agpu_int4_gemm_rows_any_supported(const void *x, int M, int N, int K, int group) {
    return M >= 3 && (M > 16 || K <= 4096 || (long long)M * N >= 4000) && K % 8 == 0 && group % 32 == 0 && ((group / 32) & (group / 32 - 1)) == 0 && ((uintptr_t)x % 16) == 0;
}
int32_t agpu_int4_gemm_rows_any_launch(agpu_ctx *ctx, const float *x, const uint32_t *packed, const float *scales, const float *bias, const float *residual, float *y, int M, int N,
                                        int K, int group, uint32_t flags) {
    RowsParams p{};
    p.x = x; p.packed = packed; p.scales = scales; p.bias = bias; p.residual = residual; p.y = y;
    p.M = M; p.N = N; p.K = K; p.chunk_shift = __builtin_ctz((unsigned)(group / 32)); p.flags = flags;
    auto go = [&](auto tail) -> int32_t {
        constexpr bool TAIL = decltype(tail)::value;
        const long long rows = ceil_div(M, 32), cus = ctx->num_cus;
        if (rows * ceil_div(N, 32) <= cus) return rows_launch<1, 16, 2, 0, false, false, TAIL>(ctx, p);
        if (rows * ceil_div(N, 64) <= cus) return rows_launch<2, 8, 2, 0, false, false, TAIL>(ctx, p);
        return rows_launch<3, 8, 2, 0, false, false, TAIL>(ctx, p);
    };
    return K % 32 ? go(std::true_type{}) : go(std::false_type{});
}

int32_t agpu_int4_gemm_rows_launch(agpu_ctx *ctx, const float *x, const uint32_t *packed, const float *scales, const float *bias,
                                   const float *residual, float *y, int M, int N, int K, int group, uint32_t flags, const KvScatter *kv, const RowsLn *ln) {
    RowsParams p{};
    if (kv) p.kv = *kv;
    if (ln) { p.stats_in = ln->in; p.gamma = ln->gamma; p.beta = ln->beta; p.eps = ln->eps; p.inv_k = 1.0f / (float)K; p.inv_chunks = 32.0f / (float)K; p.stats_out = ln->out; }
    if (p.stats_in && (p.stats_out || !agpu_int4_gemm_rows_can_norm(ctx, M, N, K))) return agpu_fail(ctx, AGPU_ERR_UNSUPPORTED, "int4_gemm_rows: no LayerNorm for M=%d N=%d K=%d", M, N, K);
    p.x = x; p.packed = packed; p.scales = scales; p.bias = bias; p.residual = residual; p.y = y;
    p.M = M; p.N = N; p.K = K; p.chunk_shift = __builtin_ctz((unsigned)(group / 32)); p.flags = flags;
    const RowsTile tile = rows_tile(ctx, M, N, K);
    p.slices = p.stats_in ? 1 : rows_slices(ctx, M, N, K);
    if (p.slices > 1) {
        p.partial = reinterpret_cast<float *>(ctx->workspace); p.counters = ctx->counters; p.strict = ctx->strict_sync;
        return rows_split_go(ctx, p);
    }
    if (tile == RowsTile::Cols32 && p.stats_in) return rows_launch<1, 8, 2, 16, false>(ctx, p);
    if (tile == RowsTile::Cols32) return rows_go<1, 16, 2>(ctx, p);
    if (tile == RowsTile::Cols96) return rows_go<3, 8, 2>(ctx, p);
    // a wave's chunks are padded to a multiple of those on their way: three or two, whichever pads less
    const int steps = ceil_div(K / 32, 8);
    return ceil_div(steps, 3) * 3 < ceil_div(steps, 2) * 2 ? rows_go<2, 8, 3>(ctx, p) : rows_go<2, 8, 2>(ctx, p);
}
