// Prefill GEMM of the int4 weight-only Linear for many rows, on the f16 matrix cores of gfx950 at fp32 accuracy.
//
// x arrives as pairs of f16 numbers with a power-of-two scale per row (gemm_pairs.h), made once by pair_rows_kernel (with the LayerNorm
// in front, where there is one) instead of by every column tile; the weights (q - 8) / 128 are f16 numbers as they are.  Products are exact in
// fp32, so per 64 k and output
//     acc += scale[0] * u0 + scale[1] * u1,   u = sum over 32 k of (lo + hi) * (q - 8) / 128, smallest pieces first
// takes 8 v_mfma_f32_32x32x16_f16 per 32 x 32 tile (three bf16 pieces: 12).  The right-hand side joins acc by two chained v_fma_f32, a rounding of
// the sum over K per 32 k, or, with K long enough for it to count (LONG), by three vector instructions and a rounding per 64 k.  The row's factor
// comes in at the end.
//
// A wave owns 64 x 64 outputs, two waves share a SIMD.  A tile is 64 x 128: two waves side by side are a group, and two (KS = 2) or four (KS = 4)
// groups take the tile's K blocks in turn and meet in LDS at the end, so that a workgroup is four waves, two of them to a CU, or eight, the CU's
// only one.  Lane j of a half wave owns columns 2 j and 2 j + 1, one per column block, so the words of 64 k are four 8-byte loads.  The pairs of a
// K block come into LDS by loads that write it directly, a block ahead, double buffered.  Tiles with rows that are not for pairs (kPairShort) take another way (pair_general_sums).
// A block is four units (row block, column block) of 8 MFMAs.  Beside the MFMAs of a unit stand, written out one by one, the scaling of
// the unit before and the LDS reads of the next row block's operands; in the last unit the next block's words become operands.  The one
// barrier per block stands before its last unit, when the block's last operands are in registers.
#include "gemm_pairs.h"
#include <algorithm>
#include <atomic>
#include <cmath>
#include <type_traits>

namespace {

struct PairGemmParams {
    const char *frags;
    const float *factors;    // per row, or null: `factor`
    float factor;
    PairMarks marks;                // without: which rows stand as floats in which blocks
    const float *x, *gamma, *beta;  // with `factors`: the rows themselves, K floats each, and the LayerNorm in front of them (or null)
    float eps;
    const uint32_t *packed;
    const float *scales;
    GemmOut out;
    int K, chunk_shift;
    int row_blocks, k_blocks;
    int row_tiles, col_tiles;
    int full_tiles;          // tiles 0 .. full_tiles - 1 have one workgroup each, the others tail_ks workgroups (slices of K)
    int tail_ks, n_tail;     // ... and how many tiles those others are
    int blocks_per_split;
    float *partial;          // [tail_ks, n_tail tiles] partial results
    unsigned int *counters;  // one ticket per sliced tile, left at zero
    int strict;
};

// Where rows come from and go to: kPlain: rows with a factor and flags each -> y; kKv: the same, K and V columns to the cache as well; kHandOn: the same -> pairs
// instead of y; kHanded: rows that were handed on, with one scale for all and marks -> y.  (In one kernel for all of them the checks of kKv and kHandOn
// cost every launch 0.6 us.)
enum class PairKind { kPlain, kKv, kHandOn, kHanded };

// 1 KiB of global memory straight into LDS, lane l's 16 bytes to lds + OFF + 16 l.  Written out, because the compiler lets every LDS read
// wait for all such loads in flight.  M0 needs one wait state.
template <int OFF>
__device__ __forceinline__ void pair_load_1k(uint32_t lds, uint32_t lane_off, const char *src) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 offset:%3" ::"s"(lds), "v"(lane_off), "s"(src), "n"(OFF) : "memory");
}

// WC waves of 64 x 64 outputs per group, KS groups
template <int WC, int KS>
struct PairTile {
    static constexpr int BM = 64, BN = 64 * WC, T = 64 * WC * KS;
    static constexpr int STAGE = 2 * kPairBlockBytes;       // pairs of one K block
    static constexpr int PER = 64 / KS;                     // registers a lane finishes
    static constexpr int LOOP_BYTES = KS * 2 * STAGE;
    static constexpr int RED_BYTES = KS * (KS - 1) * WC * PER * 64 * 4;
    static constexpr int TR_LD = 68, TR_BYTES = 16 * TR_LD * 4;  // the epilogue's K rows, per wave
    static constexpr int LDS = LOOP_BYTES > RED_BYTES + WC * KS * TR_BYTES ? LOOP_BYTES : RED_BYTES + WC * KS * TR_BYTES;
    static_assert(LDS <= 160 * 1024 - 64, "LDS of a CU");
    static_assert(KS == 2 || KS == 4, "a group finishes row blocks or halves of one");
};

// two floats that need not lie on eight bytes (N may be odd)
struct __attribute__((packed, aligned(4))) Float2 {
    float x, y;
};

// What the epilogue reads of one half of a row block, requested before the sums are complete.
struct PairEarly {
    float4 factor[2];
    Float2 res[8];
};

// 32 rows of a row block are 2 x 8 registers x 2 half waves: half s of them, 16 rows x 64 columns, in v[register][column of the lane]:
// row m0 + 8 (r / 4) + 4 hh + r % 4 with r = 8 s + register, column nb + c; the lane stores columns n and n + 1 below N (nb = n unless
// the last column stands alone: then nb = n - 1).
template <int TR_LD, PairKind KIND>
__device__ __forceinline__ void pair_finish_half(const GemmOut &o, float (&v)[8][2], const float (&bias)[2], const PairEarly &in, int m0, int s, int n0, int j, int hh,
                                                 int kv_pos, float *tr) {
    const int n = n0 + 2 * j, lane = 32 * hh + j;
    auto row_of = [&](int i) { return m0 + 16 * s + 8 * (i >> 2) + 4 * hh + (i & 3); };
    const int dm = o.N / 3;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int m = row_of(i);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            v[i][c] += bias[c];
            if (o.flags & AGPU_EPI_GELU_TANH) v[i][c] = gelu_tanh_dev(v[i][c]);
            else if (o.flags & AGPU_EPI_GELU_QUICK) v[i][c] = gelu_quick_dev(v[i][c]);
        }
        if (KIND != PairKind::kHandOn && m < o.M && n < o.N) {
            const Float2 out = {v[i][0] + in.res[i].x, v[i][1] + in.res[i].y};
            float *y = o.y + (size_t)m * o.N;
            if (n + 1 < o.N) *reinterpret_cast<Float2 *>(y + n) = out;
            else y[n] = out.y;
            if (KIND == PairKind::kKv && n >= dm) {  // (N is even then, and both columns are within one head's K or V)
                const int in_v = n >= 2 * dm ? 1 : 0, e = n - dm - in_v * dm;
                const int b = m / o.kv.new_len, pos = m - b * o.kv.new_len;
                float *dst = in_v ? o.kv.vcache : o.kv.kcache;
                *reinterpret_cast<Float2 *>(dst + ((size_t)(b * o.kv.n_heads + (e >> 6)) * o.kv.n_positions + kv_pos + pos) * 64 + (e & 63)) = out;
            }
        }
    }
    if (KIND == PairKind::kHandOn && m0 < o.M) {  // uniform; (a row block that begins at or past M has no place)
#pragma unroll
        for (int i = 0; i < 8; ++i) *reinterpret_cast<float2 *>(tr + (8 * (i >> 2) + 4 * hh + (i & 3)) * TR_LD + 2 * j) = make_float2(v[i][0], v[i][1]);
        // same wave: LDS operations complete in order
        char *block = o.pairs + ((size_t)(m0 >> 5) * (o.N >> 6) + (n0 >> 6)) * kPairBlockBytes;
        // 16 rows x 8 runs of eight columns, two a lane: a row's 64 bytes of a step go out together
        const int row = (lane >> 1) & 15, run0 = (lane & 1) | (lane >> 5) << 1;
        float a[2][8], most = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float4 lo4 = *reinterpret_cast<const float4 *>(tr + row * TR_LD + 8 * (run0 + 4 * i)), hi4 = *reinterpret_cast<const float4 *>(tr + row * TR_LD + 8 * (run0 + 4 * i) + 4);
            const float x[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                a[i][e] = x[e];
                most = fmaxf(most, fabsf(x[e]));
            }
        }
        most = fmaxf(most, dpp_move<0xb1, 0xf>(most, most));  // quad_perm [1,0,3,2]
        const auto halves = __builtin_amdgcn_permlane32_swap(__float_as_uint(most), __float_as_uint(most), false, false);
        const bool raw = pair_raw(fmaxf(__uint_as_float(halves[0]), __uint_as_float(halves[1])) * o.pairs_up);
        auto store_pairs = [&](int i) {
            const int run = run0 + 4 * i;
            uint4 lo, hi;
            split_pair(a[i], o.pairs_up, lo, hi);
            *reinterpret_cast<uint4 *>(block + pair_offset(16 * s + row, run >> 1, 0, run & 1)) = lo;
            *reinterpret_cast<uint4 *>(block + pair_offset(16 * s + row, run >> 1, 1, run & 1)) = hi;
        };
        if (__builtin_expect(!__any(raw), 1)) {
            store_pairs(0);
            store_pairs(1);
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (raw) {
#pragma unroll
                    for (int e = 0; e < 8; e += 4)
                        *reinterpret_cast<float4 *>(block + pair_raw_offset(16 * s + row, 8 * (run0 + 4 * i) + e)) = make_float4(a[i][e], a[i][e + 1], a[i][e + 2], a[i][e + 3]);
                } else {
                    store_pairs(i);
                }
            }
            if (raw) o.marks.tiles[m0 >> 6] = o.marks.epoch;
        }
        if (run0 == 0 && m0 + 16 * s + row < o.M) o.marks.marks[(size_t)(n0 >> 6) * 32 * ((o.M + 31) >> 5) + m0 + 16 * s + row] = raw;
    }
    // The K and V columns once more as the f16 operand fragments of the prefill attention (rows = key positions from 0; a row block
    // that begins at or past M belongs to no sequence).  V: a lane holds two dimensions and the eight keys of its registers, which are
    // operands as they are.  K: a lane needs 8 dimensions of one key, so the rows go through LDS.
    if (KIND == PairKind::kKv && o.kv.kfrag && n0 + 64 > dm && m0 < o.M) {  // wave-uniform
        // Rows past M are sums over zeros, that is the bias, for which k_up and v_up are no bound.  They are never visible, but their weight of
        // zero meets V in a product, which an infinity would make NaN: zeros instead.
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int c = 0; c < 2; ++c) v[i][c] = row_of(i) < o.M ? v[i][c] : 0.0f;
        const int seq = m0 / o.kv.new_len, tile = (m0 - seq * o.kv.new_len) >> 5;  // sequences are whole numbers of 32-row blocks
        auto base = [&](int e) { return ((size_t)(seq * o.kv.n_heads + (e >> 6)) * o.kv.tiles_cap + tile) * kKvFragsPerTile; };
        if (n >= 2 * dm && n < o.N) {
            const int e = n - 2 * dm, d = e & 63;
            bool small = false;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                float a[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) a[i] = v[i][c];
                small = small || v_is_small(a, o.kv.v_up, m0 + 32 <= o.M);
                store_kv_frags(o.kv.vfrag + base(e) + (size_t)(((d >> 5) * 4 + s) * 2 + hh) * 32 + (d & 31) + c, 2 * 2 * 32, a, o.kv.v_up);
            }
            if (__builtin_expect(small, 0)) o.kv.v_small[seq * o.kv.n_heads + (e >> 6)] = o.kv.epoch;
        }
        if (n0 < 2 * dm) {  // wave-uniform
#pragma unroll
            for (int i = 0; i < 8; ++i) *reinterpret_cast<float2 *>(tr + (8 * (i >> 2) + 4 * hh + (i & 3)) * TR_LD + 2 * j) = make_float2(v[i][0], v[i][1]);
            // same wave: LDS operations complete in order
#pragma unroll
            for (int i = 0; i < 2; ++i) {  // 16 rows x 8 runs of eight dimensions
                const int item = lane + 64 * i, row = item & 15, run = item >> 4, col = n0 + 8 * run;
                if (col < dm || col >= 2 * dm) continue;
                const float4 lo = *reinterpret_cast<const float4 *>(tr + row * TR_LD + 8 * run), hi = *reinterpret_cast<const float4 *>(tr + row * TR_LD + 8 * run + 4);
                const float a[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                const int e = col - dm, d = e & 63;
                store_kv_frags(o.kv.kfrag + base(e) + (size_t)((d >> 4) * 4 + ((d >> 3) & 1)) * 32 + 16 * s + row, 2 * 32, a, o.kv.k_up);
            }
        }
    }
}

// sum += v with what the addition rounds off collected in rest (Knuth's two-sum): a few partial sums meet here, and each would
// otherwise round at the size of the result.  Infinities stay what they are.
__device__ __forceinline__ void add_exactly(float &sum, float &rest, float v) {
    const float t = sum + v, z = t - sum, e = (sum - (t - z)) + (v - z);
    rest += fabsf(t) < INFINITY ? e : 0.0f;
    sum = t;
}

template <int N, class F>
__device__ __forceinline__ void static_for(F f) {
    if constexpr (N > 0) {
        static_for<N - 1>(f);
        f(std::integral_constant<int, N - 1>{});
    }
}

// Sums of 64 rows x `blocks` blocks of 32 columns on three bf16 pieces, as int4_gemm_bf16.hip forms them, for tiles with rows that are not for pairs: wave by
// wave a block of 32 x 32 at a time, operands straight from memory.  `sums` [64][32 blocks + 4] and `stats` [64] are LDS.  All waves of the workgroup.
// us with the pass in front, all rows for pairs / no tile / int4_gemm_bf16.hip: 1000 rows 1280 -> 3840 36 / 90 / 43; 2048 rows 1600 -> 4800 88 / 284 / 134; 1000
// rows 5120 -> 1280 53 / 166 / 75.
template <bool HANDED>
__device__ __forceinline__ void pair_general_sums(const PairGemmParams &p, int m0, int n0, int blocks, float *sums, float2 *stats, int waves, int wave, int lane) {
    const int c = lane & 31, h2 = lane >> 5, N = p.out.N, chunks = p.K / 32, ld = 32 * blocks + 4;
    if (!HANDED && p.gamma) {  // mean and variance in two passes, as pair_rows_kernel does it
#pragma unroll 1
        for (int r = wave; r < 64; r += waves) {
            const float *row = p.x + (size_t)min(m0 + r, p.out.M - 1) * p.K;
            float s = 0.0f, q = 0.0f;
            for (int k = lane; k < p.K; k += 64) s += row[k];
            const float mean = wave_sum(s) / (float)p.K;
            for (int k = lane; k < p.K; k += 64) q += (row[k] - mean) * (row[k] - mean);
            const float rstd = 1.0f / sqrtf(wave_sum(q) / (float)p.K + p.eps);
            if (lane == 0) stats[r] = make_float2(mean, rstd);
        }
        __syncthreads();
    }
#pragma unroll 1
    for (int b = wave; b < 2 * blocks; b += waves) {
        const int rb = b / blocks, cb = b - rb * blocks;
        const int n = min(n0 + 32 * cb + c, N - 1);
        const int m = min(m0 + 32 * rb + c, p.out.M - 1);
        const float *row = p.x + (size_t)m * p.K + 8 * h2, unit = p.factor / kPairWeightUnit;
        const float2 st = !HANDED && p.gamma ? stats[32 * rb + c] : make_float2(0.0f, 1.0f);
        floatx16 acc = {0};
        // what 32 k take, requested one turn ahead
        float4 x[2][2];  // (of rows that were handed on: lo and hi, or floats)
        uint32_t words[2];
        float scale;
        int mark = 0;
        auto request = [&](int ch) {
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                if (!HANDED) {
#pragma unroll
                    for (int e = 0; e < 2; ++e) x[s][e] = *reinterpret_cast<const float4 *>(row + 32 * ch + 16 * s + 4 * e);
                } else {
                    const int step = 2 * (ch & 1) + s;
                    mark = p.marks.marks[(size_t)(ch >> 1) * 32 * p.row_blocks + m];
                    const char *block = p.frags + ((size_t)(m >> 5) * p.k_blocks + (ch >> 1)) * kPairBlockBytes;
#pragma unroll
                    for (int e = 0; e < 2; ++e)
                        x[s][e] = *reinterpret_cast<const float4 *>(block + (mark ? pair_raw_offset(m & 31, 16 * step + 8 * h2 + 4 * e) : pair_offset(m & 31, step, e, h2)));
                }
                words[s] = p.packed[(size_t)(4 * ch + 2 * s + h2) * N + n];
            }
            scale = p.scales[(size_t)(ch >> p.chunk_shift) * N + n] * GB_NIBBLE_UNIT;
        };
        request(0);
#pragma unroll 1
        for (int ch = 0; ch < chunks; ++ch) {
            floatx16 gs = {0};
            bf16x8 a[2][3], w[2];
            const float sc = scale;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                const int k = 32 * ch + 16 * s + 8 * h2;
                float v[8] = {x[s][0].x, x[s][0].y, x[s][0].z, x[s][0].w, x[s][1].x, x[s][1].y, x[s][1].z, x[s][1].w};
                if (HANDED && !mark) {  // lo and hi, in the order of split_pair
                    const f16x8 lo = __builtin_bit_cast(f16x8, x[s][0]), hi = __builtin_bit_cast(f16x8, x[s][1]);
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[(e >> 1) + 4 * (e & 1)] = ((float)hi[e] + (float)lo[e]) * unit;
                }
                if (!HANDED && p.gamma) {
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = (v[e] - st.x) * st.y * p.gamma[k + e] + p.beta[k + e];
                }
                split_pieces(v, a[s]);
                w[s] = nibbles_to_bf16(words[s]);
            }
            request(min(ch + 1, chunks - 1));
#pragma unroll
            for (int piece = 0; piece < 3; ++piece)
#pragma unroll
                for (int s = 0; s < 2; ++s) gs = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s][piece], w[s], gs, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = fmaf(sc, gs[r], acc[r]);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) sums[(32 * rb + 8 * (r >> 2) + 4 * h2 + (r & 3)) * ld + 32 * cb + c] = acc[r];
    }
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

template <int WC, int KS, bool LONG, PairKind KIND>
__global__ __launch_bounds__(64 * WC * KS, 2) void int4_gemm_pairs_kernel(const PairGemmParams p) {
    using Tile = PairTile<WC, KS>;
    constexpr bool HANDED = KIND == PairKind::kHanded;
    extern __shared__ __align__(16) unsigned char pg_smem[];
    __shared__ int s_last;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)pg_smem;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 31, hh = lane >> 5;
    const int group = wave / WC, wc = wave - group * WC;
    // Workgroup b runs on XCD b % 8, each with an L2 of its own: an XCD takes a run of consecutive tiles (then of slices), and tiles are
    // numbered column by column within bands of four rows of tiles, so the 32 tiles at work in an XCD share rows and columns.
    const int full_grid = 8 * ((p.full_tiles + 7) / 8);
    int tile_no, split, ksplit, bps;
    if ((int)blockIdx.x < full_grid) {
        tile_no = ((int)blockIdx.x & 7) * (full_grid >> 3) + ((int)blockIdx.x >> 3);
        if (tile_no >= p.full_tiles) return;
        split = 0; ksplit = 1; bps = p.k_blocks;
    } else {
        const int items = p.n_tail * p.tail_ks, per = (items + 7) / 8, b = (int)blockIdx.x - full_grid;
        const int item = (b & 7) * per + (b >> 3);
        if ((b >> 3) >= per || item >= items) return;
        split = item / p.n_tail; tile_no = p.full_tiles + (item - split * p.n_tail); ksplit = p.tail_ks; bps = p.blocks_per_split;
    }
    const int band = tile_no / (4 * p.col_tiles), in_band = tile_no - band * 4 * p.col_tiles, band_rows = min(4, p.row_tiles - 4 * band);
    const int tile_col = in_band / band_rows, tile_row = 4 * band + (in_band - tile_col * band_rows);
    const int m0 = tile_row * Tile::BM, n0 = tile_col * Tile::BN + 64 * wc;
    const int kb0 = split * bps, kb1 = min(p.k_blocks, kb0 + bps);
    const int N = p.out.N, chunks = p.K / 32;

    // ---- what a wave brings of a K block, in requests of 1 KiB ----
    constexpr int REQUESTS = Tile::STAGE / 1024 / WC;
    static_assert(REQUESTS == 8, "one request beside each instruction, a row block per wave");
    const uint32_t lane_off = lane * 16;
    const uint32_t my_lds = lds0 + group * 2 * Tile::STAGE + wc * kPairBlockBytes;
    const char *const my_frags = p.frags + (size_t)min(2 * tile_row + wc, p.row_blocks - 1) * p.k_blocks * kPairBlockBytes;  // row blocks past the last repeat it
    auto request_pairs = [&](int kb, int buf, auto i) {
        constexpr int I = decltype(i)::value;
        pair_load_1k<(I & 3) * 1024>(my_lds + buf * Tile::STAGE + (I >> 2) * 4096, lane_off, my_frags + (size_t)kb * kPairBlockBytes + (I >> 2) * 4096);
    };
    auto request_all_pairs = [&](int kb, int buf) {
        static_for<REQUESTS>([&](auto i) { request_pairs(kb, buf, i); });
    };
    // ---- weight words and scales: buffer loads (scalar row, the lane's two columns; columns beyond the last repeat the last two) ----
    const uint32_t row_bytes = (uint32_t)N * 4u;
    const __amdgpu_buffer_rsrc_t words_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t *>(p.packed), 0, (uint32_t)(p.K / 8) * row_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t scales_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p.scales), 0, (uint32_t)(((chunks - 1) >> p.chunk_shift) + 1) * row_bytes, 0x00020000);
    const uint32_t soff = (uint32_t)min(n0 + 2 * j, N - 2) * 4u, woff = soff + (uint32_t)hh * row_bytes;
    u32x2 bw[4], bs[2];  // [16 k], [32 k]: words and scales of the next block
    auto request_words = [&](int kb, int st) {  // K % 64 == 32: the last block's second half does not exist (its pairs are zeros)
        bw[st] = __builtin_amdgcn_raw_buffer_load_b64(words_rsrc, woff, __builtin_amdgcn_readfirstlane((uint32_t)(8 * kb + (st < 2 || 2 * kb + 1 < chunks ? 2 * st : 2 * st - 4)) * row_bytes), 0);
    };
    auto request_scales = [&](int kb, int h) {
        bs[h] = __builtin_amdgcn_raw_buffer_load_b64(scales_rsrc, soff, __builtin_amdgcn_readfirstlane((uint32_t)((2 * kb + (2 * kb + 1 < chunks ? h : 0)) >> p.chunk_shift) * row_bytes), 0);
    };
    f16x8 b[2][4];       // [column][16 k]
    float sc[2][2];      // [column][32 k]
    auto take_scale = [&](int kb, int c, int h) {  // blocks beyond this group's last and halves beyond K count for nothing
        sc[c][h] = kb < kb1 && 2 * kb + h < chunks ? __uint_as_float(bs[h][c]) : 0.0f;
    };
    const unsigned char *const stage[2] = {pg_smem + group * 2 * Tile::STAGE + pair_offset(j, 0, 0, hh), pg_smem + group * 2 * Tile::STAGE + pair_offset(j, 0, 1, hh)};
    f16x8 a[4][2];       // one row block's [16 k][lo, hi]
    auto read_pair = [&](int buf, int rb, int st, int pc) {
        a[st][pc] = *reinterpret_cast<const f16x8 *>(stage[pc] + buf * Tile::STAGE + rb * kPairBlockBytes + st * 2048);
    };

    floatx16 acc[2][2], u[2][2];  // [row block][column], [unit parity][32 k]
    const floatx16 zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int rb = 0; rb < 2; ++rb)
#pragma unroll
        for (int c = 0; c < 2; ++c) acc[rb][c] = zero;
    u[1][0] = u[1][1] = zero;
    float last_sc[2] = {0.0f, 0.0f};  // of the unit before a block's first

    // what this wave asked for a block ago has arrived, then what every wave did; and every wave's reads of the block before are done
    auto block_barrier = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    // group g takes blocks kb0 + g, kb0 + g + KS, ...; all groups run the same number of turns, those past the last repeat a block
    int turns = (kb1 - kb0 + KS - 1) / KS;
    auto block_of = [&](int turn) { return kb0 + turn * KS + group; };
    auto source = [&](int turn) { return min(block_of(turn), kb1 - 1); };
    request_all_pairs(source(0), 0);
    bool general;  // the tile has rows that are not for pairs
    uint32_t row_flags = 0;
    if constexpr (HANDED) general = *(const __attribute__((address_space(4))) uint32_t *)(uintptr_t)(p.marks.tiles + tile_row) == p.marks.epoch;
    else if (m0 + lane < 32 * p.row_blocks) row_flags = reinterpret_cast<const uint32_t *>(p.factors + 32 * p.row_blocks)[m0 + lane];
#pragma unroll
    for (int st = 0; st < 4; ++st) request_words(source(0), st);
#pragma unroll
    for (int h = 0; h < 2; ++h) request_scales(source(0), h);
    block_barrier();
    if constexpr (!HANDED) general = __any(row_flags != 0);  // (every wave sees all 64)
    if (__builtin_expect(general, 0)) {
        // The tile's sums on three bf16 pieces, in place of those of the first slice and group; nothing comes from the others.  (Here and out of the
        // way of the others: behind the loop it cost every launch 0.3 us, in line 0.5 us.)
        constexpr int LD = Tile::BN + 4;
        static_assert((64 * LD + 2 * 64) * 4 <= Tile::LOOP_BYTES, "");
        float *sums = reinterpret_cast<float *>(pg_smem);
        if (split == 0) pair_general_sums<HANDED>(p, m0, tile_col * Tile::BN, Tile::BN / 32, sums, reinterpret_cast<float2 *>(sums + 64 * LD), WC * KS, wave, lane);
        __syncthreads();
        if (split == 0 && group == 0) {
            const int col = max(min(n0 + 2 * j, N - 2) - tile_col * Tile::BN, 0);  // (this lane's first column; waves beyond the last: any)
#pragma unroll
            for (int rb = 0; rb < 2; ++rb)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = 32 * rb + 8 * (r >> 2) + 4 * hh + (r & 3);
                    const float f = !HANDED ? p.factors[min(m0 + row, 32 * p.row_blocks - 1)] : p.factor, inv = f > 0.0f ? 1.0f / f : 0.0f;  // a power of two
#pragma unroll
                    for (int c = 0; c < 2; ++c) acc[rb][c][r] = sums[row * LD + min(col + c, Tile::BN - 1)] * inv;
                }
        }
        __syncthreads();
        turns = 0;
    }
    request_all_pairs(source(1), 1);
#pragma unroll
    for (int st = 0; st < 4; ++st) {
        read_pair(0, 0, st, 0);
        read_pair(0, 0, st, 1);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            b[c][st] = nibbles_to_f16(bw[st][c]);
            if (st < 2) take_scale(block_of(0), c, st);
        }
    }
#pragma unroll
    for (int st = 0; st < 4; ++st) request_words(source(1), st);
#pragma unroll
    for (int h = 0; h < 2; ++h) request_scales(source(1), h);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): nothing from before the loop is waited for inside it
    for (int turn = 0; turn < turns; ++turn) {
        const int buf = turn & 1, next = source(turn + 2);
#pragma unroll
        for (int unit = 0; unit < 4; ++unit) {  // unit = (row block, column)
            const int rb = unit >> 1, c = unit & 1, P = unit & 1, prb = ((unit + 3) & 3) >> 1, pc_ = c ^ 1;
            if (unit == 3) block_barrier();
            const float s0 = unit == 0 ? last_sc[0] : sc[pc_][0], s1 = unit == 0 ? last_sc[1] : sc[pc_][1];
            static_for<8>([&](auto slice) {
                constexpr int i = decltype(slice)::value, h = i & 1, st = 2 * h + ((i >> 1) & 1), pc = i >> 2;  // smallest pieces first
                u[P][h] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[st][pc], b[c][st], i < 2 ? zero : u[P][h], 0, 0, 0);
                // the operand's last use: the next row block's (the next block's) in its place
                if (c == 1) read_pair(rb == 0 ? buf : buf ^ 1, rb ^ 1, st, pc);
                // beside it: the unit before joins the accumulators, its first half first
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (LONG) {
                        if (q < 2) acc[prb][pc_][2 * i + q] += fmaf(s1, u[P ^ 1][1][2 * i + q], s0 * u[P ^ 1][0][2 * i + q]);
                    } else {
                        const int e = 4 * i + q, r = e & 15;
                        acc[prb][pc_][r] = fmaf(e < 16 ? s0 : s1, u[P ^ 1][e >> 4][r], acc[prb][pc_][r]);
                    }
                }
                if (unit == 3) {  // the other column's operands of this block have been used, this one's with this instruction
                    if constexpr (i < 4) {
                        b[0][i] = nibbles_to_f16(bw[i][0]);
                    } else {
                        b[1][st] = nibbles_to_f16(bw[st][1]);
                        request_words(next, st);
                    }
                    request_pairs(next, buf, slice);  // one by one: in a burst they stall the waves
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if (unit == 3) {
                last_sc[0] = sc[1][0];
                last_sc[1] = sc[1][1];
#pragma unroll
                for (int h = 0; h < 2; ++h) {
#pragma unroll
                    for (int cc = 0; cc < 2; ++cc) take_scale(block_of(turn + 1), cc, h);
                    request_scales(next, h);
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        if constexpr (LONG) acc[1][1][r] += fmaf(last_sc[1], u[1][1][r], last_sc[0] * u[1][0][r]);
        else acc[1][1][r] = fmaf(last_sc[1], u[1][1][r], fmaf(last_sc[0], u[1][0][r], acc[1][1][r]));
    }

    // ---- the groups' sums meet in LDS; group g finishes the registers g PER .. of every lane, in the order [row block][16][column] ----
    constexpr int PER = Tile::PER;
    float *red = reinterpret_cast<float *>(pg_smem);
    auto reg_of = [&](int i) { return acc[i >> 5][i & 1][(i >> 1) & 15]; };
    float fin[PER / 2][2];
    block_barrier();  // the requests past the end have landed, the last operands have been read
    // what the epilogue reads is requested now and arrives while the sums meet (columns beyond the last, rows past M: any)
    constexpr int HALVES = PER / 16;
    PairEarly early[HALVES];
    const int nb = min(n0 + 2 * j, N - 2);
    const Float2 bias2 = p.out.bias ? *reinterpret_cast<const Float2 *>(p.out.bias + nb) : Float2{0.0f, 0.0f};
    const int kv_pos = KIND == PairKind::kKv ? *p.out.kv.pos_dev : 0;
    auto half_row = [&](int half) { return m0 + 16 * (group * HALVES + half); };  // halves of row blocks in the order of the registers
#pragma unroll
    for (int half = 0; half < HALVES; ++half) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
            early[half].factor[q] = !HANDED ? *reinterpret_cast<const float4 *>(p.factors + min(half_row(half) + 8 * q + 4 * hh, 32 * p.row_blocks - 4))
                                              : make_float4(p.factor, p.factor, p.factor, p.factor);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int m = min(half_row(half) + 8 * (i >> 2) + 4 * hh + (i & 3), p.out.M - 1);
            early[half].res[i] = p.out.residual ? *reinterpret_cast<const Float2 *>(p.out.residual + (size_t)m * N + nb) : Float2{0.0f, 0.0f};
        }
    }
    {
        // [finishing group][contribution][wave of the group][register][lane]
        auto place = [&](int g, int slot) { return red + (size_t)(((g * (KS - 1) + slot) * WC + wc) * PER) * 64 + lane; };
#pragma unroll
        for (int g = 0; g < KS; ++g) {
            if (g == group) {
#pragma unroll
                for (int i = 0; i < PER; ++i) fin[i >> 1][i & 1] = reg_of(g * PER + i);
            } else {
                float *dst = place(g, group < g ? group : group - 1);
#pragma unroll
                for (int i = 0; i < PER; ++i) dst[i * 64] = reg_of(g * PER + i);
            }
        }
        __syncthreads();
        if constexpr (KS == 2) {
            const float *src = place(group, 0);
#pragma unroll
            for (int i = 0; i < PER; ++i) fin[i >> 1][i & 1] += src[i * 64];
        } else {
            float rest[PER / 2][2] = {};
#pragma unroll
            for (int s = 0; s < KS - 1; ++s) {
                const float *src = place(group, s);
#pragma unroll
                for (int i = 0; i < PER; ++i) add_exactly(fin[i >> 1][i & 1], rest[i >> 1][i & 1], src[i * 64]);
            }
#pragma unroll
            for (int i = 0; i < PER; ++i) fin[i >> 1][i & 1] += rest[i >> 1][i & 1];
        }
    }
    if (ksplit > 1) {
        // Partial sums in the order of the registers: [slice][tile][wave][pair of registers][lane] 8-byte words
        const int tile = tile_no - p.full_tiles;
        constexpr int kWaveWords = PER / 2 * 64;
        unsigned long long *mine = reinterpret_cast<unsigned long long *>(p.partial) + ((size_t)(split * p.n_tail + tile) * WC * KS + wave) * kWaveWords + lane;
#pragma unroll
        for (int q = 0; q < PER / 2; ++q) {
            const unsigned long long v = (unsigned long long)__float_as_uint(fin[q][0]) |
                                         ((unsigned long long)__float_as_uint(fin[q][1]) << 32);
            __hip_atomic_store(mine + q * 64, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        partials_published(p.strict);
        __syncthreads();
        if (tid == 0) {
            const unsigned int tk = take_ticket(&p.counters[tile], p.strict);
            s_last = (tk == (unsigned int)(ksplit - 1));
            if (s_last) __hip_atomic_store(&p.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (!s_last) return;
        const size_t slice_words = (size_t)p.n_tail * WC * KS * kWaveWords;
        const unsigned long long *first = mine - (size_t)split * slice_words;
        float rest[PER / 2][2] = {};
#pragma unroll
        for (int i = 0; i < PER; ++i) fin[i >> 1][i & 1] = 0.0f;
        for (int sp = 0; sp < ksplit; ++sp) {  // slice order: the same sum every run
            unsigned long long part[PER / 2];
#pragma unroll
            for (int q = 0; q < PER / 2; ++q) part[q] = __hip_atomic_load(first + (size_t)sp * slice_words + q * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int q = 0; q < PER / 2; ++q) {
                add_exactly(fin[q][0], rest[q][0], __uint_as_float((uint32_t)part[q]));
                add_exactly(fin[q][1], rest[q][1], __uint_as_float((uint32_t)(part[q] >> 32)));
            }
        }
#pragma unroll
        for (int i = 0; i < PER; ++i) fin[i >> 1][i & 1] += rest[i >> 1][i & 1];
    }
    if (n0 >= N) return;
    float *tr = red + Tile::RED_BYTES / 4 + wave * (Tile::TR_BYTES / 4);
    // the last column of an odd N is the second one of its lane (nb = N - 2)
    const float bias[2] = {bias2.x, bias2.y};
#pragma unroll
    for (int half = 0; half < HALVES; ++half) {  // eight registers x two columns
        float v[8][2];
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const float4 f = early[half].factor[q];
            const float fs[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < 2; ++c) v[4 * q + i][c] = fin[8 * half + 4 * q + i][c] * fs[i];
        }
        const int idx = group * HALVES + half;
        pair_finish_half<Tile::TR_LD, KIND>(p.out, v, bias, early[half], m0 + 32 * (idx >> 1), idx & 1, n0, j, hh, kv_pos, tr);
    }
}

// Rows (LN: normalised first) -> pairs.  A workgroup takes two rows, four waves; thread t holds of row (t / 2) % 2 the runs of eight k
// number 2 (t / 4) + t % 2, + 128, ..., so a store of four lanes is 128 consecutive bytes.  Mean and variance in two passes over the
// registers, as the LayerNorm kernels do it.
template <bool LN, int IT>
__global__ __launch_bounds__(256) void pair_rows_kernel(const float *__restrict__ x, const float *__restrict__ gamma, const float *__restrict__ beta,
                                                        float eps, char *__restrict__ frags, float *__restrict__ factors, int M, int K, int k_blocks) {
    __shared__ float s_part[3][4][2];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r = (tid >> 1) & 1, first = 2 * (tid >> 2) + (tid & 1), runs = K >> 3;
    const int row = 2 * (int)blockIdx.x + r;
    const bool row_ok = row < M;
    const float *src = x + (size_t)min(row, M - 1) * K;
    float v[IT][8];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int k = 8 * min(first + 128 * i, runs - 1);
        const float4 a = *reinterpret_cast<const float4 *>(src + k), b = *reinterpret_cast<const float4 *>(src + k + 4);
        v[i][0] = a.x; v[i][1] = a.y; v[i][2] = a.z; v[i][3] = a.w; v[i][4] = b.x; v[i][5] = b.y; v[i][6] = b.z; v[i][7] = b.w;
    }
    // over the lanes of a row among 16, then over the wave, then over the waves
    auto of_16 = [](float part, auto op) {
        part = op(part, dpp_move<0xb1, 0xf>(part, part));      // quad_perm [1,0,3,2]
        part = op(part, dpp_move<0x124, 0xf>(part, part));     // row_ror:4
        return op(part, dpp_move<0x128, 0xf>(part, part));     // row_ror:8
    };
    auto all = [&](float part, int slot, auto op) {
        part = of_16(part, op);
        part = op(part, __shfl_xor(part, 16, kWave));
        part = op(part, __shfl_xor(part, 32, kWave));
        if ((lane & ~2) == 0) s_part[slot][wave][r] = part;
        __syncthreads();
        return op(op(s_part[slot][0][r], s_part[slot][1][r]), op(s_part[slot][2][r], s_part[slot][3][r]));
    };
    auto add = [](float a, float b) { return a + b; };
    if constexpr (LN) {
        float s = 0.0f;
#pragma unroll
        for (int i = 0; i < IT; ++i)
            if (first + 128 * i < runs) s += ((v[i][0] + v[i][1]) + (v[i][2] + v[i][3])) + ((v[i][4] + v[i][5]) + (v[i][6] + v[i][7]));
        const float mean = all(s, 0, add) / (float)K;
        float q = 0.0f;
#pragma unroll
        for (int i = 0; i < IT; ++i)
            if (first + 128 * i < runs)
#pragma unroll
                for (int e = 0; e < 8; ++e) q += (v[i][e] - mean) * (v[i][e] - mean);
        const float rstd = 1.0f / sqrtf(all(q, 1, add) / (float)K + eps);
#pragma unroll
        for (int i = 0; i < IT; ++i) {
            const int k = 8 * min(first + 128 * i, runs - 1);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float4 g = *reinterpret_cast<const float4 *>(gamma + k + 4 * h), be = *reinterpret_cast<const float4 *>(beta + k + 4 * h);
                v[i][4 * h] = (v[i][4 * h] - mean) * rstd * g.x + be.x;
                v[i][4 * h + 1] = (v[i][4 * h + 1] - mean) * rstd * g.y + be.y;
                v[i][4 * h + 2] = (v[i][4 * h + 2] - mean) * rstd * g.z + be.z;
                v[i][4 * h + 3] = (v[i][4 * h + 3] - mean) * rstd * g.w + be.w;
            }
        }
    }
    float amax = 0.0f;  // runs beyond the last repeat it
#pragma unroll
    for (int i = 0; i < IT; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(v[i][e]));
    amax = all(amax, 2, [](float a, float b) { return fmaxf(a, b); });
    const int s = pair_exponent(amax);
    const float up = pow2f(s);
    char *base = frags + (size_t)(row >> 5) * k_blocks * kPairBlockBytes;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int run = first + 128 * i;
        if (run >= 8 * k_blocks) continue;
        uint4 lo = make_uint4(0, 0, 0, 0), hi = lo;
        if (run < runs && row_ok) split_pair(v[i], up, lo, hi);
        char *dst = base + (size_t)(run >> 3) * kPairBlockBytes;
        *reinterpret_cast<uint4 *>(dst + pair_offset(row & 31, (run >> 1) & 3, 0, run & 1)) = lo;
        *reinterpret_cast<uint4 *>(dst + pair_offset(row & 31, (run >> 1) & 3, 1, run & 1)) = hi;
    }
    if ((tid & ~2) == 0) factors[row] = row_ok ? pow2f(7 - s) : 0.0f;  // kPairWeightUnit / up
    // elements below kPairShort once scaled that are not zero (which goes round to the largest number)
    const uint32_t below = s < 124 ? ((uint32_t)(124 - s) << 24) - 1u : 0u;
    uint32_t few = 0;
#pragma unroll
    for (int i = 0; i < IT; ++i)
        if (first + 128 * i < runs)
#pragma unroll
            for (int e = 0; e < 8; ++e) few += 2u * __float_as_uint(v[i][e]) - 1u < below ? 1u : 0u;
    const uint64_t many = __ballot(of_16((float)few, add) > pair_short_allowed(K));
    if ((lane & ~2) == 0) reinterpret_cast<uint8_t *>(factors + 2 * gridDim.x)[4 * row + wave] = row_ok && (many & (r ? 0xccccccccccccccccull : 0x3333333333333333ull)) ? 1 : 0;
}

// A workgroup takes 64 columns of one Linear, its 16 waves the packed rows in turn, four of them requested at a time.
__global__ __launch_bounds__(1024) void pair_bound_kernel(const PairBoundBatch batch, int K, int N, int first, int count, int part_columns, int group, uint32_t *out, uint32_t *out2) {
    __shared__ float part[2][16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = (int)blockIdx.x * 64 + lane, n = first + min(c, count - 1), rows = K / 8;
    const uint32_t *packed = batch.packed[blockIdx.y] + n;
    const float *scales = batch.scales[blockIdx.y] + n, *gamma = batch.gamma[blockIdx.y], *beta = batch.beta[blockIdx.y], *bias = batch.bias[blockIdx.y];
    float sq = 0.0f, off = 0.0f;
    for (int kp0 = wave; kp0 < rows; kp0 += 64) {
        uint32_t w[4];
        float sc[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kp = min(kp0 + 16 * u, rows - 1);
            w[u] = packed[(size_t)kp * N];
            sc[u] = kp0 + 16 * u < rows ? scales[(size_t)(8 * kp / group) * N] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int kp = min(kp0 + 16 * u, rows - 1);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float q = (float)((int)((w[u] >> (4 * i)) & 15u) - 8) * sc[u], g = gamma[8 * kp + i] * q;
                sq = fmaf(g, g, sq);
                off = fmaf(beta[8 * kp + i], q, off);
            }
        }
    }
    part[0][wave][lane] = sq;
    part[1][wave][lane] = off;
    __syncthreads();
    if (wave > 0) return;
    float s2 = 0.0f, t = 0.0f;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        s2 += part[0][w][lane];
        t += part[1][w][lane];
    }
    const float bound = c < count ? 1.001f * (sqrtf((float)K * s2) + fabsf(t + (bias ? bias[n] : 0.0f))) : 0.0f;
    const float largest = wave_max(bound != bound ? INFINITY : bound);
    const float smallest = -wave_max(bound > 0.0f ? -bound : -INFINITY);
    if (lane == 0) {  // bits of floats that are not negative are ordered like the floats
        uint32_t *o = ((int)blockIdx.x * 64 < part_columns ? out : out2) + 2 * blockIdx.y;
        atomicMax(o, __float_as_uint(largest));
        if (smallest < INFINITY) atomicMax(o + 1, ~__float_as_uint(smallest));
    }
}

}  // namespace

int32_t agpu_pair_bound_launch(agpu_ctx *ctx, const PairBoundBatch &batch, int n, int K, int N, int first, int count, int part, int group, uint32_t *out, uint32_t *out2) {
    hipLaunchKernelGGL(pair_bound_kernel, dim3((unsigned)ceil_div(count, 64), (unsigned)n), dim3(1024), 0, ctx->stream, batch, K, N, first, count, part, group, out, out2);
    return AGPU_LAUNCH_CHECK(ctx, "pair_bound_kernel");
}

template <int WC, int KS, bool LONG, PairKind KIND>
static int32_t pairs_launch(agpu_ctx *ctx, PairGemmParams &p, int full_tiles, int tail_ks, size_t scratch_bytes) {
    using Tile = PairTile<WC, KS>;
    p.row_tiles = ceil_div(p.out.M, Tile::BM);
    p.col_tiles = ceil_div(p.out.N, Tile::BN);
    const int tiles = p.row_tiles * p.col_tiles;
    p.full_tiles = std::min(full_tiles, tiles);
    p.n_tail = tiles - p.full_tiles;
    // partial sums fit the scratch and tickets are there for all sliced tiles, or nothing is sliced
    while (tail_ks > 1 && ((size_t)tail_ks * p.n_tail * Tile::BM * Tile::BN * sizeof(float) > scratch_bytes || p.n_tail > ctx->n_counters)) --tail_ks;
    p.blocks_per_split = ceil_div(p.k_blocks, tail_ks);
    p.tail_ks = ceil_div(p.k_blocks, p.blocks_per_split);
    if (p.tail_ks == 1) {
        p.full_tiles = tiles;
        p.n_tail = 0;
    }
    const unsigned grid = 8u * (unsigned)ceil_div(p.full_tiles, 8) + 8u * (unsigned)ceil_div(p.n_tail * p.tail_ks, 8);
    static std::atomic<unsigned long long> lds_raised{0};  // one bit per device
    const unsigned long long bit = 1ull << (ctx->device & 63);
    if (!(lds_raised.load(std::memory_order_relaxed) & bit)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(int4_gemm_pairs_kernel<WC, KS, LONG, KIND>), hipFuncAttributeMaxDynamicSharedMemorySize, Tile::LDS);
        if (e != hipSuccess) return agpu_hip(ctx, e, "hipFuncSetAttribute");
        lds_raised.fetch_or(bit, std::memory_order_relaxed);
    }
    hipLaunchKernelGGL((int4_gemm_pairs_kernel<WC, KS, LONG, KIND>), dim3(grid), dim3(Tile::T), Tile::LDS, ctx->stream, p);
    return AGPU_LAUNCH_CHECK(ctx, "int4_gemm_pairs_kernel");
}

template <int WC, int KS, bool LONG>
static int32_t pairs_go(agpu_ctx *ctx, PairGemmParams &p, int full_tiles, int tail_ks, size_t scratch_bytes) {
    if (!p.factors) return pairs_launch<WC, KS, LONG, PairKind::kHanded>(ctx, p, full_tiles, tail_ks, scratch_bytes);
    if (p.out.pairs) return pairs_launch<WC, KS, LONG, PairKind::kHandOn>(ctx, p, full_tiles, tail_ks, scratch_bytes);
    if (p.out.kv.kcache) return pairs_launch<WC, KS, LONG, PairKind::kKv>(ctx, p, full_tiles, tail_ks, scratch_bytes);
    return pairs_launch<WC, KS, LONG, PairKind::kPlain>(ctx, p, full_tiles, tail_ks, scratch_bytes);
}

template <bool LN, int IT>
static void pair_rows_go(agpu_ctx *ctx, const float *x, const float *gamma, const float *beta, float eps, int M, int K, void *pairs) {
    const PairLayout l(M, K);
    char *frags = static_cast<char *>(pairs);
    hipLaunchKernelGGL((pair_rows_kernel<LN, IT>), dim3(16u * (unsigned)l.row_blocks), dim3(256), 0, ctx->stream, x, gamma, beta, eps, frags,
                       reinterpret_cast<float *>(frags + l.frag_bytes()), M, K, l.k_blocks);
}
template <bool LN>
static void pair_rows_pick(agpu_ctx *ctx, const float *x, const float *gamma, const float *beta, float eps, int M, int K, void *pairs) {
    if (K <= 1024) pair_rows_go<LN, 1>(ctx, x, gamma, beta, eps, M, K, pairs);
    else if (K <= 1024 * 2) pair_rows_go<LN, 2>(ctx, x, gamma, beta, eps, M, K, pairs);
    else if (K <= 1024 * 4) pair_rows_go<LN, 4>(ctx, x, gamma, beta, eps, M, K, pairs);
    else pair_rows_go<LN, 8>(ctx, x, gamma, beta, eps, M, K, pairs);
}

int32_t agpu_pair_rows_launch(agpu_ctx *ctx, const float *x, const float *gamma, const float *beta, float eps, int M, int K, void *pairs) {
    if (gamma) pair_rows_pick<true>(ctx, x, gamma, beta, eps, M, K, pairs);
    else pair_rows_pick<false>(ctx, x, gamma, beta, eps, M, K, pairs);
    return AGPU_LAUNCH_CHECK(ctx, "pair_rows_kernel");
}

// Tiles of 64 x 128 against the kernels on three bf16 pieces (us per launch, theirs / this one, without the pass in front).  K below
// 2048: 333 rows 768 -> 3072 (144 tiles) 12.6 / 11.5, 1000 rows 1280 -> 1280 (160) 20.3 / 14.5, 256 rows 1280 -> 3840 (120) 16.1 / 14.3;
// but 333 rows 768 -> 2304 (108) 11.5 / 11.3, 512 rows 1280 -> 1280 (80) 13.1 / 14.1.  A second tile for some CUs changes nothing: 768 -> 3072
// under the profiler 640 rows (240 tiles) 17.9 / 15.8, 704 (264) 22.0 / 19.6, 768 (288) 21.8 / 19.8, 960 (360) 22.2 / 19.5, 1280 (480) 28.2 / 21.2.  Longer K, by K blocks over all tiles: 256 rows 5120 -> 1280 (3200) 22.3 / 20.5, 333 rows 4096 -> 1024 (3072)
// 20.9 / 19.2, 768 rows 3072 -> 768 (3456) 22.8 / 18.9; 512 rows 3072 -> 768 (2304) 16.2 / 17.6.  Up: 1000 rows 1280 -> 3840 41.0 / 27.2,
// 2048 rows 1600 -> 4800 107 / 72, 4096 rows 196 / 140.  With K below 768 it gains little, and the split of x to 23 bits would show
// (fewer roundings of the sum stand against it).
// Rows that need a pass of their own (3.3 us + 2.2 us per million elements: 1000 x 1280 5.7, 2048 x 1600 9.5, 1000 x 5120 11.5) have to make up for
// it.  K below 2048: the estimated time of pass and GEMM against one of the other kernels', which their sizes give within 10 %; what decides besides
// the size is how the tiles fill their rounds (1024 -> 3072, us in a graph: 768 rows, 288 tiles, 21.7 on three pieces and 26.2 on pairs, 1280 rows,
// 480 tiles, 37.6 and 31.5).  Longer K: the GEMM saves about 0.3 us per 1.3e8 products, from 3072 on 0.4 with 6500 K blocks or more (512 rows
// 5120 -> 1280 29.9 / 34.6 us; 640 rows 36.4 / 34.6).  Over 533 Linears of 64 to 2048 rows (K 768 to 6400, N 64 to 6400) that is 0.960 of the time on three
// pieces, with the best of both 0.957; six are 3 to 9 % slower on it than on three pieces.
namespace {
// Two groups of waves a tile (two workgroups a CU) or four (one), in us: K blocks in turn, a turn 1.15 - 2.0 (1.5 - 2.0) as the chip
// fills and its clock comes down, about 4 for a tile's start and end.  Tiles beyond whole rounds of one per CU are sliced along K
// where that is long (320 tiles of 5120 -> 1280: 66.6 against 70.7 unsliced with two groups; 120 tiles 29.7 against 37.5).
struct PairPlan {
    float us2, us4;
    int tiles, rest4, ks;  // with four groups: all tiles, those beyond whole rounds, their slices
    PairPlan(int cus, int M, int N, int K) {
        tiles = ceil_div(M, 64) * ceil_div(N, 128);
        const int k_blocks = ceil_div(K, kPairBlockK), turns2 = ceil_div(k_blocks, 2), turns4 = ceil_div(k_blocks, 4);
        const int rest2 = tiles % (2 * cus);
        rest4 = tiles % cus;
        us2 = (float)(tiles / (2 * cus)) * (2.0f * turns2 + 4.0f);
        if (rest2 > 0) us2 += (rest2 <= cus ? 1.15f : 1.15f + 0.85f * std::sqrt((float)(rest2 - cus) / cus)) * turns2 + 4.0f;
        ks = rest4 > 0 && turns4 >= 8 ? std::min(4, cus / rest4) : 1;
        const float fill = (float)(rest4 * ks) / cus;
        us4 = (float)(tiles / cus) * (2.0f * turns4 + 4.0f);
        if (rest4 > 0) us4 += (1.5f + 0.5f * fill * fill) * ceil_div(turns4, ks) + 4.0f + (ks > 1 ? 2.0f + 0.5f * ks : 0.0f);
    }
    bool four() const { return us4 <= us2; }
};
}  // namespace

bool agpu_int4_gemm_pairs_wanted(const agpu_ctx *ctx, int M, int N, int K, int group, bool pass) {
    if (M <= 16 || N < 2 || K < 768 || K > kPairMaxK || K % 32 != 0 || group % 32 != 0 || ((group / 32) & (group / 32 - 1)) != 0) return false;
    if ((size_t)(K / 8) * N * 4 >= size_t(1) << 31) return false;  // offsets in the matrix are 32 bits
    const long long tiles = (long long)ceil_div(M, 64) * ceil_div(N, 128), cus = ctx->num_cus;
    if (K >= 2048 ? tiles * ceil_div(K, kPairBlockK) < 3000 : tiles < 116) return false;
    if (!pass) return true;
    const double products = (double)M * N * K, elements = (double)M * K;
    if (K >= 3072 && tiles * ceil_div(K, kPairBlockK) < 6500) return false;
    if (K >= 2048) return (K >= 3072 ? 0.4 : 0.3) * products / 1.3e8 >= 1.1 * (3.3 + 2.2e-6 * elements);
    const PairPlan plan((int)cus, M, N, K);
    return (plan.four() ? 0.95 * plan.us4 + 5.5 : 0.85 * plan.us2 + 9.0) + 2.3e-6 * elements < 5.0 + 7e-9 * products;
}

int32_t agpu_int4_gemm_pairs_launch(agpu_ctx *ctx, const PairIn &in, const uint32_t *packed, const float *scales, const GemmOut &out, int K, int group,
                                    void *scratch, size_t scratch_bytes) {
    const PairLayout l(out.M, K);
    PairGemmParams p{};
    p.frags = static_cast<const char *>(in.pairs);
    p.factors = in.up == 0.0f ? reinterpret_cast<const float *>(p.frags + l.frag_bytes()) : nullptr;
    p.factor = in.up == 0.0f ? 0.0f : kPairWeightUnit / in.up;
    p.marks = in.marks;
    p.x = in.x; p.gamma = in.gamma; p.beta = in.beta; p.eps = in.eps;
    p.packed = packed; p.scales = scales; p.out = out; p.K = K; p.chunk_shift = __builtin_ctz((unsigned)(group / 32));
    p.row_blocks = l.row_blocks; p.k_blocks = l.k_blocks;
    p.partial = static_cast<float *>(scratch);
    p.counters = ctx->counters;
    p.strict = ctx->strict_sync;
    const PairPlan plan(ctx->num_cus, out.M, out.N, K);
    if (K >= 3072) {  // a rounding of the sum per 64 k instead of one per 32: 2.0e-7 -> 1.7e-7 (K = 6400, two groups), 8 % of the time
        if (plan.four()) return pairs_go<2, 4, true>(ctx, p, plan.tiles - plan.rest4, plan.ks, scratch_bytes);
        return pairs_go<2, 2, true>(ctx, p, plan.tiles, 1, scratch_bytes);
    }
    if (plan.four()) return pairs_go<2, 4, false>(ctx, p, plan.tiles - plan.rest4, plan.ks, scratch_bytes);
    return pairs_go<2, 2, false>(ctx, p, plan.tiles, 1, scratch_bytes);
}
