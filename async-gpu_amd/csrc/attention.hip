// Causal attention for gfx950, d_head = 64, fp32.
//   * attn_rows_kernel: prefill / chunked prefill.  One wave per 32 query rows; S^T = K Q^T and
//     O^T = V^T P^T on v_mfma_f32_32x32x16_f16 with every operand as the sum of two f16 numbers, online softmax; K/V tiles of 32 keys.
//     Blocks whose operands are not fit for that: on v_mfma_f32_32x32x2_f32 (AttWave::exact_tiles), here and in attn_f16_kernel.
//   * attn_tile_kernel: the same for at most 32 queries and keys, in fp32.
//   * attn_f16_kernel: the same for prompts of 256 queries or more at position 0; K and V come as operand fragments (written by
//     split_kv_kernel here or by the Linear that produces them).
//   * attn_decode_kernel: decode (few query rows).  One workgroup per (head, query row); its waves
//     split the keys, 16 lanes share one key (float4 each), partial (m, l, o) merge in a fixed order.
#include "agpu_internal.h"
#include "attention.h"
#include "gemm_pairs.h"

#include <algorithm>
#include <type_traits>

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int DH = 64;
constexpr int KLD = 68;  // K tile row stride in floats: 8 consecutive lanes' b128 reads hit distinct banks

__device__ __forceinline__ void resolve_positions(const AttnParams &p, int &kv_len, int &q_offset) {
    kv_len = p.kv_len;
    q_offset = p.q_offset;
    if (p.pos_dev) {
        const int pos = *p.pos_dev;
        kv_len = pos + p.q_len;
        q_offset = pos;
    }
}

constexpr int ATT_TILE_FLOATS = 32 * KLD;  // per wave: the K tile (padded rows), then the V tile, at the end the partial result, in the same place
// exp of the prefill kernel: v_exp_f32 on x * log2(e), relative error about 2^-22 at the arguments that matter
// (the reference kernels use ex2.approx the same way, compute_transformer.rs:837-1065); 13 % of the kernel's time
// against the correctly rounded expf, which the decode kernel keeps.
#define ATT_EXP __expf

// Where a wave leaves the 64 outputs of a (query, head), lane = output dimension: a row of o, or pairs.  All of it is the same for the
// whole workgroup.
struct AttRows {
    float *o;  // the head's columns of row 0
    long long row_stride;
    __device__ __forceinline__ AttRows(const AttnParams &p, int b, int h)
        : o(p.o + (size_t)b * p.o_batch_stride + (size_t)h * p.o_head_stride), row_stride(p.o_row_stride) {}
    // rows i, i + STEP, ... of the sequence, those below `end`: v[n][lane]
    template <int N, int STEP>
    __device__ __forceinline__ void store(int i, int end, int lane, const float (&v)[N]) const {
#pragma unroll
        for (int n = 0; n < N; ++n)
            if (i + STEP * n < end) (o + (size_t)(i + STEP * n) * row_stride)[lane] = v[n];
    }
};
// Either.  (Handed to merge_partials in registers: more than 16, with its other arguments, and it would go over memory.)
struct AttOut {
    char *to;         // the head's columns of row 0, or its K block of row block 0
    long long where;  // row stride, or the head's marks
    uint32_t *tiles, epoch;
    float up;         // 0: a row of o
    int row0, k_blocks;  // the sequence's first row, K blocks of a row
    __device__ __forceinline__ AttOut(const AttnParams &p, int b, int h)
        : to(p.pairs ? p.pairs + (size_t)h * kPairBlockBytes : reinterpret_cast<char *>(p.o + (size_t)b * p.o_batch_stride + (size_t)h * p.o_head_stride)),
          where(p.pairs ? (long long)(p.pair_marks + (size_t)h * 32 * ((p.batch * p.q_len + 31) >> 5)) : p.o_row_stride), tiles(p.pair_tiles), epoch(p.epoch),
          up(p.pairs ? p.pairs_up : 0.0f), row0(b * p.q_len), k_blocks(p.n_heads) {}
    template <int N, int STEP>
    __device__ __forceinline__ void store(int i, int end, int lane, const float (&v)[N]) const {
        if (up == 0.0f) {
#pragma unroll
            for (int n = 0; n < N; ++n)
                if (i + STEP * n < end) (reinterpret_cast<float *>(to) + (size_t)(i + STEP * n) * where)[lane] = v[n];
            return;
        }
        // which rows are for floats (pair_raw); looked at together, because a branch a row is 1.4 us of 21 (20 heads of 1000)
        const float full = 1.0f / up;
        unsigned raw = 0;
#pragma unroll
        for (int n = 0; n < N; ++n) raw |= (__any(!(fabsf(v[n]) < full)) || !__any(v[n] != 0.0f) ? 0u : 1u) << n;
        if (__builtin_expect(raw == 0, 1)) {
#pragma unroll
            for (int n = 0; n < N; ++n)
                if (i + STEP * n < end) store_pair_element(to, k_blocks, row0 + i + STEP * n, lane, v[n] * up);
        } else {
#pragma unroll 1
            for (int n = 0; n < N; ++n) {
                const int row = row0 + i + STEP * n;
                if (i + STEP * n >= end) break;
                float x = v[0];
#pragma unroll
                for (int k = 1; k < N; ++k) x = n == k ? v[k] : x;
                if (raw >> n & 1) {
                    *reinterpret_cast<float *>(to + (size_t)(row >> 5) * k_blocks * kPairBlockBytes + pair_raw_offset(row & 31, lane)) = x;
                    if (lane == 0) tiles[row >> 6] = epoch;
                } else {
                    store_pair_element(to, k_blocks, row, lane, x * up);
                }
            }
        }
        if (lane < N && i + STEP * lane < end) reinterpret_cast<uint8_t *>(where)[row0 + i + STEP * lane] = raw >> lane & 1;
    }
};

// Sum of the S waves' partial results of one query block: O^T (64 x 32) at o[w], at the place att_place says, m and l per query at
// ml[w].  Lane = output dimension, so that a wave stores whole rows; wave w
// takes queries w, w + S, ...  Lane x first works out the weight exp(m_v - m) / l of partial v = x % S for the wave's query number
// x / S; the sums then take the weights from those lanes.  S is a constant here so that no read waits for another.
__device__ __forceinline__ int att_place(int d, int query) { return d * 32 + (query ^ (d & 31)); }  // neither rows nor columns meet in a bank
template <int S, bool TOGETHER = true, class Out>
__device__ __forceinline__ void merge_partials_at(const float *const (&o)[S], const float *const (&ml)[S], unsigned parts, int lane, int wave,
                                                  int i0, int q_len, const Out &out) {
    constexpr int NQ = (32 + S - 1) / S;
    float wgt;
    {
        const int qc = min(wave + S * (lane / S), 31), v = lane % S;
        float mv[S], lv[S], m_all = -INFINITY, l_all = 0.0f, mine = 0.0f;
#pragma unroll
        for (int w = 0; w < S; ++w) {
            mv[w] = ml[w][qc];
            lv[w] = ml[w][32 + qc];
            if (!(parts >> w & 1)) mv[w] = -INFINITY;  // weight 0
        }
#pragma unroll
        for (int w = 0; w < S; ++w) m_all = fmaxf(m_all, mv[w]);
#pragma unroll
        for (int w = 0; w < S; ++w) {
            const float f = mv[w] == -INFINITY ? 0.0f : ATT_EXP(mv[w] - m_all);
            l_all += lv[w] * f;
            mine = w == v ? f : mine;
        }
        wgt = mine / l_all;
    }
    float rows[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int qc = wave + S * i;
        float acc = 0.0f;
#pragma unroll
        for (int w = 0; w < S; ++w) {
            const float part = o[w][att_place(lane, min(qc, 31))] * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wgt), i * S + w));
            acc += parts >> w & 1 ? part : 0.0f;  // (what stands in for a missing one may be infinite)
        }
        rows[i] = acc;
        if (!TOGETHER) {  // (a function of its own has registers for one at a time)
            const float row[1] = {acc};
            out.template store<1, S>(i0 + qc, min(i0 + 32, q_len), lane, row);
        }
    }
    if (TOGETHER) out.template store<NQ, S>(i0 + wave, min(i0 + 32, q_len), lane, rows);
}

template <int S, class Out>
__device__ __noinline__ void merge_partials(const float *att_smem, int lane, int wave, int i0, int q_len, const Out out) {
    const float *o[S], *ml[S];
#pragma unroll
    for (int w = 0; w < S; ++w) {
        o[w] = att_smem + w * ATT_TILE_FLOATS;
        ml[w] = o[w] + 64 * 32;
    }
    merge_partials_at<S, false>(o, ml, (1u << S) - 1, lane, wave, i0, q_len, out);
}

// ---- prefill attention on the f16 matrix cores, at fp32 accuracy ----
// A number times a power of two that brings the largest of its kind (a tile's K, a tile's V, a query) to 2^14 .. 2^15 is the
// sum of two f16 numbers, hi and lo, up to 2^-24 of
// itself (smaller ones, below 2^-17 of the largest, up to 2^-41 of the largest), so a product is hi hi + hi lo + lo hi up to 2^-22 of itself (the
// lo lo left out; 2^-24.6 rms);
// S^T = K Q^T and O^T = V^T P^T take 3 v_mfma_f32_32x32x16_f16 per 16 terms of the sum (8 passes each) where fp32 operands take 8
// v_mfma_f32_32x32x2_f32 (16 passes each), and three exact bf16 pieces, six of the 16-bit kind.  Half the instructions of those pieces
// also are half the roundings of a running sum, and the terms with lo in them are added up first: 25 heads of 2048 random queries, keys
// and values are off by 1.8e-7 (rms, of the results') against 3.1e-7 with bf16 pieces, 12 of 1024 by 1.6e-7 against 2.1e-7.  The operands come as
// fragments, 16 bytes per lane and instruction, pieces 0 = hi, 1 = lo:
//   K: [head][tile of 32 keys][d step ds of 16][piece][half hh][key i]     8 f16: d = 16 ds + 8 hh + e
//   V: [head][tile][d block of 32][piece][key step s][half hh][d i]         8 f16: key = att_vkey(s, hh, e)
// written once per prefill (by split_kv_kernel, or by the GEMM that produces K and V), read with one 1 KiB request per wave and
// instruction.  att_vkey is the order in which a 32 x 32 MFMA result holds its rows: the probabilities of a key tile
// come out of the first product in exactly the layout the second one wants.
constexpr int ATT_FRAGS_PER_TILE = kKvFragsPerTile;  // uint4 per (head, tile), the same for K and for V

__device__ __forceinline__ int att_vkey(int s, int hh, int e) { return 16 * s + 8 * (e >> 2) + 4 * hh + (e & 3); }

// the sum, or the larger, of the two halves of a wave
__device__ __forceinline__ float att_other_half(float v, float &own) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    own = __uint_as_float(r[0]);
    return __uint_as_float(r[1]);
}
__device__ __forceinline__ float att_max_halves(float v) {
    float own;
    const float other = att_other_half(v, own);
    return fmaxf(own, other);
}
__device__ __forceinline__ float att_sum_halves(float v) {
    float own;
    const float other = att_other_half(v, own);
    return own + other;
}

// Operands that pairs do not do justice to, from the exponents that their largest values get (an infinity's: kExpOfInf).
// Scores: what is left out of the elements of q and k below 2^-17 of the largest comes to 2^-(exponent of q + exponent of k + 6) of a score at most,
// which is to stay below what the exponential is off by: 2^-22.  An infinity may still be a weight of zero.
constexpr int kExpOfInf = 141 - 255;
constexpr int kLeastScoreExp = 16;

// Values: an element below 2^-17 of its tile's largest is off by up to 2^-41 of that one, and a weight below 2^-11 by 2^-34.  That is to stay
// below 2^-24 of what a result is made of, dimension by dimension.  So it is fp32 operands
// * where in one of the four runs of eight keys that a tile's lanes hold (att_vkey) a dimension has nothing as large as 2^-kColumnSpread of the tile's
//   largest (random numbers: 10^-14 a run): small dimensions, keys far out, and dimensions that are zero but for a few keys, whose results may be as
//   small as the weights of those (a one-hot V reads them off).  Of a tile of less than 16 keys, whose runs are no runs, the dimension as a whole, with
//   kFewSpread;
// * where a dimension is all zeros in some tiles only, and where tiles are further apart than AttWave::kSpread;
// * where a query sees only a part of a tile and a key's V is below 2^-kRowSpread of the largest.
constexpr int kColumnSpread = 8, kFewSpread = 16, kRowSpread = 14;
// A dimension of a tile of `keys` keys against the tile's largest; most: its largest |v|, least: the smallest of its runs' largest
__device__ __forceinline__ bool att_uneven(float most, float least, float all, int keys) {
    return most > 0.0f && (keys >= 16 ? least < all * pow2f(-kColumnSpread) : most < all * pow2f(-kFewSpread));
}
// The largest |v| of a key, of which this lane has 32 dimensions at `half` and the other half wave the rest (in turn c, so that 32 rows of 256
// bytes meet in no bank)
__device__ __forceinline__ float att_key_most(const float *half, int c) {
    float most = 0.0f;
#pragma unroll 4
    for (int i = 0; i < 8; ++i) {
        const float4 v = *reinterpret_cast<const float4 *>(half + 4 * ((i + c) & 7));
        most = fmaxf(most, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
    }
    return att_max_halves(most);
}

// K and V rows [head][kv_stride][64] -> fragments of the tiles 0 .. gridDim.x - 1 and, per tile, the exponents of K and of V (kExpOfInf: not for
// pairs) and which dimensions of V are not all zeros; rows from kv_len on count as zeros.  grid (tiles, heads), 256 threads.
__global__ __launch_bounds__(256) void split_kv_kernel(const float *k, const float *v, uint4 *kfrag, uint4 *vfrag, int4 *exps, int kv_len, int kv_stride, int tiles_cap) {
    __shared__ float largest[4], column[2][4][64];
    const int t = threadIdx.x, tile = blockIdx.x, hb = blockIdx.y, wave = t >> 6, lane = t & 63;
    const int i = t & 31, hh = (t >> 5) & 1, last = kv_len - 1;
    // every request first (rows past the end read another one of the tile and count as zeros), then the arithmetic
    const int ds = t >> 6, key = tile * 32 + i;
    const float *ksrc = k + ((size_t)hb * kv_stride + min(key, last)) * DH + 16 * ds + 8 * hh, *vsrc = v + (size_t)hb * kv_stride * DH;
    const float4 klo = *reinterpret_cast<const float4 *>(ksrc), khi = *reinterpret_cast<const float4 *>(ksrc + 4);
    const int s = (t >> 6) & 1, dblk = t >> 7, d = 32 * dblk + i;
    float xv[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int j = tile * 32 + att_vkey(s, hh, e);
        xv[e] = vsrc[(size_t)(j <= last ? j : last - tile * 32 >= 15 ? j - 16 : last) * DH + d];  // (so that a run of eight is one of eight keys, where there are 16)
    }
    const bool ok = key < kv_len;
    const float xk[8] = {ok ? klo.x : 0.f, ok ? klo.y : 0.f, ok ? klo.z : 0.f, ok ? klo.w : 0.f, ok ? khi.x : 0.f, ok ? khi.y : 0.f, ok ? khi.z : 0.f, ok ? khi.w : 0.f};
    float mk = 0.0f, mv = 0.0f, lv = INFINITY;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        mk = fmaxf(mk, fabsf(xk[e]));
        mv = fmaxf(mv, fabsf(xv[e]));
        lv = fminf(lv, fabsf(xv[e]));
        xv[e] = tile * 32 + att_vkey(s, hh, e) < kv_len ? xv[e] : 0.0f;
    }
    column[0][2 * s + hh][d] = mv;
    column[1][2 * s + hh][d] = lv;
    mk = wave_max(mk);
    if (lane == 0) largest[wave] = mk;
    __syncthreads();
    const int ek = min(pair_exponent(fmaxf(fmaxf(largest[0], largest[1]), fmaxf(largest[2], largest[3]))), kMaxFragExpK);
    // lane = dimension, every wave the same
    const float most = fmaxf(fmaxf(column[0][0][lane], column[0][1][lane]), fmaxf(column[0][2][lane], column[0][3][lane]));
    const float least = fminf(fminf(column[0][0][lane], column[0][1][lane]), fminf(column[0][2][lane], column[0][3][lane]));
    const float smallest = fminf(fminf(column[1][0][lane], column[1][1][lane]), fminf(column[1][2][lane], column[1][3][lane]));
    const float all = wave_max(most);
    const int ev = min(pair_exponent(all), kMaxFragExpV);
    const size_t at = (size_t)hb * tiles_cap + tile;
    if (wave == 0) {
        bool uneven = __any(att_uneven(most, least, all, kv_len - tile * 32));
        if (!uneven && __any(most > 0.0f && smallest < all * 0x1p-16f)) uneven = __any(att_key_most(vsrc + (size_t)min(key, last) * DH + 32 * hh, 0) < all * pow2f(-kRowSpread));
        const uint64_t some = __ballot(most > 0.0f);
        if (lane == 0) exps[at] = make_int4(ek, uneven ? kExpOfInf : ev, (int)(uint32_t)some, (int)(uint32_t)(some >> 32));
    }
    store_kv_frags(kfrag + at * ATT_FRAGS_PER_TILE + (ds * 4 + hh) * 32 + i, 2 * 32, xk, pow2f(ek));
    store_kv_frags(vfrag + at * ATT_FRAGS_PER_TILE + ((dblk * 4 + s) * 2 + hh) * 32 + i, 2 * 2 * 32, xv, pow2f(ev));
}

constexpr int ATT_TILE_BYTES = ATT_FRAGS_PER_TILE * 16;  // the fragments of one key tile of K, or of V
constexpr int ATT_PART_BYTES = 64 * 32 * 4;              // O^T of one query block
constexpr int ATT_QUERY_BYTES = 4 * 2 * 64 * 16;         // the fragments of a block's queries: [d step][piece][lane]
// a tile of K and one of V of every wave (over them, at the end, its partial results), the queries (over them all m and l)
constexpr size_t att_rows_lds(int waves) { return waves * ATT_TILE_FLOATS * sizeof(float) + ATT_QUERY_BYTES + 32 * sizeof(int) + waves * sizeof(int); }
constexpr int att_lds(int blocks, int waves) { return waves * 2 * ATT_TILE_BYTES + blocks * ATT_QUERY_BYTES; }
static_assert(2 * ATT_PART_BYTES <= 2 * ATT_TILE_BYTES && 8 * 64 * 4 <= ATT_QUERY_BYTES, "");

// 8 KiB of global memory straight into LDS, lane l's 16 bytes of each KiB to lds + 16 l, once the wave's LDS reads are done.  Written out,
// because the compiler lets every LDS read wait for all such loads in flight.  M0 needs one wait state.
__device__ __forceinline__ void att_load_tile(uint32_t lds, uint32_t lane_off, const char *from) {
    // (uniform, but under pressure kept in vector registers)
    const uint64_t at = (uint64_t)from;
    const char *src = (const char *)((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)at));
    asm volatile("s_waitcnt lgkmcnt(0)\n\t"
                 "s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\tglobal_load_lds_dwordx4 %2, %3 offset:1024\n\t"
                 "global_load_lds_dwordx4 %2, %3 offset:2048\n\tglobal_load_lds_dwordx4 %2, %3 offset:3072\n\t"
                 "s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %4\n\tglobal_load_lds_dwordx4 %2, %4 offset:1024\n\t"
                 "global_load_lds_dwordx4 %2, %4 offset:2048\n\tglobal_load_lds_dwordx4 %2, %4 offset:3072"
                 ::"s"(lds), "s"(lds + 4096), "v"(lane_off), "s"(src), "s"(src + 4096) : "memory");
}

// the exponents of a tile: of its own, or one for all.  (Through the constant address space, so that they come by scalar loads: a vector
// load would have to wait for all of the fragments on their way.)
__device__ __forceinline__ int2 att_exponents(const AttFrags &f, size_t tile) {
    if (!f.exps) return make_int2(f.k_exp, f.v_exp);
    const auto *at = (const __attribute__((address_space(4))) int *)(uintptr_t)(f.exps + tile);
    return make_int2(at[0], at[1]);
}

// A wave's NB blocks of 32 queries, lane (c, h2) holding query c of each, against tiles of 32 keys.
template <int NB>
struct AttWave {
    f16x8 q[NB][4][2];  // the queries times 2^their exponent, as fragments of the second operand: [block][d step][piece]
    int qe[NB];         // that exponent
    floatx16 o[NB][2], s[NB];  // o: [block][32 dimensions]; s: scores, then weights
    float m[NB], l[NB];  // reference of the weights; their sum, this half of the wave's
    int e;             // o is in units of 2^-(e + kBase): e is no larger than any exponent that V of the tiles so far has
    float up;          // what the weights of the tile at hand are multiplied by for that unit
    // Weights are exp(score - m), where m may lag behind the largest score by kLag (six powers of two) before everything is rescaled.  As
    // operands they are multiplied by 2^kBase: they stay below 2^15, and even those of 2^-11 have a lo of full length.  (Not within the
    // exponential: an argument around 9 is rounded to 2^-21.)
    static constexpr int kBase = 9;
    // The exponents of V's tiles lie within this much of each other, or the block is worked out in fp32 (exact_tiles): so many bits of a weight of 2^-11
    // and less go to a tile of smaller V.
    static constexpr int kSpread = 8;
    static constexpr float kLag = 6.0f * 0.693147f, kLog2e = 1.44269504f;

    __device__ __forceinline__ void clear(int b) {
        o[b][0] = o[b][1] = floatx16{0};
        m[b] = -INFINITY;
        l[b] = 0.0f;
    }
    __device__ __forceinline__ void start(int unit) {
#pragma unroll
        for (int b = 0; b < NB; ++b) clear(b);
        e = unit;
    }
    __device__ __forceinline__ void take_queries(const f16x8 *frags, const int *exps, int lane) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
#pragma unroll
            for (int ds = 0; ds < 4; ++ds)
#pragma unroll
                for (int pc = 0; pc < 2; ++pc) q[b][ds][pc] = frags[((b * 4 + ds) * 2 + pc) * 64 + lane];
            qe[b] = exps[32 * b + (lane & 31)];
        }
    }

    // s = K Q^T; k(d step, piece): the fragments of the tile
    template <class F>
    __device__ __forceinline__ void scores(F k) {
        f16x8 kf[4];
        for (int b = 0; b < NB; ++b) s[b] = floatx16{0};
#pragma unroll
        for (int ds = 0; ds < 4; ++ds) {
            const f16x8 lo = k(ds, 1);
            kf[ds] = k(ds, 0);
#pragma unroll
            for (int b = 0; b < NB; ++b) s[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo, q[b][ds][0], s[b], 0, 0, 0);
#pragma unroll
            for (int b = 0; b < NB; ++b) s[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ds], q[b][ds][1], s[b], 0, 0, 0);
        }
#pragma unroll
        for (int ds = 0; ds < 4; ++ds)
#pragma unroll
            for (int b = 0; b < NB; ++b) s[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[ds], q[b][ds][0], s[b], 0, 0, 0);
    }

    // register r of s holds key j0 + 8*(r/4) + 4*h2 + r%4: keys from `keys` on, and those behind the query's own, i0 + 32 b + c, are hidden
    __device__ __forceinline__ void hide(int j0, int h2, int keys, int i) {
        for (int b = 0; b < NB; ++b) {
            const int last = min(i + 32 * b, keys - 1) - j0 - 4 * h2;
#pragma unroll
            for (int r = 0; r < 16; ++r) s[b][r] = 8 * (r >> 2) + (r & 3) <= last ? s[b][r] : -INFINITY;
        }
    }

    // s = the weights; ek, ev: the tile's exponents (uniform)
    __device__ __forceinline__ void weights(int ek, int ev) {
        float down[NB], ref[NB], top[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int es = min(100, qe[b] + ek + 3);  // with the factor 1/8 (beyond 100 the scores are nothing, below 2^-64, either way)
            down[b] = pow2f(-es);  // of the scores
            ref[b] = pow2f(es);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) top[b] = s[b][0];
#pragma unroll
        for (int r = 1; r < 16; ++r)
#pragma unroll
            for (int b = 0; b < NB; ++b) top[b] = fmaxf(top[b], s[b][r]);
        // V smaller than what sets the unit goes in as smaller weights.  (No way back up: what has been summed up may be as large as the V that
        // it came from, or nothing of it, and no power of two fits both.)
        const int to = min(e, ev);
        bool ahead = false;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            top[b] = att_max_halves(top[b]) * down[b];
            ahead = ahead || top[b] - m[b] > kLag;
        }
        if (to != e || __any(ahead)) {  // (a query that has seen no key yet: an infinite difference, or NaN)
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const float m_new = fmaxf(m[b], top[b]), alpha = m_new == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f((m[b] - m_new) * kLog2e);
                const float move = alpha * pow2f(to - e);  // (e - to is kSpread at most where the result counts)
                l[b] *= alpha;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    o[b][0][r] *= move;
                    o[b][1][r] *= move;
                }
                m[b] = m_new;
            }
            e = to;
        }
        up = pow2f(kBase + to - ev);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const float r0 = (m[b] == -INFINITY ? 0.0f : m[b]) * ref[b], f = down[b] * kLog2e;
            float sum = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[b][r] = __builtin_amdgcn_exp2f((s[b][r] - r0) * f);
                sum += s[b][r];
            }
            l[b] += sum;
        }
    }

    // o += V^T P^T; v(32 dimensions, piece, key step): the fragments of the tile; first: block 0 takes part (uniform)
    template <class F>
    __device__ __forceinline__ void outputs(F v, bool first) {
        f16x8 p[NB][2][2];  // [block][key step][piece]
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int st = 0; st < 2; ++st) {
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = s[b][8 * st + i] * up;  // element i of key step st (an exponential's result is no operand of inline assembly)
                uint32_t hi[4], lo[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) split_f16(x[2 * i], x[2 * i + 1], hi[i], lo[i]);
                p[b][st][0] = __builtin_bit_cast(f16x8, make_uint4(hi[0], hi[1], hi[2], hi[3]));
                p[b][st][1] = __builtin_bit_cast(f16x8, make_uint4(lo[0], lo[1], lo[2], lo[3]));
            }
#pragma unroll
        for (int pv = 1; pv >= 0; --pv) {
            f16x8 vf[2][2];
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int st = 0; st < 2; ++st) vf[db][st] = v(db, pv, st);
            auto block = [&](int b) {
#pragma unroll
                for (int pp = 1 - pv; pp >= 0; --pp)  // V lo P hi; V hi P lo, V hi P hi
#pragma unroll
                    for (int st = 0; st < 2; ++st)
#pragma unroll
                        for (int db = 0; db < 2; ++db) o[b][db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[db][st], p[b][st][pp], o[b][db], 0, 0, 0);
            };
            block(NB - 1);
            if (NB == 2 && first) block(0);
        }
    }

    // The general path: block B against the tiles first, first + step, ... below `end` of K and V rows kh, vh, on v_mfma_f32_32x32x2_f32, as
    // operands come (five times the matrix cycles of the pairs).  q_row: this lane's query; `tile`: the wave's own place in LDS; o is
    // in units of 1 then.  HALVES: a score is the sum of two sums, with half the roundings each (16 more registers, which attn_rows_kernel does not have).
    template <int B, bool HALVES>
    __device__ __forceinline__ void exact_tiles(const float *q_row, const float *kh, const float *vh, int first, int step, int end, int kv_len, int my_limit, float *tile,
                                                int lane) {
        const int c = lane & 31, h2 = lane >> 5, at = (lane >> 4) * KLD + 4 * (lane & 15);
        clear(B);
        float qf[32];
#pragma unroll
        for (int i = 0; i < 32; i += 4) {
            const float4 t = *reinterpret_cast<const float4 *>(q_row + 32 * h2 + i);
            qf[i] = t.x * 0.125f; qf[i + 1] = t.y * 0.125f; qf[i + 2] = t.z * 0.125f; qf[i + 3] = t.w * 0.125f;
        }
#pragma unroll 1
        for (int t = first; t < end; t += step) {
            const int j0 = 32 * t;
            float4 kt[8], vt[8];  // rows 4 it + lane / 16, zeros beyond the last
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                const int j = j0 + 4 * it + (lane >> 4);
                const size_t off = (size_t)min(j, kv_len - 1) * DH + 4 * (lane & 15);
                kt[it] = *reinterpret_cast<const float4 *>(kh + off);
                vt[it] = *reinterpret_cast<const float4 *>(vh + off);
                if (j >= kv_len) kt[it] = vt[it] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
            // (one wave: its LDS operations complete in order)
#pragma unroll
            for (int it = 0; it < 8; ++it) *reinterpret_cast<float4 *>(tile + it * 4 * KLD + at) = kt[it];
            floatx16 x = {0}, half = {0};
            floatx16 &y = HALVES ? half : x;
#pragma unroll
            for (int i = 0; i < 32; i += 4) {
                const float4 k4 = *reinterpret_cast<const float4 *>(tile + c * KLD + 32 * h2 + i);
                x = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.x, qf[i], x, 0, 0, 0);
                y = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.y, qf[i + 1], y, 0, 0, 0);
                x = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.z, qf[i + 2], x, 0, 0, 0);
                y = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.w, qf[i + 3], y, 0, 0, 0);
            }
#pragma unroll
            for (int it = 0; it < 8; ++it) *reinterpret_cast<float4 *>(tile + it * 4 * KLD + at) = vt[it];
            const int last = min(my_limit, kv_len - 1) - j0 - 4 * h2;
            float top = -INFINITY, sum = 0.0f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (HALVES) x[r] += half[r];
                x[r] = 8 * (r >> 2) + (r & 3) <= last ? x[r] : -INFINITY;
                top = fmaxf(top, x[r]);
            }
            // a query that has seen no key yet stays empty
            const float m_new = fmaxf(m[B], att_max_halves(top)), ref = m_new == -INFINITY ? 0.0f : m_new, alpha = ATT_EXP(m[B] - ref);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                x[r] = ATT_EXP(x[r] - ref);
                sum += x[r];
            }
            l[B] = l[B] * alpha + sum;
            m[B] = m_new;
            floatx16 of_tile[2] = {};  // in sums of their own: fewer roundings at the size of the whole
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float *row = tile + (8 * (r >> 2) + 4 * h2 + (r & 3)) * KLD;
                of_tile[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(row[c], x[r], of_tile[0], 0, 0, 0);
                of_tile[1] = __builtin_amdgcn_mfma_f32_32x32x2f32(row[32 + c], x[r], of_tile[1], 0, 0, 0);
            }
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[B][db][r] = fmaf(o[B][db][r], alpha, of_tile[db][r]);
        }
    }

    __device__ __forceinline__ float unit() const { return pow2f(-e - kBase); }
    __device__ __forceinline__ void store_outputs(int b, float *part, int c, int h2, float unit) const {
        int column = c ^ (4 * h2);
        asm volatile("" : "+v"(column));  // the places are worked out here, not kept in registers from the kernel's start on
        part += 4 * h2 * 32;
#pragma unroll
        for (int r = 0; r < 16; ++r) {  // att_place of dimension 8 * (r / 4) + 4 * h2 + r % 4
            const int d = 8 * (r >> 2) + (r & 3);
            part[d * 32 + (column ^ d)] = o[b][0][r] * unit;
            part[(d + 32) * 32 + (column ^ d)] = o[b][1][r] * unit;
        }
    }
    __device__ __forceinline__ float sum(int b) const { return att_sum_halves(l[b]); }
};

// At most 32 queries and 32 keys: one wave a head, on v_mfma_f32_32x32x2_f32.  Nothing but the chain of its steps
// counts here, and that of fp32 operands is shorter than the way over f16 pairs, with its scales, shares and merge: 17 tokens 6.3 us against 7.4.
// grid (n_heads * batch), 64 threads.
__global__ __launch_bounds__(64) void attn_tile_kernel(const AttnParams p) {
    __shared__ __align__(16) float tile[3][32 * KLD];  // K, Q, V
    const int lane = threadIdx.x, c = lane & 31, h2 = lane >> 5, hb = blockIdx.x, b = hb / p.n_heads, h = hb % p.n_heads;
    int kv_len, q_offset;
    resolve_positions(p, kv_len, q_offset);
    // rows it*4 + lane/16, 4 floats at column 4*(lane%16); rows beyond the last count as zeros
    float4 k[8], q[8], v[8];
    auto fetch = [&](float4 (&to)[8], const float *from, long long stride, int rows) {
#pragma unroll
        for (int it = 0; it < 8; ++it) {
            const int r = it * 4 + (lane >> 4);
            to[it] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (r < rows) to[it] = *reinterpret_cast<const float4 *>(from + (size_t)r * stride + 4 * (lane & 15));
        }
    };
    fetch(q, p.q + (size_t)b * p.q_batch_stride + (size_t)h * p.q_head_stride, p.q_row_stride, p.q_len);
    fetch(k, p.k + (size_t)hb * p.kv_stride * DH, DH, kv_len);
    fetch(v, p.v + (size_t)hb * p.kv_stride * DH, DH, kv_len);
    auto store = [&](float *to, const float4 (&from)[8]) {  // (one wave: its LDS operations complete in order)
#pragma unroll
        for (int it = 0; it < 8; ++it) *reinterpret_cast<float4 *>(to + (it * 4 + (lane >> 4)) * KLD + 4 * (lane & 15)) = from[it];
    };
    store(tile[1], q);
    store(tile[0], k);
    // S^T[key][query]: A = K[key = c][32*h2 + s], B = Q[query = c][32*h2 + s]
    floatx16 s = {0}, o0 = {0}, o1 = {0};
#pragma unroll
    for (int i = 0; i < 32; i += 4) {
        const float4 k4 = *reinterpret_cast<const float4 *>(tile[0] + c * KLD + 32 * h2 + i), q4 = *reinterpret_cast<const float4 *>(tile[1] + c * KLD + 32 * h2 + i);
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.x, q4.x * 0.125f, s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.y, q4.y * 0.125f, s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.z, q4.z * 0.125f, s, 0, 0, 0);
        s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4.w, q4.w * 0.125f, s, 0, 0, 0);
    }
    store(tile[2], v);
    // register r holds key 8*(r/4) + 4*h2 + r%4 for query c; the first key is visible to every query
    const int last = min(kv_len - 1, p.causal ? q_offset + c : kv_len) - 4 * h2;
    float top = -INFINITY, sum = 0.0f;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        s[r] = 8 * (r >> 2) + (r & 3) <= last ? s[r] : -INFINITY;
        top = fmaxf(top, s[r]);
    }
    top = fmaxf(top, __shfl_xor(top, 32, kWave));
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        s[r] = ATT_EXP(s[r] - top);
        sum += s[r];
    }
    sum += __shfl_xor(sum, 32, kWave);
    // O^T[d][query] = V^T[d][key] P^T[key][query]: A = V[key(r,h2)][32*dt + c], B = p[r]
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float *row = tile[2] + (8 * (r >> 2) + 4 * h2 + (r & 3)) * KLD;
        o0 = __builtin_amdgcn_mfma_f32_32x32x2f32(row[c], s[r], o0, 0, 0, 0);
        o1 = __builtin_amdgcn_mfma_f32_32x32x2f32(row[32 + c], s[r], o1, 0, 0, 0);
    }
    const float scale = 1.0f / sum;
    bool raw = false;
    if (p.pairs) {
        float most = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) most = fmaxf(most, fmaxf(fabsf(o0[r]), fabsf(o1[r])));
        raw = pair_raw(att_max_halves(most * scale) * p.pairs_up);
    }
    if (c >= p.q_len) return;
    // O^T element (d, query c) of lane (c, h2): o0[r] at d = 8*(r/4) + 4*h2 + r%4, o1[r] at d + 32
#pragma unroll
    for (int r = 0; r < 16; r += 4) {
        const int d = 2 * r + 4 * h2;
        const float4 a = make_float4(o0[r] * scale, o0[r + 1] * scale, o0[r + 2] * scale, o0[r + 3] * scale);
        const float4 e = make_float4(o1[r] * scale, o1[r + 1] * scale, o1[r + 2] * scale, o1[r + 3] * scale);
        if (p.pairs) {
            const int row = b * p.q_len + c;
            char *block = p.pairs + (size_t)h * kPairBlockBytes;
            const float x[8] = {a.x, a.y, a.z, a.w, e.x, e.y, e.z, e.w};
            if (raw) {
                char *dst = block + (size_t)(row >> 5) * p.n_heads * kPairBlockBytes;
                *reinterpret_cast<float4 *>(dst + pair_raw_offset(row & 31, d)) = a;
                *reinterpret_cast<float4 *>(dst + pair_raw_offset(row & 31, d + 32)) = e;
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) store_pair_element(block, p.n_heads, row, d + (i & 3) + 32 * (i >> 2), x[i] * p.pairs_up);
            }
            if (r == 0 && h2 == 0) p.pair_marks[(size_t)h * 32 * ((p.batch * p.q_len + 31) >> 5) + row] = raw;
            if (raw && r == 0) p.pair_tiles[row >> 6] = p.epoch;
        } else {
            float *row = p.o + (size_t)b * p.o_batch_stride + (size_t)h * p.o_head_stride + (size_t)c * p.o_row_stride;
            *reinterpret_cast<float4 *>(row + d) = a;
            *reinterpret_cast<float4 *>(row + 32 + d) = e;
        }
    }
}

// The queries of NB blocks, from row `row0` of the head's `src` on, become fragments in LDS (AttWave::q, [block][d step][piece][lane]) once for all
// `waves` waves; copy(row, exponent), called by the 16 lanes that share a row, leaves the exponents where they are wanted.  16 lanes a row, so
// that whole lines are read: read by every wave for itself, row by lane, they are 512 lines a block and wave.
struct AttQueries {
    const float *src;
    long long row_stride;
    int row0, rows;  // rows from `rows` on repeat the last one
    __device__ __forceinline__ float4 load(int group, int lane) const {  // of four rows
        return *reinterpret_cast<const float4 *>(src + (size_t)min(row0 + 4 * group + (lane >> 4), rows - 1) * row_stride + 4 * (lane & 15));
    }
    template <class F>
    static __device__ __forceinline__ void store(f16x8 *frags, int group, int lane, float4 v, F copy) {
        const int row = 4 * group + (lane >> 4), d = 4 * (lane & 15);
        const float largest = row16_max(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        const int up = min(pair_exponent(largest), kMaxFragExpK);
        const float scale = pow2f(up);
        uint2 hi, lo;
        split_f16(v.x, v.y, scale, hi.x, lo.x);
        split_f16(v.z, v.w, scale, hi.y, lo.y);
        uint2 *to = reinterpret_cast<uint2 *>(frags + (((row >> 5) * 4 + (d >> 4)) * 2 * 2 + ((d >> 3) & 1)) * 32 + (row & 31)) + ((d >> 2) & 1);
        to[0] = hi;
        to[2 * 64] = lo;
        copy(row, up);
    }
};

// grid (ceil(q_len/32), n_heads * batch), 64 * S threads, S = 4 .. 8.  A workgroup owns 32 query rows; its S waves
// split the key tiles of 32 (wave w takes tiles w, w + S, ...), each with its own running (m, l, O) and its
// own K/V tile in LDS, so no barrier is needed inside the key loop; the next tile travels from global
// memory into registers while the matrix cores work on the current one.  The S partials are merged
// through LDS in wave order.  Query blocks are issued last-first: the causal mask makes the last blocks
// the long ones.
// K and V come as fp32 rows (the cache) and become f16 pairs in every wave that reads them, 64 values a lane and visit: about 450 vector
// instructions beside 24 matrix instructions of 32 cycles, where fp32 operands took 64 of 64 cycles, and two waves share a SIMD.  Their
// exponents, and whether the tile is fit for pairs at all, are worked out a tile at a time (about 40 instructions), unless bounds are KNOWN (the
// model, whose cache holds what its QKV Linears can give).  A block that meets a tile unfit for them is worked out a second time, on fp32
// operands (12 heads of 320 queries 18.9 us instead of 9.7).  us per launch, fp32 operands throughout / now: 16 heads of 150 queries, 150 to 750
// keys, in the model 15.7 / 12.2; without bounds 16 of 150 with 750 keys 19.4 / 15.4, 12 of 320 11.5 / 9.7, 25 of 256 9.7 / 8.5, 12 of 128 7.2 / 7.1.
// Errors against float64 fall by a third (64 terms of 3 products rounded once per 16).
// HAND_ON: the outputs may go on as pairs (what that takes is 0.5 us of 12 with 12 heads of 333).
template <bool KNOWN, bool HAND_ON>
__global__ __launch_bounds__(512) void attn_rows_kernel(const AttnParams p) {
    extern __shared__ __align__(16) float att_smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), S = blockDim.x >> 6;
    const int c = lane & 31, h2 = lane >> 5;
    float *tile = att_smem + wave * ATT_TILE_FLOATS;  // K, then V once the wave has read K (LDS operations of one wave complete in order)
    f16x8 *queries = reinterpret_cast<f16x8 *>(att_smem + S * ATT_TILE_FLOATS);
    int *exps = reinterpret_cast<int *>(queries + ATT_QUERY_BYTES / 16), *votes = exps + 32;
    const int hb = blockIdx.y, b = hb / p.n_heads, h = hb % p.n_heads;
    int kv_len, q_offset;
    resolve_positions(p, kv_len, q_offset);
    const float *kh = p.k + (size_t)hb * p.kv_stride * DH;
    const float *vh = p.v + (size_t)hb * p.kv_stride * DH;
    // rows it*4 + lane/16 of a tile, 4 floats at column 4*(lane%16): 8 x (K, V) float4 per lane
    float4 kpre[8], vpre[8];
    const int lane_off = (lane >> 4) * DH + (lane & 15) * 4;  // this lane's place in rows 0..3 of a tile
    auto fetch_tile = [&](const float *base, float4 (&pre)[8], int j0) {
        const float *t = base + (size_t)j0 * DH + lane_off;
        if (j0 + 32 <= kv_len) {  // a whole tile (uniform): constant offsets from one address
#pragma unroll
            for (int it = 0; it < 8; ++it) pre[it] = *reinterpret_cast<const float4 *>(t + it * 4 * DH);
        } else {
#pragma unroll
            for (int it = 0; it < 8; ++it) {
                pre[it] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (j0 + it * 4 + (lane >> 4) < kv_len) pre[it] = *reinterpret_cast<const float4 *>(t + it * 4 * DH);
            }
        }
    };
    // the exponent of the tile (uniform)
    auto exponent = [](const float4 (&v)[8], int most) {
        float largest = 0.0f;
#pragma unroll
        for (int it = 0; it < 8; ++it) largest = fmaxf(largest, fmaxf(fmaxf(fabsf(v[it].x), fabsf(v[it].y)), fmaxf(fabsf(v[it].z), fabsf(v[it].w))));
        return min(__builtin_amdgcn_readfirstlane(pair_exponent(wave_max(largest))), most);
    };
    // Query blocks of this workgroup: with pairing, block nb-1-x and then block x, so that under the causal mask
    // every workgroup walks through the same number of key tiles; otherwise one block, the long ones first.
    const int nb = (p.q_len + 31) >> 5;
    for (int rep = 0; rep < (p.pair_blocks ? 2 : 1); ++rep) {
        const int qb = rep == 0 ? nb - 1 - (int)blockIdx.x : (int)blockIdx.x;
        if (rep == 1 && qb >= nb - 1 - (int)blockIdx.x) break;  // the middle block of an odd count was done already
        const int i0 = qb * 32, last_q = min(p.q_len, i0 + 32) - 1;
        const int jmax = p.causal ? min(kv_len, q_offset + last_q + 1) : kv_len;  // keys [0, jmax)
        const int my_limit = p.causal ? q_offset + i0 + c : 0x3fffffff;           // last visible key of my query
        const AttQueries rows{p.q + (size_t)b * p.q_batch_stride + (size_t)h * p.q_head_stride, p.q_row_stride, i0, p.q_len};
        const float4 q0 = rows.load(wave, lane), q1 = rows.load(min(wave + S, 7), lane);  // (at least four waves)
        // the first tile's requests go out before the wave waits for its queries
        if (wave * 32 < jmax) {
            fetch_tile(kh, kpre, wave * 32);
            fetch_tile(vh, vpre, wave * 32);
        }
        auto store = [&](int group, float4 v) { AttQueries::store(queries, group, lane, v, [&](int row, int up) { exps[row] = up; }); };
        store(wave, q0);
        if (wave + S < 8) store(wave + S, q1);
        __syncthreads();
        AttWave<1> w;
        w.take_queries(queries, exps, lane);
        w.start(p.v_exp);
        int first_ev = 0;         // of V in the wave's first tile
        uint64_t first_some = 0;  // which of dimensions c and c + 32 are not all zeros there, a bit a lane
        votes[wave] = KNOWN && __any(w.qe[0] + p.k_exp < kLeastScoreExp);  // what this wave has met is not for pairs
        for (int j0 = wave * 32; j0 < jmax; j0 += 32 * S) {
            const bool more = j0 + 32 * S < jmax;
            f16x8 f[4][2];  // fragments of K [d step][piece], then of V [32 dimensions, key step][piece]
            const int ek = KNOWN ? p.k_exp : exponent(kpre, kMaxFragExpK);
            if (!KNOWN && __any(w.qe[0] + ek < kLeastScoreExp)) votes[wave] = 1;
#pragma unroll
            for (int it = 0; it < 8; ++it) *reinterpret_cast<float4 *>(tile + (it * 4 + (lane >> 4)) * KLD + 4 * (lane & 15)) = kpre[it];
            if (more) fetch_tile(kh, kpre, j0 + 32 * S);
#pragma unroll
            for (int ds = 0; ds < 4; ++ds) {
                const float *at = tile + c * KLD + 16 * ds + 8 * h2;
                const float4 lo = *reinterpret_cast<const float4 *>(at), hi = *reinterpret_cast<const float4 *>(at + 4);
                const float x[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                split_f16(x, pow2f(ek), f[ds][0], f[ds][1]);
            }
            w.scores([&](int ds, int pc) { return f[ds][pc]; });
            // K has been read: V goes into the same tile, the next V into the registers it leaves
            if (!KNOWN && j0 + 32 > kv_len) {  // (a run of eight keys is to be one of eight, where there are 16: instead of zeros)
#pragma unroll
                for (int it = 4; it < 8; ++it) {
                    const bool past = j0 + 16 <= kv_len && j0 + it * 4 + (lane >> 4) >= kv_len;
                    vpre[it].x = past ? vpre[it - 4].x : vpre[it].x;
                    vpre[it].y = past ? vpre[it - 4].y : vpre[it].y;
                    vpre[it].z = past ? vpre[it - 4].z : vpre[it].z;
                    vpre[it].w = past ? vpre[it - 4].w : vpre[it].w;
                }
            }
#pragma unroll
            for (int it = 0; it < 8; ++it) *reinterpret_cast<float4 *>(tile + (it * 4 + (lane >> 4)) * DH + 4 * (lane & 15)) = vpre[it];
            if (more) fetch_tile(vh, vpre, j0 + 32 * S);
            // only the tiles on the diagonal or at the end of the context hide anything (uniform over the wave)
            const bool hidden = j0 + 32 > kv_len || (p.causal && j0 + 31 > q_offset + i0);
            if (hidden) w.hide(j0, h2, kv_len, my_limit);
            float key_most = INFINITY;  // of key c, where that counts
            if (!KNOWN && hidden) {
                int key = c;
                asm volatile("" : "+v"(key));  // the places are worked out here, not kept in registers from the kernel's start on
                const float v = att_key_most(tile + key * DH + 32 * h2, key);
                key_most = j0 + key < kv_len ? v : INFINITY;
            }
            float x[2][2][8];  // [32 dimensions][key step]
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int st = 0; st < 2; ++st)
#pragma unroll
                    for (int e = 0; e < 8; ++e) x[db][st][e] = tile[att_vkey(st, h2, e) * DH + 32 * db + c];
            int ev = p.v_exp;
            if constexpr (KNOWN) {
                const uint32_t least = v_least(pow2f(p.v_exp), j0 + 32 <= kv_len);
                const uint32_t most[4] = {v_most(x[0][0]), v_most(x[0][1]), v_most(x[1][0]), v_most(x[1][1])};
                if (__builtin_expect(__any(min(min(most[0], most[1]), min(most[2], most[3])) < least), 0) &&  // (zeros, or small)
                    __any(v_is_small(most[0], least) || v_is_small(most[1], least) || v_is_small(most[2], least) || v_is_small(most[3], least)))
                    votes[wave] = 1;
            } else {
                float most[2], least[2];  // of dimensions c and c + 32, which both halves of the wave have
#pragma unroll
                for (int db = 0; db < 2; ++db) {
                    float run[2] = {0.0f, 0.0f};
#pragma unroll
                    for (int st = 0; st < 2; ++st)
#pragma unroll
                        for (int e = 0; e < 8; ++e) run[st] = fmaxf(run[st], fabsf(x[db][st][e]));
                    most[db] = att_max_halves(fmaxf(run[0], run[1]));
                    least[db] = -att_max_halves(-fminf(run[0], run[1]));
                }
                const float all = wave_max(fmaxf(most[0], most[1]));
                ev = min(__builtin_amdgcn_readfirstlane(pair_exponent(all)), kMaxFragExpV);
                const uint64_t some = __ballot(h2 == 0 ? most[0] > 0.0f : most[1] > 0.0f);
                if (j0 == wave * 32) {
                    w.e = first_ev = ev;
                    first_some = some;
                }
                bool uneven = abs(ev - first_ev) > AttWave<1>::kSpread / 2 || ev == kExpOfInf || some != first_some ||
                              __any(att_uneven(most[0], least[0], all, kv_len - j0) || att_uneven(most[1], least[1], all, kv_len - j0) || key_most < all * pow2f(-kRowSpread));
                if (uneven) votes[wave] = 1;
            }
            w.weights(ek, ev);
#pragma unroll
            for (int db = 0; db < 2; ++db)
#pragma unroll
                for (int st = 0; st < 2; ++st) split_f16(x[db][st], pow2f(ev), f[2 * db + st][0], f[2 * db + st][1]);
            w.outputs([&](int db, int pc, int st) { return f[2 * db + st][pc]; }, true);
        }
        // ---- merge the S partials: each wave leaves its O^T, m and l in its own tile ----
        w.store_outputs(0, tile, c, h2, w.unit());
        const float sum = w.sum(0);
        if (h2 == 0) {
            tile[64 * 32 + c] = w.m[0];
            tile[64 * 32 + 32 + c] = sum;
        }
        __syncthreads();
        if (__any(lane < S && votes[lane])) {  // one wave's tiles are not for pairs: the block once more
            int ln = lane;
            asm volatile("" : "+v"(ln));  // the places are worked out here, not kept in registers from the kernel's start on
            const int cc = ln & 31, hh = ln >> 5;
            AttWave<1> x;
            x.exact_tiles<0, false>(rows.src + (size_t)min(i0 + cc, p.q_len - 1) * rows.row_stride, kh, vh, wave, S, (jmax + 31) >> 5, kv_len,
                             p.causal ? q_offset + i0 + cc : 0x3fffffff, tile, ln);
            x.store_outputs(0, tile, cc, hh, 1.0f);
            const float all = x.sum(0);
            if (hh == 0) {
                tile[64 * 32 + cc] = x.m[0];
                tile[64 * 32 + 32 + cc] = all;
            }
            __syncthreads();
        }
        const std::conditional_t<HAND_ON, AttOut, AttRows> out(p, b, h);
        switch (S) {
            case 4: merge_partials<4>(att_smem, lane, wave, i0, p.q_len, out); break;
            case 5: merge_partials<5>(att_smem, lane, wave, i0, p.q_len, out); break;
            case 6: merge_partials<6>(att_smem, lane, wave, i0, p.q_len, out); break;
            case 7: merge_partials<7>(att_smem, lane, wave, i0, p.q_len, out); break;
            default: merge_partials<8>(att_smem, lane, wave, i0, p.q_len, out); break;
        }
        if (p.pair_blocks) __syncthreads();  // the tiles and the queries are reused by the second block
    }
}

// Causal attention of a prompt: queries and keys start at position 0 (q_offset = 0, kv_len >= q_len).  grid: a workgroup of NW waves for
// every NB (1 or 2) blocks of 32 queries of a head, rounded up to a multiple of 8 (one dimension).  Its waves take equal runs of the key
// tiles and merge what they have summed up at the end.
//
// A visit (64 queries, 32 keys) takes a wave 48 matrix instructions, 1500 cycles of the matrix cores, about 260 vector instructions and
// 16 KiB of K and V fragments.
// * A tile comes by loads that write the wave's own LDS directly: K of the next visit while this
//   one is at its softmax and V^T P, V of the next from then on.  Waves wait for nobody until the merge, so that the two of a SIMD drift
//   apart and one's matrix instructions meet the other's vector instructions; two waves sharing a tile between their 32 queries each and
//   kept in step by a barrier per phase took 2200 cycles for a phase of 12 matrix instructions (25 heads of 2048: 71 us against 63).
// * The queries become fragments once per workgroup (2 heads of 1024: 19.8 us, and 22.4 with each wave reading all rows).
// * A workgroup is one pair of blocks, the longest pairs first: two pairs a workgroup (a long one and a short one) balance worse, with
//   fewer workgroups than places for them (25 heads of 2048: 400 for 512; 75 us against 73).
// us per launch in the model or block, bf16 pieces before / now: 25 heads of 2048 92 / 63, 20 of 1000 27.0 / 21.2.  At the first of these all CUs
// run 1.26 M matrix instructions, 30 us at the 24 ns that two waves taking turns at a matrix core need for one on random operands (one wave: 17.4).
template <int NB, int NW>
__global__ __launch_bounds__(64 * NW, 2) void attn_f16_kernel(const AttnParams p, const AttFrags fr) {
    extern __shared__ __align__(16) float att_smem[];  // [wave][K, V] tiles
    unsigned char *const lds = reinterpret_cast<unsigned char *>(att_smem);
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c = lane & 31, h2 = lane >> 5;
    // Workgroup -> (head, pair).  Consecutive workgroup numbers go round the eight XCDs, and an XCD takes a run of consecutive entries of the
    // list of all heads' pairs: the fragments of a few heads stay in its L2.  Within its run it takes the longest
    // pairs first: entry by entry of the list, with pairs counted from the last, it has `skip` fewer of its first head.
    constexpr int QUERIES = 32 * NB;
    const int np = (p.q_len + QUERIES - 1) / QUERIES, total = np * p.n_heads * p.batch, per_xcd = (total + 7) >> 3;
    const int xcd = (int)blockIdx.x & 7, first = xcd * per_xcd, count = min(per_xcd, total - first), at = (int)blockIdx.x >> 3;
    if (at >= count) return;
    const int head0 = first / np, skip = first - head0 * np, end = skip + count;  // entries skip .. end - 1 from head0's first on
    const int full = end / np, tail = end - full * np;
    auto before = [&](int i) { return full * i + min(i, tail) - min(i, skip); };  // entries of the run with a number below i within their head
    int lo = 0, hi = np;  // before(lo) <= at < before(hi)
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        (before(mid) <= at ? lo : hi) = mid;
    }
    const int pair = np - 1 - lo, hb = head0 + (lo < skip ? 1 : 0) + (at - before(lo)), b = hb / p.n_heads, h = hb - b * p.n_heads;
    const int kv_len = p.kv_len, i0 = QUERIES * pair, n = (min(min(i0 + QUERIES, p.q_len), kv_len) + 31) >> 5;  // key tiles that the last query sees
    const int v0 = wave * n / NW, v1 = (wave + 1) * n / NW;

    const size_t head_bytes = (size_t)hb * fr.tiles_cap * ATT_TILE_BYTES;
    const char *k_head = reinterpret_cast<const char *>(fr.k) + head_bytes, *v_head = reinterpret_cast<const char *>(fr.v) + head_bytes;
    const uint32_t lane_off = lane * 16, k_place = wave * 2 * ATT_TILE_BYTES, v_place = k_place + ATT_TILE_BYTES;
    auto request_k = [&](int t) { att_load_tile(lds0 + k_place, lane_off, k_head + (size_t)t * ATT_TILE_BYTES); };
    auto request_v = [&](int t) { att_load_tile(lds0 + v_place, lane_off, v_head + (size_t)t * ATT_TILE_BYTES); };
    const f16x8 *ks = reinterpret_cast<const f16x8 *>(lds + k_place) + lane, *vs = reinterpret_cast<const f16x8 *>(lds + v_place) + lane;
    AttWave<NB> w;
    auto older_arrived = []() { asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); };  // all but the last tile requested
    int2 ex = make_int2(0, 0);  // the exponents of the tile, asked for one visit ahead
    const size_t tile0 = (size_t)hb * fr.tiles_cap;
    auto exponents = [&](int t) { return att_exponents(fr, tile0 + t); };
    f16x8 *const queries = reinterpret_cast<f16x8 *>(lds + NW * 2 * ATT_TILE_BYTES);
    auto query_exps = [&](int u) { return reinterpret_cast<int *>(lds + (2 * u + 1) * ATT_TILE_BYTES); };  // every wave's copy, where its V will be
    const AttQueries rows{p.q + (size_t)b * p.q_batch_stride + (size_t)h * p.q_head_stride, p.q_row_stride, i0, p.q_len};
    constexpr int kGroups = QUERIES / (4 * NW);
    float4 qv[kGroups];
#pragma unroll
    for (int i = 0; i < kGroups; ++i) qv[i] = rows.load(wave * kGroups + i, lane);
    // Every wave looks at the exponents of all tiles that a block sees, and comes to the same.  (The second of two blocks sees one tile more.)
    const int seen0 = NB == 1 ? n : min(n, (min(min(i0 + 32, p.q_len), kv_len) + 31) >> 5);
    struct Looked {
        float least, most, least_k;  // least: less the smallest exponent of V; of K
        __device__ __forceinline__ void at(int4 x, const int4 &first) {  // (dimensions that are all zeros are to be the same ones in all tiles)
            least = fmaxf(least, -(float)x.y);
            most = fmaxf(most, x.y == kExpOfInf || x.z != first.z || x.w != first.w ? 1000.0f : (float)x.y);
            least_k = fmaxf(least_k, -(float)x.x);
        }
    } looked = {-INFINITY, -INFINITY, -INFINITY};
    const uint32_t small_epoch = fr.v_small ? fr.v_small[hb] : 0u;
    int4 of_first = make_int4(0, 0, 0, 0), of_mine = of_first;  // (asked for here, looked at once the queries are on their way)
    if (fr.exps) {
        of_first = fr.exps[tile0];
        of_mine = fr.exps[tile0 + min(lane, seen0 - 1)];
    }
    if (v0 < v1) {
        request_k(v0);
        ex = exponents(v0);
    }
#pragma unroll
    for (int i = 0; i < kGroups; ++i)
        AttQueries::store(queries, wave * kGroups + i, lane, qv[i], [&](int row, int up) {
            if ((lane & 15) < NW) query_exps(lane & 15)[row] = up;
        });
    int e = fr.v_exp, ek[NB];
    bool exact[NB];
    for (int b = 0; b < NB; ++b) {
        ek[b] = fr.k_exp;
        exact[b] = fr.v_small && small_epoch == fr.epoch;
    }
    if (fr.exps) {
        looked.at(of_mine, of_first);
        for (int t = lane + 64; t < seen0; t += 64) looked.at(fr.exps[tile0 + t], of_first);
        looked = {wave_max(looked.least), wave_max(looked.most), wave_max(looked.least_k)};
        e = __builtin_amdgcn_readfirstlane(-(int)looked.least);
        for (int b = 0; b < NB; ++b) {
            if (b == 1) looked.at(fr.exps[tile0 + n - 1], of_first);
            ek[b] = -(int)looked.least_k;
            exact[b] = looked.most + looked.least > (float)AttWave<NB>::kSpread;
        }
    }
    __syncthreads();
    w.take_queries(queries, query_exps(wave), lane);
    for (int b = 0; b < NB; ++b) exact[b] = __any(exact[b] || w.qe[b] + ek[b] < kLeastScoreExp || (b == 1 && exact[0]));
    const int stop = exact[0] ? v0 : exact[NB - 1] ? min(v1, seen0) : v1;  // the tiles that are taken as pairs
    w.start(e);
    if (v0 < stop) {
        const int i = i0 + c;
        request_v(v0);
        for (int tile = v0; tile < stop; ++tile) {
            const bool more = tile + 1 < stop;
            const int j0 = tile * 32;
            older_arrived();
            w.scores([&](int ds, int pc) { return ks[(ds * 2 + pc) * 64]; });
            const int2 now = ex;
            if (more) {
                request_k(tile + 1);
                ex = exponents(tile + 1);
            }
            if (j0 + 32 > kv_len || j0 + 31 > i0) w.hide(j0, h2, kv_len, i);
            w.weights(now.x, now.y);
            if (more) older_arrived();
            else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            // the second block's last tile holds no key that the first block sees: it must not meet even weights of zero (0 x NaN)
            w.outputs([&](int db, int pc, int st) { return vs[((db * 2 + pc) * 2 + st) * 64]; }, j0 <= i0 + 31);
            if (more) request_v(tile + 1);
        }
    }
    if (exact[NB - 1] && v0 < v1) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // a tile asked for above has landed where the fp32 ones go
        float *const place = reinterpret_cast<float *>(lds + k_place);
        const float *const k_rows = p.k + (size_t)hb * p.kv_stride * DH, *const v_rows = p.v + (size_t)hb * p.kv_stride * DH;
        int ln = lane;
        asm volatile("" : "+v"(ln));  // the places are worked out here, not kept in registers from the kernel's start on
        auto tiles = [&](auto block) {
            constexpr int B = decltype(block)::value;
            const int i = i0 + 32 * B + (ln & 31);
            w.template exact_tiles<B, true>(rows.src + (size_t)min(i, p.q_len - 1) * rows.row_stride, k_rows, v_rows, v0, 1, B + 1 == NB ? v1 : min(v1, seen0), kv_len, i, place, ln);
        };
        if (exact[0]) tiles(std::integral_constant<int, 0>{});
        if constexpr (NB == 2) tiles(std::integral_constant<int, 1>{});
    }
    const AttOut out(p, b, h);
    float *const ml = reinterpret_cast<float *>(queries);
    __syncthreads();  // everyone is done with the queries (and each wave with its tiles)
    if (v0 < v1) {
#pragma unroll
        for (int blk = 0; blk < NB; ++blk) {
            w.store_outputs(blk, reinterpret_cast<float *>(lds + (NB * wave + blk) * ATT_PART_BYTES), c, h2, exact[blk] ? 1.0f : w.unit());
            const float sum = w.sum(blk);
            if (h2 == 0) {
                ml[(NB * wave + blk) * 64 + c] = w.m[blk];
                ml[(NB * wave + blk) * 64 + 32 + c] = sum;
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int blk = 0; blk < NB; ++blk) {
        // the waves' partial results; for a wave without one (there are fewer tiles than waves then), the last one's, which has one
        const float *o_at[NW], *ml_at[NW];
        unsigned parts = 0;
#pragma unroll
        for (int u = 0; u < NW; ++u) {
            const bool has = u * n / NW < (u + 1) * n / NW;
            const int from = NB * (has ? u : NW - 1) + blk;
            parts |= (has ? 1u : 0u) << u;
            o_at[u] = reinterpret_cast<const float *>(lds + from * ATT_PART_BYTES);
            ml_at[u] = ml + from * 64;
        }
        merge_partials_at<NW>(o_at, ml_at, parts, lane, wave, i0 + 32 * blk, p.q_len, out);
    }
}

// Merge (m, l, o) of `other` into (m, l, o); empty partials have l == 0 and m == -inf.
__device__ __forceinline__ void merge_partial(float &m, float &l, float4 &o, float m2, float l2, float4 o2) {
    const float mn = fmaxf(m, m2);
    if (mn == -INFINITY) return;
    const float a = expf(m - mn), b = expf(m2 - mn);
    l = l * a + l2 * b;
    o.x = o.x * a + o2.x * b; o.y = o.y * a + o2.y * b; o.z = o.z * a + o2.z * b; o.w = o.w * a + o2.w * b;
    m = mn;
}

// grid (q_len, n_heads * batch), 64*W threads.  One workgroup per (head, query row) takes every
// visible key, so nothing crosses a workgroup.  Lane layout: 16 lanes x float4 per key (one DPP row),
// 4 keys per wave step; a lane group handles PASS keys per pass (scores first, then one rescale), the W
// waves interleave over the keys.  The launch is a chain of dependent latencies, so: K and V rows are
// loaded for every slot below kv_stride before the context length (possibly a device-side counter) is
// known, and masked afterwards; dot products reduce with DPP; the 4W lane-group partials are brought to
// the common maximum first (one exp each) and then just added, in a fixed order.
// With gridDim.z > 1 (long contexts, few workgroups) workgroup z takes the keys [z * kv_chunk, (z + 1) * kv_chunk):
// more CUs pull the cache in.  Each writes (o, m, l) past the L2 and takes a ticket; the last one of a row adds the
// partial results in the order of z.
constexpr int kPassMany = 8;  // keys of a lane group in flight per pass when few workgroups share the chip
constexpr int kPassFew = 4;   // ... when the launch has more than a workgroup per CU
constexpr int kPassSome = 3;  // ... when it has more than 64 and up to one per CU
constexpr int kMaxKeySplits = 8;

// Wave 0 of a workgroup that has finished head h of sequence b: the 64 outputs, one per lane, also as bf16 pieces
// (8 consecutive values per 16 bytes; `row` is LDS of the wave's own, and a wave's LDS operations complete in order).
__device__ __forceinline__ void decode_pieces(const AttnParams &p, float *row, float val, int b, int h, int lane) {
    row[lane] = val;
    if (lane < 8) {
        const float4 f0 = *reinterpret_cast<const float4 *>(row + 8 * lane), f1 = *reinterpret_cast<const float4 *>(row + 8 * lane + 4);
        const float v[8] = {f0.x, f0.y, f0.z, f0.w, f1.x, f1.y, f1.z, f1.w};
        px_store_pieces(p.px_pieces, h * DH + 8 * lane, b, v);
    }
}

// SPLIT: keys split over gridDim.z workgroups.  PASS: keys of a lane group in flight per pass.
template <bool SPLIT, int PASS = kPassMany>
__global__ __launch_bounds__(1024) void attn_decode_kernel(const AttnParams p) {
    __shared__ float sm[64], sl[64];
    __shared__ __align__(16) float so[64][DH];  // one row per lane group
    __shared__ __align__(16) float so2[16][DH];  // one row per wave
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, W = blockDim.x >> 6;
    const int gq = lane >> 4, sub = lane & 15;
    const int qi = blockIdx.x, hb = blockIdx.y;
    const int b = hb / p.n_heads, h = hb % p.n_heads;

    const float *kh = p.k + (size_t)hb * p.kv_stride * DH + 4 * sub;
    const float *vh = p.v + (size_t)hb * p.kv_stride * DH + 4 * sub;
    const float *qrow = p.q + (size_t)b * p.q_batch_stride + (size_t)h * p.q_head_stride + (size_t)qi * p.q_row_stride;
    float4 q4 = *reinterpret_cast<const float4 *>(qrow + 4 * sub);
    const int stride = 4 * W;  // keys between two consecutive keys of one lane group
    const int Z = SPLIT ? (int)gridDim.z : 1, lo = SPLIT ? (int)blockIdx.z * p.kv_chunk : 0;
    const int first = lo + wave * 4 + gq;
    float4 k4[PASS], v4[PASS];
    auto fetch = [&](int base, int limit) {  // rows below kv_stride exist whatever the context length is; others read row 0
#pragma unroll
        for (int i = 0; i < PASS; ++i) {
            const int j = base + i * stride;
            const int jr = j < limit ? j : 0;
            k4[i] = *reinterpret_cast<const float4 *>(kh + (size_t)jr * DH);
            v4[i] = *reinterpret_cast<const float4 *>(vh + (size_t)jr * DH);
        }
    };
    if (p.speculate) fetch(first, p.kv_stride);
    int kv_len, q_offset;
    resolve_positions(p, kv_len, q_offset);
    const int vis_all = p.causal ? min(kv_len, q_offset + qi + 1) : kv_len;  // keys [0, vis_all)
    const int vis = SPLIT ? min(vis_all, lo + p.kv_chunk) : vis_all;          // this workgroup's keys: [lo, vis)
    if (!p.speculate && first < vis) fetch(first, vis);
    q4.x *= 0.125f; q4.y *= 0.125f; q4.z *= 0.125f; q4.w *= 0.125f;

    float m = -INFINITY, l = 0.0f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int base = first; base < vis; base += PASS * stride) {
        if (base != first) fetch(base, vis);  // the first pass is already in registers
        float s[PASS];
        float bm = -INFINITY;
#pragma unroll
        for (int i = 0; i < PASS; ++i) {
            const float d = (q4.x * k4[i].x + q4.y * k4[i].y) + (q4.z * k4[i].z + q4.w * k4[i].w);
            s[i] = base + i * stride < vis ? row16_sum(d) : -INFINITY;
            bm = fmaxf(bm, s[i]);
        }
        const float mn = fmaxf(m, bm);  // finite: the first key of the pass is visible
        const float a = expf(m - mn);
        l *= a;
        o.x *= a; o.y *= a; o.z *= a; o.w *= a;
#pragma unroll
        for (int i = 0; i < PASS; ++i) {
            const float pj = expf(s[i] - mn);  // exp(-inf) = 0 for masked keys
            l += pj;
            // a masked slot holds whatever the row contains (possibly NaN): select, do not multiply by 0
            const bool ok = base + i * stride < vis;
            o.x += ok ? pj * v4[i].x : 0.0f; o.y += ok ? pj * v4[i].y : 0.0f;
            o.z += ok ? pj * v4[i].z : 0.0f; o.w += ok ? pj * v4[i].w : 0.0f;
        }
        m = mn;
    }
    // ---- merge the 4W lane-group partials (m, l, o) ----
    const int g = wave * 4 + gq;
    if (sub == 0) sm[g] = m;
    if (tid >= 4 * W && tid < 64) sm[tid] = -INFINITY;
    __syncthreads();
    const float m_all = wave_max(sm[lane]);  // finite when the workgroup has a key (without a split: key 0)
    const float fac = SPLIT && m_all == -INFINITY ? 0.0f : expf(m - m_all);  // 0 for an empty partial
    if (sub == 0) sl[g] = l * fac;
    if (tid >= 4 * W && tid < 64) sl[tid] = 0.0f;
    *reinterpret_cast<float4 *>(&so[g][4 * sub]) = make_float4(o.x * fac, o.y * fac, o.z * fac, o.w * fac);
    // the wave's four rows, column-wise (LDS operations of one wave complete in order)
    const float ow = (so[wave * 4][lane] + so[wave * 4 + 1][lane]) + (so[wave * 4 + 2][lane] + so[wave * 4 + 3][lane]);
    so2[wave][lane] = ow;
    __syncthreads();
    if (wave == 0) {
        const float l_all = wave_sum(sl[lane]);
        float acc = 0.0f;
        for (int w = 0; w < W; ++w) acc += so2[w][lane];
        float *orow = p.o + (size_t)b * p.o_batch_stride + (size_t)h * p.o_head_stride + (size_t)qi * p.o_row_stride;
        if constexpr (!SPLIT) {
            const float val = acc / l_all;
            orow[lane] = val;
            if (p.px_pieces) decode_pieces(p, so2[0], val, b, h, lane);
            return;
        }
        const int row = qi * gridDim.y + hb;
        float *part = p.kv_partial + (size_t)row * kMaxKeySplits * 66;
        __hip_atomic_store(part + blockIdx.z * 66 + lane, acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (lane == 0) {
            __hip_atomic_store(part + blockIdx.z * 66 + 64, m_all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(part + blockIdx.z * 66 + 65, l_all, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        partials_published(p.strict);
        unsigned int tk = 0;
        if (lane == 0) {
            tk = take_ticket(&p.counters[row], p.strict);
            if (tk == (unsigned int)(Z - 1)) __hip_atomic_store(&p.counters[row], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        tk = __builtin_amdgcn_readfirstlane(tk);
        if (tk != (unsigned int)(Z - 1)) return;
        float mz[kMaxKeySplits], lz[kMaxKeySplits], oz[kMaxKeySplits];
#pragma unroll
        for (int zz = 0; zz < kMaxKeySplits; ++zz) {
            mz[zz] = -INFINITY;
            lz[zz] = oz[zz] = 0.0f;
            if (zz < Z) {
                oz[zz] = __hip_atomic_load(part + zz * 66 + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                mz[zz] = __hip_atomic_load(part + zz * 66 + 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                lz[zz] = __hip_atomic_load(part + zz * 66 + 65, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
        float mm = -INFINITY;
#pragma unroll
        for (int zz = 0; zz < kMaxKeySplits; ++zz) mm = fmaxf(mm, mz[zz]);
        float lsum = 0.0f, osum = 0.0f;
#pragma unroll
        for (int zz = 0; zz < kMaxKeySplits; ++zz) {
            const float f = mz[zz] == -INFINITY ? 0.0f : expf(mz[zz] - mm);
            lsum += lz[zz] * f;
            osum += oz[zz] * f;
        }
        const float val = osum / lsum;
        orow[lane] = val;
        if (p.px_pieces) decode_pieces(p, so2[0], val, b, h, lane);
    }
}

}  // namespace

template <bool KNOWN, bool HAND_ON>
static int32_t att_rows_go(agpu_ctx *ctx, const AttnParams &p, int S, int heads) {
    static std::atomic<unsigned long long> lds_raised{0};  // one bit per device: the attribute belongs to the device's code object
    const unsigned long long dev_bit = 1ull << (ctx->device & 63);
    if (att_rows_lds(S) > 65536 && !(lds_raised.load(std::memory_order_relaxed) & dev_bit)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(attn_rows_kernel<KNOWN, HAND_ON>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)att_rows_lds(8));
        if (e != hipSuccess) return agpu_hip(ctx, e, "hipFuncSetAttribute");
        lds_raised.fetch_or(dev_bit, std::memory_order_relaxed);
    }
    const int nb = ceil_div(p.q_len, 32);
    hipLaunchKernelGGL((attn_rows_kernel<KNOWN, HAND_ON>), dim3(p.pair_blocks ? (nb + 1) / 2 : nb, heads), dim3(64 * S), att_rows_lds(S), ctx->stream, p);
    return AGPU_LAUNCH_CHECK(ctx, "attn_rows_kernel");
}

int32_t agpu_attention_launch(agpu_ctx *ctx, const AttnParams &p, int max_kv_len) {
    const int hb = p.n_heads * p.batch;
    if (p.q_len <= 8) {
        // waves per workgroup: one per 32 keys of the longest possible context, 1..16
        int W = ceil_div(max_kv_len, 32);
        W = W < 1 ? 1 : (W > 16 ? 16 : W);
        // More workgroups than CUs (batched decode: one per head and sequence) fill the chip by themselves: four waves each
        // (XL shape, 16 sequences, context 300: 15 us per layer against 18.4 us with sixteen waves).  Up to one a CU, what a CU has in flight sets the time:
        // a wave per 16 keys, twelve at most, three keys a lane group (us, four waves and four keys / this: 66 workgroups of 300 keys 7.2 / 5.4,
        // 96 of 600 13.9 / 10.0, 192 of 300 9.8 / 8.2, 256 of 300 10.8 / 10.0; 300 of 300 12.4 / 13.2).
        const int workgroups = p.q_len * hb;
        const bool crowded = workgroups > ctx->num_cus;
        if (crowded) W = std::min(W, 4);
        else if (workgroups > 64) W = std::min(12, std::max(1, ceil_div(max_kv_len, 16)));
        // up to 512 keys eight waves in two passes beat sixteen in one (XL shape, context 300: 3 % of the step);
        // at 1024 keys sixteen waves are faster (8.0 against 9.0 us)
        else if (max_kv_len <= 512) W = std::min(W, 8);
        AttnParams pd = p;
        pd.speculate = p.q_len * hb <= 64 ? 1 : 0;  // latency matters for a few workgroups, bandwidth for many
        // Beyond 512 keys a few workgroups cannot pull the cache in fast enough: 256 keys per workgroup, eight waves
        // (12 heads, 1024 keys: 6.3 us against 8.0 us with one workgroup of sixteen waves per head; 128 keys each: 6.4 us;
        // at 512 keys two workgroups per head take 6.1 us against 5.7 us for one)
        int Z = 1;
        if (p.q_len * hb <= 64 && max_kv_len > 512 && p.q_len * hb <= ctx->n_counters) {
            Z = ceil_div(max_kv_len, 256);
            if (Z > kMaxKeySplits) Z = kMaxKeySplits;
            pd.kv_chunk = ceil_div(max_kv_len, Z);
            pd.kv_partial = reinterpret_cast<float *>(ctx->workspace);
            pd.counters = ctx->counters;
            pd.strict = ctx->strict_sync;
            W = ceil_div(pd.kv_chunk, 32);
            W = W > 16 ? 16 : W;
        }
        if (Z > 1) hipLaunchKernelGGL(attn_decode_kernel<true>, dim3(p.q_len, hb, Z), dim3(64 * W), 0, ctx->stream, pd);
        // many workgroups (batched decode) stream the cache at HBM speed: half the keys in flight per lane group arrive
        // sooner (XL shape, 16 sequences: 2.27 ms per step against 2.31; a quarter: the same)
        else if (crowded) hipLaunchKernelGGL((attn_decode_kernel<false, kPassFew>), dim3(p.q_len, hb), dim3(64 * W), 0, ctx->stream, pd);
        else if (workgroups > 64) hipLaunchKernelGGL((attn_decode_kernel<false, kPassSome>), dim3(p.q_len, hb), dim3(64 * W), 0, ctx->stream, pd);
        else hipLaunchKernelGGL(attn_decode_kernel<false>, dim3(p.q_len, hb), dim3(64 * W), 0, ctx->stream, pd);
        return AGPU_LAUNCH_CHECK(ctx, "attn_decode_kernel");
    }
    // Under the causal mask query block i walks through i + 1 key tiles.  When there are more workgroups than CUs, the
    // long ones share their SIMDs with others and set the time; pairing block nb-1-x with block x gives every
    // workgroup the same nb + 1 tiles (12 heads x 1024: 32.3 us against 44.2 us unpaired).  With fewer workgroups
    // pairing only lengthens the chains (12 heads x 256: 15.6 us against 10.0 us).
    AttnParams pm = p;
    const int nb = ceil_div(p.q_len, 32);
    pm.pair_blocks = (p.causal && nb >= 4 && nb * hb > ctx->num_cus) ? 1 : 0;
    const int wgs = (pm.pair_blocks ? (nb + 1) / 2 : nb) * hb;
    // key split: one wave per key tile of the longest query block.  The registers allow two waves per SIMD: one
    // workgroup of eight waves fills them when every workgroup has a CU of its own, two of four waves otherwise
    // (25 heads x 1024, 400 workgroups: 54.4 us with four waves, 63.1 us with eight)
    const int tiles = ceil_div(max_kv_len, 32);
    const int cap = wgs <= ctx->num_cus ? 8 : 4;
    const int S = std::max(4, std::min(tiles, cap));  // (waves without a tile still take their part of the queries and the merge)
    // Splitting K and V into fragments first (split_kv_kernel, 3 to 10 us with its launch) pays from 512 queries on, and where each tile
    // would be split by several query blocks a CU (us, rows / fragments: 12 heads of 400 12.4 / 12.9, 2 of 512 12.1 / 11.5, 2 of 700 15.4 / 13.1, 25 of 300,
    // 250 blocks, 10.9 / 13.1, 25 of 400 18.2 / 15.0, 64 of 300 24.5 / 23.7).
    if (p.causal && !p.pos_dev && p.q_offset == 0 && p.kv_len >= p.q_len && (p.q_len >= 512 || (p.q_len >= 288 && nb * hb > ctx->num_cus))) {
        const int tiles_cap = ceil_div(p.kv_len, 32);
        const size_t frag_bytes = agpu_attention_fragment_bytes(hb, p.kv_len), tiles_all = (size_t)hb * tiles_cap;
        if (2 * frag_bytes + tiles_all * sizeof(int4) <= ctx->ws_bytes / 2) {
            uint4 *kfrag = reinterpret_cast<uint4 *>(ctx->workspace), *vfrag = kfrag + frag_bytes / sizeof(uint4);
            int4 *exps = reinterpret_cast<int4 *>(vfrag + frag_bytes / sizeof(uint4));
            hipLaunchKernelGGL(split_kv_kernel, dim3(tiles_cap, hb), dim3(256), 0, ctx->stream, p.k, p.v, kfrag, vfrag, exps, p.kv_len, p.kv_stride,
                               tiles_cap);
            return agpu_attention_fragments_launch(ctx, p, AttFrags{kfrag, vfrag, exps, 0, 0, tiles_cap});
        }
    }
    if (max_kv_len <= 32 && p.q_len <= 32) {
        hipLaunchKernelGGL(attn_tile_kernel, dim3(hb), dim3(64), 0, ctx->stream, p);
        return AGPU_LAUNCH_CHECK(ctx, "attn_tile_kernel");
    }
    if (p.kv_known) return p.pairs ? att_rows_go<true, true>(ctx, pm, S, hb) : att_rows_go<true, false>(ctx, pm, S, hb);
    return p.pairs ? att_rows_go<false, true>(ctx, pm, S, hb) : att_rows_go<false, false>(ctx, pm, S, hb);
}

size_t agpu_attention_fragment_bytes(int heads, int kv_len) {
    return (size_t)heads * ceil_div(kv_len, 32) * ATT_FRAGS_PER_TILE * sizeof(uint4);
}

template <int NB, int NW>
static int32_t att_f16_go(agpu_ctx *ctx, const AttnParams &p, const AttFrags &fr) {
    static std::atomic<unsigned long long> lds_raised{0};  // one bit per device
    const unsigned long long bit = 1ull << (ctx->device & 63);
    if (!(lds_raised.load(std::memory_order_relaxed) & bit)) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(attn_f16_kernel<NB, NW>), hipFuncAttributeMaxDynamicSharedMemorySize, att_lds(NB, NW));
        if (e != hipSuccess) return agpu_hip(ctx, e, "hipFuncSetAttribute");
        lds_raised.fetch_or(bit, std::memory_order_relaxed);
    }
    const int grid = 8 * ceil_div(ceil_div(p.q_len, 32 * NB) * p.n_heads * p.batch, 8);
    hipLaunchKernelGGL((attn_f16_kernel<NB, NW>), dim3(grid), dim3(64 * NW), att_lds(NB, NW), ctx->stream, p, fr);
    return AGPU_LAUNCH_CHECK(ctx, "attn_f16_kernel");
}

int32_t agpu_attention_fragments_launch(agpu_ctx *ctx, const AttnParams &p, const AttFrags &fr) {
    if (!p.causal || p.pos_dev || p.q_offset != 0 || p.kv_len < p.q_len || p.q_len < 256 || fr.tiles_cap < ceil_div(p.kv_len, 32))
        return agpu_fail(ctx, AGPU_ERR_UNSUPPORTED, "attention on fragments: causal, from position 0, 256 queries or more");
    // A workgroup of eight waves per block of 32 queries while each has a CU of its own; then two of four waves share one (their LDS), and
    // from about three blocks a CU on, the fragments being read twice as often counts for more than the last round being nearly empty, they take two blocks
    // each.  us per launch with those three (splitting K and V included): 2 heads of 1024 14.0 / 15.3 / 21.4, 6 of 768 13.4 / 14.2 / 19.4,
    // 12 of 1024 23.4 / 20.3 / 25.3, 20 of 1000 34.8 / 29.0 / 31.7, 16 of 1500 42.9 / 38.0 / 39.8, 25 of 1024 43.8 / 35.4 / 34.2,
    // 64 of 1000 82.6 / 60.2 / 53.2, 25 of 2048 91.7 / 75.6 / 70.0.
    const long long blocks = (long long)ceil_div(p.q_len, 32) * p.n_heads * p.batch;
    if (blocks <= ctx->num_cus) return att_f16_go<1, 8>(ctx, p, fr);
    return blocks <= 3 * ctx->num_cus ? att_f16_go<1, 4>(ctx, p, fr) : att_f16_go<2, 4>(ctx, p, fr);
}

AGPU_EXPORT int32_t agpu_attention(agpu_ctx *ctx, const float *q, const float *k, const float *v, float *o,
                                   int32_t n_heads, int32_t q_len, int32_t kv_len, int32_t q_offset,
                                   int32_t kv_stride, int32_t d_head, int32_t causal) {
    AGPU_REQUIRE_CTX(ctx);
    if (!q || !k || !v || !o) return agpu_fail(ctx, AGPU_ERR_NULL_POINTER, "attention: null pointer");
    if (d_head != DH)
        return agpu_fail(ctx, AGPU_ERR_SHAPE_MISMATCH, "attention: expected d_head = 64, got d_head = %d", d_head);
    if (n_heads <= 0 || q_len < 0 || kv_len < 1 || q_offset < 0 || kv_stride < kv_len)
        return agpu_fail(ctx, AGPU_ERR_SHAPE_MISMATCH,
                         "attention: bad dims heads=%d q_len=%d kv_len=%d q_offset=%d kv_stride=%d", n_heads, q_len,
                         kv_len, q_offset, kv_stride);
    if (q_len == 0) return AGPU_OK;
    AttnParams p{};
    p.q = q; p.k = k; p.v = v; p.o = o;
    p.n_heads = n_heads; p.batch = 1; p.q_len = q_len; p.kv_len = kv_len; p.q_offset = q_offset;
    p.kv_stride = kv_stride; p.causal = causal ? 1 : 0;
    p.q_batch_stride = 0; p.q_head_stride = (long long)q_len * DH; p.q_row_stride = DH;
    p.o_batch_stride = 0; p.o_head_stride = (long long)q_len * DH; p.o_row_stride = DH;
    p.pos_dev = nullptr;
    return agpu_attention_launch(ctx, p, kv_len);
}

AGPU_EXPORT int32_t agpu_bench_attention(agpu_ctx *ctx, const float *q, const float *k, const float *v, float *o,
                                         int32_t n_heads, int32_t q_len, int32_t kv_len, int32_t q_offset,
                                         int32_t kv_stride, int32_t d_head, int32_t causal, int32_t reps,
                                         float *us_per_launch_out_host) {
    AGPU_REQUIRE_CTX(ctx);
    AGPU_REQUIRE_PTR(ctx, us_per_launch_out_host);
    if (reps <= 0) return agpu_fail(ctx, AGPU_ERR_SHAPE_MISMATCH, "bench_attention: reps must be positive");
    if (!ctx->stream) return agpu_fail(ctx, AGPU_ERR_UNSUPPORTED, "bench_attention: needs a context with its own stream");
    int32_t rc = agpu_attention(ctx, q, k, v, o, n_heads, q_len, kv_len, q_offset, kv_stride, d_head, causal);
    if (rc != AGPU_OK) return rc;
    hipError_t e = hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal);
    if (e != hipSuccess) return agpu_hip(ctx, e, "hipStreamBeginCapture");
    for (int i = 0; i < reps && rc == AGPU_OK; ++i)
        rc = agpu_attention(ctx, q, k, v, o, n_heads, q_len, kv_len, q_offset, kv_stride, d_head, causal);
    hipGraph_t graph = nullptr;
    e = hipStreamEndCapture(ctx->stream, &graph);
    if (rc != AGPU_OK || e != hipSuccess) {
        if (graph) (void)hipGraphDestroy(graph);
        return rc != AGPU_OK ? rc : agpu_hip(ctx, e, "hipStreamEndCapture");
    }
    hipGraphExec_t exec = nullptr;
    e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
    (void)hipGraphDestroy(graph);
    if (e != hipSuccess) return agpu_hip(ctx, e, "hipGraphInstantiate");
    float ms = 0.0f;
    e = hipGraphLaunch(exec, ctx->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
    if (e == hipSuccess) rc = agpu_timer_start(ctx);
    if (e == hipSuccess && rc == AGPU_OK) e = hipGraphLaunch(exec, ctx->stream);
    if (e == hipSuccess && rc == AGPU_OK) rc = agpu_timer_stop(ctx, &ms);
    (void)hipGraphExecDestroy(exec);
    if (e != hipSuccess) return agpu_hip(ctx, e, "hipGraphLaunch");
    *us_per_launch_out_host = ms * 1000.0f / (float)reps;
    return rc;
}
