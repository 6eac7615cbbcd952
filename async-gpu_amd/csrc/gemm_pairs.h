// What the kernels around the prefill GEMM on f16 pairs share (csrc/int4_gemm_pairs.hip): operand types, the split of fp32 rows into
// pairs, their layout in memory, and the conversion of packed nibbles.
//
// A row is scaled by a power of two that brings its largest value into [2^14, 2^15), and every scaled value is the sum of two f16
// numbers, hi = f16(v) and lo = f16(v - hi), both rounded to nearest: 23 significant bits, up to 2^-39 of the
// row's largest value.
#pragma once
#include "gemm_bf16.h"


constexpr int kPairBlockK = 64;                 // k of one block
constexpr int kPairBlockBytes = 4 * 32 * 64;    // 32 rows x 64 k: [step of 16 k][row][64 bytes]

// Where the 16 bytes (eight k: half hh of step st) of piece pc (0 lo, 1 hi) of row `row` lie in a block.  A row's four units of a
// step are rotated by its number, so that the 16 lanes that LDS serves at a time, 16 rows of one unit, fall on different banks, and a
// row's 64 bytes stay together for whoever writes them.
__host__ __device__ constexpr int pair_offset(int row, int st, int pc, int hh) {
    return st * 2048 + row * 64 + 16 * (((2 * pc + hh) + (row >> 2)) & 3);
}

// The pairs of x [M, K]: blocks [row block of 32][K block], zeros beyond M and K, behind them a factor per row (what its sums have to be
// multiplied by: kPairWeightUnit times the inverse of its scale), and behind those four bytes a row: not zero: the row is not for pairs.
struct PairLayout {
    int row_blocks, k_blocks;
    PairLayout(int M, int K) : row_blocks(ceil_div(M, 32)), k_blocks(ceil_div(K, kPairBlockK)) {}
    size_t frag_bytes() const { return (size_t)row_blocks * k_blocks * kPairBlockBytes; }
    // Rows that are handed on have one scale for all of them, and instead a byte a K block and row, [k_blocks][rows]: not zero: there the row stands as floats
    // (pair_raw_offset).  (In that order a wave's marks are in one line.)
    size_t marks_at() const { return bytes(); }
    size_t handed_bytes() const { return marks_at() + (size_t)row_blocks * 32 * k_blocks; }
    size_t bytes() const { return frag_bytes() + (size_t)row_blocks * 32 * (sizeof(float) + sizeof(uint32_t)); }
};

// exponent of the scale for a row whose largest |x| is amax: 2^s brings it into [2^14, 2^15) (rows below 2^-112 stay smaller)
__device__ __forceinline__ int pair_exponent(float amax) {
    const int s = 141 - (int)((__float_as_uint(amax) >> 23) & 255u);
    return s < 126 ? s : 126;
}
// Scaled values below this have a lo without all of its bits (it is a multiple of 2^-24): elements below 2^-17 to 2^-18 of a row's largest, which are off
// by up to 2^-39 of that one.  That shows where the weights of the larger elements are zero.  A few such elements are in any row (of 8192 random numbers
// 0.2, of 1024 with a few 2000 times as large 9); a row with more than this in one of its 16 parts is not for pairs.
constexpr float kPairShort = 0x1p-3f;  // (its exponent field: 124)
__device__ __forceinline__ float pair_short_allowed(int K) { return (float)(8 + K / 1024); }
__device__ __forceinline__ float pow2f(int s) { return __uint_as_float((uint32_t)(s + 127) << 23); }  // -126 <= s <= 127

// 8 consecutive k of a row, scaled by `up` -> the two fragments in the order (0, 4, 1, 5, 2, 6, 3, 7) of nibbles_to_f16
__device__ __forceinline__ void split_pair(const float (&v)[8], float up, uint4 &lo, uint4 &hi) {
    f16x8 h, l;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int i = (e >> 1) + 4 * (e & 1);
        const float x = v[i] * up;
        h[e] = (_Float16)x;
        l[e] = (_Float16)(x - (float)h[e]);
    }
    hi = __builtin_bit_cast(uint4, h);
    lo = __builtin_bit_cast(uint4, l);
}

// one scaled value: element k of the K block `block` (of row block 0) of row `row`
__device__ __forceinline__ void store_pair_element(char *block, int k_blocks, int row, int k, float v) {
    const _Float16 hi = (_Float16)v, lo = (_Float16)(v - (float)hi);
    const int i = k & 7, at = 2 * ((i & 3) * 2 + (i >> 2));  // place of nibble i in the order (0, 4, 1, 5, 2, 6, 3, 7)
    char *dst = block + (size_t)(row >> 5) * k_blocks * kPairBlockBytes + at;
    *reinterpret_cast<_Float16 *>(dst + pair_offset(row & 31, k >> 4, 0, (k >> 3) & 1)) = lo;
    *reinterpret_cast<_Float16 *>(dst + pair_offset(row & 31, k >> 4, 1, (k >> 3) & 1)) = hi;
}

// What a Linear or an attention hands on has a scale that follows from a bound (agpu_pair_bound_launch), and numbers are off by up to 2^-25 once scaled.  Where
// the largest of a row's 64 in a block is below 1, 2^-14 to 2^-15 of the bound, they stand in their place as floats.  (Usual values are 2^-5 of it, in the
// smallest column 2^-13; far smaller ones come from rows whose size is in channels that the Linear ignores, or from gains for channels that are
// small in the rows: with gains of 2^20 logits were off by 2e-5 of their size, by 7e-7 on floats.)
__device__ __forceinline__ bool pair_raw(float most) { return most > 0.0f && most < 1.0f; }
__host__ __device__ constexpr int pair_raw_offset(int row, int k) { return (k >> 4) * 2048 + row * 64 + 4 * (k & 15); }

// 8 nibbles of one column -> the f16 numbers (q - 8) / 128 in the order (0, 4, 1, 5, 2, 6, 3, 7).  A nibble put into the low bits of the f16
// number 8 (into the bits above them) makes it 8 + q / 128 (8 + q / 8): one shift, four v_and_or_b32 and four packed operations.
// The power of two lies halfway between that of the rows (2^14 .. 2^15 for their largest value), which would leave sums 2^14 larger than
// the results of a row whose largest value is 1 (Inf for scales from 2^104 on), and its inverse, which would take bits from scales below 2^-110.
constexpr float kPairWeightUnit = 128.0f;  // what nibbles_to_f16 divides by
__device__ __forceinline__ f16x8 nibbles_to_f16(uint32_t w) {
    const uint32_t v = w >> 8;
    uint32_t one = 0x48004800u;
    asm("" : "+v"(one));  // in a vector register: with both constants as literals a mask and an or are two instructions
    constexpr _Float16 o = (_Float16)-8.0625f, s = (_Float16)0.0625f, o16 = (_Float16)-0.5625f;  // (all exact)
    const f16x2 off = {o, o}, sixteenth = {s, s}, off16 = {o16, o16};
    auto low = [&](uint32_t x) { return __builtin_bit_cast(f16x2, (x & 0x000f000fu) | one) + off; };
    auto high = [&](uint32_t x) { return __builtin_elementwise_fma(__builtin_bit_cast(f16x2, (x & 0x00f000f0u) | one), sixteenth, off16); };
    const f16x2 a = low(w), b = high(w), c = low(v), d = high(v);
    return f16x8{a.x, a.y, b.x, b.y, c.x, c.y, d.x, d.y};
}

// Where it is left which rows of which blocks stand as floats: `marks` a byte each (PairLayout), `tiles` per 64 rows: `epoch`, where there are any; it has to
// be another one for every launch that hands rows on (one of before costs time only).
struct PairMarks {
    uint8_t *marks = nullptr;
    uint32_t *tiles = nullptr, epoch = 0;
};

// Where the outputs of the GEMM go: y = epilogue(acc), and with kv the K and V columns of a fused QKV projection as well.
struct GemmOut {
    const float *bias;
    const float *residual;
    float *y;
    int M, N;
    uint32_t flags;
    KvScatter kv;  // kcache == nullptr: none
    // Instead of y: the outputs as the pairs of the next Linear (N % 64 == 0, no residual), all rows times `pairs_up`, a power of two
    // that keeps them within f16 (that Linear's PairIn::up).
    char *pairs = nullptr;
    PairMarks marks;
    float pairs_up = 1.0f;
};

// Rows as pairs: with a factor per row behind the blocks (PairLayout), or one scale for all of them.
struct PairIn {
    const void *pairs;
    float up = 0.0f;  // the scale; 0: per row
    PairMarks marks{};  // with one scale
    // per row: what the pairs were made of (agpu_pair_rows_launch)
    const float *x = nullptr, *gamma = nullptr, *beta = nullptr;
    float eps = 0.0f;
};

// A bound of what a Linear behind a LayerNorm can give, whatever the rows: normalised rows have a 2-norm of at most sqrt(K), so output n
// is at most sqrt(K) |gamma W_n| + |beta W_n + bias_n|.  For up to kPairBoundBatch Linears [K, N] of the same shape, over columns first ..
// first + count - 1: out[2 i] = the largest (its bits), out[2 i + 1] = the smallest of columns that are not all zero (its bits inverted; 0: there
// are none).  Columns from first + part on (part a multiple of 64) go to out2 instead.  Both have to be zeros.
constexpr int kPairBoundBatch = 32;
struct PairBoundBatch {
    const uint32_t *packed[kPairBoundBatch];
    const float *scales[kPairBoundBatch], *bias[kPairBoundBatch], *gamma[kPairBoundBatch], *beta[kPairBoundBatch];
};
int32_t agpu_pair_bound_launch(agpu_ctx *ctx, const PairBoundBatch &batch, int n, int K, int N, int first, int count, int part, int group, uint32_t *out, uint32_t *out2);
// Rows of x, normalised first where gamma is given -> pairs (K <= kPairMaxK)
constexpr int kPairMaxK = 512 * 16;
int32_t agpu_pair_rows_launch(agpu_ctx *ctx, const float *x, const float *gamma, const float *beta, float eps, int M, int K, void *pairs);
// Whether the GEMM on pairs is the faster one for this shape (pass: its rows come as fp32 and have to be turned into pairs by a launch
// of their own), and whether it takes these operands at all.
bool agpu_int4_gemm_pairs_wanted(const agpu_ctx *ctx, int M, int N, int K, int group, bool pass);
// scratch: where partial sums of sliced tiles may go (0 bytes: none are sliced)
int32_t agpu_int4_gemm_pairs_launch(agpu_ctx *ctx, const PairIn &in, const uint32_t *packed, const float *scales, const GemmOut &out, int K, int group,
                                    void *scratch, size_t scratch_bytes);
