// What the two prefill GEMMs on the bf16 matrix cores share: operand types, the split of an fp32 number into three bf16
// pieces (hi, mid, lo: each the leading bits of what the ones before it left, an exact sum), the conversion of packed
// nibbles, and the K / V operand fragments of the prefill attention.
#pragma once
#include "linear_common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

// the leading 16 bits of two floats as one register: a in the low half
__device__ __forceinline__ uint32_t pack_top(float a, float b) {
    return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u);
}

__device__ __forceinline__ float top_bits(float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); }

// 8 nibbles of one column -> the bf16 numbers (q - 8) / 16 in the order (0, 2, 4, 6, 1, 3, 5, 7).  With the top bit of a
// nibble flipped, q - 8 is the nibble read as a signed 4-bit field, and v_cvt_off_f32_i4 turns the low four bits of its
// operand, read that way, into the float field / 16; its SDWA form takes them from any byte of a register, so a word
// costs one shift for the odd nibbles and one instruction per nibble (shifts and v_cvt_f32_i32 cost three per nibble:
// 322 vector instructions per two K blocks of the 32 x 128 tile against 386; M = 1024, K = 768, N = 2304: 21.7 us
// against 22.1 us).  The factor 16 goes into the scale of the group (exact, a power of two).
#define AGPU_CVT_I4(dst, src, byte) \
    asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_" #byte : "=v"(dst) : "v"(src))
__device__ __forceinline__ bf16x8 nibbles_to_bf16(uint32_t w) {
    const uint32_t even = w ^ 0x88888888u, odd = even >> 4;
    float f[8];
    AGPU_CVT_I4(f[0], even, 0);
    AGPU_CVT_I4(f[2], even, 1);
    AGPU_CVT_I4(f[4], even, 2);
    AGPU_CVT_I4(f[6], even, 3);
    AGPU_CVT_I4(f[1], odd, 0);
    AGPU_CVT_I4(f[3], odd, 1);
    AGPU_CVT_I4(f[5], odd, 2);
    AGPU_CVT_I4(f[7], odd, 3);
    const uint4 v = make_uint4(pack_top(f[0], f[2]), pack_top(f[4], f[6]), pack_top(f[1], f[3]), pack_top(f[5], f[7]));
    return __builtin_bit_cast(bf16x8, v);
}
#undef AGPU_CVT_I4
constexpr float GB_NIBBLE_UNIT = 16.0f;  // what nibbles_to_bf16 divides by

// 8 consecutive k of a row (in the nibbles' order (0, 2, 4, 6, 1, 3, 5, 7)) -> their three pieces, lo, mid, hi.
__device__ __forceinline__ void split_pieces(const float (&v)[8], bf16x8 (&piece)[3]) {
    float r1[8], r2[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        r1[e] = v[e] - top_bits(v[e]);    // exact: what the leading 8 bits leave
        r2[e] = r1[e] - top_bits(r1[e]);  // exact, at most 8 significant bits
    }
    piece[0] = __builtin_bit_cast(bf16x8, make_uint4(pack_top(r2[0], r2[2]), pack_top(r2[4], r2[6]), pack_top(r2[1], r2[3]), pack_top(r2[5], r2[7])));
    piece[1] = __builtin_bit_cast(bf16x8, make_uint4(pack_top(r1[0], r1[2]), pack_top(r1[4], r1[6]), pack_top(r1[1], r1[3]), pack_top(r1[5], r1[7])));
    piece[2] = __builtin_bit_cast(bf16x8, make_uint4(pack_top(v[0], v[2]), pack_top(v[4], v[6]), pack_top(v[1], v[3]), pack_top(v[5], v[7])));
}

// Two values, times a power of two -> hi, the f16 numbers next to them, and lo, those next to what is left.  (v_fma_mix_* take and leave f16
// numbers in either half of a register: two and a half vector instructions a value, five when product and difference are written as such.)
__device__ __forceinline__ void split_f16(float a, float b, float up, uint32_t &hi, uint32_t &lo) {
    typedef float Float2 __attribute__((ext_vector_type(2)));
    float ra, rb;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(hi) : "v"(a), "v"(up));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(hi) : "v"(b), "v"(up));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(ra) : "v"(a), "v"(up), "v"(hi));
    asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(rb) : "v"(b), "v"(up), "v"(hi));
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(Float2{ra, rb}, f16x2));
}
// the same without the power of two
__device__ __forceinline__ void split_f16(float a, float b, uint32_t &hi, uint32_t &lo) {
    typedef float Float2 __attribute__((ext_vector_type(2)));
    float ra, rb;
    hi = __builtin_bit_cast(uint32_t, __builtin_convertvector(Float2{a, b}, f16x2));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(ra) : "v"(hi), "v"(a));
    asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(rb) : "v"(hi), "v"(b));
    lo = __builtin_bit_cast(uint32_t, __builtin_convertvector(Float2{ra, rb}, f16x2));
}
__device__ __forceinline__ void split_f16(const float (&v)[8], float up, f16x8 &hi, f16x8 &lo) {
    uint32_t h[4], l[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) split_f16(v[2 * i], v[2 * i + 1], up, h[i], l[i]);
    hi = __builtin_bit_cast(f16x8, make_uint4(h[0], h[1], h[2], h[3]));
    lo = __builtin_bit_cast(f16x8, make_uint4(l[0], l[1], l[2], l[3]));
}

// 8 values of K (8 head dimensions of one key) or V (8 keys of one head dimension), in the attention's order, times `up` as two
// 16-byte fragments `stride` apart (hi, lo).
__device__ __forceinline__ void store_kv_frags(uint4 *dst, int stride, const float (&a)[8], float up) {
    f16x8 hi, lo;
    split_f16(a, up, hi, lo);
    dst[0] = __builtin_bit_cast(uint4, hi);
    dst[stride] = __builtin_bit_cast(uint4, lo);
}

// Eight keys of one dimension of V, under a scale that follows from a bound: whether none of them fills its fragment, that is, reaches 1 once scaled (what
// is left out of a fragment is up to 2^-25).  Of a tile that is not whole, whose eight may be a single key, 2^-8 is asked for: among 64 usual numbers,
// 2^-5 of the bound, one below 1 is nothing rare.
__device__ __forceinline__ uint32_t v_most(const float (&a)[8]) {  // the largest |a|'s bits (written out: fmaxf has its operands go through a v_max_f32 first)
    uint32_t most;
    asm("v_max3_f32 %0, |%1|, |%2|, |%3|" : "=v"(most) : "v"(a[0]), "v"(a[1]), "v"(a[2]));
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(a[3]), "v"(a[4]));
    asm("v_max3_f32 %0, %0, |%1|, |%2|" : "+v"(most) : "v"(a[5]), "v"(a[6]));
    asm("v_max_f32_e64 %0, %0, |%1|" : "+v"(most) : "v"(a[7]));
    return most;
}
__device__ __forceinline__ uint32_t v_least(float up, bool whole) { return __float_as_uint((whole ? 1.0f : 0x1p-8f) / up); }  // (a power of two)
__device__ __forceinline__ bool v_is_small(uint32_t most, uint32_t least) { return most - 1u < least - 1u; }  // (zeros are not)
__device__ __forceinline__ bool v_is_small(const float (&a)[8], float up, bool whole) { return v_is_small(v_most(a), v_least(up, whole)); }
