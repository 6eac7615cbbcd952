// What the two prefill GEMMs on the bf16 matrix cores share: operand types, the split of an fp32 number into three bf16
// pieces (hi, mid, lo: each the leading bits of what the ones before it left, an exact sum), the conversion of packed
// nibbles, and the K / V operand fragments of the prefill attention.
#pragma once
#include "linear_common.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
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

// 8 values of K (8 head dimensions of one key) or V (8 keys of one head dimension), in the attention's order, as three
// 16-byte fragments `stride` apart (hi, mid, lo).
__device__ __forceinline__ void store_kv_frags(uint4 *dst, int stride, const float (&a)[8]) {
    float b1[8], b2[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        b1[e] = a[e] - top_bits(a[e]);
        b2[e] = b1[e] - top_bits(b1[e]);
    }
    dst[0] = make_uint4(pack_top(a[0], a[1]), pack_top(a[2], a[3]), pack_top(a[4], a[5]), pack_top(a[6], a[7]));
    dst[stride] = make_uint4(pack_top(b1[0], b1[1]), pack_top(b1[2], b1[3]), pack_top(b1[4], b1[5]), pack_top(b1[6], b1[7]));
    dst[2 * stride] = make_uint4(pack_top(b2[0], b2[1]), pack_top(b2[2], b2[3]), pack_top(b2[4], b2[5]), pack_top(b2[6], b2[7]));
}
