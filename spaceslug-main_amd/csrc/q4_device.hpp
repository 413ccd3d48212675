// Device-side helpers shared by the gfx950 int4 kernels: vector types and
// nibble decoding. Layout facts (q4gemm.comp:7-19): a packed byte holds
// k even in bits 0..3 and k odd in bits 4..7, so one little-endian 32-bit word
// holds 8 consecutive K values of one column, value t in bits 4t..4t+3, each a
// two's-complement nibble.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>
#include <utility>

namespace spaceslug {

// Calls f(std::integral_constant<int, I>{}) for I = 0 .. N-1 in order (compile-time indices, so
// register arrays indexed by I stay in registers).
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// v_cvt_off_f32_i4 reads bits 3..0 of its operand as a two's-complement value v
// and returns v / 16 exactly. The SDWA forms read byte 1, 2 or 3 of the operand
// in place, so a byte's low nibble needs no shift.
#define SPACESLUG_CVT_OFF_BYTE(SEL)                                                                      \
    __device__ __forceinline__ float cvt_off_##SEL(uint32_t w) {                                          \
        float r;                                                                                         \
        asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:" #SEL : "=v"(r) \
            : "v"(w));                                                                                   \
        return r;                                                                                        \
    }
SPACESLUG_CVT_OFF_BYTE(BYTE_1)
SPACESLUG_CVT_OFF_BYTE(BYTE_2)
SPACESLUG_CVT_OFF_BYTE(BYTE_3)
#undef SPACESLUG_CVT_OFF_BYTE

// Signed decode of all 8 nibbles of w: f[t] = v_t / 16 exactly, in 9 VALU ops
// (one shift for the odd nibbles, eight conversions). A sum of x * f times 16
// (exact) is the sum of x * v.
__device__ __forceinline__ void nibbles_signed_16th(uint32_t w, float (&f)[8]) {
    const uint32_t wo = w >> 4;
    f[0] = __builtin_amdgcn_cvt_off_f32_i4(static_cast<int>(w));
    f[1] = __builtin_amdgcn_cvt_off_f32_i4(static_cast<int>(wo));
    f[2] = cvt_off_BYTE_1(w);
    f[3] = cvt_off_BYTE_1(wo);
    f[4] = cvt_off_BYTE_2(w);
    f[5] = cvt_off_BYTE_2(wo);
    f[6] = cvt_off_BYTE_3(w);
    f[7] = cvt_off_BYTE_3(wo);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// x as three bf16 limbs (bit patterns in b[0..2], low 16 bits): b0 is x truncated to its top
// 8 significant bits (truncation, so nothing rounds past the fp32 range), b1 is x - b0
// truncated the same way, and b2 = x - b0 - b1 has at most 8 significant bits. Both
// subtractions are exact in fp32, so b0 + b1 + b2 == x whenever x's lowest significant bit is
// at least 2^-133 (bf16's subnormal resolution): every |x| >= 2^-110, and zero. Below that
// the limbs drop at most 2^-133 of x. A non-finite x travels in b0 alone, with zero lower
// limbs: +-inf stays +-inf (so a product with v = 0 is NaN and with v != 0 is +-inf, as in
// IEEE arithmetic on x itself), and a NaN stays a NaN (its quiet bit is set, so no payload
// truncates to an infinity).
__device__ __forceinline__ void split_bf16_limbs(float x, uint32_t (&b)[3]) {
    const uint32_t u = __float_as_uint(x);
    const float b0 = __uint_as_float(u & 0xFFFF0000u);
    const float r1 = x - b0;
    const float b1 = __uint_as_float(__float_as_uint(r1) & 0xFFFF0000u);
    const float r2 = r1 - b1;
    const uint32_t mag = u << 1;  // exponent and mantissa, sign dropped
    const bool finite = mag < 0xFF000000u;
    b[0] = (u >> 16) | (mag > 0xFF000000u ? 0x0040u : 0u);
    b[1] = finite ? __float_as_uint(b1) >> 16 : 0u;
    b[2] = finite ? __float_as_uint(r2) >> 16 : 0u;
}

// The 8 nibbles of w as bf16 v / 16, packed in element order (element t in the
// low half of word t/2 when t is even, the high half when odd). v / 16 has at
// most three significant bits, so the high half of its fp32 form is the exact
// bf16 value and one byte permute packs two. For values written to LDS: the
// consumer is a later MFMA, not the next instruction, so the inline-asm decode
// is safe here.
__device__ __forceinline__ u32x4 nibbles_bf16_16th(uint32_t w) {
    float f[8];
    nibbles_signed_16th(w, f);
    u32x4 r;
#pragma unroll
    for (int t = 0; t < 4; ++t)
        r[t] = __builtin_amdgcn_perm(__float_as_uint(f[2 * t + 1]), __float_as_uint(f[2 * t]), 0x07060302u);
    return r;
}

// Address of the B operand of lane slot s (column s % 32, word 2 half + s / 32 of the sub-group)
// of half `half` in sub-group `sub`'s buffer: s ^ 4 ((s >> 5) & 1) ^ 8 half ^ 2 sub. gfx950 serves
// 128-bit LDS reads 16 lanes per cycle (in a half-wavefront, the 4-lane chunks whose index has even
// popcount parity together, then the odd ones) and 128-bit writes 16 consecutive lanes per cycle; two
// lanes of a cycle conflict when their addresses agree modulo 256 bytes. With this map the MFMA
// operand reads (lane l reads slot l of one half of one sub-group) and the decode writes (lane l of
// wavefront w writes word l % 4 of sub-group (l / 4) % 2 of column 8 w + l / 8 to half (l % 4) / 2,
// slot column + 32 (l % 2)) both touch 16 distinct 16-byte bank groups per cycle.
__device__ __forceinline__ int pipe_b_slot(int s, int half, int sub) {
    return s ^ (4 * ((s >> 5) & 1)) ^ (8 * half) ^ (2 * sub);
}

}  // namespace spaceslug
